// The whole Newton-Schulz chain of a matrix with a short side of at most 64, or 128, in one workgroup (see small_chain.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "common.h"

// The matrices of one shape, and a list of such buckets as one launch takes them.
struct ChainBucket {
    const bf16_t* U;             // the blend, dense in the parameter's layout, strideU elements per matrix
    long strideU;
    const float* partials;       // nparts sums of squares per matrix
    bf16_t* X;                   // work area of strideX elements per matrix; without p_ptrs and out the result, blocked with cbx column blocks
    long strideX;
    const void* const* p_ptrs;   // device table of the parameters to update; null: the result goes to `out`
    bf16_t* out;                 // the result, dense in the parameter's layout, one matrix after the other; null: it goes to X
    float scale;
    int cbx, nparts, rows, cols, batch;
};
constexpr int CHAIN_MAX_LIST = 16;
struct ChainList {
    int n;
    int start[CHAIN_MAX_LIST + 1];
    ChainBucket b[CHAIN_MAX_LIST];
};
struct ChainMath {
    int steps;
    float a, b, c;
    int p_dtype;
    float decay, alpha;  // 1 - lr*wd and -lr
};

// A short side of M, a long side of K: whether the registers of one workgroup hold the matrix.
bool chain_fits(int M, int K);
// Whether a bucket's result is better written to `out` by the chain than copied there from X, on a device of `cus` compute units.
bool chain_writes(int rows, int cols, int batch, const void* out, int cus);
// The launches of a list on a device of `cus` compute units: for each bucket the kernel (blocks of 16 rows, fragments of X per lane) and the
// launch that takes it, and the order in which the buckets start.  Returns how many launches there are, or -1 where a bucket does not fit.
struct ChainRoute {
    int blocks, frags, launch;
};
int plan_ns_chain(const ChainBucket* buckets, int n, int cus, ChainRoute* route, int* order);
// Every bucket must fit; steps >= 1.  cus: compute units of the device.
hipError_t launch_ns_chain(const ChainBucket* buckets, int n, const ChainMath& cm, int cus, hipStream_t stream);
