// Host-side description of one batched NT GEMM launch (see gemm_nt.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <atomic>
#include "common.h"

// EPI_BX_UPD is EPI_BX with the parameter update folded into the epilogue (GemmArgs::upd_*) instead of writing X';
// EPI_BX_UPD_T is the same for a parameter that is the transpose of X (rows > cols)
// EPI_MMT is EPI_SYRK with a row-major result, and a left operand that may be row-major too (matmul_transpose on its own)
enum { EPI_SYRK = 0, EPI_SYMPOLY = 1, EPI_BX = 2, EPI_BX_UPD = 3, EPI_BX_UPD_T = 4, EPI_MMT = 5 };
constexpr bool epi_is_bx(int e) { return e == EPI_BX || e == EPI_BX_UPD || e == EPI_BX_UPD_T; }
// how the B.X epilogue finishes: 0 writes X', 1 updates a parameter in the orientation of X, 2 a transposed one
constexpr int epi_fold_mode(int e) { return e == EPI_BX_UPD ? 1 : e == EPI_BX_UPD_T ? 2 : 0; }
enum {
    GEMM_CFG_128_PIPE = 0,      // 128x128 tile, 4 waves, 64-column k-tiles in two LDS stages
    GEMM_CFG_256_PIPE = 1,      // 256x256 tile, 8 waves, the same pipeline
    GEMM_CFG_256_PINGPONG = 2,  // 256x256 tile, 8 waves in two alternating groups, four stages of 32 columns
    GEMM_CFG_128_PINGPONG = 3,  // 128x128 tile, the same eight-wave kernel, two workgroups per compute unit
    GEMM_CFG_256_PERSIST = 4,   // the ping-pong loop as a persistent kernel (a workgroup per compute unit walks tiles of one or
                                // several products, the next tile's first loads land behind an epilogue without LDS): a.X + B.X,
                                // and the symmetric products with reductions up to 2048; launches of at most one round, a few
                                // rounds with a nearly empty last one, and launches that carry the parameter update run
                                // GEMM_CFG_256_PINGPONG
    GEMM_CFG_64_DEEP = 5,       // 64x64 tile, 4 waves, eight stages of 64 columns: launches that leave most compute units idle
    GEMM_CFG_COUNT = 6
};

constexpr int GEMM_UPD_RESULT = 2;
struct GemmArgs {
    const bf16_t* P;        // left operand: rows x kdim, blocked
    const bf16_t* Q;        // right operand, blocked: rows x kdim (SYRK, SYMPOLY) or kdim x columns (BX)
    long strideP, strideQ;  // elements between matrices of the batch
    int cbP;                // column blocks of P (and of Q in the symmetric kernels): its storage may be wider than the reduction
    int cbQ;                // BX: column blocks of Q
    int kdim;               // reduction length, a multiple of 128
    int rows, cols;         // of C, whole 128-tiles (symmetric kernels: rows == cols); larger tiles may overhang into the storage
    int tiles_m, tiles_n;   // set by the launcher: tile grid of one matrix
    int tiles_per_mat;      // set by the launcher: tiles_m*(tiles_m+1)/2 for the symmetric kernels, tiles_m*tiles_n for BX
    int batch;
    bf16_t* C;              // out[i][j], blocked with cbC column blocks
    long strideC;
    int cbC;
    bf16_t* Ct;             // symmetric kernels: out[j][i], the same buffer as C; BX: unused
    long strideCt;
    int cbCt;
    const bf16_t* Et;       // elementwise source, blocked: A read as Et[j][i] (symmetric), or X read as Et[i][j] (BX)
    long strideEt;
    int cbEt;
    float s0, s1;           // SYMPOLY: (b, c); BX: (a, -)
    // BX, optional: fold apply_scaling and the parameter update into the epilogue instead of writing X'
    // (EPI_BX_UPD: the parameter is X's image, rows <= cols; EPI_BX_UPD_T: its transpose, rows > cols)
    const void* const* upd_ptrs;  // device table of parameter base pointers, one per matrix; null = write X'
    int upd_dtype;                // MUON_HIP_F32 or MUON_HIP_BF16; GEMM_UPD_RESULT: no parameters, X' itself goes to the dense matrices at
                                  // upd_ptrs (bf16, upd_rows x upd_cols each, one after the other)
    int upd_rows, upd_cols;       // the parameter's own (unpadded) shape
    float upd_scale, upd_decay, upd_alpha;  // python-double scale, 1 - lr*wd and -lr, as fp32
    // EPI_MMT: C is row-major, dense_rows x dense_rows (rows, cols: in whole 128-tiles as ever).  dense_pitch: P and Q are too, with
    // that many elements from row to row and dense_rows rows; 0: they are blocked.
    int dense_rows, dense_pitch;
    unsigned* ppx;          // tile counters of the persistent kernel (GEMM_PPX_COUNTER_BYTES, zero between launches);
                            // null: the launcher takes the one-tile kernels instead
};

// One launch works on up to GEMM_MAX_LIST products of different sizes, each a batch of its own (matrices of several shapes in
// one optimizer step): tile t of the launch belongs to the entry with start[i] <= t < start[i + 1].  Passed by value, in the
// 4 KB that a kernel's arguments may take.
constexpr int GEMM_MAX_LIST = 16;
struct GemmList {
    int n;
    int xcd_shift;   // log2 of the XCD count of the device
    int big_blocks;  // split-tail kernel: workgroups that compute whole 256x256 tiles
    int start[GEMM_MAX_LIST + 1];
    GemmArgs g[GEMM_MAX_LIST];
};
static_assert(sizeof(GemmList) <= 4096, "kernel arguments");

// Tile counters of one persistent launch: a 64-byte line per XCD (tiles handed out beyond the two static rounds) and one
// for the workgroups that have left.  A launch finds them zero and leaves them zero (the last workgroup out resets them),
// so launches that share a buffer must be ordered on one stream.
constexpr int GEMM_MAX_XCDS = 8;
constexpr size_t GEMM_PPX_COUNTER_BYTES = (GEMM_MAX_XCDS + 1) * 16 * sizeof(unsigned);

// Shape of the current device, read once per device: compute units (one 256x256 workgroup each per round of tiles) and
// XCDs.  gfx950 dies carry 32 active compute units per XCD, and a partition of the part exposes whole XCDs, so the XCD
// count is the compute-unit count over 32; workgroups are dealt to the XCDs round-robin by their linear id.
struct MachineShape {
    int cus, xcd_shift;
};
hipError_t machine_shape(MachineShape& ms);

// Dynamic LDS beyond 64 KB has to be allowed per kernel, and the attribute belongs to the device that is current when
// it is set: once per (kernel instantiation, device), remembered as one bit per device in the instantiation's mask.
hipError_t allow_dynamic_lds(const void* kern, int bytes, std::atomic<unsigned long long>& done);

int gemm_cfg_tile(int cfg);
// The products args[0..n) of one kind, each with the configuration that its shape asks for, in as few launches as their
// configurations allow.  `adapt`: launches whose tiles would not fill the machine may run on smaller ones (same results bit
// for bit); without it every product runs its configuration as named.
struct GemmItem {
    GemmArgs g;
    int cfg, epi;
};
hipError_t launch_gemm_nt(const GemmItem* items, int n, bool adapt, hipStream_t stream);

// What launch_gemm_nt does with each of them on a device of `cus` compute units: the kernel, the rows of its tiles, and the
// launch of the call (from 0) that it goes with.  The number of launches, or -1 when it refuses them; touches no device.
struct GemmRoute {
    int cfg, height, launch;
};
int plan_gemm_nt(const GemmItem* items, int n, bool adapt, int cus, GemmRoute* route);

// The chain of many small matrices as one launch (gemm_nt_flow_kernel): every matrix belongs to one of `groups` groups, each of
// which runs on one XCD.  Matrices first[g] .. first[g + 1] - 1 of an entry are those of group g.
constexpr int GEMM_MAX_XCC_IDS = 16;                                       // values the hardware's XCD number can take
constexpr int GEMM_FLOW_LINE = 16;                                         // words between the counters of two matrices
constexpr size_t GEMM_FLOW_CONTROL_BYTES = (GEMM_MAX_XCDS + GEMM_MAX_XCC_IDS + 2) * 16 * sizeof(unsigned);
struct FlowEntry {
    bf16_t* X[2];              // iteration i reads X[i & 1] and writes the other; blocked, Mp x Kp
    bf16_t *A, *B;             // Mp x Mp
    long strideX, strideA;
    int Mp, Kr, Kp, batch;     // as GemmArgs: Kr columns in whole 128-tiles of storage for Kp
    unsigned* done;            // a counter per matrix, GEMM_FLOW_LINE words apart, zero before the launch
    const void* const* p_ptrs; // device table of the parameters to update (FlowList::p_dtype GEMM_UPD_RESULT: where X' goes, GemmArgs::upd_ptrs);
                               // null: the last iteration writes X'
    int rows, cols;            // of the parameter
    float scale;
    int sym, rect;             // 128-tiles of a matrix: of a symmetric product, of a.X + B.X
    int first[GEMM_MAX_XCDS + 1];
};
struct FlowList {
    int n, groups, steps, p_dtype;
    float a, b, c, decay, alpha;
    unsigned* control;         // GEMM_FLOW_CONTROL_BYTES, zero before the launch
    unsigned* alarm;           // host memory, set when a wait is given up: the results are then not what was asked for
    unsigned polls;            // after which a wait is given up
    int sym[GEMM_MAX_XCDS], rect[GEMM_MAX_XCDS];  // per group: tiles of each symmetric product, of a.X + B.X
    FlowEntry e[GEMM_MAX_LIST];
};
static_assert(sizeof(FlowList) <= 4096, "kernel arguments");

// Tiles of a group are numbered by iteration, product (0 X.Xt, 1 b.A + c.A.A, 2 a.X + B.X), entry, matrix and place in the product.
// Tile t of group g, and how many tiles of its matrix come before its product: all of them have to be finished first.
struct FlowPlace {
    int entry, matrix, tile, stage, it, before;
};
__host__ __device__ inline int flow_tiles(const FlowList& l, int g) { return l.steps * (2 * l.sym[g] + l.rect[g]); }
__host__ __device__ inline FlowPlace flow_place(const FlowList& l, int g, int t) {
    FlowPlace p;
    const int sym = l.sym[g], each_it = 2 * sym + l.rect[g];
    p.it = t / each_it;
    t -= p.it * each_it;
    p.stage = t < sym ? 0 : t < 2 * sym ? 1 : 2;
    t -= p.stage * sym;
    int each = 1;
    for (p.entry = 0;; ++p.entry) {
        const FlowEntry& e = l.e[p.entry];
        each = p.stage == 2 ? e.rect : e.sym;
        const int here = (e.first[g + 1] - e.first[g]) * each;
        if (t < here || p.entry == l.n - 1) break;
        t -= here;
    }
    const FlowEntry& e = l.e[p.entry];
    const int m = t / each;
    p.matrix = e.first[g] + m;
    p.tile = t - m * each;
    p.before = p.it * (2 * e.sym + e.rect) + p.stage * e.sym;
    return p;
}

// Deals the matrices of l.e[0 .. l.n) to the XCDs (fills groups, sym and rect, here and in the entries, and every first); false where
// launches of their own are the faster way.  recorded: the call is being recorded into a graph, its launches cost the caller nothing.
// Touches no device.
bool plan_flow(FlowList& l, int xcds, bool recorded);
hipError_t launch_flow(const FlowList& l, hipStream_t stream);
