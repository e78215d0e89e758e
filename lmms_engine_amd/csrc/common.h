// Shared device helpers for the gfx950 Muon kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef __bf16 bf16_t;
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Vectors at the address of any element: the hardware reads and writes them whole, at the cost of the cache lines that they touch.
typedef bf16x8 __attribute__((aligned(2))) bf16x8_any;
typedef f32x4 __attribute__((aligned(4))) f32x4_any;

// dtype codes shared with the C ABI (include/muon_hip.h)
#define MUON_HIP_F32 0
#define MUON_HIP_BF16 1

// Every matrix of the Newton-Schulz workspace is stored in blocks of 256 rows x BLK_COLS
// columns (rows of a block back to back): element (r, c) of a matrix with `cb` column blocks is at
//   ((r / 256) * cb + c / BLK_COLS) * BLK_ELEMS + (r % 256) * BLK_COLS + c % BLK_COLS.
// A k-tile of an operand panel is then one contiguous run of memory instead of 256 row pieces
// a row pitch apart, which is what DRAM pages, the L2 channels and the TLB all prefer.
#ifndef MUON_BLK_COLS
#define MUON_BLK_COLS 32
#endif
constexpr int BLK_ROWS = 256, BLK_COLS = MUON_BLK_COLS, BLK_SHIFT = BLK_COLS == 64 ? 6 : 5;
constexpr int BLK_ELEMS = BLK_ROWS * BLK_COLS;
static_assert(BLK_COLS == 32 || BLK_COLS == 64, "block width");

__host__ __device__ inline long blocked_offset(long r, long c, int cb) {
    return ((r >> 8) * cb + (c >> BLK_SHIFT)) * BLK_ELEMS + (r & 255) * BLK_COLS + (c & (BLK_COLS - 1));
}
// elements of a blocked rows x cols matrix (cols a multiple of BLK_COLS)
inline long blocked_elems(long rows, long cols) { return ((rows + BLK_ROWS - 1) / BLK_ROWS) * (cols / BLK_COLS) * BLK_ELEMS; }

// fp32 -> bf16, round-to-nearest-even (v_cvt_pk_bf16_f32 on gfx950), and back.
__device__ __forceinline__ bf16_t f2bf(float f) { return (bf16_t)f; }
__device__ __forceinline__ float bf2f(bf16_t h) { return (float)h; }
// round through bf16 and return the fp32 value
__device__ __forceinline__ float rbf(float f) { return (float)((bf16_t)f); }

// Square roots and divisions: sqrtf(x) and __fdiv_rn(x, y) are correctly rounded in this build (hipcc's default
// -fhip-fp32-correctly-rounded-divide-sqrt), which is what torch's GPU kernels compute; __fsqrt_rn is the
// hardware approximation despite its name (it differs from the exact root in one result out of six) and is not used.

// A value that the reference holds in a tensor of its own: the compiler must round it where it stands and not
// contract the product behind it into the next addition (hipcc fuses across statements by default).
__device__ __forceinline__ float materialized(float x) {
    asm volatile("" : "+v"(x));
    return x;
}

// Two values rounded to bf16 in one instruction, the first in the low half; and back.  Left to itself the compiler rounds most of them one by
// one, where the halves are used again: half an instruction more per element and rounding point.
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    uint32_t w = __builtin_bit_cast(uint32_t, bf16x2{f2bf(a), f2bf(b)});
    asm("" : "+v"(w));  // (what is taken out of it again is taken out of this register)
    return w;
}
__device__ __forceinline__ float low_bf16(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float high_bf16(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }
// bf(bf(a x) + v) for both halves of x and v
__device__ __forceinline__ uint32_t axpy_bf16x2(float a, uint32_t x, uint32_t v) {
    const uint32_t p = pack_bf16x2(a * low_bf16(x), a * high_bf16(x));
    return pack_bf16x2(low_bf16(p) + low_bf16(v), high_bf16(p) + high_bf16(v));
}

// bf(u / d) with IEEE division, for bf16 values u and one bf16 value d.  u times the reciprocal of d rounds to the same value: a quotient of
// two 8-bit significands is never halfway between two bf16 values (u = m d with an odd 9-bit m needs more than 8 bits) and at least 2^-17 of
// itself away from there, and the product is off by 2^-22.  What that leaves out is a quotient among the subnormal numbers, where fewer bits
// are kept, and a d whose reciprocal is one: those are divided.
struct DivideBf16 {
    float d, r;
    bool fast;
    __device__ __forceinline__ explicit DivideBf16(float d_) : d(d_), r(__fdiv_rn(1.0f, d_)), fast(d_ >= 0x1p-100f && d_ <= 0x1p100f) {}
    // out is right where true is returned
    __device__ __forceinline__ bool quick(bf16x8& out, const bf16x8& u) const {
        const u32x4 w = __builtin_bit_cast(u32x4, u);
        u32x4 o;
        bool normal = fast;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float a = low_bf16(w[e]) * r, b = high_bf16(w[e]) * r;
            normal &= !__builtin_amdgcn_classf(a, 0x90) & !__builtin_amdgcn_classf(b, 0x90);  // the subnormal numbers of either sign
            o[e] = pack_bf16x2(a, b);
        }
        out = __builtin_bit_cast(bf16x8, o);
        return normal;
    }
    __device__ __forceinline__ bf16x8 slow(const bf16x8& u) const {
        bf16x8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = f2bf(__fdiv_rn(bf2f(u[e]), d));
        return o;
    }
};

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Workgroups are dealt to the XCDs (2^xcd_shift of them) round-robin by their linear id.  Give each XCD runs of
// XCD_CHUNK consecutive logical ids instead (one round of its 32 CUs), so tiles that share operands
// share an L2, and deal those runs to the XCDs in turn, so that at any time all of them work on
// neighbouring tiles of the same matrix and the memory-side cache, which all XCDs share, serves
// the panels the others have already fetched.
#ifndef XCD_CHUNK
#define XCD_CHUNK 32
#endif
__device__ __forceinline__ int xcd_remap(int pid, int nblocks, int xcd_shift) {
    const int span = XCD_CHUNK << xcd_shift;  // one run for every XCD
    const int full = nblocks / span * span;
    const int xcds = 1 << xcd_shift, xcd = pid & (xcds - 1);
    if (pid >= full) {
        // Less than a run per XCD is left: equal runs, so that each XCD still works on neighbouring tiles and fetches the
        // panels of its own run only (dealt one by one, every XCD fetched nearly every panel).
        const int rest = nblocks - full, local = (pid - full) >> xcd_shift, each = rest >> xcd_shift, more = rest & (xcds - 1);
        return full + xcd * each + (xcd < more ? xcd : more) + local;
    }
    const int local = pid >> xcd_shift;
    return (((local / XCD_CHUNK) << xcd_shift) + xcd) * XCD_CHUNK + local % XCD_CHUNK;
}
