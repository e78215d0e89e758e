// Newton-Schulz for matrices with a short side of at most 64 (low-rank adapters), or 128 where the long one is at most 512 (toy models, heads):
// normalisation, every iteration and the parameter update in one kernel, a workgroup per matrix, X in registers from the first product to the last.
//
// The tiled products of gemm_nt.hip pad a short side to 128 rows and stream X from memory three times an iteration: for 16 rows
// that is 64 times the multiplications, eight times the bytes and 17 launches.  Here the matrix is read once and the result (or
// the parameter) written once; what bounds it is the chain of dependent steps inside a workgroup (five iterations of the sums of
// X Xt handed from wave to wave, a walk over the wave's chunks, and three barriers) times the rounds of workgroups, not memory.
// fast_newtonschulz, us, tiles | this:
//      16 x  512, 1 | 256 | 1024 matrices   97 |  191 |  609    20 |  22 |  50
//      16 x 5632                           217 | 1414 | 5461    60 |  81 | 325
//    5632 x   16                                                65 |  85 | 352
//      32 x 4096                           181 | 1087 | 4229    75 | 109 | 431
//      64 x 2048                           137 |  556 | 2322    87 | 118 | 497
//    2048 x   64                           139 |  567 | 2363    96 | 131 | 509
// What a workgroup spends (cycles, one 16 x 5632 with an fp32 parameter, 175000 in all): an iteration 20000, of which the sums of X Xt 9500 (48
// for each of 176 MFMAs, hand-over included) and X' 10000; blend and norm 22000; the parameter, 720 KB through one compute unit, 48000.
// With the blend divided element by element and the parameter in pairs of chunks these were 24000, 32000 and 60000.
// and with a short side beyond 64, one | 64 | 1024 matrices (there the tiles already run in one launch):
//     128 x  128                           80 |   85 |  239    35 |  36 | 147
//     128 x  512                           88 |  107 |  654    73 |  78 | 359
//     512 x   67                           91 |  108 |  616    79 |  86 | 388
// It wins wherever the registers hold the matrix, so that is the rule (chain_fits); larger ones take the tiled products.
//
// Eight waves share the columns of X in chunks of 32, a run of consecutive chunks each.  Lane (i = l%16, q = l/16) of a wave holds
// X[r][8q .. 8q+7] of a chunk for one row r of every block of 16 rows (chain_row): an operand fragment of
// v_mfma_f32_16x16x32_bf16 as it stands, so
//   A = X Xt      contracts such fragments with one another; the sum of a 16x16 block goes from wave to wave through LDS (beyond 64 rows all of X
//                 does, and a wave sums whole blocks);
//   B = bA + cAA  is a handful of MFMAs on A in LDS;
//   X' = aX + BX  contracts rows, for which a chunk is turned on its way through 1 KB of LDS: a transposing read gives four rows of
//                 one column, and the rows are dealt to the lanes so that two blocks make eight consecutive rows, the fragment
//                 that B's rows meet; what comes out lies as X lay.
// A matrix of a parameter that is taller than wide (X is its transpose) is read and written the same way where its rows are whole pieces
// of four: a chunk is then a run of the parameter, 2 KB of it for 16 columns in fp32, and not 32 columns element by element.
// Results are those of the tiled kernels bit for bit: the same rounding points (bf(X Xt); bf(bf(bA) + bf(c bf(AA)));
// bf(bf(aX) + bf(BX))), and every fp32 sum in their order, ascending in 32-deep MFMAs with the reduction index in its natural
// place.  That order is why a block of X Xt is one chain through the waves and not eight partial sums, which take 3 to 30 % less
// time (16 x 5632: 57 | 95 | 415 when this took 82 | 118 | 511, 64 x 2048: 87 | 160 | 621 against 97 | 165 | 660): a bf16 value that rounds the other way moves through the remaining
// iterations, up to 1e-3 of the result in norm.
#include "small_chain.h"
#include "gemm_nt.h"
#include <algorithm>
#include <atomic>
#include <type_traits>

namespace {

__device__ __forceinline__ f32x4 mfma(const bf16x8& p, const bf16x8& q, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(p, q, c, 0, 0, 0);
}

template <typename PT>
__device__ __forceinline__ float update_one(float p, bf16_t x, float scale, float decay, float alpha) {
    const float os = rbf(bf2f(x) * scale);
    const float pd = sizeof(PT) == 2 ? rbf(p * decay) : p * decay;
    return fmaf(alpha, os, pd);
}

// Four elements of the parameter that lie next to one another, and four of X (two registers) that meet them.
template <typename PT>
using FourOf = PT __attribute__((ext_vector_type(4)));
template <typename PT>
__device__ __forceinline__ FourOf<PT> update_four(const FourOf<PT>& p, uint32_t x01, uint32_t x23, float scale, float decay, float alpha) {
    FourOf<PT> o;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const uint32_t x = e ? x23 : x01, os = pack_bf16x2(low_bf16(x) * scale, high_bf16(x) * scale);
        if constexpr (sizeof(PT) == 2) {
            const uint32_t pd = pack_bf16x2(bf2f(p[2 * e]) * decay, bf2f(p[2 * e + 1]) * decay);
            o[2 * e] = f2bf(fmaf(alpha, low_bf16(os), low_bf16(pd)));
            o[2 * e + 1] = f2bf(fmaf(alpha, high_bf16(os), high_bf16(pd)));
        } else {
            o[2 * e] = fmaf(alpha, low_bf16(os), p[2 * e] * decay);
            o[2 * e + 1] = fmaf(alpha, high_bf16(os), p[2 * e + 1] * decay);
        }
    }
    return o;
}
// Where the parameter is read and written in whole pieces: rows of X are rows of it (eight columns are all there or none is), or X is its
// transpose and four rows of X lie next to one another there.
__device__ __forceinline__ bool whole_rows(const void* p, int cols, bool turn) { return !turn && cols % 8 == 0 && (((uintptr_t)p) & 15) == 0; }
__device__ __forceinline__ bool turned_pieces(const void* p, int M, bool turn, int elem) { return turn && M % 4 == 0 && ((uintptr_t)p & (4 * elem - 1)) == 0; }

// The first `left` of W elements from any address on (whole pieces where they are all there, four together and single ones where they are not),
// and back.
template <int W, typename PT, typename V>
__device__ __forceinline__ void load_cut(V& o, const PT* a, int left) {
    typedef PT __attribute__((ext_vector_type(W), aligned(sizeof(PT)))) whole_any;
    typedef FourOf<PT> __attribute__((aligned(sizeof(PT)))) four_any;
    if (left >= W) {
        o = *(const whole_any*)a;
        return;
    }
    if (W == 8 && left >= 4) {
        const FourOf<PT> f = *(const four_any*)a;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = f[e];
    }
#pragma unroll
    for (int e = 0; e < W - 1; ++e)
        if (e < left && (W == 4 || e >= 4 || left < 4) && e != 3) o[e] = a[e];
}
template <int W, typename PT, typename V>
__device__ __forceinline__ void store_cut(PT* a, const V& o, int left) {
    typedef PT __attribute__((ext_vector_type(W), aligned(sizeof(PT)))) whole_any;
    typedef FourOf<PT> __attribute__((aligned(sizeof(PT)))) four_any;
    if (left >= W) {
        *(whole_any*)a = o;
        return;
    }
    if (W == 8 && left >= 4) {
        FourOf<PT> f;
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = o[e];
        *(four_any*)a = f;
    }
#pragma unroll
    for (int e = 0; e < W - 1; ++e)
        if (e < left && (W == 4 || e >= 4 || left < 4) && e != 3) a[e] = o[e];
}

// Elsewhere in pieces from any address, or element by element, eight columns of a row of X at a time.  In two halves, so that the loads of several pieces are in flight
// before the first store (the compiler cannot know that the pieces are apart: one after the other they cost a trip to memory each, eight for
// a turned piece; see kBatch).
struct Piece {
    float v[8];
};
template <typename PT>
__device__ __forceinline__ void load_each(Piece& o, const PT* p, int row, int col, int cols, int M, int K, bool turn) {
    typedef FourOf<PT> __attribute__((aligned(sizeof(PT)))) four_any;
    if (!turn && col + 8 <= K) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const FourOf<PT> v = *(const four_any*)(p + (long)row * cols + col + 4 * h);
#pragma unroll
            for (int e = 0; e < 4; ++e) o.v[4 * h + e] = (float)v[e];
        }
        return;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
        if (col + e < K) o.v[e] = (float)p[turn ? (long)(col + e) * M + row : (long)row * cols + col + e];
}
template <typename PT>
__device__ __forceinline__ void store_each(PT* p, const Piece& o, const bf16x8& x, int row, int col, int cols, int M, int K, bool turn, float scale, float decay,
                                           float alpha) {
    typedef FourOf<PT> __attribute__((aligned(sizeof(PT)))) four_any;
    if (!turn && col + 8 <= K) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            FourOf<PT> v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (PT)update_one<PT>(o.v[4 * h + e], x[4 * h + e], scale, decay, alpha);
            *(four_any*)(p + (long)row * cols + col + 4 * h) = v;
        }
        return;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
        if (col + e < K) p[turn ? (long)(col + e) * M + row : (long)row * cols + col + e] = (PT)update_one<PT>(o.v[e], x[e], scale, decay, alpha);
}

// A block of 16 rows and 32 columns turned within a wave, through LDS of its own (a wave's LDS instructions are carried out in order,
// so it needs no barrier).  lds_read_tr16: in a group of 16 lanes, lane i receives element i%4 of the 8-byte pieces addressed by lanes
// i/4, 4 + i/4, 8 + i/4, 12 + i/4.
constexpr int TURN_ZEROS = 16, TURN_BYTES = (TURN_ZEROS + 4) * 64;
typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ bf16x4 lds_read_tr16(const unsigned char* p) {
    typedef __attribute__((address_space(3))) void* lds_void_ptr;
    return __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(lds_void_ptr)p));
}
// v: four rows 4 (l%4) .. of columns l/4 and 16 + l/4 in lane l  ->  columns 8q .. 8q+7 of row i
__device__ __forceinline__ bf16x8 turn_in(unsigned char* lds, const bf16x8& v, int lane) {
    const int i = lane & 15, q = lane >> 4;
    asm volatile("" ::: "memory");
    *(bf16x4*)(lds + lane * 8) = bf16x4{v[0], v[1], v[2], v[3]};
    *(bf16x4*)(lds + 512 + lane * 8) = bf16x4{v[4], v[5], v[6], v[7]};
    asm volatile("" ::: "memory");
    const unsigned char* r = lds + (8 * q + (i >> 2)) * 32 + (i & 3) * 8;
    const bf16x4 lo = lds_read_tr16(r), hi = lds_read_tr16(r + 128);
    asm volatile("" ::: "memory");
    return bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}
// v: columns 8q .. 8q+7 of row i in lane (i, q)  ->  rows row .. row+3 of columns 8 (i/4) + i%4 and 8 (i/4) + 4 + i%4.  Without v: of the
// block that is there.  Row TURN_ZEROS and those after it are zeros.
__device__ __forceinline__ bf16x8 turn_rows(unsigned char* lds, const bf16x8* v, int row, int lane) {
    const int i = lane & 15, q = lane >> 4;
    if (v) {
        asm volatile("" ::: "memory");
        *(bf16x8*)(lds + i * 64 + q * 16) = *v;
        asm volatile("" ::: "memory");
    }
    const unsigned char* r = lds + (row + (i >> 2)) * 64 + (i & 3) * 16;
    const bf16x4 lo = lds_read_tr16(r), hi = lds_read_tr16(r + 8);
    asm volatile("" ::: "memory");
    return bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}
// v: columns 8q .. 8q+7 of row i in lane (i, q)  ->  rows 4q .. 4q+3 of column i, then of column 16 + i
__device__ __forceinline__ bf16x8 turn_out(unsigned char* lds, const bf16x8& v, int lane) {
    const int i = lane & 15, q = lane >> 4;
    asm volatile("" ::: "memory");
    *(bf16x8*)(lds + i * 64 + q * 16) = v;
    asm volatile("" ::: "memory");
    const unsigned char* r = lds + (4 * q + (i >> 2)) * 64 + (i & 3) * 8;
    const bf16x4 lo = lds_read_tr16(r), hi = lds_read_tr16(r + 32);
    asm volatile("" ::: "memory");
    return bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

// The row that lane i of 16 holds in block t of 16 rows.  The turned fragment of a block has rows i = 4q .. 4q+3 of it in lane group
// q; in this order blocks 2p and 2p + 1 put rows 32p + 8q .. 32p + 8q + 7 there, which is where an MFMA has them.  A single block
// (MT = 1) is in natural order: its fragment is two reads of four rows, and zeros.
template <int MT>
__device__ __forceinline__ int chain_row(int t, int i) {
    return MT == 1 ? i : 32 * (t >> 1) + 8 * (i >> 2) + 4 * (t & 1) + (i & 3);
}

constexpr int CHAIN_WAVES = 8;
constexpr int CHAIN_FRAGS = 32;  // fragments of X a lane can hold: 128 of the 256 registers of a wave

// Where the parameter goes element by element: fragments that a lane asks for together, while those before them are still on their way
// (loads and stores leave the queue in order, so a load that is issued behind a store waits for it as well).
constexpr int kBatch = 2;

template <int MT>
struct ChainShared {
    static constexpr int PITCH = 32 * ((MT + 1) / 2) + 8;  // of A and B; with MT = 1 columns 16 to 31 stay zero
    f32x4 sum[MT * (MT + 1) / 2][64];
    bf16_t A[MT * 16][PITCH], B[MT * 16][PITCH];
    unsigned char turned[CHAIN_WAVES][TURN_BYTES];
    float red[4];
    int left[MT * (MT + 1) / 2];  // per leg: waves that have left it, of all iterations
};

// Eight row blocks: the fragments of X of all waves (STAGE, 16 chunks) while A is summed, A and B in their place afterwards.
template <>
struct ChainShared<8> {
    static constexpr int PITCH = 32 * 4 + 8, CHUNKS = 2 * CHAIN_WAVES;
    union {
        bf16x8 stage[CHUNKS * 8][64];
        struct {
            bf16_t A[128][PITCH], B[128][PITCH];
        };
        f32x4 sum[1][64];  // (the sums stay in registers)
    };
    unsigned char turned[CHAIN_WAVES][TURN_BYTES];
    float red[4];
    int left[1];
};
static_assert(sizeof(ChainShared<8>) <= 139 * 1024 && sizeof(ChainShared<8>) > 80 * 1024, "one workgroup of eight row blocks per compute unit, of 160 KB");

// Matrix b of bucket k.  MT blocks of 16 rows (1, 2, 4 or 8), up to NCH chunks of 32 columns per wave.
template <int MT, int NCH>
__device__ __forceinline__ void chain_matrix(const ChainBucket& k, int b, const ChainMath& cm, ChainShared<MT>& sh) {
    constexpr int NP = (MT + 1) / 2;         // 32-deep reductions over the rows
    constexpr int PITCH = ChainShared<MT>::PITCH;
    constexpr int NF = MT * (MT + 1) / 2;    // 16 x 16 blocks of A on or above the diagonal
    constexpr int BATCH = kBatch < MT ? 1 : kBatch / MT;  // chunks of the parameter that are loaded together
    constexpr bool TWO = MT < 4;             // while the next ones are on their way (with four blocks a chunk is enough, and two spill)
    // Chunks without a branch between them: 40 -> 30 ns for each MFMA of the chain through 176 chunks (16 x 5632).  Four blocks have
    // ten MFMAs between two branches anyway; and where a wave has four chunks at most, those that are not there cost as much as the
    // branches (111 of 20 x 56, one chunk: 17.5 with runs, 16.0 without).
    constexpr int RUN = MT >= 4 || NCH < 8 ? 1 : 4;
    constexpr int GROUP = MT >= 4 || RUN == 1 ? 1 : 4 / MT;  // chunks of X' that are computed together
    static_assert(NCH % RUN == 0 && RUN % GROUP == 0, "whole runs");
    constexpr int LEG = MT == 4 ? 2 : 1, NLEG = NF / LEG;  // blocks that a wave adds its chunks to at a time
    auto& sum = sh.sum;
    auto& As = sh.A;
    auto& Bs = sh.B;
    auto& turned = sh.turned;
    auto& red = sh.red;
    const bool turn = k.rows > k.cols;
    const int M = turn ? k.cols : k.rows, K = turn ? k.rows : k.cols;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i = lane & 15, q = lane >> 4;
    // The wave's chunks: `per` of them from chunk `first` on.  What is left over goes to the first waves, one chunk each: with equal runs 12
    // chunks would give six waves two, and a SIMD that has two of those four, where it has three like this.
    const int chunks = (K + 31) / 32, spare = chunks % CHAIN_WAVES;
    const int per = chunks / CHAIN_WAVES + (wave < spare ? 1 : 0), first = wave * (chunks / CHAIN_WAVES) + (wave < spare ? wave : spare);
    const int col0 = first * 32 + 8 * q;  // this lane's first column in chunk 0
    const bf16_t* u = k.U + b * k.strideU;
    bf16_t* area = k.X + b * k.strideX;
    // this lane's fragments in the work area: read and written by this lane only
    bf16x8* mine = (bf16x8*)area + (long)first * MT * 64 + lane;

    if constexpr (MT < 8)
    for (int t = tid; t < MT * 16 * PITCH; t += 64 * CHAIN_WAVES) {
        (&As[0][0])[t] = (bf16_t)0.f;
        (&Bs[0][0])[t] = (bf16_t)0.f;
    }
    *(unsigned*)&turned[wave][TURN_ZEROS * 64 + lane * 4] = 0u;
    if (MT < 8 && tid < NLEG) sh.left[tid] = 0;
    // The matrix in whole pieces (turned: four rows of two columns, turned below), every load in flight together; zero past its edges.
    const bool vec = !turn && K % 8 == 0, tvec = turned_pieces(u, M, turn, 2);
    unsigned char* const tl = turned[wave];
    float s = (tid & 255) < k.nparts ? k.partials[(long)b * k.nparts + (tid & 255)] : 0.f;  // asked for ahead of them
    bf16x8 zero8;
#pragma unroll
    for (int e = 0; e < 8; ++e) zero8[e] = (bf16_t)0.f;
    bf16x8 x[NCH][MT];
#pragma unroll
    for (int j = 0; j < NCH; ++j)
#pragma unroll
        for (int t = 0; t < MT; ++t) x[j][t] = zero8;
    if (vec) {
#pragma unroll
        for (int j = 0; j < NCH; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                const int row = chain_row<MT>(t, i), col = col0 + j * 32;
                if (j < per && row < M && col < K) x[j][t] = *(const bf16x8*)(u + (long)row * K + col);
            }
    } else if (tvec) {
#pragma unroll
        for (int j = 0; j < NCH; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                const int row = chain_row<MT>(t, 4 * (lane & 3)), col = (first + j) * 32 + (lane >> 2);
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    if (j < per && row < M && col + 16 * h < K) {
                        const bf16x4 p = *(const bf16x4*)(u + (long)(col + 16 * h) * M + row);
#pragma unroll
                        for (int e = 0; e < 4; ++e) x[j][t][4 * h + e] = p[e];
                    }
            }
    }
    // eight row blocks, elsewhere: the same pieces at the address of any element, and those that the matrix ends in element by element
    const bool cut = MT == 8 && !vec && !tvec;
    if constexpr (MT == 8)
        if (cut) {
#pragma unroll
            for (int j = 0; j < NCH; ++j)
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    if (j >= per) continue;
                    if (turn) {
                        const int row = chain_row<MT>(t, 4 * (lane & 3)), col = (first + j) * 32 + (lane >> 2);
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            bf16x4 p = {zero8[0], zero8[1], zero8[2], zero8[3]};
                            load_cut<4>(p, u + (long)(col + 16 * h) * M + row, col + 16 * h < K ? M - row : 0);
#pragma unroll
                            for (int e = 0; e < 4; ++e) x[j][t][4 * h + e] = p[e];
                        }
                    } else {
                        const int row = chain_row<MT>(t, i), col = col0 + j * 32;
                        load_cut<8>(x[j][t], u + (long)row * K + col, row < M ? K - col : 0);
                    }
                }
        }
    // d = bf(bf(sqrt(sum)) + 1e-7), in the order of the normalisation kernel: both halves of the workgroup add the same sums
    for (int t = (tid & 255) + 256; t < k.nparts; t += 256) s += k.partials[(long)b * k.nparts + t];
    s = wave_sum(s);
    if (lane == 0 && wave < 4) red[wave] = s;
    __syncthreads();
    const DivideBf16 div(rbf(rbf(sqrtf((red[0] + red[1]) + (red[2] + red[3]))) + 1e-7f));
    const bool turned_in = tvec || (cut && turn);
    bool exact = (vec || tvec || cut) && div.fast;
    if (exact) {
#pragma unroll
        for (int j = 0; j < NCH; ++j)
            if (j < per) {
#pragma unroll
                for (int t = 0; t < MT; ++t) exact &= div.quick(x[j][t], turned_in ? turn_in(tl, x[j][t], lane) : x[j][t]);
            }
    }
    if (!__all(exact)) {
        // In pieces from any address or element by element, or divided: a few fragments at a time through the work area, so that the loop
        // need not be unrolled over the register array (their loads before the first store, which the compiler cannot tell apart from them).
        constexpr int AHEAD = MT < 4 ? 4 / MT : 1;
        for (int j0 = 0; j0 < per; j0 += AHEAD) {
            bf16x8 v[AHEAD][MT];
#pragma unroll
            for (int jj = 0; jj < AHEAD; ++jj)
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    const int row = chain_row<MT>(t, i), col = col0 + (j0 + jj) * 32;
                    if (j0 + jj >= per) continue;
                    if (!turn && row < M && col + 8 <= K) {
                        v[jj][t] = *(const bf16x8_any*)(u + (long)row * K + col);
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            v[jj][t][e] = (row < M && col + e < K) ? u[turn ? (long)(col + e) * M + row : (long)row * K + col + e] : (bf16_t)0.f;
                    }
                }
#pragma unroll
            for (int jj = 0; jj < AHEAD; ++jj)
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    if (j0 + jj >= per) continue;
                    bf16x8 o;
                    if (!div.quick(o, v[jj][t])) o = div.slow(v[jj][t]);
                    mine[((j0 + jj) * MT + t) * 64] = o;
                }
        }
#pragma unroll
        for (int j = 0; j < NCH; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) x[j][t] = j < per ? mine[(j * MT + t) * 64] : zero8;
    }
    // The sum of leg `leg` (LEG blocks of A) over this wave's chunks, on top of the waves' before it.
    auto add_leg = [&](auto leg_c, int before) {
        constexpr int F0 = decltype(leg_c)::value * LEG;
        int* const left = &sh.left[decltype(leg_c)::value];
        f32x4 acc[LEG];
        for (;;) {  // the count and the sums in one trip to LDS (a wave's LDS instructions are carried out in order)
            const int n = __hip_atomic_load(left, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            asm volatile("" ::: "memory");
#pragma unroll
            for (int f = 0; f < LEG; ++f) acc[f] = sum[F0 + f][lane];
            if (n == before) break;
        }
        if (wave == 0) {
#pragma unroll
            for (int f = 0; f < LEG; ++f) acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        __builtin_amdgcn_s_setprio(3);
#pragma unroll
        for (int j0 = 0; j0 < NCH; j0 += RUN) {
            if (j0 >= per) break;
#pragma unroll
            for (int j = j0; j < j0 + RUN; ++j) {  // (past the wave's last chunk x is zero, and the sum plus zero is the sum)
                int f = 0;
#pragma unroll
                for (int ti = 0; ti < MT; ++ti)
#pragma unroll
                    for (int tj = ti; tj < MT; ++tj, ++f)
                        if (f >= F0 && f < F0 + LEG) acc[f - F0] = mfma(x[j][ti], x[j][tj], acc[f - F0]);
            }
        }
#pragma unroll
        for (int f = 0; f < LEG; ++f) sum[F0 + f][lane] = acc[f];
        __builtin_amdgcn_s_setprio(0);
        asm volatile("" ::: "memory");
        if (lane == 0) __hip_atomic_store(left, before + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };

    const int active = chunks < CHAIN_WAVES ? chunks : CHAIN_WAVES;  // waves that have columns
    for (int it = 0; it < cm.steps; ++it) {
        // A wave starts a leg when the wave before it has left it, so the legs follow one another through the waves; the first ones go
        // ahead while the last are still at X' of the iteration before.  Every wave of the workgroup runs, and waits only for the one
        // before it.
        if constexpr (MT == 8) {
            // With at most two chunks a wave there is little to add between two hand-overs.  Here all of X goes through LDS, and a wave sums its
            // own blocks of A over all chunks, the same sums: rows p and 7 - p have nine, five of row p for one wave and the others for the next.
            const int p = wave >> 1, odd = wave & 1;
            f32x4 acc[5];
#pragma unroll
            for (int f = 0; f < 5; ++f) acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
            auto row_of = [&](int f) { return odd && 5 + f >= 8 - p ? 7 - p : p; };                     // block f of this wave
            auto col_of = [&](int f) { return !odd ? p + f : 5 + f >= 8 - p ? 7 - p + (5 + f - (8 - p)) : p + 5 + f; };
            __syncthreads();  // B is no longer read
#pragma unroll
            for (int j = 0; j < NCH; ++j)
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    if (j < per) sh.stage[(first + j) * MT + t][lane] = x[j][t];
            __syncthreads();
            if (!odd) {
#pragma unroll 2
                for (int c = 0; c < chunks; ++c) {
                    const bf16x8 own = sh.stage[c * MT + p][lane];
#pragma unroll
                    for (int f = 0; f < 5; ++f) acc[f] = mfma(own, sh.stage[c * MT + p + f][lane], acc[f]);
                }
            } else {
#pragma unroll 2
                for (int c = 0; c < chunks; ++c)
#pragma unroll
                    for (int f = 0; f < 4; ++f) acc[f] = mfma(sh.stage[c * MT + row_of(f)][lane], sh.stage[c * MT + col_of(f)][lane], acc[f]);
            }
            __syncthreads();  // X is no longer read
#pragma unroll
            for (int f = 0; f < 5; ++f) {
                if (f == 4 && odd) break;
                const int ti = row_of(f), tj = col_of(f), r = chain_row<MT>(ti, q * 4), c = chain_row<MT>(tj, i);
                const u32x2 o = {pack_bf16x2(acc[f][0], acc[f][1]), pack_bf16x2(acc[f][2], acc[f][3])};
                *(u32x2*)&As[c][r] = o;
                if (ti != tj) {
                    const bf16x4 v = __builtin_bit_cast(bf16x4, o);
#pragma unroll
                    for (int e = 0; e < 4; ++e) As[r + e][c] = v[e];
                }
            }
        } else
        if (wave < active) {
            const int before = it * active + wave;
            add_leg(std::integral_constant<int, 0>{}, before);
            if constexpr (NLEG > 1) add_leg(std::integral_constant<int, 1>{}, before);
            if constexpr (NLEG > 2) add_leg(std::integral_constant<int, 2>{}, before);
            if constexpr (NLEG > 3) add_leg(std::integral_constant<int, 3>{}, before);
            if constexpr (NLEG > 4) add_leg(std::integral_constant<int, 4>{}, before);
            static_assert(NLEG <= 5 && NLEG * LEG == NF, "every leg has its branch");
        }
        __syncthreads();
        if constexpr (MT < 8) {
        for (int t = tid; t < NF * 64; t += 64 * CHAIN_WAVES) {
            const int ln = t & 63;
            int f = t >> 6, ti = 0;
            const f32x4 v = sum[f][ln];
            while (f >= MT - ti) f -= MT - ti++;
            const int tj = ti + f, r = chain_row<MT>(ti, (ln >> 4) * 4), c = chain_row<MT>(tj, ln & 15);
            bf16x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = f2bf(v[e]);
            *(bf16x4*)&As[c][r] = o;  // A is symmetric: the mirrored block in one piece, this one element by element
            if (ti != tj) {
#pragma unroll
                for (int e = 0; e < 4; ++e) As[r + e][c] = o[e];
            }
        }
        __syncthreads();
        }
        if constexpr (MT == 8) {  // a row of blocks for each wave, whole: its operand is read once
            bf16x8 own[NP];
#pragma unroll
            for (int p = 0; p < NP; ++p) own[p] = *(const bf16x8*)&As[wave * 16 + i][p * 32 + 8 * q];
#pragma unroll 4
            for (int tj = 0; tj < MT; ++tj) {
                f32x4 aa = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int p = 0; p < NP; ++p) aa = mfma(own[p], *(const bf16x8*)&As[tj * 16 + i][p * 32 + 8 * q], aa);
                u32x2 o = *(const u32x2*)&As[tj * 16 + i][wave * 16 + 4 * q];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const uint32_t w = pack_bf16x2(aa[2 * e], aa[2 * e + 1]);
                    o[e] = axpy_bf16x2(cm.b, o[e], pack_bf16x2(cm.c * low_bf16(w), cm.c * high_bf16(w)));
                }
                *(u32x2*)&Bs[tj * 16 + i][wave * 16 + 4 * q] = o;
            }
        } else
        for (int f0 = wave; f0 < NF; f0 += CHAIN_WAVES) {  // on and above the diagonal, and the mirror image
            int ti = 0, f = f0;
            while (f >= MT - ti) f -= MT - ti++;
            const int tj = ti + f;
            f32x4 aa = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int p = 0; p < NP; ++p)
                aa = mfma(*(const bf16x8*)&As[ti * 16 + i][p * 32 + 8 * q], *(const bf16x8*)&As[tj * 16 + i][p * 32 + 8 * q], aa);
            const bf16x4 av = *(const bf16x4*)&As[tj * 16 + i][ti * 16 + 4 * q];
            bf16x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = f2bf(rbf(cm.b * bf2f(av[e])) + rbf(cm.c * rbf(aa[e])));
            *(bf16x4*)&Bs[tj * 16 + i][ti * 16 + 4 * q] = o;
            if (ti != tj) {
#pragma unroll
                for (int e = 0; e < 4; ++e) Bs[ti * 16 + 4 * q + e][tj * 16 + i] = o[e];
            }
        }
        __syncthreads();
        // B's rows, in the order of X's.  Those of eight blocks do not fit beside X: they are read as they are met.
        constexpr bool KEPT = MT < 8;
        bf16x8 bfr[KEPT ? MT : 1][NP];
        auto read_b = [&](int t, bf16x8 (&w)[NP]) {
#pragma unroll
            for (int p = 0; p < NP; ++p) w[p] = *(const bf16x8*)&Bs[chain_row<MT>(t, i)][p * 32 + 8 * q];
        };
        if constexpr (KEPT) {
#pragma unroll
            for (int t = 0; t < MT; ++t) read_b(t, bfr[t]);
        }
        // GROUP chunks together, so that one's way through LDS and the products passes behind the others'
        auto next_chunks = [&](int j0, auto count_c) {
            constexpr int N = decltype(count_c)::value;
            bf16x8 xt[N][2][NP];  // xt[.][h][p]: rows 32p + 8q .. + 7 of column 8 (i/4) + 4h + i%4, the operand that B's rows meet
#pragma unroll
            for (int n = 0; n < N; ++n) {
                bf16x8(&xc)[MT] = x[j0 + n];
                if constexpr (MT == 1) {
                    const bf16x8 lo = turn_rows(tl, &xc[0], q < 2 ? 8 * q : TURN_ZEROS, lane), hi = turn_rows(tl, nullptr, q < 2 ? 8 * q + 4 : TURN_ZEROS, lane);
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        xt[n][h][0] = bf16x8{lo[4 * h], lo[4 * h + 1], lo[4 * h + 2], lo[4 * h + 3], hi[4 * h], hi[4 * h + 1], hi[4 * h + 2], hi[4 * h + 3]};
                } else {
#pragma unroll
                    for (int t = 0; t < MT; ++t) {
                        const bf16x8 v = turn_rows(tl, &xc[t], 4 * q, lane);
#pragma unroll
                        for (int h = 0; h < 2; ++h)
#pragma unroll
                            for (int e = 0; e < 4; ++e) xt[n][h][t / 2][4 * (t & 1) + e] = v[4 * h + e];
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            constexpr int TB = KEPT ? MT : 2;  // blocks whose products come before their sums with X
#pragma unroll
            for (int t0 = 0; t0 < MT; t0 += TB) {
                f32x4 v[N][TB][2];
                bf16x8 bt[KEPT ? 1 : TB][NP];
                if constexpr (!KEPT) {
#pragma unroll
                    for (int t = 0; t < TB; ++t) read_b(t0 + t, bt[t]);
                }
#pragma unroll
                for (int p = 0; p < NP; ++p)
#pragma unroll
                    for (int n = 0; n < N; ++n)
#pragma unroll
                        for (int t = 0; t < TB; ++t)
#pragma unroll
                            for (int h = 0; h < 2; ++h) v[n][t][h] = mfma(xt[n][h][p], KEPT ? bfr[KEPT ? t : 0][p] : bt[KEPT ? 0 : t][p], p ? v[n][t][h] : f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                for (int n = 0; n < N; ++n)
#pragma unroll
                    for (int t = 0; t < TB; ++t) {
                        u32x4 xw = __builtin_bit_cast(u32x4, x[j0 + n][t0 + t]);
#pragma unroll
                        for (int h = 0; h < 2; ++h)
#pragma unroll
                            for (int e = 0; e < 2; ++e) xw[2 * h + e] = axpy_bf16x2(cm.a, xw[2 * h + e], pack_bf16x2(v[n][t][h][2 * e], v[n][t][h][2 * e + 1]));
                        x[j0 + n][t0 + t] = __builtin_bit_cast(bf16x8, xw);
                    }
            }
        };
        // (waves w and w + 4 share a SIMD: the first four are done in half of the time, and the sums of the next iteration can start)
        if (wave < CHAIN_WAVES / 2) __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int j0 = 0; j0 < NCH; j0 += RUN) {
            if (j0 + RUN <= per) {
#pragma unroll
                for (int j = j0; j < j0 + RUN; j += GROUP) next_chunks(j, std::integral_constant<int, GROUP>{});
            } else {  // (nothing is computed past the last chunk: with an infinite B its zeros would not stay zero)
#pragma unroll
                for (int j = j0; j < j0 + RUN - 1; ++j)
                    if (j < per) next_chunks(j, std::integral_constant<int, 1>{});
            }
        }
        __builtin_amdgcn_s_setprio(0);
    }

    bf16_t* out = k.out + (long)b * M * K;
    const bool whole_out = !turn && K % 8 == 0 && (((uintptr_t)k.out) & 15) == 0;
    if (!k.p_ptrs && (!k.out || whole_out)) {
#pragma unroll
        for (int j = 0; j < NCH; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                const int row = chain_row<MT>(t, i), col = col0 + j * 32;
                if (j < per && row < M && col < K) *(bf16x8*)(k.out ? out + (long)row * K + col : area + blocked_offset(row, col, k.cbx)) = x[j][t];
            }
        return;
    }
    if (!k.p_ptrs && turned_pieces(k.out, M, turn, 2)) {
#pragma unroll
        for (int j = 0; j < NCH; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                if (j >= per) continue;
                const bf16x8 v = turn_out(tl, x[j][t], lane);
                const int row = chain_row<MT>(t, 4 * q), col = (first + j) * 32 + i;
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    if (row < M && col + 16 * h < K)
                        *(bf16x4*)(out + (long)(col + 16 * h) * M + row) = bf16x4{v[4 * h], v[4 * h + 1], v[4 * h + 2], v[4 * h + 3]};
            }
        return;
    }
    void* const p = k.p_ptrs ? const_cast<void*>(k.p_ptrs[b]) : nullptr;
    auto piece_update = [&](auto* pp, auto turned_c) {
        using PT = std::remove_pointer_t<decltype(pp)>;
        constexpr bool TURNED = decltype(turned_c)::value;
        // fragments whose pieces are asked for together: what the registers hold beside X
        constexpr int G = NCH * MT == 8 ? 4 : sizeof(PT) == 4 ? 8 : 16;
#pragma unroll
        for (int f0 = 0; f0 < NCH * MT; f0 += G) {
            if (f0 / MT >= per) break;
            FourOf<PT> o[G][2];
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const int j = (f0 + g) / MT, t = (f0 + g) % MT, row = chain_row<MT>(t, TURNED ? 4 * q : i), col = TURNED ? (first + j) * 32 + i : col0 + j * 32;
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    if (j < per && row < M && col + (TURNED ? 16 * h : 0) < K)
                        o[g][h] = *(const FourOf<PT>*)(pp + (TURNED ? (long)(col + 16 * h) * M + row : (long)row * K + col + 4 * h));
            }
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const int j = (f0 + g) / MT, t = (f0 + g) % MT, row = chain_row<MT>(t, TURNED ? 4 * q : i), col = TURNED ? (first + j) * 32 + i : col0 + j * 32;
                if (j >= per) continue;
                const bf16x8 v = TURNED ? turn_out(tl, x[j][t], lane) : x[j][t];
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    if (row < M && col + (TURNED ? 16 * h : 0) < K)
                        *(FourOf<PT>*)(pp + (TURNED ? (long)(col + 16 * h) * M + row : (long)row * K + col + 4 * h)) =
                            update_four<PT>(o[g][h], __builtin_bit_cast(u32x4, v)[2 * h], __builtin_bit_cast(u32x4, v)[2 * h + 1], k.scale, cm.decay, cm.alpha);
            }
        }
    };
    // Eight row blocks, elsewhere: pieces of eight bf16 or four fp32 columns (turned: of four rows) at the address of any element, straight from the
    // registers.  Element by element and through the work area, as below, such steps were slower than on the tiles: us, tiles | that | this,
    // bf16: 300 of 511 x 127 249 | 289 | 233, 16 of 399 x 127 100 | 105 | 94, 300 of 101 x 511 236 | 260 | 227, one 512 x 128 behind a boundary 98 | 106 | 99.
    // What is left is the unit that takes apart pieces behind a 4-byte boundary, lane by lane.
    auto cut_update = [&](auto* pp) {
        using PT = std::remove_pointer_t<decltype(pp)>;
        auto run = [&](auto turned_c) {
            constexpr bool TURNED = decltype(turned_c)::value;
            constexpr int W = !TURNED && sizeof(PT) == 2 ? 8 : 4, H = 8 / W;  // elements of a piece, pieces of a fragment
            constexpr int G = NCH * MT == 8 ? 4 : 8;
            typedef PT __attribute__((ext_vector_type(W))) piece_t;
            // piece h of fragment (j, t): where it lies, and how many elements from there on are the matrix's
            auto place = [&](int j, int t, int h, long& at) {
                const int row = chain_row<MT>(t, TURNED ? 4 * q : i), col = TURNED ? (first + j) * 32 + i + 16 * h : col0 + j * 32 + W * h;
                at = TURNED ? (long)col * M + row : (long)row * K + col;
                return j >= per ? 0 : TURNED ? (col < K ? M - row : 0) : row < M ? K - col : 0;
            };
#pragma unroll
            for (int f0 = 0; f0 < NCH * MT; f0 += G) {
                if (f0 / MT >= per) break;
                piece_t o[G][H];
#pragma unroll
                for (int g = 0; g < G; ++g)
#pragma unroll
                    for (int h = 0; h < H; ++h) {
                        long at;
                        const int left = place((f0 + g) / MT, (f0 + g) % MT, h, at);
                        load_cut<W>(o[g][h], pp + at, left);
                    }
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const int j = (f0 + g) / MT, t = (f0 + g) % MT;
                    if (j >= per) continue;
                    const u32x4 v = __builtin_bit_cast(u32x4, TURNED ? turn_out(tl, x[j][t], lane) : x[j][t]);
#pragma unroll
                    for (int h = 0; h < H; ++h) {
                        long at;
                        const int left = place(j, t, h, at);
                        if (left <= 0) continue;
                        piece_t n;
#pragma unroll
                        for (int w = 0; w < W / 4; ++w) {
                            FourOf<PT> f;
#pragma unroll
                            for (int e = 0; e < 4; ++e) f[e] = o[g][h][4 * w + e];
                            f = update_four<PT>(f, v[2 * (h + w)], v[2 * (h + w) + 1], k.scale, cm.decay, cm.alpha);
#pragma unroll
                            for (int e = 0; e < 4; ++e) n[4 * w + e] = f[e];
                        }
                        store_cut<W>(pp + at, n, left);
                    }
                }
            }
        };
        if (turn) run(std::true_type{});
        else run(std::false_type{});
    };
    auto try_pieces = [&](auto* pp) {
        if (turned_pieces(p, M, turn, sizeof(*pp))) piece_update(pp, std::true_type{});
        else if (whole_rows(p, k.cols, turn)) piece_update(pp, std::false_type{});
        else return false;
        return true;
    };
    if (k.p_ptrs && (cm.p_dtype == MUON_HIP_BF16 ? try_pieces((bf16_t*)p) : try_pieces((float*)p))) return;
    if constexpr (MT == 8) {
        if (k.p_ptrs) {
            if (cm.p_dtype == MUON_HIP_BF16) cut_update((bf16_t*)p);
            else cut_update((float*)p);
            return;
        }
    }
#pragma unroll
    for (int j = 0; j < NCH; ++j)
#pragma unroll
        for (int t = 0; t < MT; ++t)
            if (j < per) mine[(j * MT + t) * 64] = x[j][t];
    if (!k.p_ptrs) {  // turned, or of rows that are no whole pieces: element by element
        for (int j = 0; j < per; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                const int row = chain_row<MT>(t, i), col = col0 + j * 32;
                const bf16x8 v = mine[(j * MT + t) * 64];
                if (!turn && row < M && col + 8 <= K) *(bf16x8_any*)(out + (long)row * K + col) = v;
                else
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (row < M && col + e < K) out[turn ? (long)(col + e) * M + row : (long)row * K + col + e] = v[e];
            }
        return;
    }
    auto each_update = [&](auto* pp) {  // element by element, BATCH chunks asked for ahead of the stores of the BATCH before
        struct Batch {
            Piece o[BATCH][MT];
            bf16x8 v[BATCH][MT];
        } w[TWO ? 2 : 1];
        auto each = [&](int j0, auto f) {
#pragma unroll
            for (int jj = 0; jj < BATCH; ++jj)
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    const int row = chain_row<MT>(t, i), col = col0 + (j0 + jj) * 32;
                    if (j0 + jj < per && row < M && col < K) f(jj, t, row, col);
                }
        };
        auto load = [&](int j0, Batch& w) {
            each(j0, [&](int jj, int t, int row, int col) {
                w.v[jj][t] = mine[((j0 + jj) * MT + t) * 64];
                load_each(w.o[jj][t], pp, row, col, k.cols, M, K, turn);
            });
        };
        auto store = [&](int j0, Batch& w) {
            each(j0, [&](int jj, int t, int row, int col) { store_each(pp, w.o[jj][t], w.v[jj][t], row, col, k.cols, M, K, turn, k.scale, cm.decay, cm.alpha); });
        };
        if constexpr (TWO) load(0, w[0]);
        for (int j0 = 0; j0 < per; j0 += (TWO ? 2 : 1) * BATCH) {
            load(TWO ? j0 + BATCH : j0, w[TWO ? 1 : 0]);
            store(j0, w[0]);
            if constexpr (TWO) {
                load(j0 + 2 * BATCH, w[0]);
                store(j0 + BATCH, w[1]);
            }
        }
    };
    if (cm.p_dtype == MUON_HIP_BF16) each_update((bf16_t*)p);
    else each_update((float*)p);
}

// Workgroup `id` of a list: its bucket, and the matrix there.
__device__ __forceinline__ int chain_bucket(const ChainList& l, int id, int& b) {
    int i = 0;
    while (i + 1 < l.n && id >= l.start[i + 1]) ++i;
    i = __builtin_amdgcn_readfirstlane(i);
    b = id - l.start[i];
    return i;
}

// (with 8 fragments two workgroups share a compute unit)
template <int MT, int NCH>
__global__ void __launch_bounds__(64 * CHAIN_WAVES, MT * NCH == 8 && MT < 8 ? 4 : 2) ns_chain_kernel(const ChainList l, const ChainMath cm) {
    int b;
    const int i = chain_bucket(l, blockIdx.x, b);
    if constexpr (MT == 8) {
        extern __shared__ __align__(16) unsigned char dynamic[];
        chain_matrix<MT, NCH>(l.b[i], b, cm, *(ChainShared<MT>*)dynamic);
    } else {
        __shared__ __align__(16) unsigned char shared[sizeof(ChainShared<MT>)];
        chain_matrix<MT, NCH>(l.b[i], b, cm, *(ChainShared<MT>*)shared);
    }
}

__host__ __device__ constexpr int chain_blocks(int M) { return M <= 16 ? 1 : M <= 32 ? 2 : M <= 64 ? 4 : 8; }
__host__ __device__ constexpr int chain_per_wave(int K) { return ((K + 31) / 32 + CHAIN_WAVES - 1) / CHAIN_WAVES; }

// Fragments of X per lane that a kernel is built for.
__host__ __device__ constexpr int chain_class(int need) { return need <= 8 ? 8 : need <= 16 ? 16 : 32; }

template <int MT, int NCH>
hipError_t launch_chain(const ChainList& l, const ChainMath& cm, hipStream_t stream) {
    int lds = 0;
    if constexpr (MT == 8) {  // past the 64 KB that a kernel has without asking
        lds = sizeof(ChainShared<MT>);
        static std::atomic<unsigned long long> configured{0};  // per instantiation
        if (hipError_t e = allow_dynamic_lds((const void*)ns_chain_kernel<MT, NCH>, lds, configured); e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((ns_chain_kernel<MT, NCH>), dim3(l.start[l.n]), dim3(64 * CHAIN_WAVES), lds, stream, l, cm);
    return hipGetLastError();
}
template <int MT>
hipError_t launch_as(int frags, const ChainList& l, const ChainMath& cm, hipStream_t stream) {
    if constexpr (MT < 8)
        if (frags == 32) return launch_chain<MT, 32 / MT>(l, cm, stream);
    return frags == 8 ? launch_chain<MT, 8 / MT>(l, cm, stream) : launch_chain<MT, 16 / MT>(l, cm, stream);
}

}  // namespace

// (128 rows and four chunks a wave, 32 fragments, would fit the registers but for 100 bytes a lane.)
bool chain_fits(int M, int K) { return M <= 128 && K <= 8192 && chain_per_wave(K) * chain_blocks(M) <= (M <= 64 ? CHAIN_FRAGS : 16); }

// Whole pieces, of rows or of a turned matrix's columns, cost the chain nothing.  Element by element a workgroup pays 0.6 us for a fragment,
// which few matrices of many fragments feel more than the copy, while with many the copy, a pass over memory, costs more: the lines cross
// between 64 and 160 matrices (profiles/low_rank_result_copy.txt); at three quarters of the compute units the chain is ahead everywhere.  (Rows
// that are no whole pieces and not turned are the exception: 33 x 515, 192 matrices 60.5 with the copy, 58.4 without, 1024 229 and 237.)
bool chain_writes(int rows, int cols, int batch, const void* out, int cus) {
    if (rows <= cols && cols % 8 == 0 && ((uintptr_t)out & 15) == 0) return true;
    if (rows > cols && cols % 4 == 0 && ((uintptr_t)out & 7) == 0) return true;
    return 4L * batch >= 3L * cus || chain_per_wave(std::max(rows, cols)) * chain_blocks(std::min(rows, cols)) <= 4;
}

// One launch per number of row blocks, on the kernel that holds the widest matrices, or one per kernel (8, 16 or 32 fragments of X per
// lane: fewer registers, more workgroups in flight).
//
// The longest come first, the others on the compute units that they leave: a launch of its own per width waits for the one before.  The
// narrow ones lose a place: two workgroups of 8 fragments share a compute unit on their own kernel, on a wider one each has its own.
// Steps (us, apart | together): 308 narrow with 84 of 16 x 5632 and 5632 x 16 178 | 140, a quarter of them 134 | 100; 12 of 24 x
// 1024 to 2624 in three widths 164 | 82; 504 narrow of 24 x 1024 with 168 of 24 x 2200 189 | 199; 616 with 168 of rank 16 272 | 262.
// With eight row blocks a workgroup has a compute unit of its own on either kernel (LDS, and registers), so there is nothing to lose: 400 of
// 128 x 128 with 20 of 128 x 512 171 | 102, 1000 with 100 294 | 243, 400 of 128 x 256 with 300 of 128 x 400 347 | 269.
//
// Matrices of fewer row blocks go along, as if their rows were padded, while every workgroup of the launch has a compute unit of its own and
// their waves have no more columns than those of the launch have: then they end before those do.
int plan_ns_chain(const ChainBucket* buckets, int n, int cus, ChainRoute* route, int* order) {
    if (n < 1 || n > CHAIN_MAX_LIST) return -1;
    int per[CHAIN_MAX_LIST], blocks[CHAIN_MAX_LIST];
    for (int i = 0; i < n; ++i) {
        const ChainBucket& k = buckets[i];
        const int M = std::min(k.rows, k.cols), K = std::max(k.rows, k.cols);
        if (!chain_fits(M, K)) return -1;
        blocks[i] = chain_blocks(M);
        per[i] = chain_per_wave(K);
        order[i] = i;
        route[i].launch = -1;
    }
    std::stable_sort(order, order + n, [&](int x, int y) { return blocks[x] != blocks[y] ? blocks[x] > blocks[y] : per[x] > per[y]; });
    int launches = 0;
    for (int at = 0; at < n; ++at) {
        const int head = order[at], mt = blocks[head], frags = chain_class(per[head] * mt);
        if (route[head].launch >= 0) continue;
        long narrow = 0, used = 0;
        for (int i = 0; i < n; ++i)
            if (route[i].launch < 0 && blocks[i] == mt && chain_class(per[i] * mt) == 8) narrow += buckets[i].batch;
        const bool together = mt == 8 || 2 * narrow <= 3L * cus;
        for (int k = at; k < n; ++k) {
            const int i = order[k];
            if (route[i].launch >= 0) continue;
            if (blocks[i] == mt ? !together && chain_class(per[i] * mt) != frags : per[i] > per[head] || used + buckets[i].batch > cus) continue;
            route[i] = ChainRoute{mt, frags, launches};
            used += buckets[i].batch;
        }
        ++launches;
    }
    return launches;
}

hipError_t launch_ns_chain(const ChainBucket* buckets, int n, const ChainMath& cm, int cus, hipStream_t stream) {
    ChainRoute route[CHAIN_MAX_LIST];
    int order[CHAIN_MAX_LIST];
    const int launches = plan_ns_chain(buckets, n, cus, route, order);
    if (launches < 0 || cm.steps < 1) return hipErrorInvalidValue;
    for (int k = 0; k < launches; ++k) {
        ChainList l;
        l.n = 0;
        l.start[0] = 0;
        int mt = 0, frags = 0;
        for (int j = 0; j < n; ++j) {
            const int i = order[j];
            if (route[i].launch != k) continue;
            mt = route[i].blocks;
            frags = route[i].frags;
            l.b[l.n] = buckets[i];
            l.start[l.n + 1] = l.start[l.n] + buckets[i].batch;
            ++l.n;
        }
        if (hipError_t e = mt == 8 ? launch_as<8>(frags, l, cm, stream) : mt == 4 ? launch_as<4>(frags, l, cm, stream)
                           : mt == 2 ? launch_as<2>(frags, l, cm, stream) : launch_as<1>(frags, l, cm, stream);
            e != hipSuccess) return e;
    }
    return hipSuccess;
}
