// Newton-Schulz for matrices with a short side of at most 64 (low-rank adapters): normalisation, every iteration and the
// parameter update in one kernel, a workgroup per matrix, X in registers from the first product to the last.
//
// The tiled products of gemm_nt.hip pad a short side to 128 rows and stream X from memory three times an iteration: for 16 rows
// that is 64 times the multiplications, eight times the bytes and 17 launches.  Here the matrix is read once and the result (or
// the parameter) written once; what bounds it is the chain of dependent steps inside a workgroup (five iterations of the sums of
// X Xt handed from wave to wave, a walk over the wave's chunks, and three barriers) times the rounds of workgroups, not memory.
// fast_newtonschulz, us, tiles | this:
//      16 x  512, 1 | 256 | 1024 matrices   97 |  191 |  609    17 |  20 |  44
//      16 x 5632                           217 | 1414 | 5461    72 |  94 | 395
//      32 x 4096                           181 | 1087 | 4229    81 | 116 | 481
//      64 x 2048                           137 |  556 | 2322    97 | 134 | 558
//    2048 x   64                           139 |  567 | 2363   103 | 177 | 694
// It wins wherever the registers hold the matrix, so that is the rule (chain_fits); larger ones take the tiled products.
//
// Eight waves share the columns of X in chunks of 32, a run of consecutive chunks each.  Lane (i = l%16, q = l/16) of a wave holds
// X[r][8q .. 8q+7] of a chunk for one row r of every block of 16 rows (chain_row): an operand fragment of
// v_mfma_f32_16x16x32_bf16 as it stands, so
//   A = X Xt      contracts such fragments with one another; the sum of a 16x16 block goes from wave to wave through LDS;
//   B = bA + cAA  is a handful of MFMAs on A in LDS;
//   X' = aX + BX  contracts rows, for which a chunk is turned by multiplying it with selected columns of the identity (exact:
//                 one product is the element, the others are zero): the result's four registers are four rows of one column,
//                 and the rows are dealt to the lanes so that two blocks make eight consecutive rows, the fragment that B's rows
//                 meet; what comes out lies as X lay.
// Results are those of the tiled kernels bit for bit: the same rounding points (bf(X Xt); bf(bf(bA) + bf(c bf(AA)));
// bf(bf(aX) + bf(BX))), and every fp32 sum in their order, ascending in 32-deep MFMAs with the reduction index in its natural
// place.  That order is why a block of X Xt is one chain through the waves and not eight partial sums, which take 3 to 30 % less
// time (16 x 5632: 57 | 95 | 415 when this took 82 | 118 | 511, 64 x 2048: 87 | 160 | 621 against 97 | 165 | 660): a bf16 value that rounds the other way moves through the remaining
// iterations, up to 1e-3 of the result in norm.
#include "small_chain.h"
#include <algorithm>
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

// Eight consecutive columns of one row of X meet the parameter: a piece of its row, or (turned) of its column.  In two halves, so that
// the loads of several pieces are in flight before the first store (the compiler cannot know that the pieces are apart: one after the
// other they cost a trip to memory each, eight for a turned piece; see kBatch).
struct Piece {
    float v[8];
};
__device__ __forceinline__ bool whole_rows(const void* p, int cols, bool turn) { return !turn && cols % 8 == 0 && (((uintptr_t)p) & 15) == 0; }
template <typename PT>
__device__ __forceinline__ void load8(Piece& o, const PT* p, int row, int col, int cols, int M, int K, bool turn, bool whole) {
    if (whole) {  // eight columns are all there or none is
        const PT* d = p + (long)row * cols + col;
        if constexpr (sizeof(PT) == 2) {
            const bf16x8 v = *(const bf16x8*)d;
#pragma unroll
            for (int e = 0; e < 8; ++e) o.v[e] = bf2f(v[e]);
        } else {
            const f32x4 v = *(const f32x4*)d, w = *(const f32x4*)(d + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) o.v[e] = v[e], o.v[4 + e] = w[e];
        }
        return;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
        if (col + e < K) o.v[e] = (float)p[turn ? (long)(col + e) * M + row : (long)row * cols + col + e];
}
template <typename PT>
__device__ __forceinline__ void store8(PT* p, const Piece& o, const bf16x8& x, int row, int col, int cols, int M, int K, bool turn, bool whole, float scale,
                                       float decay, float alpha) {
    if (whole) {
        PT* d = p + (long)row * cols + col;
        if constexpr (sizeof(PT) == 2) {
            bf16x8 v;
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = f2bf(update_one<PT>(o.v[e], x[e], scale, decay, alpha));
            *(bf16x8*)d = v;
        } else {
            f32x4 v, w;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = update_one<PT>(o.v[e], x[e], scale, decay, alpha);
                w[e] = update_one<PT>(o.v[4 + e], x[4 + e], scale, decay, alpha);
            }
            *(f32x4*)d = v;
            *(f32x4*)(d + 4) = w;
        }
        return;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
        if (col + e < K) p[turn ? (long)(col + e) * M + row : (long)row * cols + col + e] = (PT)update_one<PT>(o.v[e], x[e], scale, decay, alpha);
}

// The row that lane i of 16 holds in block t of 16 rows.  The turned fragment of a block has rows i = 4q .. 4q+3 of it in lane group
// q; in this order blocks 2p and 2p + 1 put rows 32p + 8q .. 32p + 8q + 7 there, which is where an MFMA has them.  A single block
// (MT = 1) is in natural order: its fragment is put together by lane swaps instead.
template <int MT>
__device__ __forceinline__ int chain_row(int t, int i) {
    return MT == 1 ? i : 32 * (t >> 1) + 8 * (i >> 2) + 4 * (t & 1) + (i & 3);
}

// Rows 4q .. 4q+3 of a column in lane group q = l/16 become rows 8q .. 8q+7 in groups 0 and 1, and zeros in 2 and 3.
__device__ __forceinline__ bf16x8 gather_rows16(const bf16x4& v) {
    u32x2 r = __builtin_bit_cast(u32x2, v);
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const auto half = __builtin_amdgcn_permlane32_swap(r[e], 0u, false, false);      // groups 0, 1 and 2, 3, each before zeros
        const auto part = __builtin_amdgcn_permlane16_swap(half[0], half[1], false, false);  // groups 0, 2 and 1, 3
        o[e] = part[0];
        o[2 + e] = part[1];
    }
    return __builtin_bit_cast(bf16x8, o);
}

constexpr int CHAIN_WAVES = 8;
constexpr int CHAIN_FRAGS = 32;  // fragments of X a lane can hold: 128 of the 256 registers of a wave

// Fragments that a lane loads from memory (the blend; the parameter) together, while those before them are still on their way: loads and
// stores leave the queue in order, so a load that is issued behind a store waits for it as well.  One at a time, as written before, 56
// matrices of 5632 x 16 in fp32 took 142 us, now 117 (with four 117 as well, at the cost of 20 to 50 registers); 168 + 84 + 56 of 2048 and 512 columns
// 60 and 53; 256 of 2048 x 64 296 and 205 (a whole step; 256 of 64 x 2048 199 and 203 in fp32, 190 and 182 in bf16).  Asking for the parameter before the iterations, through LDS, gave nothing on top.
constexpr int kBatch = 2;

// MT blocks of 16 rows (1, 2 or 4), up to NCH chunks of 32 columns per wave.
template <int MT, int NCH>
__global__ void __launch_bounds__(64 * CHAIN_WAVES) ns_chain_kernel(const ChainList l, const ChainMath cm) {
    constexpr int NP = (MT + 1) / 2;         // 32-deep reductions over the rows
    constexpr int PITCH = 32 * NP + 8;       // of A and B in LDS; with MT = 1 columns 16 to 31 stay zero
    constexpr int NF = MT * (MT + 1) / 2;    // 16 x 16 blocks of A on or above the diagonal
    constexpr int BATCH = kBatch < MT ? 1 : kBatch / MT;  // chunks that are loaded from memory together
    constexpr bool TWO = MT < 4;             // while the next ones are on their way (with four blocks a chunk is enough, and two spill)
    // Chunks without a branch between them: 40 -> 30 ns for each MFMA of the chain through 176 chunks (16 x 5632).  Four blocks have
    // ten MFMAs between two branches anyway; and where a wave has four chunks at most, those that are not there cost as much as the
    // branches (111 of 20 x 56, one chunk: 17.5 with runs, 16.0 without).
    constexpr int RUN = MT == 4 || NCH < 8 ? 1 : 4;
    static_assert(NCH % RUN == 0, "whole runs");
    constexpr int LEG = MT == 4 ? 2 : 1, NLEG = NF / LEG;  // blocks that a wave adds its chunks to at a time
    __shared__ __align__(16) f32x4 sum[NF][64];
    __shared__ __align__(16) bf16_t As[MT * 16][PITCH], Bs[MT * 16][PITCH];
    __shared__ float red[4];

    int bucket = 0;
    while (bucket + 1 < l.n && (int)blockIdx.x >= l.start[bucket + 1]) ++bucket;
    const ChainBucket& k = l.b[__builtin_amdgcn_readfirstlane(bucket)];
    const int b = blockIdx.x - l.start[__builtin_amdgcn_readfirstlane(bucket)];
    const bool turn = k.rows > k.cols;
    const int M = turn ? k.cols : k.rows, K = turn ? k.rows : k.cols;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i = lane & 15, q = lane >> 4;
    const int per = ((K + 31) / 32 + CHAIN_WAVES - 1) / CHAIN_WAVES;  // chunks per wave
    const int col0 = wave * per * 32 + 8 * q;                         // this lane's first column in the wave's chunk 0
    const bf16_t* u = k.U + b * k.strideU;
    bf16_t* area = k.X + b * k.strideX;
    // this lane's fragments in the work area: read and written by this lane only
    bf16x8* mine = (bf16x8*)area + (long)wave * per * MT * 64 + lane;

    for (int t = tid; t < MT * 16 * PITCH; t += 64 * CHAIN_WAVES) {
        (&As[0][0])[t] = (bf16_t)0.f;
        (&Bs[0][0])[t] = (bf16_t)0.f;
    }
    // d = bf(bf(sqrt(sum)) + 1e-7), in the order of the normalisation kernel: both halves of the workgroup add the same sums
    float s = 0.f;
    for (int t = tid & 255; t < k.nparts; t += 256) s += k.partials[(long)b * k.nparts + t];
    s = wave_sum(s);
    if (lane == 0 && wave < 4) red[wave] = s;
    __syncthreads();
    const float d = rbf(rbf(sqrtf((red[0] + red[1]) + (red[2] + red[3]))) + 1e-7f);

    // Normalised fragments, zero past the matrix's edges.  Through the work area, so that the loop over loads of every kind
    // (ragged, turned) and divisions need not be unrolled over the register array.
    const bool vec = !turn && K % 8 == 0;
    auto fetch = [&](bf16x8& v, int j, int t) {
        const int row = chain_row<MT>(t, i), col = col0 + j * 32;
        if (vec && row < M && col < K) {
            v = *(const bf16x8*)(u + (long)row * K + col);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                v[e] = (row < M && col + e < K) ? u[turn ? (long)(col + e) * M + row : (long)row * K + col + e] : (bf16_t)0.f;
        }
    };
    auto norm = [&](bf16x8& v, int j, int t) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = f2bf(__fdiv_rn(bf2f(v[e]), d));
        mine[(j * MT + t) * 64] = v;
    };
    if constexpr (TWO) {
        bf16x8 v[2][BATCH][MT];
        auto each = [&](int j0, bf16x8 (&w)[BATCH][MT], auto f) {
#pragma unroll
            for (int jj = 0; jj < BATCH; ++jj)
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    if (j0 + jj < per) f(w[jj][t], j0 + jj, t);
        };
        each(0, v[0], fetch);
        for (int j0 = 0; j0 < per; j0 += 2 * BATCH) {
            each(j0 + BATCH, v[1], fetch);
            each(j0, v[0], norm);
            each(j0 + 2 * BATCH, v[0], fetch);
            each(j0 + BATCH, v[1], norm);
        }
    } else {
        // Four blocks in one order: a chunk's loads together would gain 4 % at 256 of 64 x 2048 and lose 9 % at 2048 x 64 (its elements
        // come one by one) and 5 % at 111 of 34 x 56.
#pragma unroll 4
        for (int j = 0; j < per; ++j) {
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                bf16x8 v;
                fetch(v, j, t);
                norm(v, j, t);
            }
        }
    }
    bf16x8 zero8, unit[2];  // unit[h]: selects columns 8q' + 4h + 0..3 (q' = 0..3) of a chunk
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        zero8[e] = (bf16_t)0.f;
#pragma unroll
        for (int h = 0; h < 2; ++h) unit[h][e] = (bf16_t)((q == i >> 2 && e == 4 * h + (i & 3)) ? 1.f : 0.f);
    }
    bf16x8 x[NCH][MT];
#pragma unroll
    for (int j = 0; j < NCH; ++j)
#pragma unroll
        for (int t = 0; t < MT; ++t) x[j][t] = j < per ? mine[(j * MT + t) * 64] : zero8;
    // The sum of leg `leg` (LEG blocks of A) over this wave's chunks, on top of the waves' before it.
    auto add_leg = [&](auto leg_c) {
        constexpr int F0 = decltype(leg_c)::value * LEG;
        f32x4 acc[LEG];
#pragma unroll
        for (int f = 0; f < LEG; ++f) acc[f] = wave == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : sum[F0 + f][lane];
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
    };

    for (int it = 0; it < cm.steps; ++it) {
        // A wave starts a leg when the wave before it has left it, so the legs follow one another through the waves.
        for (int slot = 0; slot < NLEG + CHAIN_WAVES - 1; ++slot) {
            const int leg = slot - wave;
            if (leg == 0) add_leg(std::integral_constant<int, 0>{});
            if constexpr (NLEG > 1) if (leg == 1) add_leg(std::integral_constant<int, 1>{});
            if constexpr (NLEG > 2) if (leg == 2) add_leg(std::integral_constant<int, 2>{});
            if constexpr (NLEG > 3) if (leg == 3) add_leg(std::integral_constant<int, 3>{});
            if constexpr (NLEG > 4) if (leg == 4) add_leg(std::integral_constant<int, 4>{});
            static_assert(NLEG <= 5 && NLEG * LEG == NF, "every leg has its branch");
            __syncthreads();
        }
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
        for (int f = wave; f < MT * MT; f += CHAIN_WAVES) {
            const int ti = f / MT, tj = f % MT;
            f32x4 aa = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int p = 0; p < NP; ++p)
                aa = mfma(*(const bf16x8*)&As[ti * 16 + i][p * 32 + 8 * q], *(const bf16x8*)&As[tj * 16 + i][p * 32 + 8 * q], aa);
            const bf16x4 av = *(const bf16x4*)&As[tj * 16 + i][ti * 16 + 4 * q];
            bf16x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = f2bf(rbf(cm.b * bf2f(av[e])) + rbf(cm.c * rbf(aa[e])));
            *(bf16x4*)&Bs[tj * 16 + i][ti * 16 + 4 * q] = o;
        }
        __syncthreads();
        bf16x8 bfr[MT][NP];  // B's rows, in the order of X's
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int p = 0; p < NP; ++p) bfr[t][p] = *(const bf16x8*)&Bs[chain_row<MT>(t, i)][p * 32 + 8 * q];
        auto next_chunk = [&](bf16x8 (&xc)[MT]) {
            bf16x8 xt[2][NP];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    const f32x4 v = mfma(xc[t], unit[h], f32x4{0.f, 0.f, 0.f, 0.f});
                    if constexpr (MT == 1) {
                        xt[h][0] = gather_rows16(bf16x4{f2bf(v[0]), f2bf(v[1]), f2bf(v[2]), f2bf(v[3])});
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) xt[h][t / 2][4 * (t & 1) + e] = f2bf(v[e]);
                    }
                }
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int p = 0; p < NP; ++p) v = mfma(xt[h][p], bfr[t][p], v);
#pragma unroll
                    for (int e = 0; e < 4; ++e) xc[t][4 * h + e] = f2bf(rbf(cm.a * bf2f(xc[t][4 * h + e])) + rbf(v[e]));
                }
        };
#pragma unroll
        for (int j0 = 0; j0 < NCH; j0 += RUN) {
            if (j0 + RUN <= per) {
#pragma unroll
                for (int j = j0; j < j0 + RUN; ++j) next_chunk(x[j]);
            } else {  // (nothing is computed past the last chunk: with an infinite B its zeros would not stay zero)
#pragma unroll
                for (int j = j0; j < j0 + RUN - 1; ++j)
                    if (j < per) next_chunk(x[j]);
            }
        }
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
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (row < M && col + e < K) out[turn ? (long)(col + e) * M + row : (long)row * K + col + e] = v[e];
            }
        return;
    }
    void* p = const_cast<void*>(k.p_ptrs[b]);
    const bool whole = whole_rows(p, k.cols, turn);
    auto update = [&](auto* pp) {
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
                load8(w.o[jj][t], pp, row, col, k.cols, M, K, turn, whole);
            });
        };
        auto store = [&](int j0, Batch& w) {
            each(j0, [&](int jj, int t, int row, int col) {
                store8(pp, w.o[jj][t], w.v[jj][t], row, col, k.cols, M, K, turn, whole, k.scale, cm.decay, cm.alpha);
            });
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
    if (cm.p_dtype == MUON_HIP_BF16) update((bf16_t*)p);
    else update((float*)p);
}

int chain_blocks(int M) { return M <= 16 ? 1 : M <= 32 ? 2 : 4; }
int chain_per_wave(int K) { return ((K + 31) / 32 + CHAIN_WAVES - 1) / CHAIN_WAVES; }

template <int MT>
void launch_as(int nch, const ChainList& l, const ChainMath& cm, hipStream_t stream) {
    const dim3 grid(l.start[l.n]), block(64 * CHAIN_WAVES);
    if (nch * MT == 8) hipLaunchKernelGGL((ns_chain_kernel<MT, 8 / MT>), grid, block, 0, stream, l, cm);
    else if (nch * MT == 16) hipLaunchKernelGGL((ns_chain_kernel<MT, 16 / MT>), grid, block, 0, stream, l, cm);
    else hipLaunchKernelGGL((ns_chain_kernel<MT, 32 / MT>), grid, block, 0, stream, l, cm);
}

}  // namespace

bool chain_fits(int M, int K) { return M <= 64 && K <= 8192 && chain_per_wave(K) * chain_blocks(M) <= CHAIN_FRAGS; }

// Measured (profiles/low_rank_result_copy.txt, iterations and result), with the copy | written by the chain.  Whole pieces of rows cost the
// chain nothing: 32 x 4096, one | 256 matrices 78 | 77 and 124 | 95 us.  Element by element a workgroup pays 0.6 us for a fragment, which
// few matrices of many fragments feel more than the copy: one of 4096 x 32 (32 fragments) 93 | 112, of 512 x 64 (eight) 40.5 | 42.8, of
// 512 x 16 (two) 18.1 | 16.5.  With many matrices the copy, a pass over memory, costs more.  The lines cross between 64 matrices (5632 x 16,
// 512 x 64) and 160 (2048 x 64); at three quarters of the compute units the chain is ahead everywhere: 192 of 5632 x 16 144 | 106, of
// 4096 x 32 147 | 130, of 2048 x 64 143 | 135.  (Rows that are no whole pieces and not turned are the exception: 33 x 515, 192 matrices
// 60.5 | 58.4, 1024 229 | 237.)
bool chain_writes(int rows, int cols, int batch, const void* out, int cus) {
    if (rows <= cols && cols % 8 == 0 && ((uintptr_t)out & 15) == 0) return true;
    return 4L * batch >= 3L * cus || chain_per_wave(std::max(rows, cols)) * chain_blocks(std::min(rows, cols)) <= 4;
}

// One launch per kernel: blocks of rows, and 8, 16 or 32 fragments of X per lane (fewer registers, more workgroups in flight).
hipError_t launch_ns_chain(const ChainBucket* buckets, int n, const ChainMath& cm, hipStream_t stream) {
    if (n < 1 || n > CHAIN_MAX_LIST || cm.steps < 1) return hipErrorInvalidValue;
    for (int mt = 4; mt >= 1; mt /= 2)
        for (int frags = CHAIN_FRAGS; frags >= 8; frags /= 2) {
            ChainList l;
            l.n = 0;
            l.start[0] = 0;
            for (int i = 0; i < n; ++i) {
                const ChainBucket& k = buckets[i];
                const int M = k.rows < k.cols ? k.rows : k.cols, K = k.rows < k.cols ? k.cols : k.rows;
                if (!chain_fits(M, K)) return hipErrorInvalidValue;
                const int need = chain_per_wave(K) * chain_blocks(M);
                if (chain_blocks(M) != mt || (need <= 8 ? 8 : need <= 16 ? 16 : 32) != frags) continue;
                l.b[l.n] = k;
                l.start[l.n + 1] = l.start[l.n] + k.batch;
                ++l.n;
            }
            if (!l.n) continue;
            if (mt == 4) launch_as<4>(frags / 4, l, cm, stream);
            else if (mt == 2) launch_as<2>(frags / 2, l, cm, stream);
            else launch_as<1>(frags, l, cm, stream);
            if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
        }
    return hipSuccess;
}
