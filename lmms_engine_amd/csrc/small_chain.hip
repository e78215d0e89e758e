// Newton-Schulz for matrices with a short side of at most 64 (low-rank adapters): normalisation, every iteration and the
// parameter update in one kernel, a workgroup per matrix, X in registers from the first product to the last.
//
// The tiled products of gemm_nt.hip pad a short side to 128 rows and stream X from memory three times an iteration: for 16 rows
// that is 64 times the multiplications, eight times the bytes and 17 launches.  Here the matrix is read once and the result (or
// the parameter) written once; what bounds it is the chain of dependent steps inside a workgroup (five iterations of a walk over
// the wave's chunks and four barriers) times the rounds of workgroups, not memory.  fast_newtonschulz, us, tiles | this:
//      16 x  512, 1 | 256 | 1024 matrices   97 |  191 |  609    22 |  22 |  42
//      16 x 5632                           217 | 1414 | 5461    58 |  95 | 416
//      32 x 4096                           181 | 1087 | 4229    78 | 149 | 586
//      64 x 2048                           137 |  556 | 2322    87 | 159 | 623
//    2048 x   64                           139 |  567 | 2363   100 | 182 | 705
// It wins wherever the registers hold the matrix, so that is the rule (chain_fits); larger ones take the tiled products.
//
// Eight waves share the columns of X in chunks of 32.  Lane (i = l%16, q = l/16) of a wave holds X[16 t + i][8q .. 8q+7] of a
// chunk for every block t of 16 rows: an operand fragment of v_mfma_f32_16x16x32_bf16 as it stands, so
//   A = X Xt      contracts such fragments with one another; the eight partial sums meet in LDS;
//   B = bA + cAA  is a handful of MFMAs on A in LDS;
//   X' = aX + BX  contracts rows, for which a chunk is turned by multiplying it with selected columns of the identity (exact:
//                 one product is the element, the others are zero): the result's four registers are four rows of one column,
//                 the fragment that B's rows meet, and what comes out lies as X lay.
// Rounding points are those of the tiled kernels (bf(X Xt); bf(bf(bA) + bf(c bf(AA))); bf(bf(aX) + bf(BX))), sums are fp32.
#include "small_chain.h"

namespace {

typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma(const bf16x8& p, const bf16x8& q, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(p, q, c, 0, 0, 0);
}

template <typename PT>
__device__ __forceinline__ float update_one(float p, bf16_t x, float scale, float decay, float alpha) {
    const float os = rbf(bf2f(x) * scale);
    const float pd = sizeof(PT) == 2 ? rbf(p * decay) : p * decay;
    return fmaf(alpha, os, pd);
}

// Eight consecutive columns of one row of X to the parameter: a piece of its row, or (turned) of its column.
template <typename PT>
__device__ __forceinline__ void update8(PT* p, const bf16x8& x, int row, int col, int cols, int M, int K, bool turn, float scale,
                                        float decay, float alpha) {
    if (turn) {
        for (int e = 0; e < 8 && col + e < K; ++e) {
            PT* d = p + (long)(col + e) * M + row;
            *d = (PT)update_one<PT>((float)*d, x[e], scale, decay, alpha);
        }
        return;
    }
    PT* d = p + (long)row * cols + col;
    if (cols % 8 == 0 && (((uintptr_t)p) & 15) == 0) {  // eight columns are all there or none is
        if constexpr (sizeof(PT) == 2) {
            bf16x8 v = *(const bf16x8*)d;
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = f2bf(update_one<PT>(bf2f(v[e]), x[e], scale, decay, alpha));
            *(bf16x8*)d = v;
        } else {
            f32x4 v = *(const f32x4*)d, w = *(const f32x4*)(d + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = update_one<PT>(v[e], x[e], scale, decay, alpha);
                w[e] = update_one<PT>(w[e], x[4 + e], scale, decay, alpha);
            }
            *(f32x4*)d = v;
            *(f32x4*)(d + 4) = w;
        }
        return;
    }
    for (int e = 0; e < 8 && col + e < K; ++e) d[e] = (PT)update_one<PT>((float)d[e], x[e], scale, decay, alpha);
}

constexpr int CHAIN_WAVES = 8;
constexpr int CHAIN_FRAGS = 32;  // fragments of X a lane can hold: 128 of the 256 registers of a wave

// MT blocks of 16 rows (1, 2 or 4), up to NCH chunks of 32 columns per wave.
template <int MT, int NCH>
__global__ void __launch_bounds__(64 * CHAIN_WAVES) ns_chain_kernel(const ChainList l, const ChainMath cm) {
    constexpr int NP = (MT + 1) / 2;         // 32-deep reductions over the rows
    constexpr int PITCH = 32 * NP + 8;       // of A and B in LDS; with MT = 1 columns 16 to 31 stay zero
    constexpr int NF = MT * (MT + 1) / 2;    // 16 x 16 blocks of A on or above the diagonal
    constexpr int HALF = CHAIN_WAVES / 2;
    __shared__ __align__(16) f32x4 part[HALF][NF][64];
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
#pragma unroll 4
    for (int j = 0; j < per; ++j) {
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const int row = t * 16 + i, col = col0 + j * 32;
            bf16x8 v;
            if (vec && row < M && col < K) {
                v = *(const bf16x8*)(u + (long)row * K + col);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    v[e] = (row < M && col + e < K) ? u[turn ? (long)(col + e) * M + row : (long)row * K + col + e] : (bf16_t)0.f;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = f2bf(__fdiv_rn(bf2f(v[e]), d));
            mine[(j * MT + t) * 64] = v;
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
    f32x4 acc[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto gram = [&](const bf16x8 (&xc)[MT]) {
        int f = 0;
#pragma unroll
        for (int ti = 0; ti < MT; ++ti)
#pragma unroll
            for (int tj = ti; tj < MT; ++tj, ++f) acc[f] = mfma(xc[ti], xc[tj], acc[f]);
    };
#pragma unroll
    for (int j = 0; j < NCH; ++j)
#pragma unroll
        for (int t = 0; t < MT; ++t) x[j][t] = j < per ? mine[(j * MT + t) * 64] : zero8;
#pragma unroll
    for (int j = 0; j < NCH; ++j) gram(x[j]);

    for (int it = 0; it < cm.steps; ++it) {
        // the eight partial sums, in a fixed order
        if (wave >= HALF) {
#pragma unroll
            for (int f = 0; f < NF; ++f) part[wave - HALF][f][lane] = acc[f];
        }
        __syncthreads();
        if (wave < HALF) {
#pragma unroll
            for (int f = 0; f < NF; ++f) part[wave][f][lane] = part[wave][f][lane] + acc[f];
        }
        __syncthreads();
        for (int t = tid; t < NF * 64; t += 64 * CHAIN_WAVES) {
            const int ln = t & 63;
            int f = t >> 6, ti = 0;
            const f32x4 sum = (part[0][f][ln] + part[1][f][ln]) + (part[2][f][ln] + part[3][f][ln]);
            while (f >= MT - ti) f -= MT - ti++;
            const int tj = ti + f, r = ti * 16 + (ln >> 4) * 4, c = tj * 16 + (ln & 15);
            bf16x4_t o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = f2bf(sum[e]);
            *(bf16x4_t*)&As[c][r] = o;  // A is symmetric: the mirrored block in one piece, this one element by element
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
            const bf16x4_t av = *(const bf16x4_t*)&As[tj * 16 + i][ti * 16 + 4 * q];
            bf16x4_t o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = f2bf(rbf(cm.b * bf2f(av[e])) + rbf(cm.c * rbf(aa[e])));
            *(bf16x4_t*)&Bs[tj * 16 + i][ti * 16 + 4 * q] = o;
        }
        __syncthreads();
        bf16x8 bfr[MT][NP];  // B's rows, in the order that the turned chunks have their rows in
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                const bf16x4_t lo = *(const bf16x4_t*)&Bs[t * 16 + i][p * 32 + 4 * q], hi = *(const bf16x4_t*)&Bs[t * 16 + i][p * 32 + 16 + 4 * q];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    bfr[t][p][e] = lo[e];
                    bfr[t][p][4 + e] = hi[e];
                }
            }
#pragma unroll
        for (int f = 0; f < NF; ++f) acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto next_chunk = [&](bf16x8 (&xc)[MT]) {
            bf16x8 xt[2][NP];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int t = 0; t < 2 * NP; ++t) {
                    const f32x4 v = t < MT ? mfma(xc[t < MT ? t : 0], unit[h], f32x4{0.f, 0.f, 0.f, 0.f}) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int e = 0; e < 4; ++e) xt[h][t / 2][4 * (t & 1) + e] = f2bf(v[e]);
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
            gram(xc);
        };
#pragma unroll
        for (int j = 0; j < NCH; ++j)
            if (j < per) next_chunk(x[j]);
    }

    if (!k.p_ptrs) {
#pragma unroll
        for (int j = 0; j < NCH; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                const int row = t * 16 + i, col = col0 + j * 32;
                if (j < per && row < M && col < K) *(bf16x8*)(area + blocked_offset(row, col, k.cbx)) = x[j][t];
            }
        return;
    }
#pragma unroll
    for (int j = 0; j < NCH; ++j)
#pragma unroll
        for (int t = 0; t < MT; ++t)
            if (j < per) mine[(j * MT + t) * 64] = x[j][t];
    void* p = const_cast<void*>(k.p_ptrs[b]);
    for (int j = 0; j < per; ++j)
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const int row = t * 16 + i, col = col0 + j * 32;
            if (row >= M || col >= K) continue;
            const bf16x8 v = mine[(j * MT + t) * 64];
            if (cm.p_dtype == MUON_HIP_BF16) update8((bf16_t*)p, v, row, col, k.cols, M, K, turn, k.scale, cm.decay, cm.alpha);
            else update8((float*)p, v, row, col, k.cols, M, K, turn, k.scale, cm.decay, cm.alpha);
        }
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
