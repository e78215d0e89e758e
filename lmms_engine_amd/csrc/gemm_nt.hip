// GEMM family for the Newton-Schulz chain on gfx950, built on v_mfma_f32_16x16x32_bf16.
//
// Why the 16x16x32 instruction: under matrix-pipe load the part lowers its clock to stay inside its power
// limit, and on operands with random mantissas a loop of nothing but MFMAs (probe.hip, a measurement library of its own) sustains about
// 1.85 PFLOP/s with 32x32x16 and about 2.09 with 16x16x32 (both reach 2.45 on constant operands): the deeper dot
// product updates each fp32 accumulator half as often per FLOP.  The same kernels built on 32x32x16 ran 4 to 8 %
// slower at a 3 to 9 % lower clock.  Operand fragment: lane l holds row l%16, eight consecutive k from 8*(l/16)
// (16 bytes).  Accumulator fragment: lane l holds column l%16, rows 4*(l/16)+0..3 (f32x4).
//
// The three products of one NS iteration:
//   SYRK     A  = bf(X Xt)                         P = Q = X   (M x K)           C[i][j] = sum_k P[i][k] Q[j][k]
//   SYMPOLY  B  = bf(bf(b A) + bf(c bf(A A)))      P = Q = A   (M x M, symmetric so A A = A At)      same
//   BX       X' = bf(bf(a X) + bf(B X))            P = B (M x M), Q = X (M x K)  C[i][j] = sum_k P[i][k] Q[k][j]
// SYRK/SYMPOLY contract rows with rows and compute only tiles on or above the diagonal, mirrored in the
// epilogue, which makes the result symmetric bit for bit.  BX contracts rows of B with columns of X: its Q
// fragments come out of LDS through the transposing read ds_read_b64_tr_b16, so X is kept in one
// orientation only.
//
// Every bf16 rounding point of the reference's torch expressions
// (/root/reference/src/lmms_engine/utils/muon_utils.py:149-152) is applied in registers.
//
// Operands and results live in the blocked layout of common.h (256 x 32 blocks), zero padded
// by the producers to whole tiles, so there is no masking here; the host launcher checks that
// the shapes it is given are whole tiles before launching.
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "common.h"
#include "gemm_nt.h"

namespace {

// Upper-triangle tile order in row groups of GM: inside a group, column by column, so the
// ~32 tiles an XCD works on at a time touch few distinct row panels.
template <int GM>
__device__ __forceinline__ void tri_decode(int t, int T, int& ti, int& tj) {
    int r0 = 0, gm, cnt;
    for (;;) {  // find the row group that holds tile t
        gm = (T - r0 < GM) ? (T - r0) : GM;
        cnt = gm * (T - r0) - gm * (gm - 1) / 2;
        if (t < cnt || r0 + gm >= T) break;
        t -= cnt;
        r0 += gm;
    }
    const int tri = gm * (gm + 1) / 2;
    int c = 0, u = t;  // column c of the leading gm x gm triangle holds c+1 tiles
    while (u >= c + 1 && c < gm - 1) { u -= c + 1; ++c; }
    const int rest = t - tri;
    const bool in_tri = t < tri;
    ti = r0 + (in_tri ? u : rest % gm);
    tj = r0 + (in_tri ? c : gm + rest / gm);
}

template <int GM>
__device__ __forceinline__ void rect_decode(int t, int TM, int TN, int& ti, int& tj) {
    const int per_group = GM * TN;
    const int gidx = t / per_group;
    const int first = gidx * GM;
    const int gm = (TM - first < GM) ? (TM - first) : GM;
    const int r = t - gidx * per_group;
    ti = first + r % gm;
    tj = r / gm;
}

struct TileCoord {
    int bidx, ti, tj;
};

// A pointer that is the same in every lane, moved into scalar registers.
template <typename T>
__device__ __forceinline__ const T* uniform_ptr(const T* p) {
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return (const T*)(((unsigned long long)hi << 32) | lo);
}

// Tile `logical` (0 .. tiles_per_mat * batch - 1) in the launch order: matrix by matrix, 4-row groups.
template <int EPI>
__device__ __forceinline__ TileCoord tile_of(const GemmArgs& g, int logical) {
    const int bidx = logical / g.tiles_per_mat;
    const int t = logical - bidx * g.tiles_per_mat;
    int ti = 0, tj = 0;  // plain locals: references into the struct kept it in scratch memory
    if (epi_is_bx(EPI)) rect_decode<4>(t, g.tiles_m, g.tiles_n, ti, tj);
    else tri_decode<4>(t, g.tiles_m, ti, tj);
    return TileCoord{bidx, ti, tj};
}

// Tile `logical` of a list: its entry, and its place in that entry.
__device__ __forceinline__ int list_entry(const GemmList& l, int logical) {
    int i = 0;
    while (i + 1 < l.n && logical >= l.start[i + 1]) ++i;
    return __builtin_amdgcn_readfirstlane(i);
}

typedef __attribute__((address_space(3))) void* lds_void_ptr;
typedef const __attribute__((address_space(1))) void* glb_void_ptr;

// The thread's number.  COH: in a form that the compiler cannot take out of the loop over tiles, with everything that each kind of
// tile computes from it (which it did, and spilled).
template <bool COH>
__device__ __forceinline__ int thread_number() {
    int t = threadIdx.x;
    if constexpr (COH) asm volatile("" : "+v"(t));
    return t;
}

// 16 bytes at base + off elements.  COH: read at device scope, past this compute unit's vector cache, which may still hold what
// the address contained before another compute unit of the same launch wrote it (gemm_nt_flow_kernel).
typedef unsigned u32x4a __attribute__((ext_vector_type(4)));
template <bool COH>
__device__ __forceinline__ bf16x8 load16(const bf16_t* base, long off) {
    if constexpr (COH) {
        constexpr int kDeviceScope = 16;  // sc1
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, 0xffffffffu, 0x00027000);
        const u32x4a v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(off * 2), 0, kDeviceScope);
        return *(const bf16x8*)&v;
    } else {
        return *(const bf16x8*)(base + off);
    }
}

#define WAIT_LGKM0() __builtin_amdgcn_s_waitcnt(0xC07F)
// s_waitcnt with only vmcnt set: vmcnt is split over bits [3:0] and [15:14] (N < 64)
#define WAIT_VM(N) __builtin_amdgcn_s_waitcnt(0x0F70 | ((N) & 15) | (((N) >> 4) << 14))

// Start of row panel `row0` (a multiple of the tile edge, so the panel lies inside one row of
// blocks) of a blocked matrix with cb column blocks: add kblock * BLK_ELEMS to reach a k-tile.
__device__ __forceinline__ long panel_offset(int row0, int cb) {
    return (long)(row0 >> 8) * cb * BLK_ELEMS + (row0 & 255) * BLK_COLS;
}

// EPI_MMT: rows of a row-major C.  Pieces of 16 and 8 bytes where its rows are whole numbers of them, element by element otherwise
// and at the edge.
__device__ __forceinline__ bool dense_vec(const GemmArgs& g) { return g.dense_rows % 8 == 0 && (((uintptr_t)g.C) & 15) == 0; }
template <typename V>
__device__ __forceinline__ void dense_store(const GemmArgs& g, bool vec, int row, int col, const V& v) {
    constexpr int N = sizeof(V) / 2;
    bf16_t* p = g.C + (long)row * g.dense_rows + col;
    if (row >= g.dense_rows) return;
    if (vec && col + N <= g.dense_rows) {
        *(V*)p = v;
    } else {
        const bf16_t* e = (const bf16_t*)&v;
#pragma unroll
        for (int k = 0; k < N; ++k)
            if (col + k < g.dense_rows) p[k] = e[k];
    }
}

// EPI_MMT of a row-major X: where the panel of rows row0.. starts, and row r of it from there.  Past the last row of X that row
// again: what it gives lies outside C.
__device__ __forceinline__ long dense_panel(const GemmArgs& g, int row0) {
    return (long)(row0 < g.dense_rows ? row0 : g.dense_rows - 1) * g.dense_pitch;
}
__device__ __forceinline__ int dense_row(const GemmArgs& g, int row0, int r) {
    const int left = row0 < g.dense_rows ? g.dense_rows - 1 - row0 : 0;
    return (r < left ? r : left) * g.dense_pitch;
}

// ---- epilogue ------------------------------------------------------------------------------
// One LDS copy of the tile, both output orientations written as 16-byte vectors.  The tile
// lives in LDS as Tt[n][m] (n = local column, m = local row of the accumulator tile), the
// orientation of Ct and of the elementwise source Et.  Every lane writes its rounded accumulators
// as 8-byte pieces (4 consecutive m of one n, exactly what an accumulator lane holds: lane&15 owns
// column n, its four registers are rows 4*(lane>>4) + 0..3 of the 16x16 fragment); after one barrier rows of Tt
// leave as rows of Ct (SYMPOLY adds the b.A term there, from pieces of Et that each thread loaded
// into registers before the accumulators were written, and puts the sums back), while rows of C
// are gathered with ds_read_b64_tr_b16: in a group of 16 lanes, lane i receives element i%4 of the
// 8-byte pieces addressed by lanes i/4, 4+i/4, 8+i/4, 12+i/4.
// Diagonal tiles of the symmetric kernels: only the 32x32 fragments on or above the diagonal need to be
// computed; the Ct pass writes them as the lower half (and the diagonal fragments) of the tile, the gather
// writes the upper half.  Inside a diagonal fragment acc(i,j) and acc(j,i) are sums of the same exact products
// in the same order, so the result is symmetric bit for bit.
template <int BM, int BN>
constexpr int epilogue_bytes() { return BN * (BM * 2 + 16); }

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ s16x4 lds_read_tr16(const unsigned char* p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(lds_void_ptr)p);
}

//
// The epilogues come in two parts: EPI_LOADS fetches the elementwise term into `ev` (16-byte pieces, tile_pieces of them for a
// thread), EPI_REST does everything else.  On 128-tiles the registers have room for the term beside the accumulators: it is
// fetched in front of the k loop and its latency passes behind the first k-tiles'.
enum { EPI_LOADS = 1, EPI_REST = 2, EPI_ALL = 3 };
template <int BM, int BN, int WGM, int WGN>
constexpr int tile_pieces() { return BM * BN / 8 / (WGM * WGN * 64); }

template <int BM, int BN, int WGM, int WGN, int EPI, bool MASKED, bool COH, int PART, int NEV>
__device__ __forceinline__ void epilogue(const GemmArgs& g, const TileCoord& tc,
                                         f32x4 (&acc)[BM / WGM / 16][BN / WGN / 16], unsigned char* smem, bf16x8 (&ev)[NEV]) {
    constexpr int NT = WGM * WGN * 64;
    constexpr int WTM = BM / WGM, WTN = BN / WGN;
    constexpr int FM = WTM / 16, FN = WTN / 16;
    constexpr int S = BM * 2 + 16;      // Tt row pitch (bytes): conflict-free for the 8-byte pieces
    constexpr int NLE = BN * (BM / 8) / NT;  // 16-byte chunks per thread for a whole tile
    static_assert((BN * (BM / 8)) % NT == 0 && BM % 64 == 0, "even split");
    const int tid = thread_number<COH>(), lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WGN, wn = wave % WGN, quad = lane >> 4;
    const int m0 = tc.ti * BM, n0 = tc.tj * BN;
    const bool diag = (!epi_is_bx(EPI)) && (tc.ti == tc.tj);
    // Et and Ct hold the tile as rows n0.. (BN of them) x columns m0.. (BM of them).  Chunk c of a
    // thread: 16 bytes j = c%8 of the 128-byte row piece of row n = (c/8)%BN in column block c/8/BN,
    // so that a wave touches 8 rows x 128 bytes = 1 KB of one block, contiguous in memory.
    // The return value says whether the chunk is a computed one: in a diagonal tile of a MASKED caller (the
    // ping-pong kernel, which skips the others) only the 32x32 fragments on or above the diagonal are, i.e. column
    // block m/32 <= row block n/32 of Tt.  A caller that computes whole diagonal tiles writes them in the Ct pass.
    auto tile_chunk = [&](int c, int cb, long& goff, int& loff) {
        constexpr int CPB = BLK_COLS / 8;  // 16-byte chunks per row of a block
        static_assert(BLK_COLS == 32, "a column block is one fragment wide");
        const int j = c % CPB, n = (c / CPB) % BN, cbk = (c / CPB) / BN;
        goff = panel_offset(n0, cb) + (long)((m0 >> BLK_SHIFT) + cbk) * BLK_ELEMS + n * BLK_COLS + j * 8;
        loff = n * S + (cbk * CPB + j) * 16;
        return !MASKED || !diag || cbk <= (n >> 5);
    };
    // SYMPOLY: this thread's 16-byte pieces of the b.A term, in the layout of the Ct pass, go to registers
    // first, so that the loads are in flight while the accumulators are rounded into LDS
    static_assert(NEV >= (EPI == EPI_SYMPOLY ? NLE : 1), "pieces of the b.A term");
    if constexpr (EPI == EPI_SYMPOLY && (PART & EPI_LOADS)) {
        const bf16_t* Et = g.Et + tc.bidx * g.strideEt;
#pragma unroll
        for (int u = 0; u < NLE; ++u) {
            long goff;
            int loff;
            tile_chunk(tid + u * NT, g.cbEt, goff, loff);
            ev[u] = load16<COH>(Et, goff);
        }
    }
    if constexpr (!(PART & EPI_REST)) return;
    __syncthreads();  // the operand stages are no longer read
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            bf16x4 o;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float v = rbf(acc[i][j][r]);
                if (EPI == EPI_SYMPOLY) v = g.s1 * v;
                o[r] = f2bf(v);
            }
            *(bf16x4*)(smem + (wn * WTN + j * 16 + (lane & 15)) * S + (wm * WTM + i * 16 + quad * 4) * 2) = o;
        }
    __syncthreads();
    {
        // rows of Tt leave as rows of Ct; SYMPOLY adds the rounded b.A term here and, when the tile itself is
        // gathered from LDS afterwards, puts the finished pieces back
        bf16_t* Ct = g.Ct + tc.bidx * g.strideCt;
        if constexpr (EPI == EPI_MMT) {  // whole tile rows: a wave covers 64 pieces of a row, 256 or 512 bytes at a time
            const bool vec = dense_vec(g);
#pragma unroll
            for (int u = 0; u < NLE; ++u) {
                const int c = tid + u * NT, n = c / (BM / 8), piece = c % (BM / 8);
                if (MASKED && diag && (piece >> 2) > (n >> 5)) continue;
                dense_store(g, vec, n0 + n, m0 + piece * 8, *(const u32x4*)(smem + n * S + piece * 16));
            }
        } else
#pragma unroll
        for (int u = 0; u < NLE; ++u) {
            long goff;
            int loff;
            const bool computed = tile_chunk(tid + u * NT, g.cbCt, goff, loff);
            bf16x8 t = *(const bf16x8*)(smem + loff);
            if (EPI == EPI_SYMPOLY) {
#pragma unroll
                for (int k = 0; k < 8; ++k) t[k] = f2bf(rbf(g.s0 * bf2f(ev[u][k])) + bf2f(t[k]));
                if (MASKED ? computed : !diag) *(bf16x8*)(smem + loff) = t;
            }
            if (g.Ct && computed) *(bf16x8*)(Ct + goff) = t;
        }
        if (EPI == EPI_SYMPOLY && (MASKED || !diag)) __syncthreads();
    }
    if (g.C && (MASKED || !diag)) {
        // lane j = 4r+s of a group addresses row n + 8s + r (then + 4), pieces m = 4c..4c+3: lane i = 4s+e
        // receives Tt[n+8s .. n+8s+7][4c+e], 16 bytes of row 4c+e of C.  The four groups of a wave sit
        // side by side along n (128 columns = two column blocks): 4 rows x 128 bytes per block and store.
        const int grp = lane >> 4, i16 = lane & 15;
        const unsigned char* src = smem + ((i16 & 3) * 8 + (i16 >> 2) + grp * 32) * S;
        bf16_t* dst = g.C + tc.bidx * g.strideC + panel_offset(m0, g.cbC) +
                      (long)((n0 >> BLK_SHIFT) + ((grp * 32) >> BLK_SHIFT)) * BLK_ELEMS + (i16 & 3) * BLK_COLS +
                      ((grp * 32) & (BLK_COLS - 1)) + (i16 >> 2) * 8;
        constexpr int NSTRIP = BN / 128, NQUAD = BM / 4, NW = NT / 64;
        constexpr int NUNIT = NSTRIP * NQUAD / NW;
        static_assert(BN % 128 == 0 && (NSTRIP * NQUAD) % NW == 0, "whole 128-column strips per wave");
#pragma unroll 8
        for (int u = 0; u < NUNIT; ++u) {
            const int wu = wave + u * NW, strip = wu % NSTRIP, c = wu / NSTRIP;
            const unsigned char* q = src + strip * 128 * S + c * 8;
            const s16x4 lo = lds_read_tr16(q), hi4 = lds_read_tr16(q + 4 * S);
            const s16x8 o = {lo[0], lo[1], lo[2], lo[3], hi4[0], hi4[1], hi4[2], hi4[3]};
            // a diagonal tile: the pieces strictly above the diagonal fragments (row block c/8 < column block);
            // the Ct pass has written the rest
            if (diag && (c >> 3) >= strip * 4 + grp) continue;
            if constexpr (EPI == EPI_MMT)
                dense_store(g, dense_vec(g), m0 + c * 4 + (i16 & 3), n0 + strip * 128 + grp * 32 + (i16 >> 2) * 8, o);
            else
                *(s16x8*)(dst + (long)strip * (128 / BLK_COLS) * BLK_ELEMS + c * 4 * BLK_COLS) = o;
        }
    }
}

// Epilogue of BX.  The accumulators were built with the MFMA operands swapped, so a lane holds 4
// consecutive columns n of one row m (lane&15 owns row m of its P fragment, its four registers are columns
// 4*(lane>>4) + 0..3 of its Q fragment): 8-byte pieces of rows of X'.  Every thread first issues the
// loads of its share of the a.X tile (16-byte pieces of rows, the layout of the output pass) into registers,
// then the rounded accumulators go to LDS as T[m][n] while those loads are in flight; after one barrier each
// thread reads its pieces of T, adds the rounded a.X term and stores rows of X' (1 KB contiguous per wave
// instruction).
template <int BM, int BN>
constexpr int epilogue_nn_bytes() { return BM * (BN * 2 + 16); }

// Folded parameter update: eight consecutive elements of one parameter row, o = bf16(X' * scale);
// p <- rnd(p * decay); p <- rnd(p + alpha * o), the arithmetic of the stand-alone update kernel (elementwise.hip).
// The parameter piece is fetched into registers early (fold_load) and applied after the tile has been through LDS.
template <bool WHOLE>
struct FoldPiece {
    f32x4 lo;                 // bf16 parameter: the eight values; fp32 parameter: the first four
    f32x4 hi[WHOLE ? 1 : 0];  // the other four; without them they are fetched when the piece is applied, from the cache line that
                              // the fetch of `lo` brought in
};
template <typename PT, bool WHOLE>
__device__ __forceinline__ void fold_load(FoldPiece<WHOLE>& f, const PT* p, int left) {
    if (left < 8) return;
    if constexpr (sizeof(PT) == 2) {
        const bf16x8 v = __builtin_nontemporal_load((const bf16x8_any*)p);
        f.lo = *(const f32x4*)&v;
    } else {
        f.lo = __builtin_nontemporal_load((const f32x4_any*)p);
        if constexpr (WHOLE) f.hi[0] = __builtin_nontemporal_load((const f32x4_any*)(p + 4));
    }
}
template <typename PT, bool WHOLE>
__device__ __forceinline__ void fold_apply(PT* p, const FoldPiece<WHOLE>& f, const bf16x8& x, int left, const GemmArgs& g) {
    constexpr bool PBF = std::is_same<PT, bf16_t>::value;
    auto one = [&](float pv, bf16_t xv) {
        const float os = rbf(bf2f(xv) * g.upd_scale);
        const float pd = PBF ? rbf(pv * g.upd_decay) : pv * g.upd_decay;
        return fmaf(g.upd_alpha, os, pd);
    };
    if (left >= 8) {
        if constexpr (PBF) {
            bf16x8 pv = *(const bf16x8*)&f.lo;
#pragma unroll
            for (int k = 0; k < 8; ++k) pv[k] = f2bf(one(bf2f(pv[k]), x[k]));
            __builtin_nontemporal_store(pv, (bf16x8_any*)p);
        } else {
            f32x4 a = f.lo, b;
            if constexpr (WHOLE) b = f.hi[0];
            else b = __builtin_nontemporal_load((const f32x4_any*)(p + 4));
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                a[k] = one(a[k], x[k]);
                b[k] = one(b[k], x[4 + k]);
            }
            __builtin_nontemporal_store(a, (f32x4_any*)p);
            __builtin_nontemporal_store(b, (f32x4_any*)(p + 4));
        }
    } else {  // the ragged end of a row: element by element
        for (int k = 0; k < 8 && k < left; ++k) {
            if constexpr (PBF) p[k] = f2bf(one(bf2f(p[k]), x[k]));
            else p[k] = one(p[k], x[k]);
        }
    }
}

__device__ __forceinline__ void result_store(bf16_t* p, const bf16x8& x, int left) {
    if (left >= 8) {
        *(bf16x8_any*)p = x;
    } else {
        for (int k = 0; k < 8 && k < left; ++k) p[k] = x[k];
    }
}

// pv: the parameter's pieces, fetched with the a.X term.  PRELOAD: they are, with EPI_LOADS; otherwise this part comes later, with
// the accumulators in LDS.
template <int BM, int BN, int WGM, int WGN, int FOLD, bool COH, int PART, int NEV, bool PRELOAD, int NPV>
__device__ __forceinline__ void epilogue_nn(const GemmArgs& g, const TileCoord& tc, f32x4 (&acc)[BM / WGM / 16][BN / WGN / 16],
                                            unsigned char* smem, bf16x8 (&ev)[NEV], FoldPiece<PRELOAD> (&pv)[NPV]) {
    constexpr int NT = WGM * WGN * 64;
    constexpr int WTM = BM / WGM, WTN = BN / WGN;
    constexpr int FM = WTM / 16, FN = WTN / 16;
    constexpr int S = BN * 2 + 16;           // T row pitch (bytes)
    constexpr int CPB = BLK_COLS / 8;        // 16-byte chunks per row of a block
    constexpr int NLE = BM * (BN / 8) / NT;  // 16-byte chunks per thread for a whole tile
    static_assert((BM * (BN / 8)) % NT == 0 && BN % BLK_COLS == 0, "even split");
    const int tid = thread_number<COH>(), lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WGN, wn = wave % WGN, quad = lane >> 4;
    const int m0 = tc.ti * BM, n0 = tc.tj * BN;
    // Last iteration of a step, parameter in the orientation of X: the scaled update goes straight into the
    // parameter (apply_scaling and the decay / update lines, muon_utils.py:167-175, :324-325) and X' is not written.
    constexpr bool fold = FOLD == 1;
    // chunk c: 16 bytes j of the row piece of row m in column block cbk of the tile.  Writing X' a wave covers
    // 16 rows of one block = 1 KB contiguous in the blocked layout; writing the parameter (row-major) it covers
    // whole tile rows instead, 2 x 512 B of bf16, and reads E in 64-byte pieces.
    auto decode = [&](int c, int& j, int& m, int& cbk) {
        if constexpr (fold) {
            const int piece = c % (BN / 8);
            m = c / (BN / 8);
            cbk = piece / CPB;
            j = piece % CPB;
        } else {
            j = c % CPB;
            m = (c / CPB) % BM;
            cbk = (c / CPB) / BM;
        }
    };
    auto tile_chunk = [&](int c, int cb, long& goff, int& loff) {
        int j, m, cbk;
        decode(c, j, m, cbk);
        goff = panel_offset(m0, cb) + (long)((n0 >> BLK_SHIFT) + cbk) * BLK_ELEMS + m * BLK_COLS + j * 8;
        loff = m * S + (cbk * CPB + j) * 16;
    };
    const bf16_t* Et = g.Et + tc.bidx * g.strideEt;
    static_assert(NEV == NLE && NPV >= (FOLD ? NLE : 1), "pieces of the tile");
    if constexpr (PART & EPI_LOADS) {
#pragma unroll
        for (int u = 0; u < NLE; ++u) {
            long goff;
            int loff;
            tile_chunk(tid + u * NT, g.cbEt, goff, loff);
            ev[u] = load16<COH>(Et, goff);
        }
    }
    // FOLD: the parameter, and this thread's piece u of the tile in it
    // (launch_gemm_nt: no other kernel is given a result to write)
    const bool result = FOLD && BM == 128 && NT == 512 && g.upd_dtype == GEMM_UPD_RESULT;
    void* pbase = !FOLD ? nullptr : result ? (bf16_t*)g.upd_ptrs + (long)tc.bidx * g.upd_rows * g.upd_cols : const_cast<void*>(g.upd_ptrs[tc.bidx]);
    const bool pbf = g.upd_dtype == MUON_HIP_BF16;
    constexpr int NSTRIP = BM / 128, NWV = NT / 64;
    const int grp = lane >> 4, i16 = lane & 15;
    auto piece = [&](int u, long& poff, int& left) {
        int row, col;
        if constexpr (FOLD == 2) {
            const int wu = wave + u * NWV, strip = wu % NSTRIP, c = wu / NSTRIP;
            row = n0 + c * 4 + (i16 & 3), col = m0 + strip * 128 + grp * 32 + (i16 >> 2) * 8;
        } else {
            int j, m, cbk;
            decode(tid + u * NT, j, m, cbk);
            row = m0 + m, col = n0 + cbk * BLK_COLS + j * 8;
        }
        poff = (long)row * g.upd_cols + col;
        left = g.upd_cols - col;
        return row < g.upd_rows && left > 0;
    };
    auto load_param = [&]() {
        if (result) return;
#pragma unroll
        for (int u = 0; u < NLE; ++u) {
            long poff;
            int left;
            if (!piece(u, poff, left)) continue;
            if (pbf) fold_load(pv[u], (const bf16_t*)pbase + poff, left);
            else fold_load(pv[u], (const float*)pbase + poff, left);
        }
    };
    if constexpr (FOLD && PRELOAD && (PART & EPI_LOADS)) load_param();
    if constexpr (!(PART & EPI_REST)) return;
    __syncthreads();  // the operand stages are no longer read
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            bf16x4 t;
#pragma unroll
            for (int r = 0; r < 4; ++r) t[r] = f2bf(acc[i][j][r]);
            *(bf16x4*)(smem + (wm * WTM + i * 16 + (lane & 15)) * S + (wn * WTN + j * 16 + quad * 4) * 2) = t;
        }
    bf16_t* C = g.C + tc.bidx * g.strideC;
    if constexpr (FOLD == 0) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < NLE; ++u) {
            long goff;
            int loff;
            tile_chunk(tid + u * NT, g.cbC, goff, loff);
            const bf16x8 t = *(const bf16x8*)(smem + loff);
            bf16x8 o;
#pragma unroll
            for (int k = 0; k < 8; ++k) o[k] = f2bf(rbf(g.s0 * bf2f(ev[u][k])) + bf2f(t[k]));
            *(bf16x8*)(C + goff) = o;
        }
        return;
    }
    if constexpr (FOLD == 2) {
        // The parameter is the transpose of X (rows > cols): row n0 + n of the parameter is column n of the tile.  The
        // finished X' values go back into T in place, and after a barrier a wave gathers them the other way round with
        // ds_read_b64_tr_b16 (the gather of the symmetric epilogue): lane i16 of a group of 16 receives
        // T[m .. m+7][4c + i16 % 4] with m = strip * 128 + grp * 32 + (i16 / 4) * 8, i.e. 16 bytes of row 4c + i16 % 4
        // of the parameter tile; a wave instruction covers 4 parameter rows x 128 columns.
        constexpr int NQUAD = BN / 4, NUNIT = NSTRIP * NQUAD / NWV;
        static_assert(BM % 128 == 0 && NUNIT * NWV == NSTRIP * NQUAD && NUNIT == NLE, "whole 128-row strips per wave");
        if constexpr (!PRELOAD) load_param();
        __syncthreads();
#pragma unroll
        for (int u = 0; u < NLE; ++u) {
            long goff;
            int loff;
            tile_chunk(tid + u * NT, g.cbC, goff, loff);
            const bf16x8 t = *(const bf16x8*)(smem + loff);
            bf16x8 o;
#pragma unroll
            for (int k = 0; k < 8; ++k) o[k] = f2bf(rbf(g.s0 * bf2f(ev[u][k])) + bf2f(t[k]));
            *(bf16x8*)(smem + loff) = o;
        }
        __syncthreads();
        // lane j = 4r+s of a group addresses row m + 8s + r of T (then + 4), columns 4c..4c+3
        const unsigned char* src = smem + ((i16 & 3) * 8 + (i16 >> 2) + grp * 32) * S;
#pragma unroll  // fully: the parameter pieces are indexed by u and must stay in registers
        for (int u = 0; u < NUNIT; ++u) {
            const int wu = wave + u * NWV, strip = wu % NSTRIP, c = wu / NSTRIP;
            const unsigned char* q = src + strip * 128 * S + c * 8;
            const s16x4 lo = lds_read_tr16(q), hi4 = lds_read_tr16(q + 4 * S);
            const s16x8 t8 = {lo[0], lo[1], lo[2], lo[3], hi4[0], hi4[1], hi4[2], hi4[3]};
            long poff;
            int left;
            if (piece(u, poff, left)) {
                const bf16x8 o = *(const bf16x8*)&t8;
                if (result) result_store((bf16_t*)pbase + poff, o, left);
                else if (pbf) fold_apply((bf16_t*)pbase + poff, pv[u], o, left, g);
                else fold_apply((float*)pbase + poff, pv[u], o, left, g);
            }
        }
        return;
    }
    // The parameter pieces are fetched here, with the accumulators already in LDS, so that their latency passes
    // behind the barrier.
    if constexpr (!PRELOAD) load_param();
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NLE; ++u) {
        long goff, poff;
        int loff, left;
        tile_chunk(tid + u * NT, g.cbC, goff, loff);
        const bf16x8 t = *(const bf16x8*)(smem + loff);
        bf16x8 o;
#pragma unroll
        for (int k = 0; k < 8; ++k) o[k] = f2bf(rbf(g.s0 * bf2f(ev[u][k])) + bf2f(t[k]));
        if (piece(u, poff, left)) {
            if (result) result_store((bf16_t*)pbase + poff, o, left);
            else if (pbf) fold_apply((bf16_t*)pbase + poff, pv[u], o, left, g);
            else fold_apply((float*)pbase + poff, pv[u], o, left, g);
        }
    }
}

// The same result for EPI_BX without LDS and without a barrier.  A lane holds, of fragment (i, j), columns 4q..4q+3
// (q = lane / 16) of row lane % 16 as two packed registers.  v_permlane16_swap_b32 exchanges the odd 16-lane rows of
// its first operand with the even rows of its second: applied to the registers of fragments j = 2t and 2t+1 it leaves
// a lane of row 0 / 2 with columns 0..7 / 8..15 of fragment 2t and a lane of row 1 / 3 with those of fragment 2t+1,
// i.e. 16 consecutive bytes of a row of X', and the 64 lanes of a wave with 16 rows x 64 bytes = one contiguous KB of
// the blocked layout, the same store the LDS version issues.  The a.X pieces are loaded in the same pattern.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ unsigned pack_bf16x2(float a, float b) {
    const bf16x2 p = {f2bf(a), f2bf(b)};
    return *(const unsigned*)&p;
}
//
// SPLIT: rows of the tile that the first of its two wave rows holds.  The wave rows may differ (variable-height tiles of the
// persistent kernel).  FMU: fragment rows this wave holds.  IN_BLOCK: the tile lies inside one row block, so that fragment rows
// are instruction offsets apart; otherwise each is addressed on its own, with scalar arithmetic.
template <int BN, int WGN, int SPLIT, int FMU, bool IN_BLOCK, bool COH, int PART, int FM, int FN, int NEV>
__device__ __forceinline__ void epilogue_nn_reg(const GemmArgs& g, int bidx, int m0, int n0, f32x4 (&acc)[FM][FN], bf16x8 (&ev)[NEV]) {
    constexpr int WTN = BN / WGN;
    static_assert(FN % 2 == 0 && FN * 16 == WTN && BLK_COLS == 32, "a pair of fragments is one column block");
    const int tid = thread_number<COH>(), lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN, row = lane >> 4;
    // piece (i, t): row m0 + wm*SPLIT + 16 i + lane%16, columns n0 + wn*WTN + 32 t + 16 (row & 1) + 8 (row >> 1) .. + 7
    const int lane_off = (lane & 15) * BLK_COLS + (row & 1) * 16 + (row >> 1) * 8;
    const int m = m0 + wm * SPLIT;
    auto at = [&](int i, int cb) { return IN_BLOCK ? panel_offset(m, cb) + i * 16 * BLK_COLS : panel_offset(m + i * 16, cb); };
    const long et_off = (long)((n0 >> BLK_SHIFT) + wn * (WTN / 32)) * BLK_ELEMS + lane_off;
    const bf16_t* Et = g.Et + bidx * g.strideEt + (COH ? 0 : et_off);  // (COH: the same in every lane)
    bf16_t* C = g.C + bidx * g.strideC + (long)((n0 >> BLK_SHIFT) + wn * (WTN / 32)) * BLK_ELEMS + lane_off;
    static_assert(PART == EPI_ALL || NEV >= FMU * (FN / 2), "pieces of the a.X term");
    // Where nothing comes between the two parts the pieces are an array of this function's own: in the caller's they cost the 224-row
    // persistent kernel (251 registers like this) four more registers, 12 bytes of scratch a lane and 0.5 to 1 % (median us: 60 of 640 x
    // 2560 159.0 and 157.6 like this, 48 of 896 x 896 77.7 and 76.7).
    bf16x8 own[PART == EPI_ALL ? FMU : 1][FN / 2];
    auto piece = [&](int i, int t) -> bf16x8& {
        if constexpr (PART == EPI_ALL) return own[i][t];
        else return ev[i * (FN / 2) + t];
    };
    if constexpr (PART & EPI_LOADS) {
#pragma unroll
        for (int i = 0; i < FMU; ++i)
#pragma unroll
            for (int t = 0; t < FN / 2; ++t)
                piece(i, t) = load16<COH>(Et, (COH ? et_off : 0) + at(i, g.cbEt) + (long)t * BLK_ELEMS);
    }
    if constexpr (!(PART & EPI_REST)) return;
#pragma unroll
    for (int i = 0; i < FMU; ++i)
#pragma unroll
        for (int t = 0; t < FN / 2; ++t) {
            const f32x4 a = acc[i][2 * t], b = acc[i][2 * t + 1];
            const u32x2v lo = __builtin_amdgcn_permlane16_swap(pack_bf16x2(a[0], a[1]), pack_bf16x2(b[0], b[1]), false, false);
            const u32x2v hi = __builtin_amdgcn_permlane16_swap(pack_bf16x2(a[2], a[3]), pack_bf16x2(b[2], b[3]), false, false);
            const u32x4 tw = {lo[0], hi[0], lo[1], hi[1]};
            const bf16x8 tv = *(const bf16x8*)&tw;
            bf16x8 o;
#pragma unroll
            for (int k = 0; k < 8; ++k) o[k] = f2bf(rbf(g.s0 * bf2f(piece(i, t)[k])) + bf2f(tv[k]));
            *(bf16x8*)(C + at(i, g.cbC) + (long)t * BLK_ELEMS) = o;
        }
}

// Symmetric products without LDS and without a barrier.  A lane holds, of fragment (i, j), rows 4q..4q+3 (q = lane / 16)
// of column lane % 16: 8-byte pieces of rows of the mirror image Ct, which leave exactly as the rows of X' above, with
// fragments i = 2t and 2t+1 paired by v_permlane16_swap_b32 (SYMPOLY adds the b.A term to the paired pieces, read from
// the mirror tile of A in the same pattern).  For the tile itself the finished values return to the fragment layout
// (the swap is its own inverse) and every group of four lanes transposes its 4 x 4 elements in two exchanges:
//   with the lane one away (DPP quad_perm [1,0,3,2]) the 16-bit halves of each register,
//   with the lane two away (quad_perm [2,3,0,1]) one of the two registers,
// after which lane 4a+s of row q holds columns 4a..4a+3 of row 4q+s of the fragment: 8-byte pieces of rows of C, a wave
// store covering 16 rows x 32 bytes.  In a diagonal tile only the 32x32 blocks on or above the diagonal hold computed
// values: they go out as Ct pieces (the lower half and the diagonal blocks) and, strictly above it, as C pieces.
__device__ __forceinline__ void quad_transpose_b16(unsigned& p0, unsigned& p1, unsigned sel, bool upper) {
    const unsigned t0 = (unsigned)__builtin_amdgcn_update_dpp(0, (int)p0, 0xB1, 0xF, 0xF, false);
    const unsigned t1 = (unsigned)__builtin_amdgcn_update_dpp(0, (int)p1, 0xB1, 0xF, 0xF, false);
    p0 = __builtin_amdgcn_perm(t0, p0, sel);
    p1 = __builtin_amdgcn_perm(t1, p1, sel);
    const unsigned send = upper ? p0 : p1;
    const unsigned recv = (unsigned)__builtin_amdgcn_update_dpp(0, (int)send, 0x4E, 0xF, 0xF, false);
    p0 = upper ? recv : p0;
    p1 = upper ? p1 : recv;
}
template <int BM, int BN, int WGM, int WGN, int EPI, unsigned MASK, bool COH, int PART, int NEV>
__device__ __forceinline__ void epilogue_sym_reg(const GemmArgs& g, const TileCoord& tc,
                                                 f32x4 (&acc)[BM / WGM / 16][BN / WGN / 16], bf16x8 (&ev)[NEV]) {
    constexpr int WTM = BM / WGM, WTN = BN / WGN;
    constexpr int FM = WTM / 16, FN = WTN / 16;
    static_assert(FM % 2 == 0 && FN % 2 == 0 && BLK_COLS == 32, "a pair of fragments is one column block");
    static_assert(EPI == EPI_SYRK || EPI == EPI_SYMPOLY || EPI == EPI_MMT, "symmetric products");
    constexpr bool DENSE = EPI == EPI_MMT;
    const bool vec = DENSE && dense_vec(g);
    const int tid = thread_number<COH>(), lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN, row = lane >> 4;
    const int m0 = tc.ti * BM, n0 = tc.tj * BN;
    const bool diag = tc.ti == tc.tj;
    // Ct piece (t, j): row n0 + wn*WTN + 16 j + lane%16, columns m0 + wm*WTM + 32 t + 16 (row & 1) + 8 (row >> 1) .. + 7
    const long ct_off = (long)((m0 >> BLK_SHIFT) + wm * (WTM / 32)) * BLK_ELEMS + (wn * WTN + (lane & 15)) * BLK_COLS +
                        (row & 1) * 16 + (row >> 1) * 8;
    bf16_t* Ct = g.Ct + tc.bidx * g.strideCt + panel_offset(n0, g.cbCt) + ct_off;
    // C piece of fragment (i, j): row m0 + wm*WTM + 16 i + 4 row + lane%4, columns n0 + wn*WTN + 16 j + 4 (lane/4 % 4) .. + 3
    bf16_t* C = g.C + tc.bidx * g.strideC + panel_offset(m0, g.cbC) + (long)((n0 >> BLK_SHIFT) + wn * (WTN / 32)) * BLK_ELEMS +
                (wm * WTM + 4 * row + (lane & 3)) * BLK_COLS + ((lane >> 2) & 3) * 4;
    const unsigned sel = (lane & 1) ? 0x03020706u : 0x05040100u;
    const bool upper = (lane & 2) != 0;
    // SYMPOLY: the b.A pieces of EV_AHEAD rows of pairs are in flight at a time; those of row t + EV_AHEAD are fetched
    // when row t starts (all of them at once do not fit beside the accumulators in the persistent kernel)
    static_assert(NEV >= (EPI == EPI_SYMPOLY ? FM / 2 * FN : 1), "pieces of the b.A term");
    const bf16_t* Et = g.Et + tc.bidx * g.strideEt + panel_offset(n0, g.cbEt) + (COH ? 0 : ct_off);  // (COH: the same in every lane)
    constexpr int EV_AHEAD = PART == EPI_REST ? FM / 2 : 2 < FM / 2 ? 2 : FM / 2;  // measured: 3 no faster, 4 spills an accumulator fragment
    auto load_ev = [&](int t) {
#pragma unroll
        for (int j = 0; j < FN; ++j) ev[t * FN + j] = load16<COH>(Et, (COH ? ct_off : 0) + j * 16 * BLK_COLS + (long)t * BLK_ELEMS);
    };
    if constexpr (EPI == EPI_SYMPOLY && (PART & EPI_LOADS)) {
#pragma unroll
        for (int t = 0; t < (PART == EPI_LOADS ? FM / 2 : EV_AHEAD); ++t) load_ev(t);
    }
    if constexpr (!(PART & EPI_REST)) return;
    auto rounded = [&](float v) {
        v = rbf(v);
        if (EPI == EPI_SYMPOLY) v = g.s1 * v;
        return v;
    };
#pragma unroll
    for (int t = 0; t < FM / 2; ++t) {
        if constexpr (EPI == EPI_SYMPOLY) {
            if (t + EV_AHEAD < FM / 2) load_ev(t + EV_AHEAD);
        }
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            // MASK: the fragments that this copy of a diagonal tile's loop has not computed (pp_skip_mask), known when
            // the caller has one copy of the epilogue per mask; the test on the block indices covers the other callers
            if ((MASK >> (2 * t * FN + j)) & 1) continue;
            const int mblk = wm * (WTM / 32) + t, nblk = wn * (WTN / 32) + (j >> 1);
            if (diag && mblk > nblk) continue;  // not computed: the mirror image of a block another wave holds
            const f32x4 a = acc[2 * t][j], b = acc[2 * t + 1][j];
            unsigned a01 = pack_bf16x2(rounded(a[0]), rounded(a[1])), a23 = pack_bf16x2(rounded(a[2]), rounded(a[3]));
            unsigned b01 = pack_bf16x2(rounded(b[0]), rounded(b[1])), b23 = pack_bf16x2(rounded(b[2]), rounded(b[3]));
            u32x2v lo = __builtin_amdgcn_permlane16_swap(a01, b01, false, false);
            u32x2v hi = __builtin_amdgcn_permlane16_swap(a23, b23, false, false);
            if constexpr (EPI == EPI_SYMPOLY) {
                const u32x4 tw = {lo[0], hi[0], lo[1], hi[1]};
                const bf16x8 tv = *(const bf16x8*)&tw;
                bf16x8 o;
#pragma unroll
                for (int k = 0; k < 8; ++k) o[k] = f2bf(rbf(g.s0 * bf2f(ev[t * FN + j][k])) + bf2f(tv[k]));
                *(bf16x8*)(Ct + j * 16 * BLK_COLS + (long)t * BLK_ELEMS) = o;
                if (diag && mblk == nblk) continue;
                const u32x4 ow = *(const u32x4*)&o;
                lo = __builtin_amdgcn_permlane16_swap(ow[0], ow[2], false, false);
                hi = __builtin_amdgcn_permlane16_swap(ow[1], ow[3], false, false);
                a01 = lo[0], b01 = lo[1], a23 = hi[0], b23 = hi[1];
            } else {
                const u32x4 tw = {lo[0], hi[0], lo[1], hi[1]};
                if constexpr (DENSE)
                    dense_store(g, vec, n0 + wn * WTN + 16 * j + (lane & 15), m0 + wm * WTM + 32 * t + 16 * (row & 1) + 8 * (row >> 1), tw);
                else *(u32x4*)(Ct + j * 16 * BLK_COLS + (long)t * BLK_ELEMS) = tw;
                if (diag && mblk == nblk) continue;
            }
            quad_transpose_b16(a01, a23, sel, upper);
            quad_transpose_b16(b01, b23, sel, upper);
            if constexpr (DENSE) {
                const int r = m0 + wm * WTM + 32 * t + 4 * row + (lane & 3), c = n0 + wn * WTN + 16 * j + ((lane >> 2) & 3) * 4;
                dense_store(g, vec, r, c, u32x2v{a01, a23});
                dense_store(g, vec, r + 16, c, u32x2v{b01, b23});
                continue;
            }
            bf16_t* cp = C + (2 * t) * 16 * BLK_COLS + (long)(j >> 1) * BLK_ELEMS + (j & 1) * 16;
            *(u32x2v*)cp = u32x2v{a01, a23};
            *(u32x2v*)(cp + 16 * BLK_COLS) = u32x2v{b01, b23};
        }
    }
}

// Transposing LDS read of a Q fragment of BX: the stage holds the k-tile of X as pieces of 32 columns,
// [piece][k][32 columns] with 64-byte rows, and a fragment is 16 columns x 32 k.  ds_read_b64_tr_b16 works in
// groups of 16 lanes: lane j = 4r+s addresses row k+r, columns 4s..4s+3 of the group's 16 columns, and lane
// i = 4s+e receives rows k..k+3 of column 4s+e; a second read takes rows k+4..k+7.  Group g = lane/16 starts at
// k = 8g, which gives the MFMA operand layout (lane l: column l%16, eight consecutive k from 8*(l/16)).
// Two groups that are served together (g and g^1) would read the same 32-byte window of rows 64*8 bytes = two
// bank rounds apart, so the two 32-byte halves of a row are stored swapped in rows whose k has bit 3 set (the
// global side of the load applies the swap): fragment half h of group g sits at byte (h ^ (g & 1)) * 32.
// qt_lane_offset(lane, h): byte offset of this lane's first read inside the piece, k-step 0.
__device__ __forceinline__ int qt_lane_offset(int lane, int h) {
    const int grp = lane >> 4, i16 = lane & 15;
    return (grp * 8 + (i16 >> 2)) * 64 + ((h ^ (grp & 1)) * 32) + (i16 & 3) * 8;
}
__device__ __forceinline__ bf16x8 lds_read_qt(const unsigned char* q) {
    const s16x4 lo = lds_read_tr16(q), hi4 = lds_read_tr16(q + 4 * 64);
    const s16x8 t = {lo[0], lo[1], lo[2], lo[3], hi4[0], hi4[1], hi4[2], hi4[3]};
    return *(const bf16x8*)&t;
}

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// ---- kernel 1: 64-column k-tiles in two LDS stages, one barrier per k-tile -------------------
// Operand panels go from global memory straight into LDS (global_load_lds_dwordx4): one wave
// instruction fills 1 KB of LDS in lane order, i.e. 8 rows of 128 bytes, so the XOR swizzle
// that keeps the fragment reads conflict free (16-byte chunk c of row r sits at c ^ ((r>>1)&7))
// is applied on the global side: lane L fetches the chunk whose swizzled position is L&7.
// Per k-tile (two 32-column MFMA steps) a wave issues FM*FN*2 MFMAs, (FM+FN)*2 LDS fragment reads and
// LA+LB loads.  Every non-MFMA instruction is placed between two MFMAs so that it issues in their shadow:
//   k-step 0 : MFMAs of step 0 interleaved with the fragment reads of step 1;
//   k-step 1 : the wave has now read everything it needs from this stage, so it waits
//              for its own loads of the next k-tile, crosses the one barrier, and then
//              interleaves the last MFMAs with the loads of k-tile t+2 (into the stage just
//              released) and with the fragment reads of step 0 of k-tile t+1.
// The fences (sched_barrier) pin that order; without them the scheduler sinks every LDS read
// next to its first use and the MFMA pipe idles for an LDS round trip per k-step.  Barriers are
// raw s_barrier with explicit s_waitcnt: __syncthreads() would wait for the loads in flight.
constexpr int ROW_BYTES = 128;

template <int BM, int BN, int WGM, int WGN, int EPI>
__global__ void __launch_bounds__(WGM* WGN * 64) gemm_nt_pipe_kernel(const GemmList l) {
    constexpr int NW = WGM * WGN;
    constexpr int WTM = BM / WGM, WTN = BN / WGN;
    constexpr int FM = WTM / 16, FN = WTN / 16;
    constexpr int A_BYTES = BM * ROW_BYTES, B_BYTES = BN * ROW_BYTES, STAGE = A_BYTES + B_BYTES;
    constexpr int LA = BM / 8 / NW, LB = BN / 8 / NW;
    constexpr int KS = 2;  // 32-column MFMA steps per k-tile
    constexpr int NMF = FM * FN, NRD = FM + FN, NLD = LA + LB;
    static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "dma split");
    static_assert(epi_is_bx(EPI) || BM == BN, "triangular tiles are square");

    extern __shared__ __align__(16) unsigned char smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int logical = xcd_remap(blockIdx.x, gridDim.x, l.xcd_shift), entry = list_entry(l, logical);
    const GemmArgs& g = l.g[entry];
    const TileCoord tc = tile_of<EPI>(g, logical - l.start[entry]);
    constexpr bool QT = epi_is_bx(EPI);  // Q is X itself, rows = reduction index
    const int kb = g.cbP;
    const bf16_t* Pb = g.P + tc.bidx * g.strideP + panel_offset(tc.ti * BM, kb);
    const bf16_t* Qb = g.Q + tc.bidx * g.strideQ +
                       (QT ? (long)(tc.tj * BN >> BLK_SHIFT) * BLK_ELEMS : panel_offset(tc.tj * BN, kb));

    const int drow = lane >> 3;
    const bf16_t* pa = Pb + (wave * 8 * LA + drow) * BLK_COLS;
    // BX: a k-tile of Q is BN/32 pieces of 64 rows x 32 columns, each a contiguous 4 KB run of one block;
    // load instruction t of the tile (1 KB) is the quarter t%4 of piece t/4, in lane order, with the two halves
    // of a row swapped in rows whose k has bit 3 set (see qt_lane_offset)
    const bf16_t* pb = QT ? Qb + (lane >> 2) * BLK_COLS + ((lane & 3) ^ (((lane >> 5) & 1) << 1)) * 8
                          : Qb + (wave * 8 * LB + drow) * BLK_COLS;
    const int lds_a = wave * 8 * LA * ROW_BYTES;
    const int lds_b = A_BYTES + wave * 8 * LB * ROW_BYTES;
    // element offset of the 16-byte chunk this lane fetches inside a row of the 64-column k-tile, as an offset
    // in the blocked layout (a k-tile is 64 / BLK_COLS column blocks)
    auto chunk_off = [](int e) { return (long)(e >> BLK_SHIFT) * BLK_ELEMS + (e & (BLK_COLS - 1)); };
    const long ch_even = chunk_off(((lane & 7) ^ (drow >> 1)) * 8), ch_odd = chunk_off(((lane & 7) ^ (4 | (drow >> 1))) * 8);
    constexpr int KT_BLOCKS = 64 / BLK_COLS;

    // load instruction n (0..NLD-1) of k-tile kt: A rows first, then B rows
    auto issue_one = [&](int n, int stage, int kt) {
        unsigned char* s = smem + stage * STAGE;
        if (n < LA) {
            const long ch = ((wave * LA + n) & 1) ? ch_odd : ch_even;
            __builtin_amdgcn_global_load_lds((glb_void_ptr)(pa + (long)kt * KT_BLOCKS * BLK_ELEMS + n * 8 * BLK_COLS + ch),
                                             (lds_void_ptr)(s + lds_a + n * 8 * ROW_BYTES), 16, 0, 0);
        } else if (QT) {
            const int i = n - LA, t = wave * LB + i, k0 = kt * 64;
            const long off = ((long)(k0 >> 8) * g.cbQ + (t >> 2)) * BLK_ELEMS + ((k0 & 255) + (t & 3) * 16) * BLK_COLS;
            __builtin_amdgcn_global_load_lds((glb_void_ptr)(pb + off), (lds_void_ptr)(s + lds_b + i * 8 * ROW_BYTES), 16, 0, 0);
        } else {
            const int i = n - LA;
            const long ch = ((wave * LB + i) & 1) ? ch_odd : ch_even;
            __builtin_amdgcn_global_load_lds((glb_void_ptr)(pb + (long)kt * KT_BLOCKS * BLK_ELEMS + i * 8 * BLK_COLS + ch),
                                             (lds_void_ptr)(s + lds_b + i * 8 * ROW_BYTES), 16, 0, 0);
        }
    };

    f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

    // fragment reads: lane l takes row l%16 of the fragment, 16-byte chunk 4*ks + l/16 of the 128-byte row
    const int sw = (lane >> 1) & 7, kq = lane >> 4;
    const int a_off = (wm * WTM + (lane & 15)) * ROW_BYTES;
    const int b_off = A_BYTES + (wn * WTN + (lane & 15)) * ROW_BYTES;
    const int q_off[2] = {A_BYTES + (wn * WTN / 32) * 4096 + qt_lane_offset(lane, 0),
                          A_BYTES + (wn * WTN / 32) * 4096 + qt_lane_offset(lane, 1)};

    bf16x8 fr[2][NRD];  // fragment double buffer: [0..FM) rows of P, [FM..NRD) rows (BX: columns) of Q
    auto read_one = [&](int buf, int n, const unsigned char* st, int ks) {
        const int co = (((ks << 2) | kq) ^ sw) << 4;
        if (n < FM) fr[buf][n] = *(const bf16x8*)(st + a_off + n * 16 * ROW_BYTES + co);
        else if (QT) fr[buf][n] = lds_read_qt(st + q_off[(n - FM) & 1] + ((n - FM) >> 1) * 4096 + ks * 32 * 64);
        else fr[buf][n] = *(const bf16x8*)(st + b_off + (n - FM) * 16 * ROW_BYTES + co);
    };
    auto mfma_one = [&](int buf, int idx) {
        const int i = idx / FN, j = idx % FN;
        if (QT)  // operands swapped: a lane then holds 4 consecutive columns of one row of the tile
            acc[i][j] = mfma16(fr[buf][FM + j], fr[buf][i], acc[i][j]);
        else
            acc[i][j] = mfma16(fr[buf][i], fr[buf][FM + j], acc[i][j]);
    };

    const int nk = g.kdim / 64;
#pragma unroll
    for (int n = 0; n < NLD; ++n) issue_one(n, 0, 0);
#pragma unroll
    for (int n = 0; n < NLD; ++n) issue_one(n, 1, 1);  // kdim >= 128: there are at least two k-tiles
    WAIT_VM(NLD);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int n = 0; n < NRD; ++n) read_one(0, n, smem, 0);

    for (int kt = 0; kt < nk; ++kt) {
        const unsigned char* st = smem + (kt & 1) * STAGE;
        const unsigned char* stn = smem + ((kt + 1) & 1) * STAGE;
#pragma unroll
        for (int ks = 0; ks < KS - 1; ++ks) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int idx = 0; idx < NMF; ++idx) {
                mfma_one(ks & 1, idx);
                if (idx < NRD) {
                    __builtin_amdgcn_sched_barrier(0);
                    read_one((ks + 1) & 1, idx, st, ks + 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // Fragments of the last k-step are in: this wave is done with stage kt&1.  The tail is
        // branch free: past the end it re-loads the last k-tile into a stage nobody reads and
        // pre-reads fragments nobody uses, which costs 2 of nk loads and keeps the MFMAs in
        // one basic block (a branch here makes the register allocator spill the accumulators).
        WAIT_LGKM0();
        WAIT_VM(0);  // its loads of k-tile kt+1 (the only ones in flight) have landed
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int k2 = kt + 2 < nk ? kt + 2 : nk - 1;
        constexpr int PER = (NLD + NRD + NMF - 1) / NMF;  // loads and reads per MFMA slot
#pragma unroll
        for (int idx = 0; idx < NMF; ++idx) {
            mfma_one((KS - 1) & 1, idx);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < PER; ++u) {
                const int o = idx * PER + u;
                if (o < NRD) read_one(KS & 1, o, stn, 0);
                else if (o < NRD + NLD) issue_one(o - NRD, kt & 1, k2);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    WAIT_VM(0);  // the dummy loads of the last two tails must not land in the epilogue's tile
    bf16x8 ev[tile_pieces<BM, BN, WGM, WGN>()];
    FoldPiece<false> pv[tile_pieces<BM, BN, WGM, WGN>()];
    if constexpr (QT) epilogue_nn<BM, BN, WGM, WGN, epi_fold_mode(EPI), false, EPI_ALL>(g, tc, acc, smem, ev, pv);
    else epilogue<BM, BN, WGM, WGN, EPI, false, false, EPI_ALL>(g, tc, acc, smem, ev);
}

// 16x16 fragments (i, j) of wave `wave` of a WGM x WGN wave grid whose enclosing 32x32 block lies entirely below
// the diagonal of a diagonal tile (the epilogue masks at that granularity).
template <int WTM, int WTN, int FM, int FN, int WGN>
constexpr unsigned pp_skip_mask(int wave) {
    const int wm = wave / WGN, wn = wave % WGN;
    unsigned m = 0;
    for (int i = 0; i < FM; ++i)
        for (int j = 0; j < FN; ++j)
            if ((wm * WTM + i * 16) / 32 > (wn * WTN + j * 16) / 32) m |= 1u << (i * FN + j);
    return m;
}
template <int WTM, int WTN, int FM, int FN, int WGN>
constexpr bool pp_first_with_mask(int wave) {
    for (int w = 0; w < wave; ++w)
        if (pp_skip_mask<WTM, WTN, FM, FN, WGN>(w) == pp_skip_mask<WTM, WTN, FM, FN, WGN>(wave)) return false;
    return true;
}

// Where the 16-byte chunks of a 64-byte LDS row go: chunk c of a row in row group rg = (row / 4) % 4 sits at
// c ^ pp_swizzle(rg) = c ^ [0, 2, 3, 1][rg].  ds_read_b128 serves a wave in four passes of 16 lanes, and the
// passes are not lanes 0-15, 16-31, ...: the first takes lanes 0-3, 12-15, 20-23, 24-27, the second 4-7, 8-11,
// 16-19, 28-31, the other two the same plus 32.  With fragment lane l on row l%16, chunk l/16, this table is the
// one that gives every pass sixteen different 16-byte bank groups: 256 bytes per clock measured, against 144
// with the plain c ^ rg, which collides two ways in every pass.
__device__ __forceinline__ int pp_swizzle(int rg) { return (0x78 >> (2 * rg)) & 3; }

// ---- kernel 2: eight waves in two groups that alternate between memory and MFMA phases --------
// Every wave runs the same loop  { M(t): read its fragments of k-tile t from LDS, issue its
// share of the loads of k-tile t+3, wait;  barrier;  C(t): FM*FN*2 MFMAs;  barrier }  over
// 32-column k-tiles in four LDS stages, but waves 4..7 enter it one barrier later than waves
// 0..3.  Wave w and wave w+4 share a SIMD, so at any time one of them is issuing nothing but
// MFMAs from registers while the other does all the LDS and address-path work and absorbs the
// waits; the barrier is crossed when the MFMA wave has issued its last MFMA.
// Timeline (phase p between two barriers): group 0 runs M(t) in p=2t and C(t) in p=2t+1,
// group 1 runs M(t) in p=2t+1 and C(t) in p=2t+2.  Stage t&3 is last read in p=2t+1, the
// loads of k-tile t+4 into it are issued in p=2t+2 / 2t+3, each wave waits for its own at the
// end of its M phase two k-tiles later (p=2t+6 / 2t+7), and k-tile t+4 is first read in p=2t+8.
//
// COH: operands and elementwise terms are read at device scope (load16).  before_loads() runs in front of the first load, after_loop()
// between the k loop and the epilogue.  Where wanted(), asked with the first loads on their way, says no in every wave, the tile ends there:
// nothing is stored, and the loads are still in flight.
struct Nothing {
    __device__ void operator()() const {}
};
struct Always {
    __device__ bool operator()() const { return true; }
};
template <int BM, int BN, int WGM, int WGN, int EPI, bool COH = false, typename F0 = Nothing, typename F1 = Nothing, typename F2 = Always>
__device__ __forceinline__ void pp_tile(const GemmArgs& g, const TileCoord& tc, unsigned char* smem, F0 before_loads = F0(), F1 after_loop = F1(),
                                        F2 wanted = F2()) {
    constexpr int NW = WGM * WGN;
    constexpr int BK4 = 32, ROWB = 64;
    constexpr int WTM = BM / WGM, WTN = BN / WGN;
    constexpr int FM = WTM / 16, FN = WTN / 16;
    constexpr int A_BYTES = BM * ROWB, B_BYTES = BN * ROWB, STAGE = A_BYTES + B_BYTES;
    constexpr int LA = BM / 16 / NW, LB = BN / 16 / NW;
    constexpr int NLD = LA + LB;
    static_assert(FM * FN <= 32, "one mask bit per fragment");
    static_assert(NW == 8, "two groups of four waves, one of each per SIMD");
    static_assert(BM % (16 * NW) == 0 && BN % (16 * NW) == 0, "dma split");
    static_assert(epi_is_bx(EPI) || BM == BN, "triangular tiles are square");

    const int tid = thread_number<COH>(), lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 2;
    const int wm = wave / WGN, wn = wave % WGN;
    constexpr bool QT = epi_is_bx(EPI);  // Q is X itself, rows = reduction index
    const int kb = g.cbP;
    const bool dense = EPI == EPI_MMT && g.dense_pitch != 0;
    auto panel = [&](int row0) { return dense ? dense_panel(g, row0) : panel_offset(row0, kb); };
    auto in_panel = [&](int row0, int r, int ch) {  // element offset of row r, column ch of a k-tile from the panel's start
        return dense ? dense_row(g, row0, r) + ch : r * BLK_COLS + ch;
    };
    const bf16_t* Pb = uniform_ptr(g.P + tc.bidx * g.strideP + panel(tc.ti * BM));
    const bf16_t* Qb = uniform_ptr(g.Q + tc.bidx * g.strideQ +
                                   (QT ? (long)(tc.tj * BN >> BLK_SHIFT) * BLK_ELEMS : panel(tc.tj * BN)));

    // Loads: a wave-uniform base pointer (advanced along k with scalar adds) plus a 32-bit byte
    // offset per lane, so that no vector ALU instruction is needed per load: in the memory phase
    // every VALU instruction would queue behind the sibling wave's MFMAs.
    const int drow = lane >> 2;
    const int dch = ((lane & 3) ^ pp_swizzle((lane >> 4) & 3)) * 8;
    unsigned offa[LA], offb[LB];
#pragma unroll
    for (int n = 0; n < LA; ++n) offa[n] = (unsigned)in_panel(tc.ti * BM, wave * 16 * LA + n * 16 + drow, dch) * 2;
    // BX: a k-tile of Q is BN/32 pieces of 32 rows x 32 columns, each a contiguous 2 KB run of one block; load
    // instruction t of the tile (1 KB) is the half t%2 of piece t/2, in lane order, with the two 32-byte halves
    // of a row swapped in rows whose k has bit 3 set (see qt_lane_offset)
    const int qch = ((lane & 3) ^ (((drow >> 3) & 1) << 1)) * 8;
#pragma unroll
    for (int n = 0; n < LB; ++n) {
        const int t = wave * LB + n;
        offb[n] = QT ? (unsigned)(((t >> 1) * BLK_ELEMS + ((t & 1) * 16 + drow) * BLK_COLS + qch) * 2)
                     : (unsigned)in_panel(tc.tj * BN, wave * 16 * LB + n * 16 + drow, dch) * 2;
    }
    const int lds_a = wave * 16 * LA * ROWB;
    const int lds_b = A_BYTES + wave * 16 * LB * ROWB;
    const int nk = g.kdim / BK4;
    const int kstep = dense ? BK4 : BLK_ELEMS;  // elements from k-tile to k-tile

    // global_load_lds_dwordx4 with a scalar base and a 32-bit vector offset; the LDS destination
    // of lane 0 goes through M0 (the wave's 64 lanes fill 1 KB from there in lane order).
    auto dma = [&](const char* base, unsigned voff, unsigned lds_byte) {
        if constexpr (COH)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 sc1"
                         :
                         : "s"(lds_byte), "v"(voff), "s"(base)
                         : "memory");
        else
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                         :
                         : "s"(lds_byte), "v"(voff), "s"(base)
                         : "memory");
    };
    const unsigned lds_base = (unsigned)(uintptr_t)(lds_void_ptr)smem;
    auto issue_tile = [&](int kt) {  // kt may run past the end: re-load the last k-tile
        const int k0 = (kt < nk ? kt : nk - 1) * BK4;
        static_assert(BLK_COLS == BK4, "a k-tile is one block of columns");
        const long koff = (long)(k0 >> BLK_SHIFT) * kstep;
        const char* ba = (const char*)(Pb + koff);
        const char* bb = (const char*)(Qb + (QT ? (long)(k0 >> 8) * g.cbQ * BLK_ELEMS + (k0 & 255) * BLK_COLS : koff));
        const unsigned st = lds_base + (kt & 3) * STAGE;
#pragma unroll
        for (int n = 0; n < LA; ++n) dma(ba, offa[n], st + lds_a + n * 16 * ROWB);
#pragma unroll
        for (int n = 0; n < LB; ++n) dma(bb, offb[n], st + lds_b + n * 16 * ROWB);
    };

    f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

    // Diagonal tile of a symmetric product: a fragment of a wave that lies entirely below the diagonal is the
    // mirror image of one another wave computes, and the epilogue does not read it.  Bit i*FN+j of a wave's mask:
    // skip that fragment's MFMAs (and the fragment reads nobody needs).
    const bool diag = !epi_is_bx(EPI) && tc.ti == tc.tj;
    // fragment reads: lane l takes row l%16 of the fragment and the 16-byte chunk l/16 of its 64-byte row
    // (chunk c of row r sits at c ^ pp_swizzle((r>>2)&3))
    const int sw = pp_swizzle((lane >> 2) & 3), kq = lane >> 4;
    const int co = (kq ^ sw) << 4;
    const int a_off = (wm * WTM + (lane & 15)) * ROWB + co;
    const int b_off = A_BYTES + (wn * WTN + (lane & 15)) * ROWB + co;

    // The elementwise term and the parameter's pieces first, where they fit (128-tiles).  They lie before the k-tiles in the queue,
    // which returns in order, so the counts below stay what they are.
    constexpr bool PRE = BM == 128;
    // The epilogues that need no LDS.  Measured: on whole 256-tiles b.A + c.A.A is 0.5 % faster without it, X.Xt 0.6 % slower; on
    // 128-tiles a launch of either is 1 % slower, but in the kernel with COH, where every tile is waited for, two barriers fewer are
    // worth 2 % of the chain's launch in the mean and up to 8 % (56 drawn sets, profiles/flow_chain_or_launches.txt).
    constexpr bool REG = EPI == EPI_BX;
    constexpr bool SREG = (EPI == EPI_SYMPOLY && BM == 256) || (!QT && COH);
    constexpr int NEV = tile_pieces<BM, BN, WGM, WGN>(), LATE = PRE ? EPI_REST : EPI_ALL;
    bf16x8 ev[NEV];
    FoldPiece<PRE> pv[NEV];
    before_loads();
    if constexpr (PRE) {
        if constexpr (REG) epilogue_nn_reg<BN, WGN, WTM, FM, true, COH, EPI_LOADS>(g, tc.bidx, tc.ti * BM, tc.tj * BN, acc, ev);
        else if constexpr (QT) epilogue_nn<BM, BN, WGM, WGN, epi_fold_mode(EPI), COH, EPI_LOADS>(g, tc, acc, smem, ev, pv);
        else if constexpr (SREG) epilogue_sym_reg<BM, BN, WGM, WGN, EPI, 0, COH, EPI_LOADS>(g, tc, acc, ev);
        else epilogue<BM, BN, WGM, WGN, EPI, true, COH, EPI_LOADS>(g, tc, acc, smem, ev);
    }

    issue_tile(0);
    issue_tile(1);
    issue_tile(2);
    if (!wanted()) return;
    WAIT_VM(2 * NLD);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (grp) __builtin_amdgcn_s_barrier();

    // LDS read addresses: one register per operand (BX: per half of a piece) and pair of stages; the stage
    // inside the pair and the fragment index are instruction offsets (below 64 KB) once the k loop is unrolled
    // by the four stages.
    const unsigned char* ra[2];
    const unsigned char* rb[2][2];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        ra[half] = smem + half * 2 * STAGE + a_off;
#pragma unroll
        for (int h = 0; h < 2; ++h)
            rb[half][h] = QT ? smem + half * 2 * STAGE + A_BYTES + (wn * WTN / 32) * 2048 + qt_lane_offset(lane, h)
                             : smem + half * 2 * STAGE + b_off;
    }
    // LATER: k-tiles behind kt that are still to come, as far as it matters: 3 where kt + 3 is (or, on 256-tiles, the last k-tile
    // is loaded once more in its place, into a stage that nobody reads: a straight loop), fewer in the last three of a 128-tile,
    // where a short loop would wait for such loads in front of its epilogue.
    auto body = [&](int kt, auto stage_c, auto mask_c, auto later_c) {
        constexpr int SIDX = decltype(stage_c)::value, LATER = decltype(later_c)::value;
        constexpr unsigned MASK = decltype(mask_c)::value;
        auto kept = [](int i, int j) { return !((MASK >> (i * FN + j)) & 1); };
        // ---- M(kt)
        bf16x8 fa[FM], fb[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            bool used = false;
#pragma unroll
            for (int j = 0; j < FN; ++j) used |= kept(i, j);
            if (used) fa[i] = *(const bf16x8*)(ra[SIDX >> 1] + (SIDX & 1) * STAGE + i * 16 * ROWB);
        }
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            bool used = false;
#pragma unroll
            for (int i = 0; i < FM; ++i) used |= kept(i, j);
            if (!used) continue;
            if (QT) fb[j] = lds_read_qt(rb[SIDX >> 1][j & 1] + (SIDX & 1) * STAGE + (j >> 1) * 2048);
            else fb[j] = *(const bf16x8*)(rb[SIDX >> 1][0] + (SIDX & 1) * STAGE + j * 16 * ROWB);
        }
        if constexpr (LATER == 3) issue_tile(kt + 3);
        WAIT_LGKM0();
        if constexpr (LATER > 0) WAIT_VM((LATER - 1) * NLD);  // own loads of k-tile kt+1 have landed
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        // ---- C(kt): column fragment outermost, so that consecutive MFMAs share the Q fragment (measured +1 to 2 %
        // for B.X against rows outermost)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int ii = 0; ii < FM; ++ii) {
                const int i = (j & 1) ? FM - 1 - ii : ii;
                if (QT)  // operands swapped: a lane then holds 4 consecutive columns of one row of the tile
                    acc[i][j] = mfma16(fb[j], fa[i], acc[i][j]);
                else if (kept(i, j))
                    acc[i][j] = mfma16(fa[i], fb[j], acc[i][j]);
            }
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // nk is a multiple of 4 (k extents are multiples of 128)
    auto k_loop = [&](auto mask_c) {
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        using I2 = std::integral_constant<int, 2>;
        using I3 = std::integral_constant<int, 3>;
        constexpr bool PEEL = BM == 128 && !epi_fold_mode(EPI);  // (with the parameter's pieces held as well a second copy spills)
        const int whole = PEEL ? nk - 4 : nk;
        for (int kt = 0; kt < whole; kt += 4) {
            body(kt, I0{}, mask_c, I3{});
            body(kt + 1, I1{}, mask_c, I3{});
            body(kt + 2, I2{}, mask_c, I3{});
            body(kt + 3, I3{}, mask_c, I3{});
        }
        if constexpr (PEEL) {
            body(nk - 4, I0{}, mask_c, I3{});
            body(nk - 3, I1{}, mask_c, I2{});
            body(nk - 2, I2{}, mask_c, I1{});
            body(nk - 1, I3{}, mask_c, I0{});
        }
    };
    // One copy of the loop per distinct mask (the masks are compile-time facts of the wave grid), chosen once per
    // tile: no test inside the loop.  Tiles off the diagonal, nearly all, take the first.
    if (!diag) {
        k_loop(std::integral_constant<unsigned, 0>{});
    } else {
        auto run_if_mine = [&](auto wave_c) {
            constexpr int W = decltype(wave_c)::value;
            constexpr unsigned M = pp_skip_mask<WTM, WTN, FM, FN, WGN>(W);
            if constexpr (pp_first_with_mask<WTM, WTN, FM, FN, WGN>(W)) {
                if (pp_skip_mask<WTM, WTN, FM, FN, WGN>(wave) == M) k_loop(std::integral_constant<unsigned, M>{});
            }
        };
        run_if_mine(std::integral_constant<int, 0>{});
        run_if_mine(std::integral_constant<int, 1>{});
        run_if_mine(std::integral_constant<int, 2>{});
        run_if_mine(std::integral_constant<int, 3>{});
        run_if_mine(std::integral_constant<int, 4>{});
        run_if_mine(std::integral_constant<int, 5>{});
        run_if_mine(std::integral_constant<int, 6>{});
        run_if_mine(std::integral_constant<int, 7>{});
    }
    if (!grp) __builtin_amdgcn_s_barrier();
    after_loop();
    if constexpr (REG) {
        // no LDS in this epilogue: the loads issued past the end may land while it runs (its own loads are behind
        // them in the queue, so they have landed before the wave ends)
        epilogue_nn_reg<BN, WGN, WTM, FM, true, COH, LATE>(g, tc.bidx, tc.ti * BM, tc.tj * BN, acc, ev);
        return;
    }
    if constexpr (SREG) {
        epilogue_sym_reg<BM, BN, WGM, WGN, EPI, 0, COH, LATE>(g, tc, acc, ev);
        return;
    }
    WAIT_VM(0);  // the loads issued past the end must not land in the epilogue's tile
    if constexpr (QT) epilogue_nn<BM, BN, WGM, WGN, epi_fold_mode(EPI), COH, LATE>(g, tc, acc, smem, ev, pv);
    else epilogue<BM, BN, WGM, WGN, EPI, true, COH, LATE>(g, tc, acc, smem, ev);
}

template <int BM, int BN, int WGM, int WGN, int EPI>
__global__ void __launch_bounds__(WGM* WGN * 64, BM == 128 ? 4 : 2) gemm_nt_pp_kernel(const GemmList l) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int logical = xcd_remap(blockIdx.x, gridDim.x, l.xcd_shift), entry = list_entry(l, logical);
    pp_tile<BM, BN, WGM, WGN, EPI>(l.g[entry], tile_of<EPI>(l.g[entry], logical - l.start[entry]), smem);
}

// ---- kernel 2b: a deep pipeline on 64x64 tiles, for launches that leave compute units idle --------
// One matrix makes few tiles: 896 x 4864 has 28 triangular 128-tiles for 256 compute units, and a lone workgroup is paced by
// the latency of its three k-tiles in flight (157 ns per 32 columns).  64-tiles are four times the workgroups at half the
// bytes each, and with at most one workgroup per compute unit all of its LDS can hold stages: eight of 64 columns, 112 KB in
// flight.  Four waves of 2x2 fragments, one barrier per k-tile; the fragment reads of k-tile t+1 and the loads of k-tile t+7
// issue between the MFMAs of k-tile t.  What bounds it then is the L2 (136 workgroups pull 12 TB/s).  Nothing is loaded past
// the end (short reductions are the common case): the last eight k-tiles are a straight line of their own with the counts of
// what is still in flight.  Measured against 128-tiles: X.Xt of 896 x 4864 30 -> 17.7 us, of 1024 x 1024 9.8 -> 6.5,
// b.A + c.A.A of 896 rows 9.9 -> 6.4; the same structure on 128-tiles was no faster than the ping-pong kernel (34 against
// 25 us for 1024 x 4096).  Stage layout, swizzle and transposing reads are those of kernel 1, the register epilogues those of
// the persistent kernel, and every element sums its products in the same order: the results are the other kernels' bit for bit.
template <int EPI>
__global__ void __launch_bounds__(256) gemm_nt_deep_kernel(const GemmList l) {
    static_assert(EPI == EPI_BX || EPI == EPI_SYRK || EPI == EPI_SYMPOLY || EPI == EPI_MMT, "the epilogues that need no LDS");
    constexpr int BM = 64, BN = 64, WGM = 2, WGN = 2, NW = 4;
    constexpr int WTM = BM / WGM, WTN = BN / WGN, FM = WTM / 16, FN = WTN / 16;
    constexpr int A_BYTES = BM * ROW_BYTES, STAGE = A_BYTES + BN * ROW_BYTES, NST = 8;
    constexpr int LA = BM / 8 / NW, LB = BN / 8 / NW, NLD = LA + LB;  // 1 KB load instructions per wave and k-tile
    constexpr int KS = 2, NRD = FM + FN;
    constexpr bool QT = EPI == EPI_BX;
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int logical = xcd_remap(blockIdx.x, gridDim.x, l.xcd_shift), entry = list_entry(l, logical);
    const GemmArgs& g = l.g[entry];
    const TileCoord tc = tile_of<EPI>(g, logical - l.start[entry]);
    const int kb = g.cbP;
    // a row-major X of EPI_MMT: as in pp_tile
    const bool dense = EPI == EPI_MMT && g.dense_pitch != 0;
    auto panel = [&](int row0) { return dense ? dense_panel(g, row0) : panel_offset(row0, kb); };
    auto in_panel = [&](int row0, int r) { return dense ? dense_row(g, row0, r) : r * BLK_COLS; };
    const bf16_t* Pb = uniform_ptr(g.P + tc.bidx * g.strideP + panel(tc.ti * BM));
    const bf16_t* Qb = uniform_ptr(g.Q + tc.bidx * g.strideQ +
                                   (QT ? (long)(tc.tj * BN >> BLK_SHIFT) * BLK_ELEMS : panel(tc.tj * BN)));
    const int drow = lane >> 3;
    // byte offsets of this lane's 16 bytes of each load instruction, from the scalar base of the k-tile (ping-pong kernel: no
    // vector ALU work per load)
    const int kstep = dense ? BLK_COLS : BLK_ELEMS;  // elements from 32 columns to the next 32
    auto chunk_off = [&](int e) { return (e >> BLK_SHIFT) * kstep + (e & (BLK_COLS - 1)); };
    unsigned offa[LA], offb[LB];
#pragma unroll
    for (int n = 0; n < LA; ++n)  // LA is even: instruction n of a wave covers an even or an odd group of eight rows
        offa[n] = (unsigned)(in_panel(tc.ti * BM, (wave * LA + n) * 8 + drow) + chunk_off(((lane & 7) ^ (((n & 1) << 2) | (drow >> 1))) * 8)) * 2;
#pragma unroll
    for (int n = 0; n < LB; ++n) {
        const int t = wave * LB + n;
        offb[n] = QT ? (unsigned)((t >> 2) * BLK_ELEMS + ((t & 3) * 16 + (lane >> 2)) * BLK_COLS + ((lane & 3) ^ (((lane >> 5) & 1) << 1)) * 8) * 2
                     : (unsigned)(in_panel(tc.tj * BN, t * 8 + drow) + chunk_off(((lane & 7) ^ (((n & 1) << 2) | (drow >> 1))) * 8)) * 2;
    }
    constexpr int KT_BLOCKS = 64 / BLK_COLS;
    const unsigned lds_base = (unsigned)(uintptr_t)(lds_void_ptr)smem;
    auto dma = [&](const char* base, unsigned voff, unsigned lds_byte) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :
                     : "s"(lds_byte), "v"(voff), "s"(base)
                     : "memory");
    };
    auto issue_one = [&](int n, int kt) {  // load instruction n of k-tile kt: rows of P first, then Q
        const unsigned st = lds_base + (kt & (NST - 1)) * STAGE;
        const long koff = (long)kt * KT_BLOCKS * kstep;
        const int k0 = kt * 64;
        if (n < LA) dma((const char*)(Pb + koff), offa[n], st + (wave * LA + n) * 8 * ROW_BYTES);
        else
            dma((const char*)(Qb + (QT ? (long)(k0 >> 8) * g.cbQ * BLK_ELEMS + (k0 & 255) * BLK_COLS : koff)), offb[n - LA],
                st + A_BYTES + (wave * LB + n - LA) * 8 * ROW_BYTES);
    };
    const int sw = (lane >> 1) & 7, kq = lane >> 4;
    const int a_off = (wm * WTM + (lane & 15)) * ROW_BYTES;
    const int b_off = A_BYTES + (wn * WTN + (lane & 15)) * ROW_BYTES;
    const int q_off[2] = {A_BYTES + wn * (WTN / 32) * 4096 + qt_lane_offset(lane, 0),
                          A_BYTES + wn * (WTN / 32) * 4096 + qt_lane_offset(lane, 1)};
    bf16x8 fr[2][KS * NRD];
    auto read_one = [&](auto buf_c, int o, const unsigned char* st) {
        constexpr int BUF = decltype(buf_c)::value;
        const int ks = o / NRD, n = o % NRD, co = (((ks << 2) | kq) ^ sw) << 4;
        if (n < FM) fr[BUF][o] = *(const bf16x8*)(st + a_off + n * 16 * ROW_BYTES + co);
        else if (QT) fr[BUF][o] = lds_read_qt(st + q_off[(n - FM) & 1] + ((n - FM) >> 1) * 4096 + ks * 32 * 64);
        else fr[BUF][o] = *(const bf16x8*)(st + b_off + (n - FM) * 16 * ROW_BYTES + co);
    };
    f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // k-tile kt: its fragments are in flight from LDS.  WAIT: k-tiles after kt+1 whose loads may be outstanding (-1: there is
    // no k-tile kt+1).  After the barrier every wave has read k-tile kt-1, so its stage takes k-tile kt+NST-1.  The fragment
    // reads of k-tile kt+1 and the loads stand between the MFMAs and issue in their shadow (a lone wave per SIMD has nothing
    // else to hide them behind); the fences pin that order.
    auto body = [&](int kt, auto buf_c, auto issue_c, auto wait_c) {
        constexpr int BUF = decltype(buf_c)::value, WAIT = decltype(wait_c)::value;
        constexpr int NRD2 = WAIT >= 0 ? KS * NRD : 0, NOTH = NRD2 + (decltype(issue_c)::value ? NLD : 0);
        constexpr int NMF = KS * FM * FN, PER = (KS * NRD + NLD + NMF - 1) / NMF;
        WAIT_LGKM0();
        if constexpr (WAIT >= 0) {
            WAIT_VM(WAIT * NLD);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
        const unsigned char* stn = smem + ((kt + 1) & (NST - 1)) * STAGE;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < NMF; ++m) {
            const int ks = m / (FM * FN), j = m % (FM * FN) / FM, ii = m % FM, i = (j & 1) ? FM - 1 - ii : ii;
            const bf16x8 p = fr[BUF][ks * NRD + i], q = fr[BUF][ks * NRD + FM + j];
            acc[i][j] = QT ? mfma16(q, p, acc[i][j]) : mfma16(p, q, acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < PER; ++u) {
                const int o = m * PER + u;
                if (o < NRD2) read_one(std::integral_constant<int, BUF ^ 1>{}, o, stn);
                else if (o < NOTH) issue_one(o - NRD2, kt + NST - 1);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    const int nk = g.kdim / 64;  // even: reductions are multiples of 128
    // k-tiles nk-R and nk-R+1, the first of the last R
    auto tail_pair = [&](auto r_c) {
        constexpr int R = decltype(r_c)::value;
        if (nk < R) return;
        constexpr int W0 = R - 2 < NST - 3 ? R - 2 : NST - 3, W1 = R - 3 < NST - 3 ? R - 3 : NST - 3;
        body(nk - R, I0{}, std::integral_constant<bool, R == NST>{}, std::integral_constant<int, W0>{});
        body(nk - R + 1, I1{}, std::false_type{}, std::integral_constant<int, W1>{});
    };
    const int first = nk < NST - 1 ? nk : NST - 1;
    for (int t = 0; t < first; ++t)
#pragma unroll
        for (int n = 0; n < NLD; ++n) issue_one(n, t);
    if (nk >= NST) WAIT_VM((NST - 2) * NLD);
    else if (nk == 6) WAIT_VM(5 * NLD);
    else if (nk == 4) WAIT_VM(3 * NLD);
    else WAIT_VM(NLD);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int o = 0; o < KS * NRD; ++o) read_one(I0{}, o, smem);
    for (int kt = 0; kt + NST < nk; kt += 2) {
        body(kt, I0{}, std::true_type{}, std::integral_constant<int, NST - 3>{});
        body(kt + 1, I1{}, std::true_type{}, std::integral_constant<int, NST - 3>{});
    }
    tail_pair(std::integral_constant<int, 8>{});
    tail_pair(std::integral_constant<int, 6>{});
    tail_pair(std::integral_constant<int, 4>{});
    tail_pair(std::integral_constant<int, 2>{});
    bf16x8 ev[tile_pieces<BM, BN, WGM, WGN>()];
    if constexpr (QT) epilogue_nn_reg<BN, WGN, WTM, FM, true, false, EPI_ALL>(g, tc.bidx, tc.ti * BM, tc.tj * BN, acc, ev);
    else epilogue_sym_reg<BM, BN, WGM, WGN, EPI, 0, false, EPI_ALL>(g, tc, acc, ev);
}

// The same with a split tail: when the tile count leaves the last round of the compute units mostly empty,
// the first big_blocks workgroups compute 256x256 tiles as above and every remaining tile is cut
// into four 128x128 tiles, one workgroup each, which fill the CUs that would otherwise idle for a
// whole tile time.  The lower-left quarter of a diagonal tile of the symmetric kernels is the mirror
// of the upper-right one and is skipped.
template <int EPI>
__global__ void __launch_bounds__(512) gemm_nt_pp_tail_kernel(const GemmList l) {
    extern __shared__ __align__(16) unsigned char smem[];
    const bool big = (int)blockIdx.x < l.big_blocks;
    const int s = blockIdx.x - l.big_blocks, quarter = s & 3;
    const int logical = big ? xcd_remap(blockIdx.x, l.big_blocks, l.xcd_shift) : l.big_blocks + (s >> 2);
    const int entry = list_entry(l, logical);
    const GemmArgs& g = l.g[entry];
    TileCoord tc = tile_of<EPI>(g, logical - l.start[entry]);
    if (big) {
        pp_tile<256, 256, 2, 4, EPI>(g, tc, smem);
    } else {
        if (!epi_is_bx(EPI) && tc.ti == tc.tj && quarter == 2) return;
        tc.ti = tc.ti * 2 + (quarter >> 1);
        tc.tj = tc.tj * 2 + (quarter & 1);
        pp_tile<128, 128, 2, 4, EPI>(g, tc, smem);
    }
}

// ---- kernel 3: the ping-pong loop as a persistent kernel ----------------------------------------
// With an epilogue that needs no LDS (epilogue_nn_reg, epilogue_sym_reg) nothing stands between the k loops of two tiles: one
// workgroup per compute unit walks tiles, the last three memory phases of a tile issue the first three k-tiles of the
// workgroup's NEXT tile into the stages the current one has finished with, and they land while the waves drain their
// accumulators.  What a one-tile workgroup pays around its k loop on top of the epilogue - the cold first loads (2 to
// 3 us) and the hand-over of the compute unit to the next workgroup (2 to 3 us) - is a sixth of a tile when the
// reduction is 24 k-tiles long (a 768-row expert matrix) and 4 % at 128.
//
// Tiles are handed out per XCD, in the order xcd_remap gives a one-tile-per-workgroup launch: workgroup b sits on
// XCD b % 8 and takes "virtual workgroup ids" 8 n + b % 8.  Its first two n are static (b / 8 and b / 8 + grid / 8),
// later ones come from an atomic counter of its XCD, asked for during the epilogue of the tile before the one whose
// last phases need it.  The counters are the caller's (GemmArgs::ppx, a piece of the workspace of the call): a launch
// finds them zero, and the last workgroup to leave puts them back to zero, so the library keeps no state of its own
// and calls with different workspaces do not meet.
struct PpxCounters {
    unsigned next[GEMM_MAX_XCDS][16];  // a cache line per XCD: tiles handed out beyond the two static rounds
    unsigned done[16];                 // workgroups that have left
};
static_assert(sizeof(PpxCounters) == GEMM_PPX_COUNTER_BYTES, "the size the header promises");

// The products of a launch share one walk over the tiles of all of them (12 of 2731 x 1000, 6 of 1000 x 2731 and 12 of
// 1000 x 1000, 3.8 rounds: 172 us in launches of their own, 123 in one).
//
// F0, F1: fragment rows (16 rows each) of the two wave rows of a tile, 8 + 8 for the 256x256 tile.  a.X + B.X also has tiles
// of 8 + 6 (224 rows) and 6 + 6 (192 rows), for short sides that leave half of a last 256-tile empty (896 = 4 x 224, 1152 =
// 6 x 192).  Waves w and w + 4 share a SIMD and belong to different wave rows, so every SIMD has the same work.
// LIST: the launch holds several products (one: its extents stay out of the per-tile state).
template <int EPI, int F0, int F1, bool LIST>
__global__ void __launch_bounds__(512) gemm_nt_ppx_kernel(const GemmList l) {
    static_assert(EPI == EPI_BX || EPI == EPI_SYRK || EPI == EPI_SYMPOLY, "the epilogues that need no LDS");
    constexpr bool QT = EPI == EPI_BX;  // Q is X itself, rows = reduction index
    static_assert(F0 >= F1 && F0 <= 8 && (QT || (F0 == 8 && F1 == 8)), "tile heights");
    constexpr int BM = 16 * (F0 + F1), BN = 256, WGM = 2, WGN = 4, NW = 8;
    constexpr int BK4 = 32, ROWB = 64;
    constexpr int WTM = 16 * F0, WTN = BN / WGN;
    constexpr int FM = F0, FN = WTN / 16;
    constexpr bool WHOLE = BM == 256;  // a tile is a row block; otherwise its panels may cross from one to the next
    constexpr int A_BYTES = 256 * ROWB, B_BYTES = BN * ROWB, STAGE = A_BYTES + B_BYTES;
    constexpr int LA = 256 / 16 / NW, LB = BN / 16 / NW;
    constexpr int NLD = LA + LB;
    constexpr int SLOT_OFF = 4 * STAGE;  // behind the four stages: where lane 0 leaves the next tile's id for the others

    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 2;
    const int wm = wave / WGN, wn = wave % WGN;
    const int total = l.start[l.n];
    const int grid = gridDim.x, xcd_shift = l.xcd_shift, xcds = 1 << xcd_shift, xcd = blockIdx.x & (xcds - 1);
    PpxCounters& ctr = *(PpxCounters*)l.g[0].ppx;

    // A tile: its product, its place there, and where its operands start.  p: this wave's load instructions of P, 16 rows each.
    // A tile that is a row block needs one pointer; in the others every instruction has its own, and the last waves, past the
    // end of the tile, fetch rows of it once more into a part of the stage that nobody reads.
    struct Tile {
        int entry, nk, cbQ;  // nk: k-tiles, a multiple of 4, at least 8 (the launcher checks)
        TileCoord tc;
        const bf16_t* p[WHOLE ? 1 : LA];
        const bf16_t* q;
    };
    auto tile_at = [&](int pid) {
        Tile t;
        const int logical = xcd_remap(pid, total, xcd_shift);
        t.entry = LIST ? list_entry(l, logical) : 0;
        const GemmArgs& g = l.g[LIST ? t.entry : 0];
        t.tc = tile_of<EPI>(g, LIST ? logical - l.start[t.entry] : logical);
        t.nk = g.kdim / BK4;
        t.cbQ = g.cbQ;
        const bf16_t* P = g.P + t.tc.bidx * g.strideP;
        if constexpr (WHOLE) {
            t.p[0] = uniform_ptr(P + panel_offset(t.tc.ti * BM, g.cbP));
        } else {
#pragma unroll
            for (int n = 0; n < LA; ++n) {
                const int grp16 = wave * LA + n < BM / 16 ? wave * LA + n : BM / 16 - 1;
                t.p[n] = uniform_ptr(P + panel_offset(t.tc.ti * BM + grp16 * 16, g.cbP));
            }
        }
        t.q = uniform_ptr(g.Q + t.tc.bidx * g.strideQ +
                          (QT ? (long)(t.tc.tj * BN >> BLK_SHIFT) * BLK_ELEMS : panel_offset(t.tc.tj * BN, g.cbP)));
        return t;
    };

    // per-lane load offsets and LDS addresses: as in pp_tile
    const int drow = lane >> 2;
    const int dch = ((lane & 3) ^ pp_swizzle((lane >> 4) & 3)) * 8;
    unsigned offa[LA], offb[LB];
#pragma unroll
    for (int n = 0; n < LA; ++n) offa[n] = (unsigned)((((WHOLE ? wave * 16 * LA + n * 16 : 0) + drow) * BLK_COLS + dch) * 2);
    const int qch = ((lane & 3) ^ (((drow >> 3) & 1) << 1)) * 8;
#pragma unroll
    for (int n = 0; n < LB; ++n) {
        const int t = wave * LB + n;
        offb[n] = QT ? (unsigned)(((t >> 1) * BLK_ELEMS + ((t & 1) * 16 + drow) * BLK_COLS + qch) * 2)
                     : (unsigned)(((wave * 16 * LB + n * 16 + drow) * BLK_COLS + dch) * 2);
    }
    const int lds_a = wave * 16 * LA * ROWB;
    const int lds_b = A_BYTES + wave * 16 * LB * ROWB;

    auto dma = [&](const char* base, unsigned voff, unsigned lds_byte) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :
                     : "s"(lds_byte), "v"(voff), "s"(base)
                     : "memory");
    };
    const unsigned lds_base = (unsigned)(uintptr_t)(lds_void_ptr)smem;
    // k-tile kt of tile t, into stage kt & 3
    auto issue_tile = [&](const Tile& t, int kt) {
        const int k0 = kt * BK4;
        const long koff = (long)(k0 >> BLK_SHIFT) * BLK_ELEMS + (k0 & (BLK_COLS - 1));
        const char* bb = (const char*)(t.q + (QT ? (long)(k0 >> 8) * (LIST ? t.cbQ : l.g[0].cbQ) * BLK_ELEMS + (k0 & 255) * BLK_COLS : koff));
        const unsigned st = lds_base + (kt & 3) * STAGE;
#pragma unroll
        for (int n = 0; n < LA; ++n) dma((const char*)(t.p[WHOLE ? 0 : n] + koff), offa[n], st + lds_a + n * 16 * ROWB);
#pragma unroll
        for (int n = 0; n < LB; ++n) dma(bb, offb[n], st + lds_b + n * 16 * ROWB);
    };

    const int sw = pp_swizzle((lane >> 2) & 3), kq = lane >> 4;
    const int co = (kq ^ sw) << 4;
    const int a_off = (wm * WTM + (lane & 15)) * ROWB + co;
    const int b_off = A_BYTES + (wn * WTN + (lane & 15)) * ROWB + co;
    const unsigned char* ra[2];
    const unsigned char* rb[2][2];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        ra[half] = smem + half * 2 * STAGE + a_off;
#pragma unroll
        for (int h = 0; h < 2; ++h)
            rb[half][h] = QT ? smem + half * 2 * STAGE + A_BYTES + (wn * WTN / 32) * 2048 + qt_lane_offset(lane, h)
                             : smem + half * 2 * STAGE + b_off;
    }

    // this workgroup's tiles: the current one, the one after it (virtual ids; >= total means none)
    int pid_cur = blockIdx.x, pid_nxt = blockIdx.x + grid;
    Tile cur = tile_at(pid_cur);

    issue_tile(cur, 0);
    issue_tile(cur, 1);
    issue_tile(cur, 2);
    WAIT_VM(0);  // a tile starts with its k-tiles 0, 1 and 2 in LDS
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (grp) __builtin_amdgcn_s_barrier();

    for (;;) {
        const bool has_next = pid_nxt < total;
        // without a next tile the last phases load this tile's first k-tiles again, into stages nobody reads any more
        const Tile next = tile_at(has_next ? pid_nxt : pid_cur);
        const GemmArgs& g = l.g[LIST ? cur.entry : 0];
        const int nk = LIST ? cur.nk : l.g[0].kdim / BK4;
        const bool diag = !QT && cur.tc.ti == cur.tc.tj;
        unsigned fetched = 0;
        // One tile, k loop and epilogue, for the waves whose skip mask in a diagonal tile is `mask_c` (pp_tile): a copy of
        // its own per mask, each with its own accumulators from the first MFMA to the last store.
        auto run_tile = [&](auto mask_c) {
            f32x4 acc[FM][FN];  // defined by the MFMAs of the tile's first k-tile, which add to zero

            // NEXT: the memory phase issues k-tile kt+3-nk of the next tile instead of k-tile kt+3 of this one.
            // NOWAIT: the first two phases of a tile wait for no load: its k-tiles 0, 1 and 2 are in LDS when it starts
            // (a count would make them wait for the stores of the epilogue before).
            constexpr unsigned MASK = decltype(mask_c)::value;  // fragments a wave skips in a diagonal tile
            auto body = [&](int kt, auto stage_c, auto next_c, auto nowait_c, auto first_c) {
                constexpr int SIDX = decltype(stage_c)::value;
                constexpr bool NEXT = decltype(next_c)::value;
                constexpr bool NOWAIT = decltype(nowait_c)::value;
                constexpr bool FIRST = decltype(first_c)::value;
                auto kept = [](int i, int j) { return !((MASK >> (i * FN + j)) & 1); };
                bf16x8 fa[FM], fb[FN];
    #pragma unroll
                for (int i = 0; i < FM; ++i) {
                    bool used = false;
    #pragma unroll
                    for (int j = 0; j < FN; ++j) used |= kept(i, j);
                    if (used) fa[i] = *(const bf16x8*)(ra[SIDX >> 1] + (SIDX & 1) * STAGE + i * 16 * ROWB);
                }
    #pragma unroll
                for (int j = 0; j < FN; ++j) {
                    bool used = false;
    #pragma unroll
                    for (int i = 0; i < FM; ++i) used |= kept(i, j);
                    if (!used) continue;
                    if (QT) fb[j] = lds_read_qt(rb[SIDX >> 1][j & 1] + (SIDX & 1) * STAGE + (j >> 1) * 2048);
                    else fb[j] = *(const bf16x8*)(rb[SIDX >> 1][0] + (SIDX & 1) * STAGE + j * 16 * ROWB);
                }
                if constexpr (NEXT) issue_tile(next, kt + 3 - nk);
                else issue_tile(cur, kt + 3);
                WAIT_LGKM0();
                if constexpr (!NOWAIT) WAIT_VM(2 * NLD);  // own loads of k-tile kt+1 have landed
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
    #pragma unroll
                for (int j = 0; j < FN; ++j)
    #pragma unroll
                    for (int ii = 0; ii < FM; ++ii) {
                        const int i = (j & 1) ? FM - 1 - ii : ii;  // back and forth: consecutive MFMAs share an operand
                        const f32x4 c = FIRST ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[i][j];
                        if (!kept(i, j)) continue;
                        acc[i][j] = QT ? mfma16(fb[j], fa[i], c) : mfma16(fa[i], fb[j], c);
                    }
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            };
            using I0 = std::integral_constant<int, 0>;
            using I1 = std::integral_constant<int, 1>;
            using I2 = std::integral_constant<int, 2>;
            using I3 = std::integral_constant<int, 3>;
            using No = std::false_type;
            using Yes = std::true_type;
            body(0, I0{}, No{}, Yes{}, Yes{});
            body(1, I1{}, No{}, Yes{}, No{});
            body(2, I2{}, No{}, No{}, No{});
            body(3, I3{}, No{}, No{}, No{});
            for (int kt = 4; kt < nk - 4; kt += 4) {
                body(kt, I0{}, No{}, No{}, No{});
                body(kt + 1, I1{}, No{}, No{}, No{});
                body(kt + 2, I2{}, No{}, No{}, No{});
                body(kt + 3, I3{}, No{}, No{}, No{});
            }
            body(nk - 4, I0{}, No{}, No{}, No{});
            body(nk - 3, I1{}, Yes{}, No{}, No{});
            body(nk - 2, I2{}, Yes{}, No{}, No{});
            body(nk - 1, I3{}, Yes{}, No{}, No{});
            if (!grp) __builtin_amdgcn_s_barrier();  // the two groups leave the k loop together

            // Every wave drains its accumulators on its own.  One lane asks for the id of the tile after the next (an
            // increment with wrap-around at 2^32 - 1: a plain atomicAdd of a uniform value is turned into a wave-wide
            // reduction by the compiler, which then waits for the answer on the spot); the answer is needed at the end.
            if (has_next && tid == 0) fetched = atomicInc(&ctr.next[xcd][0], 0xffffffffu);
            if constexpr (QT) {
                bf16x8 none[1];
                epilogue_nn_reg<BN, WGN, WTM, MASK == 0 ? F0 : F1, WHOLE, false, EPI_ALL>(g, cur.tc.bidx, cur.tc.ti * BM, cur.tc.tj * BN, acc, none);
            } else {
                bf16x8 ev[FM * FN / 2];
                epilogue_sym_reg<BM, BN, WGM, WGN, EPI, MASK, false, EPI_ALL>(g, cur.tc, acc, ev);
                // What says that this wave's share of the next tile's first k-tiles has landed: B.X and b.A + c.A.A consume
                // loads that were issued after them (the queue returns in order).  X.Xt loads nothing, and in a diagonal
                // tile a wave may have nothing to finish at all: there the count is explicit (48 stores went out after the
                // loads off the diagonal, an unknown number on it).
                asm volatile("" ::: "memory");
                if (diag) WAIT_VM(0);
                else if (EPI == EPI_SYRK) WAIT_VM(FM * FN / 2 * 3);
                asm volatile("" ::: "memory");
            }
        };  // run_tile
        if constexpr (F1 < F0) {
            if (wm == 0) run_tile(std::integral_constant<unsigned, 0>{});
            else run_tile(std::integral_constant<unsigned, (unsigned)((1ull << (F0 * FN)) - (1ull << (F1 * FN)))>{});
        } else if (!diag) {
            run_tile(std::integral_constant<unsigned, 0>{});
        } else {
            auto run_if_mine = [&](auto wave_c) {
                constexpr int W = decltype(wave_c)::value;
                constexpr unsigned M = pp_skip_mask<WTM, WTN, FM, FN, WGN>(W);
                if constexpr (pp_first_with_mask<WTM, WTN, FM, FN, WGN>(W)) {
                    if (pp_skip_mask<WTM, WTN, FM, FN, WGN>(wave) == M) run_tile(std::integral_constant<unsigned, M>{});
                }
            };
            run_if_mine(std::integral_constant<int, 0>{});
            run_if_mine(std::integral_constant<int, 1>{});
            run_if_mine(std::integral_constant<int, 2>{});
            run_if_mine(std::integral_constant<int, 3>{});
            run_if_mine(std::integral_constant<int, 4>{});
            run_if_mine(std::integral_constant<int, 5>{});
            run_if_mine(std::integral_constant<int, 6>{});
            run_if_mine(std::integral_constant<int, 7>{});
        }
        // (the answer stays untouched until here: any arithmetic on it would be scheduled next to the atomic, with a
        // wait for it)
        asm volatile("" : "+v"(fetched));
        if (tid == 0) *(int*)(smem + SLOT_OFF) = has_next ? (((2 * (grid >> xcd_shift) + (int)fetched)) << xcd_shift) + xcd : total;
        // The loads of the epilogue are behind those of the next tile's first k-tiles in the queue and have been
        // consumed, so every wave's share of those k-tiles has landed: publish them, and the id.
        __syncthreads();
        if (!has_next) break;
        pid_cur = pid_nxt;
        pid_nxt = __builtin_amdgcn_readfirstlane(*(const int*)(smem + SLOT_OFF));
        cur = next;
        if (grp) __builtin_amdgcn_s_barrier();  // and enter the next tile a phase apart again
    }
    if (tid == 0) {
        // every workgroup has its last answer from `next` before it counts itself out, so the last one out may reset
        if (atomicAdd(&ctr.done[0], 1u) == (unsigned)grid - 1) {
            for (int x = 0; x < xcds; ++x) atomicExch(&ctr.next[x][0], 0u);
            atomicExch(&ctr.done[0], 0u);
        }
    }
}

// ---- kernel 4: the whole chain of many small matrices in one launch ------------------------------
// A set of a few dozen matrices makes fifteen dependent launches of one to three rounds of tiles, and in each of them most compute
// units wait for the last tiles and for the next launch to start.  Here a matrix belongs to one XCD for all of its products:
// what one compute unit writes, another of the same XCD reads out of the L2 that they share, so that a product may start as
// soon as the one before it has finished for that matrix, with a counter in memory between them and no launch.  (The same over all
// XCDs has to write through to memory: a hand-over of 8 KB each between 32 workgroups of an XCD takes 1.9 us, between all 256 with
// written-through stores 6.4, with cache write-backs 77; a launch without any work 2.4.  profiles/flow_chain_hand_over.txt)
//
// The host deals the matrices to as many groups as there are XCDs.  A workgroup finds out which XCD it runs on, takes that
// XCD's group (the first of an XCD to ask fetches a group for it; an XCD that has finished one fetches another, so the groups
// are served whatever XCDs the workgroups land on) and then tiles of it by a counter, in the order iteration, product, matrix,
// tile.  A tile waits until its matrix has finished every tile of the product before.  Tiles are taken in order, and a tile waits
// only for tiles that come before its own, which workgroups that are running hold: the earliest unfinished tile never waits, so
// every wait ends.  Each is bounded all the same, by some minutes: then the tile that waited stores nothing and is not counted, every
// other workgroup leaves at its next wait in vain, and FlowList::alarm, a word of host memory, says so to the next call.
//
// Memory order.  Producer: the tile's stores, `s_waitcnt vmcnt(0)` in every wave (they are in L2), the workgroup's barrier, the
// matrix's counter.  Consumer: the counter, the barrier, then loads that read past the compute unit's own vector cache (load16,
// sc1 on the operand loads; the buffers of X are written again two iterations later and may be in it).  Measured, sc1 costs the
// loads nothing: the XCD's L2 serves them.
//
// 128x128 tiles on the ping-pong loop, two workgroups per compute unit: one waits, starts and drains while the other computes.
struct FlowControl {
    unsigned tile[GEMM_MAX_XCDS][16];           // per group: tiles handed out
    unsigned group_of[GEMM_MAX_XCC_IDS][16];    // the n-th group of an XCD: 0 nobody has asked, 1 being fetched, group + 2
    unsigned next_group[16];
    unsigned abandoned[16];                     // a wait has given up: everybody leaves
};
static_assert(sizeof(FlowControl) == GEMM_FLOW_CONTROL_BYTES && GEMM_MAX_XCDS < 16, "the size the header promises");

__device__ __forceinline__ unsigned flow_load(const unsigned* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Waits until *p, a count, has reached `want`; false if the launch is being abandoned.  Polls seldom while much is missing: on the
// line that sixty workgroups poll the increments themselves have to queue.
__device__ __forceinline__ bool flow_wait(const FlowList& l, const unsigned* p, unsigned want, unsigned* abandoned) {
    for (unsigned spins = 0;; ++spins) {
        const unsigned have = flow_load(p);
        if (have >= want) return true;
        if (want - have > 16) __builtin_amdgcn_s_sleep(32);
        else if (want - have > 4) __builtin_amdgcn_s_sleep(8);
        else __builtin_amdgcn_s_sleep(2);
        if ((spins & 1023) == 1023 && flow_load(abandoned)) return false;
        if (spins >= l.polls) {
            atomicExch(abandoned, 1u);
            __hip_atomic_store(l.alarm, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            return false;
        }
    }
}

constexpr int kFlowStages = 4 * (128 + 128) * 64;
// What thread 0 of a workgroup keeps, and what it tells the others: the tile (entry, matrix, tile, product, iteration; entry < 0: none
// is left).
struct FlowSlot {
    int entry, matrix, tile, stage, it;
    int gone;            // a wait has been given up
    int epoch, group;    // the XCD's group that the workgroup takes tiles of, -1 before it knows
    unsigned want;       // tiles of the matrix that come before the tile's product
    unsigned* done;      // the matrix's counter
};
// The next tile of this XCD, in order: false when there is none left.  have: tile `t` of the group has been asked for already.
__device__ __forceinline__ bool flow_next(const FlowList& l, FlowControl& ctl, FlowSlot* slot, bool have, int t) {
    int g = slot->group, epoch = slot->epoch;
    if (slot->gone) return false;
    for (;;) {
        if (g < 0) {
            if (epoch == l.groups) return false;
            unsigned id;
            asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(id));
            unsigned* const mine = &ctl.group_of[id & (GEMM_MAX_XCC_IDS - 1)][epoch];
            unsigned v = atomicCAS(mine, 0u, 1u);
            if (v == 0) {
                v = atomicAdd(&ctl.next_group[0], 1u) + 2;
                atomicExch(mine, v);
            } else if (v == 1) {
                if (!flow_wait(l, mine, 2, &ctl.abandoned[0])) return false;
                v = flow_load(mine);
            }
            g = (int)v - 2;
            if (g >= l.groups) return false;
        }
        if (!have) t = (int)atomicAdd(&ctl.tile[g][0], 1u);
        have = false;
        if (t < flow_tiles(l, g)) break;
        g = -1;
        ++epoch;
    }
    slot->group = g;
    slot->epoch = epoch;
    const FlowPlace p = flow_place(l, g, t);
    slot->entry = p.entry;
    slot->matrix = p.matrix;
    slot->tile = p.tile;
    slot->stage = p.stage;
    slot->it = p.it;
    slot->done = l.e[p.entry].done + p.matrix * GEMM_FLOW_LINE;
    slot->want = (unsigned)p.before;
    return true;
}

__global__ void __launch_bounds__(512, 4) gemm_nt_flow_kernel(const FlowList l) {
    extern __shared__ __align__(16) unsigned char smem[];
    FlowSlot* const slot = (FlowSlot*)(smem + kFlowStages);  // behind the four stages
    FlowControl& ctl = *(FlowControl*)l.control;
    const int tid = threadIdx.x;
    if (tid == 0) slot->epoch = 0, slot->group = -1, slot->gone = 0;
    int fetched = 0;             // thread 0: the tile asked for while the one before was in its epilogue
    unsigned* finished = nullptr;  // the counter of the matrix that the tile before belongs to
    auto ask = [&]() {
        // (atomicInc: an atomicAdd of a uniform value becomes a wave-wide reduction whose result the compiler waits for on the spot)
        if (tid == 0) fetched = (int)atomicInc(&ctl.tile[slot->group][0], 0xffffffffu);
    };
    auto wait = [&]() {  // everything in front of this is done while the matrix is not ready yet
        if (tid == 0 && !flow_wait(l, slot->done, slot->want, &ctl.abandoned[0])) slot->gone = 1;
        __syncthreads();
    };
    auto ready = [&]() {  // whether that wait found the matrix ready; if not, the workgroup leaves
        const bool yes = !__builtin_amdgcn_readfirstlane(slot->gone);
        if (!yes) finished = nullptr;
        return yes;
    };
    for (;;) {
        if (tid == 0 && !flow_next(l, ctl, slot, finished != nullptr, fetched)) slot->entry = -1;
        // every wave's stores of the tile before are in L2, and every wave has read what it needs from LDS
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0 && finished) __hip_atomic_fetch_add(finished, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int entry = __builtin_amdgcn_readfirstlane(slot->entry);
        if (entry < 0) break;
        const FlowEntry& e = l.e[entry];
        const int tile = __builtin_amdgcn_readfirstlane(slot->tile), stage = __builtin_amdgcn_readfirstlane(slot->stage);
        const int it = __builtin_amdgcn_readfirstlane(slot->it), cur = it & 1;
        GemmArgs a = {};
        a.cbP = e.Mp / BLK_COLS;
        a.kdim = e.Mp;
        TileCoord tc{__builtin_amdgcn_readfirstlane(slot->matrix), 0, 0};
        finished = e.done + tc.bidx * GEMM_FLOW_LINE;
        auto run = [&](auto epi_c) { pp_tile<128, 128, 2, 4, decltype(epi_c)::value, true>(a, tc, smem, wait, ask, ready); };
        if (stage == 2) {
            a.tiles_m = e.Mp / 128;
            a.tiles_n = e.Kr / 128;
            rect_decode<4>(tile, a.tiles_m, a.tiles_n, tc.ti, tc.tj);
            a.P = e.B;
            a.strideP = e.strideA;
            a.Q = a.Et = e.X[cur];
            a.C = e.X[cur ^ 1];
            a.strideQ = a.strideEt = a.strideC = e.strideX;
            a.cbQ = a.cbEt = a.cbC = e.Kp / BLK_COLS;
            a.s0 = l.a;
            if (!e.p_ptrs || it < l.steps - 1) {
                run(std::integral_constant<int, EPI_BX>{});
            } else {
                a.upd_ptrs = e.p_ptrs;
                a.upd_dtype = l.p_dtype;
                a.upd_rows = e.rows;
                a.upd_cols = e.cols;
                a.upd_scale = e.scale;
                a.upd_decay = l.decay;
                a.upd_alpha = l.alpha;
                if (e.rows <= e.cols) run(std::integral_constant<int, EPI_BX_UPD>{});
                else run(std::integral_constant<int, EPI_BX_UPD_T>{});
            }
        } else {
            tri_decode<4>(tile, e.Mp / 128, tc.ti, tc.tj);
            a.strideC = a.strideCt = e.strideA;
            a.cbC = a.cbCt = e.Mp / BLK_COLS;
            if (stage == 0) {
                a.P = a.Q = e.X[cur];
                a.strideP = a.strideQ = e.strideX;
                a.cbP = e.Kp / BLK_COLS;
                a.kdim = e.Kr;
                a.C = a.Ct = e.A;
                run(std::integral_constant<int, EPI_SYRK>{});
            } else {
                a.P = a.Q = a.Et = e.A;
                a.strideP = a.strideQ = a.strideEt = e.strideA;
                a.cbEt = e.Mp / BLK_COLS;
                a.C = a.Ct = e.B;
                a.s0 = l.b;
                a.s1 = l.c;
                run(std::integral_constant<int, EPI_SYMPOLY>{});
            }
        }
    }
}

}  // namespace
hipError_t allow_dynamic_lds(const void* kern, int bytes, std::atomic<unsigned long long>& done) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const unsigned long long bit = 1ull << (dev & 63);
    if (done.load(std::memory_order_acquire) & bit) return hipSuccess;
    e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return e;
    done.fetch_or(bit, std::memory_order_release);
    return hipSuccess;
}
namespace {

template <int EPI, int F0, int F1, bool LIST>
hipError_t launch_ppx_as(const GemmList& l, int nblocks, int cus, hipStream_t stream) {
    constexpr int smem = 4 * (256 + 256) * 64 + 64;
    static std::atomic<unsigned long long> configured{0};  // per instantiation
    const auto kern = gemm_nt_ppx_kernel<EPI, F0, F1, LIST>;
    if (hipError_t e = allow_dynamic_lds((const void*)kern, smem, configured); e != hipSuccess) return e;
    const int grid = nblocks < cus ? nblocks : cus;  // a whole number of XCDs: the caller launches more tiles than CUs
    hipLaunchKernelGGL(kern, dim3(grid), dim3(512), smem, stream, l);
    return hipGetLastError();
}
template <int EPI, int F0 = 8, int F1 = 8>
hipError_t launch_ppx(const GemmList& l, int nblocks, int cus, hipStream_t stream) {
    return l.n > 1 ? launch_ppx_as<EPI, F0, F1, true>(l, nblocks, cus, stream) : launch_ppx_as<EPI, F0, F1, false>(l, nblocks, cus, stream);
}

template <int BM, int BN, int WGM, int WGN, int EPI, int FEED>
hipError_t launch_one(const GemmList& l, int nblocks, hipStream_t stream) {
    constexpr int stages = 2 * (BM + BN) * ROW_BYTES;
    constexpr int epi = epi_is_bx(EPI) ? epilogue_nn_bytes<BM, BN>() : epilogue_bytes<BM, BN>();
    constexpr int smem = stages > epi ? stages : epi;
    static std::atomic<unsigned long long> configured{0};  // per instantiation; setting the attribute twice is harmless
    void (*kern)(const GemmList);
    if constexpr (FEED == 1) kern = gemm_nt_pp_kernel<BM, BN, WGM, WGN, EPI>;
    else kern = gemm_nt_pipe_kernel<BM, BN, WGM, WGN, EPI>;
    if (hipError_t e = allow_dynamic_lds((const void*)kern, smem, configured); e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(nblocks), dim3(WGM * WGN * 64), smem, stream, l);
    return hipGetLastError();
}

template <int EPI>
hipError_t launch_deep(const GemmList& l, int nblocks, hipStream_t stream) {
    constexpr int smem = 8 * (64 + 64) * ROW_BYTES;
    static std::atomic<unsigned long long> configured{0};
    if (hipError_t e = allow_dynamic_lds((const void*)gemm_nt_deep_kernel<EPI>, smem, configured); e != hipSuccess) return e;
    hipLaunchKernelGGL(gemm_nt_deep_kernel<EPI>, dim3(nblocks), dim3(256), smem, stream, l);
    return hipGetLastError();
}

template <int EPI>
hipError_t launch_pp_tail(GemmList& l, int nblocks, int rest, hipStream_t stream) {
    constexpr int stages = 2 * (256 + 256) * ROW_BYTES;
    constexpr int epi = epi_is_bx(EPI) ? epilogue_nn_bytes<256, 256>() : epilogue_bytes<256, 256>();
    constexpr int smem = stages > epi ? stages : epi;  // the 128-tiles need less of both
    static std::atomic<unsigned long long> configured{0};
    auto kern = gemm_nt_pp_tail_kernel<EPI>;
    if (hipError_t e = allow_dynamic_lds((const void*)kern, smem, configured); e != hipSuccess) return e;
    l.big_blocks = nblocks - rest;
    hipLaunchKernelGGL(kern, dim3(l.big_blocks + 4 * rest), dim3(512), smem, stream, l);
    return hipGetLastError();
}

template <int EPI>
hipError_t launch_cfg(int cfg, GemmList& l, int nblocks, int cus, hipStream_t stream) {
    switch (cfg) {
        case GEMM_CFG_128_PIPE: return launch_one<128, 128, 2, 2, EPI, 0>(l, nblocks, stream);
        case GEMM_CFG_256_PIPE: return launch_one<256, 256, 2, 4, EPI, 0>(l, nblocks, stream);
        case GEMM_CFG_256_PINGPONG: {
            // Split the tiles of a last round that would fill at most a quarter of the CUs (a 128x128 tile takes about 0.6 of
            // the time of a 256x256 one, so one round of quarters beats a round of whole tiles).
            const int rest = nblocks % cus;
            if (nblocks > cus && rest > 0 && rest <= cus / 4) return launch_pp_tail<EPI>(l, nblocks, rest, stream);
            return launch_one<256, 256, 2, 4, EPI, 1>(l, nblocks, stream);
        }
        case GEMM_CFG_128_PINGPONG: return launch_one<128, 128, 2, 4, EPI, 1>(l, nblocks, stream);
        case GEMM_CFG_64_DEEP:
            if constexpr (EPI == EPI_BX_UPD || EPI == EPI_BX_UPD_T) return hipErrorInvalidValue;  // the launcher takes 128-tiles
            else return launch_deep<EPI>(l, nblocks, stream);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_epi(int epi, int cfg, GemmList& l, int nblocks, int cus, hipStream_t stream) {
    switch (epi) {
        case EPI_SYRK: return launch_cfg<EPI_SYRK>(cfg, l, nblocks, cus, stream);
        case EPI_SYMPOLY: return launch_cfg<EPI_SYMPOLY>(cfg, l, nblocks, cus, stream);
        case EPI_BX: return launch_cfg<EPI_BX>(cfg, l, nblocks, cus, stream);
        case EPI_BX_UPD: return launch_cfg<EPI_BX_UPD>(cfg, l, nblocks, cus, stream);
        case EPI_BX_UPD_T: return launch_cfg<EPI_BX_UPD_T>(cfg, l, nblocks, cus, stream);
        case EPI_MMT: return launch_cfg<EPI_MMT>(cfg, l, nblocks, cus, stream);
        default: return hipErrorInvalidValue;
    }
}

// Workgroups of one launch that cuts C into square tiles of `tile`, or (a.X + B.X) into tiles of `height` x `tile`.
long count_tiles(const GemmItem& it, int tile, int height = 0) {
    const long tm = (it.g.rows + (height ? height : tile) - 1) / (height ? height : tile), tn = (it.g.cols + tile - 1) / tile;
    return (epi_is_bx(it.epi) ? tm * tn : tm * (tm + 1) / 2) * it.g.batch;
}

// Whether whole tiles of height x width cover C without leaving the storage of an operand: row blocks of 256 and, along a row,
// whole column blocks.
bool tiles_fit(const GemmItem& it, int height, int width) {
    const GemmArgs& g = it.g;
    auto up = [](int v, int m) { return (v + m - 1) / m * m; };
    if (up(g.rows, height) > up(g.rows, BLK_ROWS)) return false;
    // (the two-stage kernels read blocked operands only)
    if (it.epi == EPI_MMT && g.dense_pitch && (it.cfg == GEMM_CFG_128_PIPE || it.cfg == GEMM_CFG_256_PIPE)) return false;
    if (it.epi == EPI_MMT) return g.rows % height == 0 && g.dense_rows <= g.rows && g.dense_rows > g.rows - 128;
    if (!epi_is_bx(it.epi)) return g.rows % height == 0 && g.rows <= g.cbC * BLK_COLS;
    const int cols = up(g.cols, width);
    return cols <= g.cbC * BLK_COLS && cols <= g.cbQ * BLK_COLS && cols <= g.cbEt * BLK_COLS;
}

// Tile height of the persistent a.X + B.X for a matrix of `rows` rows: the one that covers the fewest, the tallest among equals.
// The storage of a matrix is whole row blocks of 256; a tile may overhang into it, but not past it.  The overhang reads and
// writes storage that no other product takes for anything: its values never meet a row of the matrix, because every reduction
// ends at the matrix's own extent in whole 128-tiles.
int ppx_height(int rows) {
    const int storage = (rows + 255) / 256 * 256;
    int best = 256, cover = storage;
    for (int h : {224, 192}) {
        const int c = (rows + h - 1) / h * h;
        if (c < cover) best = h, cover = c;
    }
    return best;
}

}  // namespace

int gemm_cfg_tile(int cfg) {
    switch (cfg) {
        case GEMM_CFG_64_DEEP: return 64;
        case GEMM_CFG_128_PIPE:
        case GEMM_CFG_128_PINGPONG: return 128;
        case GEMM_CFG_256_PIPE:
        case GEMM_CFG_256_PINGPONG:
        case GEMM_CFG_256_PERSIST: return 256;
        default: return 0;
    }
}

#ifndef PPX_SYRK_MAXK
#define PPX_SYRK_MAXK 2048
#endif
#ifndef PPX_SYMPOLY_MAXK
#define PPX_SYMPOLY_MAXK 2048
#endif
hipError_t machine_shape(MachineShape& ms) {
    constexpr int kMaxDevices = 64;
    static std::atomic<int> cached[kMaxDevices];  // compute units per device ordinal, 0 = not read yet
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
    int cus = (dev >= 0 && dev < kMaxDevices) ? cached[dev].load(std::memory_order_relaxed) : 0;
    if (cus == 0) {
        if (hipError_t e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev); e != hipSuccess) return e;
        if (cus <= 0) return hipErrorInvalidDevice;
        if (dev >= 0 && dev < kMaxDevices) cached[dev].store(cus, std::memory_order_relaxed);
    }
    ms.cus = cus;
    int xcds = cus / 32;  // 32 active compute units per XCD on gfx950
    ms.xcd_shift = 0;
    while ((2 << ms.xcd_shift) <= xcds && (2 << ms.xcd_shift) <= GEMM_MAX_XCDS && cus % (2 << ms.xcd_shift) == 0) ++ms.xcd_shift;
    return hipSuccess;
}

namespace {

// The launches of products with the configurations chosen[0..n).
int place_launches(const GemmItem* items, int n, bool adapt, int cus, const int* chosen, GemmRoute* route) {
    int cfg[GEMM_MAX_LIST];
    bool done[GEMM_MAX_LIST] = {};
    int launches = 0;
    std::copy(chosen, chosen + n, cfg);
    for (int i = 0; i < n; ++i)
        if (cfg[i] == GEMM_CFG_64_DEEP && epi_fold_mode(items[i].epi)) cfg[i] = GEMM_CFG_128_PINGPONG;
    // The persistent kernel: more tiles than compute units, and products with at least 8 k-tiles and a counter buffer; one launch
    // per tile height.  Short sides that are an odd number of 128-tiles take it for a.X + B.X, with tiles of their own height:
    // the loops of 128-tiles are bound by the LDS (six fragment reads per eight MFMAs against twelve per 32).  Measured, us per
    // product, 128-tiles | this: 72 of 896 x 4864 713 | 525 (224 rows; 570 with 256), 60 of 640 x 2560 190 | 155 (224), 27 of
    // 1152 x 4304 362 | 289 (192; 304 with 224), 150 of 384 x 1536 128 | 104 (192); a single row of tiles (200 of 256 x 1024)
    // 57 | 60.
    for (int epi : {EPI_SYRK, EPI_SYMPOLY, EPI_BX}) {
        for (int h : {256, 224, 192}) {
            int from[GEMM_MAX_LIST], m = 0;
            long blocks = 0, area = 0, shortest = 0x7fffffff;  // tiles, elements of C that they cover, the shortest reduction
            bool odd = false;
            for (int i = 0; i < n; ++i) {
                const GemmArgs& g = items[i].g;
                if (done[i] || items[i].epi != epi || g.kdim < 256 || !g.ppx || !tiles_fit(items[i], h, 256)) continue;
                if (cfg[i] == GEMM_CFG_256_PERSIST) {
                    if (h != 256 || (epi != EPI_BX && g.kdim > (epi == EPI_SYRK ? PPX_SYRK_MAXK : PPX_SYMPOLY_MAXK))) continue;
                } else {
                    if (!adapt || cfg[i] != GEMM_CFG_128_PINGPONG || epi != EPI_BX || g.rows < 384 || h != ppx_height(g.rows)) continue;
                    odd = true;
                }
                const long t = count_tiles(items[i], 256, h);
                if (blocks + t > 0x7fffffffL) continue;
                from[m++] = i;
                blocks += t;
                area += (long)g.rows * g.cols * g.batch;
                if (g.kdim < shortest) shortest = g.kdim;
            }
            if (blocks <= cus) continue;
            // A few rounds with a nearly empty last one: the one-tile kernel cuts that round's tiles into quarters (264 tiles of
            // 1000 x 2731 43 us against 52, 792 tiles 102 against 107; 1200 tiles of 512 x 1408 111 against 105).
            const long rest = blocks % cus, rounds = (blocks + cus - 1) / cus;
            if (!odd && adapt && rest > 0 && rest <= cus / 4 && blocks <= 4L * cus) continue;
            // Tiles of odd heights have no quarters, and their overhang is computed for nothing: 128-tiles unless the elements of
            // the matrices fill 70 % of the rounds, and a k-tile's share more for the epilogue, which short reductions show.
            // Measured on 785 batches of 384 to 2688 rows: 28 of the 590 that come here are slower than on 128-tiles, by 9 % at
            // most, and 24 of the others would have been faster here, by as much (three quarters of the tiles instead of the
            // elements took 72 that were slower, by up to 20 %: 16 of 1408 x 1408, 63 % full, 94 us on 128-tiles and 106 here; 20
            // of 1152 x 1152, 70 %, 69 and 75; 608 tiles of 896 x 4864, 79 %, 74 and 70).
            if (odd && area < (0.7 + 32.0 / shortest) * (256.0 * h) * rounds * cus) continue;
            for (int k = 0; k < m; ++k) {
                route[from[k]] = GemmRoute{GEMM_CFG_256_PERSIST, h, launches};
                done[from[k]] = true;
            }
            ++launches;
        }
    }
    for (int i = 0; i < n; ++i)
        if (cfg[i] == GEMM_CFG_256_PERSIST) cfg[i] = GEMM_CFG_256_PINGPONG;
    for (int i = 0; i < n; ++i) {  // one launch per kind and configuration
        if (done[i]) continue;
        const int tile = gemm_cfg_tile(cfg[i]);
        long blocks = 0;
        for (int k = i; k < n; ++k) {
            if (done[k] || cfg[k] != cfg[i] || items[k].epi != items[i].epi) continue;
            if (items[k].g.rows % tile || !tiles_fit(items[k], tile, tile)) return -1;
            const long t = count_tiles(items[k], tile);
            if (blocks > 0 && blocks + t > 0x7fffffffL) continue;  // goes with a later launch
            blocks += t;
            route[k] = GemmRoute{cfg[k], tile, launches};
            done[k] = true;
        }
        ++launches;
    }
    return launches;
}

}  // namespace

int plan_gemm_nt(const GemmItem* items, int n, bool adapt, int cus, GemmRoute* route) {
    if (n < 1 || n > GEMM_MAX_LIST) return -1;
    int cfg[GEMM_MAX_LIST];
    long all128 = 0, own128 = 0, all64 = 0;
    bool fold = false;
    for (int i = 0; i < n; ++i) {
        cfg[i] = items[i].cfg;
        if (gemm_cfg_tile(cfg[i]) == 0) return -1;
        all128 += count_tiles(items[i], 128);
        if (gemm_cfg_tile(cfg[i]) == 256) own128 += count_tiles(items[i], 128);
        all64 += count_tiles(items[i], 64);
        fold |= epi_fold_mode(items[i].epi) != 0;
    }
    // Smaller tiles for launches that would not fill the machine (every configuration sums in the same order, so the result
    // does not depend on the choice).  Measured on one to 48 matrices of 128 to 5120 rows, times per k-tile of 32 columns: a
    // round of 256-tiles (one workgroup per compute unit) 460 ns, of 128-tiles 157 ns alone on a compute unit and 336 ns for
    // two.  So 128-tiles win while they need no more than the two places per compute unit (X.Xt of 2048 x 5632: 84 -> 36 us,
    // of 3072 x 8192 with 300 tiles 119 -> 91) and lose beyond (4096 x 4096 with 528: 68 -> 76); 64-tiles win while each has
    // a compute unit of its own (896 x 4864: 30 -> 18) and lose with two (512 x 1408 x 8, 288 tiles: 11.7 -> 14.0).
    if (adapt) {
        for (int i = 0; i < n; ++i) {
            if (gemm_cfg_tile(cfg[i]) == 256 && own128 <= 2 * cus) cfg[i] = GEMM_CFG_128_PINGPONG;
            if (all128 <= 2 * cus && all64 <= cus && !fold) cfg[i] = GEMM_CFG_64_DEEP;
        }
    }
    // Matrices of 129 to 256 rows (keys and values beside large weights) run on 128-tiles by themselves, after the launch of the large ones and
    // on a few compute units.  Beside 256-tiles they go along, one tile a row of blocks, while that launch has eight times as many.  Steps, us,
    // apart | along: 6 layers of 1000 x 1000, 200 x 1000 and 2731 x 1000 1638 | 1511, 12 of 768, 192 and 2048 1657 | 1520, 2 of 2048, 256 and
    // 5632 3182 | 3018, 12 of 1024, 256 and 2816 3015 | 2901, 8 of 2048, 256 and 5632 (32 such matrices in 72 rounds) 10899 | 10895.
    bool along[GEMM_MAX_LIST] = {};
    for (int epi : {EPI_SYRK, EPI_SYMPOLY, EPI_BX, EPI_BX_UPD, EPI_BX_UPD_T}) {
        long large = 0, more = 0;
        bool short_side[GEMM_MAX_LIST] = {};
        for (int i = 0; i < n; ++i) {
            if (!adapt || items[i].epi != epi) continue;
            if (gemm_cfg_tile(cfg[i]) == 256) large += count_tiles(items[i], 256);
            else if (cfg[i] == GEMM_CFG_128_PINGPONG && items[i].g.rows == 256 && items[i].g.kdim >= 256 && tiles_fit(items[i], 256, 256))
                short_side[i] = true, more += count_tiles(items[i], 256);
        }
        for (int i = 0; i < n && 8 * more <= large; ++i)
            if (short_side[i]) cfg[i] = GEMM_CFG_256_PERSIST, along[i] = true;
    }
    // Large matrices and those that were to go along need not end in one launch (the persistent symmetric products take reductions of up to
    // PPX_SYRK_MAXK columns): what has too few large ones beside it in its own launch goes back to its 128-tiles.  A step over 100 of 1024 x
    // 2048 with 4 of 256 x 12288, whose four tiles of X.Xt were left alone like that: 5314 us, so 4977.
    for (;;) {
        const int launches = place_launches(items, n, adapt, cus, cfg, route);
        bool alone = false;
        for (int k = 0; k < launches; ++k) {
            long large = 0, more = 0;
            for (int i = 0; i < n; ++i)
                if (route[i].launch == k && gemm_cfg_tile(cfg[i]) == 256) (along[i] ? more : large) += count_tiles(items[i], 256);
            for (int i = 0; i < n && 8 * more > large; ++i)
                if (along[i] && route[i].launch == k) cfg[i] = GEMM_CFG_128_PINGPONG, along[i] = false, alone = true;
        }
        if (!alone) return launches;
    }
}

bool plan_flow(FlowList& l, int xcds, bool recorded) {
    l.groups = xcds;
    if (l.n < 1 || l.n > GEMM_MAX_LIST || xcds < 1 || xcds > GEMM_MAX_XCDS || l.steps < 1) return false;
    // Dearest matrices first, each to the group with the least work so far.  Work in k-tiles of 32 columns, the start and the
    // epilogue of a tile as twelve more.
    double load[GEMM_MAX_XCDS] = {}, cost[GEMM_MAX_LIST], mean = 0, most = 0, chain = 0;
    int order[GEMM_MAX_LIST];
    for (int i = 0; i < l.n; ++i) {
        FlowEntry& e = l.e[i];
        const double tm = e.Mp / 128, tn = e.Kr / 128, tri = tm * (tm + 1) / 2;
        if (tm * tn > 0xffff) return false;
        e.sym = (int)tri;
        e.rect = (int)(tm * tn);
        cost[i] = tri * (4 * tn + 12) + (tri + tm * tn) * (4 * tm + 12);
        chain = std::max(chain, 4 * tn + 8 * tm + 36);
        mean += cost[i] * e.batch / xcds;
        order[i] = i;
    }
    std::stable_sort(order, order + l.n, [&](int x, int y) { return cost[x] > cost[y]; });
    for (int k = 0; k < l.n; ++k) {
        FlowEntry& e = l.e[order[k]];
        int count[GEMM_MAX_XCDS];
        for (int g = 0; g < xcds; ++g) {
            count[g] = e.batch / xcds;
            load[g] += cost[order[k]] * count[g];
        }
        for (int r = e.batch % xcds; r > 0; --r) {
            const int least = (int)(std::min_element(load, load + xcds) - load);
            ++count[least];
            load[least] += cost[order[k]];
        }
        e.first[0] = 0;
        for (int g = 0; g < xcds; ++g) e.first[g + 1] = e.first[g] + count[g];
    }
    for (int g = 0; g < xcds; ++g) {
        long sym = 0, rect = 0;
        for (int i = 0; i < l.n; ++i) {
            const FlowEntry& e = l.e[i];
            sym += (long)(e.first[g + 1] - e.first[g]) * e.sym;
            rect += (long)(e.first[g + 1] - e.first[g]) * e.rect;
        }
        if ((2 * sym + rect) * l.steps > 0x3fffffffL) return false;  // (what is asked for past the end stays below 2^31)
        l.sym[g] = (int)sym;
        l.rect[g] = (int)rect;
        most = std::max(most, load[g]);
    }
    // The XCD with the most work and, where there is little, the chain of one matrix through an iteration set the time of one launch;
    // launches of their own share the work evenly but pay for each other's last rounds.  Measured on 500 sets of one to four shapes of 65
    // to 1536 rows, 2 to 800 matrices (recorded steps, profiles/flow_chain_or_launches.txt): the line below takes 298 of them, 13 % faster in
    // the mean (up to 32 %) and 3 slower by more than 3 % (5 % at most); of the 141 others below it 21 would be faster by more than 3 %,
    // and all of them 12 % slower in the mean.  Beyond `mean` of 30000 the 256-tiles of large launches are worth what is lost between them.
    // (The figures are of XCDs of 32 compute units, which gfx950 has however it is partitioned.)
    if (mean < 30000 && most < 1.35 * mean - 15 * chain + 600) return true;
    // A step over very little takes longer on the device, but the caller waits for his own 14 launches less.  Sets of 2 to 24 matrices of 129 x
    // 129 to 256 x 768, steps one behind the other, one launch | a launch per product: with gradient clipping and an AdamW group around them, where
    // the host sets the pace, 126 to 148 us | 156 to 177; alone, where the device does, 98 to 119 | 84 to 105.  The former are training
    // iterations.  A step that is being recorded has no such launches when it is replayed.
    return !recorded && l.e[0].p_ptrs && l.p_dtype != GEMM_UPD_RESULT && 0.032 * most + 0.64 * chain + 55 < 120;
}

hipError_t launch_flow(const FlowList& l, hipStream_t stream) {
    MachineShape ms;
    if (hipError_t e = machine_shape(ms); e != hipSuccess) return e;
    constexpr int smem = kFlowStages + (int)sizeof(FlowSlot);
    static std::atomic<unsigned long long> configured{0};
    if (hipError_t e = allow_dynamic_lds((const void*)gemm_nt_flow_kernel, smem, configured); e != hipSuccess) return e;
    // two workgroups per compute unit, but no more than have something to do: the others would only poll
    int most = 1;
    for (int g = 0; g < l.groups; ++g) most = std::max(most, l.sym[g] + l.rect[g]);
    hipLaunchKernelGGL(gemm_nt_flow_kernel, dim3(l.groups * std::min(2 * ms.cus / l.groups, most)), dim3(512), smem, stream, l);
    return hipGetLastError();
}

hipError_t launch_gemm_nt(const GemmItem* items, int n, bool adapt, hipStream_t stream) {
    MachineShape ms;
    if (hipError_t e = machine_shape(ms); e != hipSuccess) return e;
    GemmRoute route[GEMM_MAX_LIST];
    const int launches = plan_gemm_nt(items, n, adapt, ms.cus, route);
    if (launches < 0) return hipErrorInvalidValue;
    for (int k = 0; k < launches; ++k) {
        GemmList l;
        l.n = 0;
        l.xcd_shift = ms.xcd_shift;
        l.big_blocks = 0;
        l.start[0] = 0;
        int epi = 0, cfg = 0, height = 0;
        for (int i = 0; i < n; ++i) {
            if (route[i].launch != k) continue;
            epi = items[i].epi;
            cfg = route[i].cfg;
            height = route[i].height;
            const int width = gemm_cfg_tile(cfg);
            const long t = count_tiles(items[i], width, height);
            GemmArgs& g = l.g[l.n];
            g = items[i].g;
            if (g.upd_dtype == GEMM_UPD_RESULT && cfg != GEMM_CFG_128_PINGPONG) return hipErrorInvalidValue;
            g.tiles_m = (g.rows + height - 1) / height;
            g.tiles_n = (g.cols + width - 1) / width;
            g.tiles_per_mat = (int)(t / g.batch);
            l.start[l.n + 1] = l.start[l.n] + (int)t;
            ++l.n;
        }
        const int blocks = l.start[l.n];
        hipError_t e;
        if (cfg != GEMM_CFG_256_PERSIST) e = launch_epi(epi, cfg, l, blocks, ms.cus, stream);
        else if (epi == EPI_SYRK) e = launch_ppx<EPI_SYRK>(l, blocks, ms.cus, stream);
        else if (epi == EPI_SYMPOLY) e = launch_ppx<EPI_SYMPOLY>(l, blocks, ms.cus, stream);
        else if (height == 256) e = launch_ppx<EPI_BX>(l, blocks, ms.cus, stream);
        else if (height == 224) e = launch_ppx<EPI_BX, 8, 6>(l, blocks, ms.cus, stream);
        else e = launch_ppx<EPI_BX, 6, 6>(l, blocks, ms.cus, stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
