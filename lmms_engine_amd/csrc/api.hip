// C ABI of libmuon_hip.so (declared in include/muon_hip.h): argument checks, workspace
// partitioning, the grouped launch sequence of one Muon step, and per-kernel event timing.
#include <stdarg.h>
#include <stdio.h>
#include <algorithm>
#include <atomic>
#include <mutex>
#include <vector>

// The library is built with hidden visibility; the entry points declared in the public header are what it exports.
#pragma GCC visibility push(default)
#include "../../include/muon_hip.h"
#pragma GCC visibility pop
#include "common.h"
#include "elementwise.h"
#include "gemm_nt.h"
#include "multi_tensor.h"
#include "small_chain.h"

namespace {

thread_local char g_err[512] = "";
std::atomic<int> g_forced_cfg{MUON_HIP_CFG_AUTO};  // benchmarking override, read once per call

int fail(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

int hip_fail(hipError_t e, const char* what) {
    snprintf(g_err, sizeof(g_err), "%s: %s", what, hipGetErrorString(e));
    return (int)e;
}

// ---- timing ------------------------------------------------------------------------
// Event pairs come from a pool that muon_hip_timing_reserve fills ahead of the region to be measured, so that a timed
// launch costs two hipEventRecord calls and one atomic increment: no event is created and no lock is taken while the
// clock runs.  A launch that finds the pool empty goes untimed and is counted in g_untimed.
struct EventPair {
    hipEvent_t start, stop;
    int kid;
};
std::mutex g_tmu;                    // guards the pool's growth and the read-out, never a launch
std::atomic<bool> g_timing{false};
// The pool grows in chunks that are never moved or freed, so a launch may index it while another thread adds a chunk.
constexpr size_t kPoolChunk = 4096, kPoolChunks = 256, kMaxPool = kPoolChunk * kPoolChunks;
EventPair* g_chunks[kPoolChunks] = {};
std::atomic<size_t> g_pool_size{0};  // pairs that exist
std::atomic<size_t> g_used{0};       // pairs handed out since timing was enabled
std::atomic<long> g_untimed{0};
inline EventPair& pool_at(size_t i) { return g_chunks[i / kPoolChunk][i % kPoolChunk]; }

int grow_pool(size_t want) {  // under g_tmu
    if (want > kMaxPool) want = kMaxPool;
    for (size_t i = g_pool_size.load(std::memory_order_relaxed); i < want; ++i) {
        if (i % kPoolChunk == 0 && !g_chunks[i / kPoolChunk]) g_chunks[i / kPoolChunk] = new EventPair[kPoolChunk]();
        EventPair& p = pool_at(i);
        if (hipError_t e = hipEventCreate(&p.start); e != hipSuccess) return hip_fail(e, "hipEventCreate");
        if (hipError_t e = hipEventCreate(&p.stop); e != hipSuccess) {
            (void)hipEventDestroy(p.start);
            return hip_fail(e, "hipEventCreate");
        }
        g_pool_size.store(i + 1, std::memory_order_release);
    }
    return 0;
}

// Whether what is launched on the stream goes into a graph (or cannot be told to be launched now).
bool is_recorded(hipStream_t s) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cap) == hipSuccess) return cap != hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return true;
}

struct Timed {
    EventPair* ev;
    hipStream_t s;
    Timed(int kid, hipStream_t st) : ev(nullptr), s(st) {
        if (!g_timing.load(std::memory_order_acquire)) return;
        // a launch that is being recorded into a graph has no time of its own: its events would become graph nodes
        if (is_recorded(s)) {
            g_untimed.fetch_add(1, std::memory_order_relaxed);
            return;
        }
        const size_t i = g_used.fetch_add(1, std::memory_order_relaxed);
        if (i >= g_pool_size.load(std::memory_order_acquire)) {
            g_untimed.fetch_add(1, std::memory_order_relaxed);
            return;
        }
        ev = &pool_at(i);
        ev->kid = kid;
        if (hipEventRecord(ev->start, s) != hipSuccess) ev->kid = -1;
    }
    ~Timed() {
        if (ev && ev->kid >= 0 && hipEventRecord(ev->stop, s) != hipSuccess) ev->kid = -1;
    }
};

// ---- chains that were given up ---------------------------------------------------------
// A word of host memory per device, a line each, that a chain in one launch sets when it gives up a wait (gemm_nt.h).  Allocated with the
// first such launch and never freed: kernels may hold its address.
constexpr int kAlarmDevices = 64, kAlarmLine = 16;
constexpr unsigned kChainPolls = 1u << 27;  // some minutes
thread_local unsigned g_chain_polls = kChainPolls;
std::mutex g_alarm_mu;
std::atomic<unsigned*> g_alarm{nullptr};

int chain_alarm(unsigned** word) {
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return hip_fail(e, "hipGetDevice");
    if (dev >= kAlarmDevices) return fail(MUON_HIP_EINVAL, "device %d", dev);
    unsigned* p = g_alarm.load(std::memory_order_acquire);
    if (!p) {
        std::lock_guard<std::mutex> lock(g_alarm_mu);
        if (p = g_alarm.load(std::memory_order_relaxed); !p) {
            hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;  // (the launch may be one that is being recorded)
            (void)hipThreadExchangeStreamCaptureMode(&mode);
            const hipError_t e = hipHostMalloc((void**)&p, kAlarmDevices * kAlarmLine * sizeof(unsigned),
                                               hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent);
            (void)hipThreadExchangeStreamCaptureMode(&mode);
            if (e != hipSuccess) return hip_fail(e, "hipHostMalloc");
            std::fill(p, p + kAlarmDevices * kAlarmLine, 0u);
            g_alarm.store(p, std::memory_order_release);
        }
    }
    *word = p + dev * kAlarmLine;
    return 0;
}

// Reports an abandoned chain of the current device, once.
int chain_status() {
    unsigned* p = g_alarm.load(std::memory_order_acquire);
    int dev = 0;
    if (!p || hipGetDevice(&dev) != hipSuccess || dev >= kAlarmDevices) return 0;
    p += dev * kAlarmLine;
    if (!__atomic_load_n(p, __ATOMIC_RELAXED) || !__atomic_exchange_n(p, 0u, __ATOMIC_ACQ_REL)) return 0;
    return fail(MUON_HIP_ECHAIN, "an earlier chain of Newton-Schulz iterations on device %d gave up waiting for its own tiles: the parameters or "
                                 "results of that call are incomplete", dev);
}

// ---- geometry / workspace ------------------------------------------------------------
struct Plan {
    int rows, cols, batch, M, K, Mp, Kp, tile, nparts;
    int Kr;  // K in whole 128-tiles: the extent that the products work on; Kp, the extent of the storage, may be larger
    bool transposed;
    bool small;  // the whole chain runs in one workgroup per matrix (small_chain.hip) instead of as tiled products
    long n, strideU, strideX, strideA;  // elements per matrix: U dense, the others blocked
    size_t offX[2], offA, offB, offParts, offDenom, offCtr, ctrBytes, total;
};

inline long round_up(long v, long m) { return (v + m - 1) / m * m; }

// Tile edge for a matrix whose short side is M: 256 when M, padded to 128-tiles, is a whole number of 256-tiles.
bool use_tile256(int M) { return M >= 512 - 127 && round_up(M, 128) % 256 == 0; }

// A configuration, and whether the launcher may replace it by one with smaller tiles where a launch has too few (it may not
// when the caller has named it).
struct Cfg {
    int id;
    bool adapt;
};

// Configuration per kernel, from a sweep of every variant over the benchmark shapes: the ping-pong kernel
// everywhere, on 256-tiles where they fill the machine and on 128-tiles (two workgroups per compute unit) for
// short sides that, in whole 128-tiles, are no whole number of 256-tiles (for a.X + B.X the launcher has tiles of other heights
// for those) and for the symmetric products of matrices up to 512 rows.
Cfg pick_cfg(int M, int epi = EPI_BX) {
    const int forced = g_forced_cfg.load(std::memory_order_relaxed);
    if (forced >= 0) return {forced, false};
    if (!use_tile256(M)) return {GEMM_CFG_128_PINGPONG, true};
    if (epi != EPI_BX && M <= 512) return {GEMM_CFG_128_PINGPONG, true};
    // The persistent kernel where the launcher takes it: a.X + B.X, and the symmetric products with reductions of at
    // most 2048 (past that a tile is long enough that what the persistent kernel removes around it no longer shows in
    // a step that runs at the power limit); launches of at most one round of tiles and those that carry the parameter
    // update run the one-tile ping-pong kernel.
    return {GEMM_CFG_256_PERSIST, true};
}

// Where the counters of a bucket lie in their segment of its workspace.
constexpr size_t kCtrFlow = GEMM_PPX_COUNTER_BYTES, kCtrMatrix = kCtrFlow + GEMM_FLOW_CONTROL_BYTES;

int make_plan(int rows, int cols, int batch, Plan& p) {
    if (rows <= 0 || cols <= 0 || batch <= 0) return fail(MUON_HIP_EINVAL, "rows, cols and batch must be positive");
    if (batch > 65535) return fail(MUON_HIP_ESHAPE, "batch %d exceeds 65535 matrices per call", batch);
    p.rows = rows;
    p.cols = cols;
    p.batch = batch;
    p.transposed = rows > cols;
    p.M = rows < cols ? rows : cols;
    p.K = rows < cols ? cols : rows;
    const Cfg cfg = pick_cfg(p.M);
    // a configuration that the caller has named is one of the tiled kernels; without one launch for many matrices those take the larger ones
    p.small = cfg.adapt && chain_fits(p.M, p.K) && (p.M <= 64 || g_forced_cfg.load(std::memory_order_relaxed) == MUON_HIP_CFG_AUTO);
    p.tile = gemm_cfg_tile(cfg.id);
    if (p.tile == 0) return fail(MUON_HIP_EINVAL, "unknown GEMM configuration");
    if (p.tile < 128) p.tile = 128;  // the elementwise kernels move whole 128-tiles
    p.Mp = (int)round_up(p.M, p.tile);
    p.Kr = (int)round_up(p.K, 128);
    // whole tiles of the configuration, and the persistent a.X + B.X has tiles 256 wide whatever their height
    p.Kp = (int)round_up(p.K, p.Mp >= 384 ? 256 : p.tile);
    p.n = (long)rows * cols;
    p.strideU = round_up(p.n, 8);
    p.strideX = blocked_elems(p.Mp, p.Kp);
    p.strideA = blocked_elems(p.Mp, p.Mp);
    p.nparts = momentum_parts(p.n);
    const long T = p.Mp / 128, TN = p.Kp / 128;
    if (T * TN * batch > 0x7fffffffL) return fail(MUON_HIP_ESHAPE, "too many tiles for one launch");
    size_t off = 0;
    auto seg = [&](size_t bytes) {
        size_t o = off;
        off += (size_t)round_up((long)bytes, 256);
        return o;
    };
    const size_t xb = (size_t)batch * p.strideX * 2;
    const size_t ab = (size_t)batch * p.strideA * 2;
    p.offX[0] = seg(xb);
    p.offX[1] = seg(xb);  // doubles as U (the blend in the parameter's layout) before the first iteration
    p.offA = seg(ab);
    p.offB = seg(ab);
    p.offParts = seg((size_t)batch * p.nparts * sizeof(float));
    p.offDenom = seg((size_t)batch * sizeof(float));
    // counters, cleared by the normalisation stage: of the persistent kernels, of the chain in one launch, one line per matrix
    p.ctrBytes = kCtrMatrix + (size_t)batch * GEMM_FLOW_LINE * sizeof(unsigned);
    p.offCtr = seg(p.ctrBytes);
    p.total = off;
    return 0;
}

// Where `steps` iterations leave X.  The one-workgroup chain leaves it in the first buffer whatever their number: the other
// holds the blend that workgroups of other matrices may still have to read.
size_t result_offset(const Plan& p, int steps) { return p.small && steps > 0 ? p.offX[0] : p.offX[steps & 1]; }

inline bf16_t* wsp(void* ws, size_t off) { return (bf16_t*)((char*)ws + off); }

int check_ws(const void* ws) {
    if (!ws) return fail(MUON_HIP_EINVAL, "workspace is null");
    if (((uintptr_t)ws) & 255) return fail(MUON_HIP_EINVAL, "workspace must be 256-byte aligned");
    return 0;
}

int check_counters(const void* counters) {
    if (((uintptr_t)counters) & 63) return fail(MUON_HIP_EINVAL, "the counter buffer must be 64-byte aligned");
    return 0;
}

int check_gemm(int cfg, int Mp, int Kp, int batch, int& tile) {
    tile = gemm_cfg_tile(cfg);
    if (tile == 0) return fail(MUON_HIP_EINVAL, "unknown GEMM configuration %d", cfg);
    if (Mp <= 0 || Kp <= 0 || batch <= 0) return fail(MUON_HIP_EINVAL, "sizes must be positive");
    const int edge = tile < 128 ? 128 : tile;  // every kernel's reduction is a multiple of 128
    if (Mp % edge || Kp % edge) return fail(MUON_HIP_ESHAPE, "Mp=%d, Kp=%d must be multiples of the %d tile", Mp, Kp, edge);
    const long T = Mp / tile, TN = Kp / tile;
    if (T * TN * batch > 0x7fffffffL) return fail(MUON_HIP_ESHAPE, "too many tiles for one launch");
    return 0;
}

// The three products on blocked buffers; matrix b of a batch starts at b * blocked_elems(rows, cols).
// Kr: the columns of X that hold the matrix, in whole 128-tiles; Kp: the columns of its storage.
GemmItem syrk_item(int cfg, const bf16_t* X, bf16_t* A, int Mp, int Kr, int Kp, int batch, unsigned* ppx) {
    GemmItem it = {};
    GemmArgs& g = it.g;
    it.cfg = cfg;
    it.epi = EPI_SYRK;
    g.P = g.Q = X;
    g.strideP = g.strideQ = blocked_elems(Mp, Kp);
    g.cbP = Kp / BLK_COLS;
    g.kdim = Kr;
    g.rows = g.cols = Mp;
    g.batch = batch;
    g.C = g.Ct = A;
    g.strideC = g.strideCt = blocked_elems(Mp, Mp);
    g.cbC = g.cbCt = Mp / BLK_COLS;
    g.ppx = ppx;
    return it;
}

GemmItem sympoly_item(int cfg, const bf16_t* A, bf16_t* B, int Mp, int batch, double b, double c, unsigned* ppx) {
    GemmItem it = {};
    GemmArgs& g = it.g;
    it.cfg = cfg;
    it.epi = EPI_SYMPOLY;
    g.P = g.Q = A;
    g.strideP = g.strideQ = blocked_elems(Mp, Mp);
    g.cbP = Mp / BLK_COLS;
    g.kdim = Mp;
    g.rows = g.cols = Mp;
    g.batch = batch;
    g.C = g.Ct = B;
    g.strideC = g.strideCt = blocked_elems(Mp, Mp);
    g.cbC = g.cbCt = Mp / BLK_COLS;
    g.Et = A;
    g.strideEt = blocked_elems(Mp, Mp);
    g.cbEt = Mp / BLK_COLS;
    g.s0 = (float)b;
    g.s1 = (float)c;
    g.ppx = ppx;
    return it;
}

// What the last B.X of a step does to the parameters (which are X's image when rows <= cols, its transpose otherwise).
struct UpdateArgs {
    int p_dtype;
    double lr, weight_decay;
};

GemmItem bx_item(int cfg, const bf16_t* B, const bf16_t* X, bf16_t* Xout, int Mp, int Kr, int Kp, int batch, double a, unsigned* ppx) {
    GemmItem it = {};
    GemmArgs& g = it.g;
    it.cfg = cfg;
    it.epi = EPI_BX;
    g.P = B;
    g.strideP = blocked_elems(Mp, Mp);
    g.Q = X;
    g.strideQ = blocked_elems(Mp, Kp);
    g.cbQ = Kp / BLK_COLS;
    g.cbP = Mp / BLK_COLS;
    g.kdim = Mp;
    g.rows = Mp;
    g.cols = Kr;
    g.batch = batch;
    g.C = Xout;
    g.strideC = blocked_elems(Mp, Kp);
    g.cbC = Kp / BLK_COLS;
    g.Et = X;
    g.strideEt = blocked_elems(Mp, Kp);
    g.cbEt = Kp / BLK_COLS;
    g.s0 = (float)a;
    g.ppx = ppx;
    return it;
}

void fold_update(GemmItem& it, const void* const* p_ptrs, int rows, int cols, double scale, const UpdateArgs& u) {
    it.epi = rows <= cols ? EPI_BX_UPD : EPI_BX_UPD_T;
    it.g.upd_ptrs = p_ptrs;
    it.g.upd_dtype = u.p_dtype;
    it.g.upd_rows = rows;
    it.g.upd_cols = cols;
    it.g.upd_scale = (float)scale;
    it.g.upd_decay = (float)(1.0 - u.lr * u.weight_decay);
    it.g.upd_alpha = (float)(-u.lr);
}

int launch_items(int kernel_id, const char* what, const GemmItem* items, int n, bool adapt, hipStream_t s) {
    Timed t(kernel_id, s);
    hipError_t e = launch_gemm_nt(items, n, adapt, s);
    return e == hipSuccess ? 0 : hip_fail(e, what);
}

int dtype_ok(int d) { return d == MUON_HIP_F32 || d == MUON_HIP_BF16; }

// The same-shape matrices of one call, each shape with its own part of the workspace.  Every stage is one launch over all of
// them as far as the kernels' configurations allow: a set of a few matrices of several shapes would otherwise leave most of
// the machine idle in every launch, and pay 3 to 5 us of host and device time for each.
struct Bucket {
    Plan p;
    char* ws;
    const void* const* p_ptrs = nullptr;
    const void* const* g_ptrs = nullptr;
    const void* const* m_ptrs = nullptr;
    double scale = 1.0;
    int init(int rows, int cols, int batch, void* workspace) {
        ws = (char*)workspace;
        return make_plan(rows, cols, batch, p);
    }
    size_t clear_bytes = 0;  // counters that the normalisation clears
    bf16_t* at(size_t off) const { return (bf16_t*)(ws + off); }
    unsigned* counters(size_t off) const { return (unsigned*)(ws + p.offCtr + off); }
    EwBucket ew() const {
        return EwBucket{g_ptrs, m_ptrs, at(p.offX[1]), p.strideU, (float*)(ws + p.offParts), (float*)(ws + p.offDenom), at(p.offX[0]),
                        p.strideX, p.rows, p.cols, p.Mp, p.Kp, p.nparts, p.batch, counters(0), (int)(clear_bytes / sizeof(unsigned))};
    }
};
struct Work {
    int n = 0;
    Bucket b[MUON_HIP_MAX_BUCKETS];
};
static_assert(MUON_HIP_MAX_BUCKETS <= GEMM_MAX_LIST && MUON_HIP_MAX_BUCKETS <= EW_MAX_LIST && MUON_HIP_MAX_BUCKETS <= CHAIN_MAX_LIST, "a launch takes every bucket of a call");

int one_bucket(int rows, int cols, int batch, void* workspace, Work& w) {
    w.n = 1;
    if (int rc = w.b[0].init(rows, cols, batch, workspace)) return rc;
    return check_ws(workspace);
}

void ew_list(const Work& w, EwList& l) {
    l.n = w.n;
    for (int i = 0; i < w.n; ++i) l.b[i] = w.b[i].ew();
}

int do_momentum(const Work& w, int g_dtype, int m_dtype, double beta, int nesterov, int write_back_grad, hipStream_t s) {
    for (int i = 0; i < w.n; ++i)
        if (!w.b[i].g_ptrs || !w.b[i].m_ptrs) return fail(MUON_HIP_EINVAL, "pointer table is null");
    const bool combo = (g_dtype == MUON_HIP_F32 && m_dtype == MUON_HIP_F32) ||
                       (g_dtype == MUON_HIP_BF16 && (m_dtype == MUON_HIP_F32 || m_dtype == MUON_HIP_BF16));
    if (!combo) return fail(MUON_HIP_EINVAL, "unsupported (grad, momentum) dtypes (%d, %d)", g_dtype, m_dtype);
    EwList l;
    ew_list(w, l);
    Timed t(MUON_HIP_K_MOMENTUM, s);
    hipError_t e = launch_momentum_norm(l, g_dtype, m_dtype, beta, nesterov, write_back_grad, s);
    return e == hipSuccess ? 0 : hip_fail(e, "momentum_norm launch");
}

// The tile counters of the persistent kernels are those of the first bucket; the normalisation clears them.
unsigned* ppx_counters(const Work& w) { return w.b[0].counters(0); }

int do_normalize(Work& w, bool flow, hipStream_t s) {
    for (int i = 0; i < w.n; ++i) w.b[i].clear_bytes = flow ? w.b[i].p.ctrBytes : i == 0 ? kCtrFlow : 0;
    EwList l;
    ew_list(w, l);
    Timed t(MUON_HIP_K_NORMALIZE, s);
    hipError_t e = launch_normalize(l, s);
    return e == hipSuccess ? 0 : hip_fail(e, "normalize launch");
}

// The products of one stage of an iteration that reads X from buffer `cur`; whether the launcher may choose smaller tiles for
// them (the same for all: a configuration that the caller has named is named for every launch).
bool stage_items(const Work& w, int epi, int cur, double a, double b, double c, unsigned* ppx, GemmItem* items) {
    bool adapt = true;
    for (int i = 0; i < w.n; ++i) {
        const Bucket& k = w.b[i];
        const Plan& p = k.p;
        const Cfg cfg = pick_cfg(p.M, epi);
        adapt = cfg.adapt;
        if (epi == EPI_SYRK) items[i] = syrk_item(cfg.id, k.at(p.offX[cur]), k.at(p.offA), p.Mp, p.Kr, p.Kp, p.batch, ppx);
        else if (epi == EPI_SYMPOLY) items[i] = sympoly_item(cfg.id, k.at(p.offA), k.at(p.offB), p.Mp, p.batch, b, c, ppx);
        else items[i] = bx_item(cfg.id, k.at(p.offB), k.at(p.offX[cur]), k.at(p.offX[cur ^ 1]), p.Mp, p.Kr, p.Kp, p.batch, a, ppx);
    }
    return adapt;
}

// Whether a workgroup each takes the matrices of a bucket: where it holds them.  But short sides beyond 64 cost little among the tiles of larger
// matrices, in one launch or one per product; a launch of their own in front of those would come on top (a step over such a mixture: 161 us
// among the tiles, 231 with a launch of their own).
bool in_workgroups(const Work& w, int i) {
    bool tiles = false;
    for (int k = 0; k < w.n; ++k) tiles |= !w.b[k].p.small;
    return w.b[i].p.small && (w.b[i].p.M <= 64 || !tiles);
}

// The iterations as one launch (gemm_nt.h), where that is the faster way and nobody has named a configuration.
bool flow_of(const Work& w, int steps, double a, double b, double c, const UpdateArgs* upd, bf16_t* out, int xcds, bool recorded, FlowList& l) {
    if (g_forced_cfg.load(std::memory_order_relaxed) != MUON_HIP_CFG_AUTO) return false;
    l.n = w.n;
    l.steps = steps;
    l.a = (float)a;
    l.b = (float)b;
    l.c = (float)c;
    l.p_dtype = upd ? upd->p_dtype : out ? GEMM_UPD_RESULT : 0;
    l.decay = upd ? (float)(1.0 - upd->lr * upd->weight_decay) : 0.f;
    l.alpha = upd ? (float)(-upd->lr) : 0.f;
    l.control = w.b[0].counters(kCtrFlow);
    for (int i = 0; i < w.n; ++i) {
        const Bucket& k = w.b[i];
        const Plan& p = k.p;
        FlowEntry& e = l.e[i];
        for (int x : {0, 1}) e.X[x] = k.at(p.offX[x]);
        e.A = k.at(p.offA);
        e.B = k.at(p.offB);
        e.strideX = p.strideX;
        e.strideA = p.strideA;
        e.Mp = p.Mp;
        e.Kr = p.Kr;
        e.Kp = p.Kp;
        e.batch = p.batch;
        e.done = k.counters(kCtrMatrix);
        e.p_ptrs = upd ? k.p_ptrs : (const void* const*)out;
        e.rows = p.rows;
        e.cols = p.cols;
        e.scale = (float)k.scale;
    }
    return plan_flow(l, xcds, recorded);
}

// The last product of a call that returns X, as one that writes `out` itself, where that is faster; whether it is.
//
// Only tiles of 128 do that.  Those of 256 that carry an epilogue through LDS are slower than the persistent ones by more than the copy takes
// (8192 x 8192: 70 us for 53), and so are 128-tiles of large matrices where the product that writes X is a persistent one of tiles of their own
// height: the difference grows with the reduction, the copy does not.  One iteration, us, copied | written here: 60 of 640 x 2560 486 | 444, 27 of
// 1152 x 4304 833 | 783, 8 of 1664 x 6000 609 | 582, 8 of 1920 x 4096 503 | 503, 8 of 2432 x 2432 520 | 525, 6 of 2944 x 2944 652 | 673, 2 of 4480 x
// 4480 656 | 686, one 8064 x 8064 1773 | 1898.
constexpr int kResultRows = 2048;
bool write_result(const Bucket& k, bool adapt, int cus, bf16_t* out, GemmItem& item) {
    GemmItem direct = item;
    GemmRoute plain, route;
    direct.epi = k.p.rows <= k.p.cols ? EPI_BX_UPD : EPI_BX_UPD_T;
    direct.g.upd_ptrs = (const void* const*)out;
    direct.g.upd_dtype = GEMM_UPD_RESULT;
    direct.g.upd_rows = k.p.rows;
    direct.g.upd_cols = k.p.cols;
    if (!adapt || plan_gemm_nt(&direct, 1, adapt, cus, &route) != 1 || route.cfg != GEMM_CFG_128_PINGPONG) return false;
    if (k.p.Mp > kResultRows && plan_gemm_nt(&item, 1, adapt, cus, &plain) == 1 && plain.cfg == GEMM_CFG_256_PERSIST) return false;
    item = direct;
    return true;
}

// Normalise, then `steps` iterations; with `upd` the last B.X applies the parameter update instead of writing X'.
// `out`: where the result goes, dense (one bucket; null: X).  Where the last product does not write it there, *left_in_x is set.
int ns_chain(const Work& all, int steps, double a, double b, double c, const UpdateArgs* upd, hipStream_t s, bf16_t* out = nullptr,
             bool* left_in_x = nullptr) {
    if (steps < 0) return fail(MUON_HIP_EINVAL, "steps must be >= 0");
    MachineShape ms;
    if (hipError_t e = machine_shape(ms); e != hipSuccess) return hip_fail(e, "device shape");
    Work w;  // the matrices that go through the tiled products
    if (steps > 0) {
        ChainBucket small[MUON_HIP_MAX_BUCKETS];
        int n = 0;
        for (int i = 0; i < all.n; ++i) {
            const Bucket& k = all.b[i];
            if (!in_workgroups(all, i)) {
                w.b[w.n++] = k;
                continue;
            }
            small[n++] = ChainBucket{k.at(k.p.offX[1]), k.p.strideU, (const float*)(k.ws + k.p.offParts), k.at(k.p.offX[0]), k.p.strideX,
                                     upd ? k.p_ptrs : nullptr, out, (float)k.scale, k.p.Kp / BLK_COLS, k.p.nparts, k.p.rows, k.p.cols, k.p.batch};
        }
        if (n) {
            ChainMath cm{steps, (float)a, (float)b, (float)c, 0, 1.f, 0.f};
            if (upd) {
                cm.p_dtype = upd->p_dtype;
                cm.decay = (float)(1.0 - upd->lr * upd->weight_decay);
                cm.alpha = (float)(-upd->lr);
            }
            Timed t(MUON_HIP_K_SMALL_CHAIN, s);
            if (hipError_t e = launch_ns_chain(small, n, cm, ms.cus, s); e != hipSuccess) return hip_fail(e, "ns_chain launch");
        }
        if (!w.n) return 0;
    } else {
        w = all;
    }
    FlowList fl;
    const bool flow = steps > 0 && flow_of(w, steps, a, b, c, upd, out, 1 << ms.xcd_shift, upd && is_recorded(s), fl);
    if (flow)
        if (int rc = chain_alarm(&fl.alarm)) return rc;
    if (int rc = do_normalize(w, flow, s)) return rc;
    if (flow) {
        fl.polls = g_chain_polls;
        Timed t(MUON_HIP_K_FLOW_CHAIN, s);
        hipError_t e = launch_flow(fl, s);
        return e == hipSuccess ? 0 : hip_fail(e, "ns_flow launch");
    }
    unsigned* ppx = ppx_counters(w);
    GemmItem items[MUON_HIP_MAX_BUCKETS];
    for (int it = 0; it < steps; ++it) {
        const int cur = it & 1;
        bool adapt = stage_items(w, EPI_SYRK, cur, a, b, c, ppx, items);
        if (int rc = launch_items(MUON_HIP_K_SYRK, "syrk launch", items, w.n, adapt, s)) return rc;
        adapt = stage_items(w, EPI_SYMPOLY, cur, a, b, c, ppx, items);
        if (int rc = launch_items(MUON_HIP_K_SYMPOLY, "sympoly launch", items, w.n, adapt, s)) return rc;
        adapt = stage_items(w, EPI_BX, cur, a, b, c, ppx, items);
        const bool last = upd && it == steps - 1;
        if (out && it == steps - 1 && !write_result(w.b[0], adapt, ms.cus, out, items[0])) *left_in_x = true;
        if (last)
            for (int i = 0; i < w.n; ++i) fold_update(items[i], w.b[i].p_ptrs, w.b[i].p.rows, w.b[i].p.cols, w.b[i].scale, *upd);
        if (int rc = launch_items(last ? MUON_HIP_K_BX_UPDATE : MUON_HIP_K_BX, "bx launch", items, w.n, adapt, s)) return rc;
    }
    return 0;
}

// What a description of a call stands on in place of a workspace: plans hold addresses, nothing is read through them.
alignas(256) char g_nowhere[256];

// The buckets of a call whose products are tiled, as ns_chain parts them, and where they stand in the call; or the others.
int tiled_buckets(const muon_hip_bucket* buckets, int n, Work& w, int* from, bool others = false) {
    Work all;
    all.n = n;
    for (int i = 0; i < n; ++i) {
        if (int rc = all.b[i].init(buckets[i].rows, buckets[i].cols, buckets[i].batch, g_nowhere)) return rc;
        all.b[i].p_ptrs = (const void* const*)g_nowhere;
    }
    for (int i = 0; i < n; ++i)
        if (in_workgroups(all, i) == others) {
            from[w.n] = i;
            w.b[w.n++] = all.b[i];
        }
    return 0;
}

}  // namespace

extern "C" {

int muon_hip_version(void) { return 100; }

const char* muon_hip_last_error(void) { return g_err; }

int muon_hip_set_gemm_config(int cfg) {
    if (cfg != MUON_HIP_CFG_AUTO && cfg != MUON_HIP_CFG_STAGED && gemm_cfg_tile(cfg) == 0) return fail(MUON_HIP_EINVAL, "unknown GEMM configuration %d", cfg);
    g_forced_cfg.store(cfg, std::memory_order_relaxed);
    return 0;
}

int muon_hip_chain_status(void) { return chain_status(); }

int muon_hip_set_chain_polls(long polls) {
    if (polls > kChainPolls) return fail(MUON_HIP_EINVAL, "at most %u polls", kChainPolls);
    g_chain_polls = polls < 0 ? kChainPolls : (unsigned)polls;
    return 0;
}

int muon_hip_geometry(int rows, int cols, int* M, int* K, int* Mp, int* Kp, int* tile) {
    Plan p;
    if (int rc = make_plan(rows, cols, 1, p)) return rc;
    if (M) *M = p.M;
    if (K) *K = p.K;
    if (Mp) *Mp = p.Mp;
    if (Kp) *Kp = p.Kp;
    if (tile) *tile = p.tile;
    return 0;
}

size_t muon_hip_workspace_bytes(int rows, int cols, int batch) {
    Plan p;
    if (make_plan(rows, cols, batch, p)) return 0;
    return p.total;
}

int muon_hip_momentum_norm(const void* const* g_ptrs, const void* const* m_ptrs, int g_dtype, int m_dtype,
                           void* workspace, int rows, int cols, int batch, double beta, int nesterov,
                           int write_back_grad, void* stream) {
    Work w;
    if (int rc = one_bucket(rows, cols, batch, workspace, w)) return rc;
    w.b[0].g_ptrs = g_ptrs;
    w.b[0].m_ptrs = m_ptrs;
    return do_momentum(w, g_dtype, m_dtype, beta, nesterov, write_back_grad, (hipStream_t)stream);
}

int muon_hip_cast_norm(const void* G, int g_dtype, void* workspace, int rows, int cols, int batch, void* stream) {
    Plan p;
    if (int rc = make_plan(rows, cols, batch, p)) return rc;
    if (int rc = check_ws(workspace)) return rc;
    if (!G || !dtype_ok(g_dtype)) return fail(MUON_HIP_EINVAL, "bad input tensor or dtype");
    hipStream_t s = (hipStream_t)stream;
    Timed t(MUON_HIP_K_MOMENTUM, s);
    hipError_t e = launch_cast_norm(G, p.n, g_dtype, wsp(workspace, p.offX[1]), p.strideU,
                                    (float*)((char*)workspace + p.offParts), p.nparts, p.n, batch, s);
    return e == hipSuccess ? 0 : hip_fail(e, "cast_norm launch");
}

int muon_hip_normalize(void* workspace, int rows, int cols, int batch, void* stream) {
    Work w;
    if (int rc = one_bucket(rows, cols, batch, workspace, w)) return rc;
    return do_normalize(w, false, (hipStream_t)stream);
}

int muon_hip_ns_grouped(void* workspace, int rows, int cols, int batch, int steps, double a, double b, double c,
                        void* stream) {
    Work w;
    if (int rc = one_bucket(rows, cols, batch, workspace, w)) return rc;
    if (int rc = chain_status()) return rc;
    return ns_chain(w, steps, a, b, c, nullptr, (hipStream_t)stream);
}

int muon_hip_ns_result(void* workspace, int rows, int cols, int batch, int steps, double a, double b, double c, void* out, void* stream) {
    Work w;
    if (int rc = one_bucket(rows, cols, batch, workspace, w)) return rc;
    if (!out) return fail(MUON_HIP_EINVAL, "bad output pointer");
    if (int rc = chain_status()) return rc;
    MachineShape ms;
    if (hipError_t e = machine_shape(ms); e != hipSuccess) return hip_fail(e, "device shape");
    const bool direct = steps > 0 && (!w.b[0].p.small || chain_writes(rows, cols, batch, out, ms.cus));
    bool left_in_x = !direct;
    if (int rc = ns_chain(w, steps, a, b, c, nullptr, (hipStream_t)stream, direct ? (bf16_t*)out : nullptr, &left_in_x)) return rc;
    return !left_in_x ? 0 : muon_hip_ns_output(workspace, rows, cols, batch, steps, out, stream);
}

int muon_hip_apply_update(const void* const* p_ptrs, int p_dtype, void* workspace, int rows, int cols, int batch,
                          int steps, double scale, double lr, double weight_decay, void* stream) {
    Plan p;
    if (int rc = make_plan(rows, cols, batch, p)) return rc;
    if (int rc = check_ws(workspace)) return rc;
    if (!p_ptrs || !dtype_ok(p_dtype) || steps < 0) return fail(MUON_HIP_EINVAL, "bad pointer table, dtype or steps");
    hipStream_t s = (hipStream_t)stream;
    const bf16_t* O = wsp(workspace, result_offset(p, steps));  // X (M x K): the parameter's image, or its transpose when rows > cols
    Timed t(MUON_HIP_K_UPDATE, s);
    hipError_t e = launch_apply_update(p_ptrs, p_dtype, O, p.strideX, p.Kp / BLK_COLS, rows, cols, batch, scale, lr,
                                       weight_decay, s);
    return e == hipSuccess ? 0 : hip_fail(e, "apply_update launch");
}

int muon_hip_ns_output(void* workspace, int rows, int cols, int batch, int steps, void* out, void* stream) {
    Plan p;
    if (int rc = make_plan(rows, cols, batch, p)) return rc;
    if (int rc = check_ws(workspace)) return rc;
    if (!out || steps < 0) return fail(MUON_HIP_EINVAL, "bad output pointer or steps");
    hipStream_t s = (hipStream_t)stream;
    const bf16_t* O = wsp(workspace, result_offset(p, steps));
    hipError_t e = launch_unpack((bf16_t*)out, p.n, cols, O, p.strideX, p.Kp / BLK_COLS, rows, cols, p.transposed, batch, s);
    return e == hipSuccess ? 0 : hip_fail(e, "ns_output launch");
}

int muon_hip_step_multi(const muon_hip_bucket* buckets, int n, int p_dtype, int g_dtype, int m_dtype, void* workspace, double lr,
                        double weight_decay, double beta, int nesterov, int ns_steps, double a, double b, double c,
                        int write_back_grad, void* stream) {
    if (!buckets || n < 1 || n > MUON_HIP_MAX_BUCKETS)
        return fail(MUON_HIP_EINVAL, "1 to %d buckets per call", MUON_HIP_MAX_BUCKETS);
    if (int rc = check_ws(workspace)) return rc;
    if (!dtype_ok(p_dtype) || ns_steps < 0) return fail(MUON_HIP_EINVAL, "bad dtype or steps");
    Work w;
    w.n = n;
    char* base = (char*)workspace;
    for (int i = 0; i < n; ++i) {
        const muon_hip_bucket& in = buckets[i];
        if (!in.p_ptrs) return fail(MUON_HIP_EINVAL, "pointer table is null");
        if (int rc = w.b[i].init(in.rows, in.cols, in.batch, base)) return rc;
        w.b[i].p_ptrs = in.p_ptrs;
        w.b[i].g_ptrs = in.g_ptrs;
        w.b[i].m_ptrs = in.m_ptrs;
        w.b[i].scale = in.scale;
        base += w.b[i].p.total;
    }
    if (int rc = chain_status()) return rc;
    hipStream_t s = (hipStream_t)stream;
    if (int rc = do_momentum(w, g_dtype, m_dtype, beta, nesterov, write_back_grad, s)) return rc;
    // The parameter is updated by the epilogue of the last B.X (for rows > cols through a transposing gather out of
    // LDS): the final X' is then neither written nor read back.  Without an iteration there is no such product.
    const UpdateArgs u{p_dtype, lr, weight_decay};
    if (int rc = ns_chain(w, ns_steps, a, b, c, &u, s)) return rc;
    if (ns_steps == 0)
        for (int i = 0; i < n; ++i)
            if (int rc = muon_hip_apply_update(w.b[i].p_ptrs, p_dtype, w.b[i].ws, w.b[i].p.rows, w.b[i].p.cols, w.b[i].p.batch, 0,
                                               w.b[i].scale, lr, weight_decay, stream))
                return rc;
    return 0;
}

int muon_hip_routes(const muon_hip_bucket* buckets, int n, int kernel_id, int cus, muon_hip_route* out) {
    if (!buckets || !out || n < 1 || n > MUON_HIP_MAX_BUCKETS || cus < 1) return fail(MUON_HIP_EINVAL, "bad bucket list or device");
    const int epi = kernel_id == MUON_HIP_K_SYRK ? EPI_SYRK : kernel_id == MUON_HIP_K_SYMPOLY ? EPI_SYMPOLY : EPI_BX;
    const bool result = kernel_id == MUON_HIP_ROUTE_RESULT;
    if (result && n != 1) return fail(MUON_HIP_EINVAL, "a result is that of one bucket");
    const bool chain = kernel_id == MUON_HIP_K_SMALL_CHAIN;
    if (epi == EPI_BX && !result && !chain && kernel_id != MUON_HIP_K_BX && kernel_id != MUON_HIP_K_BX_UPDATE) return fail(MUON_HIP_EINVAL, "not a product");
    Work w;
    int from[MUON_HIP_MAX_BUCKETS];
    for (int i = 0; i < n; ++i) out[i] = muon_hip_route{MUON_HIP_CFG_AUTO, 0, -1};
    if (int rc = tiled_buckets(buckets, n, w, from, chain)) return rc;
    if (!w.n) return 0;
    if (chain) {
        ChainBucket small[MUON_HIP_MAX_BUCKETS] = {};
        ChainRoute r[MUON_HIP_MAX_BUCKETS];
        int order[MUON_HIP_MAX_BUCKETS];
        for (int i = 0; i < w.n; ++i) small[i].rows = w.b[i].p.rows, small[i].cols = w.b[i].p.cols, small[i].batch = w.b[i].p.batch;
        if (plan_ns_chain(small, w.n, cus, r, order) < 0) return fail(MUON_HIP_EINVAL, "no workgroup holds these matrices");
        for (int i = 0; i < w.n; ++i) out[from[i]] = muon_hip_route{MUON_HIP_CFG_AUTO, 16 * r[i].blocks, r[i].launch};
        return 0;
    }
    GemmItem items[MUON_HIP_MAX_BUCKETS];
    GemmRoute route[MUON_HIP_MAX_BUCKETS];
    const bool adapt = stage_items(w, epi, 0, 1.0, 1.0, 1.0, ppx_counters(w), items);
    if (kernel_id == MUON_HIP_K_BX_UPDATE)
        for (int i = 0; i < w.n; ++i) fold_update(items[i], nullptr, w.b[i].p.rows, w.b[i].p.cols, 1.0, UpdateArgs{});
    if (result) write_result(w.b[0], adapt, cus, (bf16_t*)g_nowhere, items[0]);
    if (plan_gemm_nt(items, w.n, adapt, cus, route) < 0) return fail(MUON_HIP_EINVAL, "no kernel takes these products");
    for (int i = 0; i < w.n; ++i) out[from[i]] = muon_hip_route{route[i].cfg, route[i].height, route[i].launch};
    return 0;
}

int muon_hip_flow_tiles(const muon_hip_bucket* buckets, int n, int steps, int update, int xcds, muon_hip_flow_tile* out, long capacity,
                        long* count) {
    const bool recorded = update & MUON_HIP_FLOW_RECORDED;
    update &= ~MUON_HIP_FLOW_RECORDED;
    if (!buckets || !count || n < 1 || n > MUON_HIP_MAX_BUCKETS || capacity < 0 || (capacity && !out) || steps < 0 || xcds < 1 || xcds > GEMM_MAX_XCDS)
        return fail(MUON_HIP_EINVAL, "bad bucket list, steps, XCDs or output");
    *count = 0;
    Work w;
    int from[MUON_HIP_MAX_BUCKETS];
    if (int rc = tiled_buckets(buckets, n, w, from)) return rc;
    FlowList l;
    const UpdateArgs u{};
    if (!w.n || steps == 0 || !flow_of(w, steps, 1.0, 1.0, 1.0, update ? &u : nullptr, nullptr, xcds, recorded, l)) return 0;
    for (int g = 0; g < l.groups; ++g)
        for (int t = 0; t < flow_tiles(l, g); ++t, ++*count) {
            if (*count >= capacity) continue;
            const FlowPlace p = flow_place(l, g, t);
            const int product = p.stage == 0 ? MUON_HIP_K_SYRK : p.stage == 1 ? MUON_HIP_K_SYMPOLY : MUON_HIP_K_BX;
            out[*count] = muon_hip_flow_tile{g, from[p.entry], p.matrix, p.it, product, p.tile, p.before};
        }
    return 0;
}

int muon_hip_step_grouped(const void* const* p_ptrs, const void* const* g_ptrs, const void* const* m_ptrs,
                          int p_dtype, int g_dtype, int m_dtype, void* workspace, int rows, int cols, int batch,
                          double lr, double weight_decay, double beta, int nesterov, int ns_steps, double scale,
                          double a, double b, double c, int write_back_grad, void* stream) {
    const muon_hip_bucket one{p_ptrs, g_ptrs, m_ptrs, rows, cols, batch, scale};
    return muon_hip_step_multi(&one, 1, p_dtype, g_dtype, m_dtype, workspace, lr, weight_decay, beta, nesterov, ns_steps, a, b, c,
                               write_back_grad, stream);
}

long muon_hip_blocked_elems(int rows, int cols) {
    if (rows <= 0 || cols <= 0 || cols % BLK_COLS) {
        fail(MUON_HIP_ESHAPE, "a blocked matrix needs positive sizes and a multiple of 32 columns (got %d x %d)", rows, cols);
        return 0;
    }
    return blocked_elems(rows, cols);
}

int muon_hip_pack_bf16(const void* src, long src_stride, int ld, int rows, int cols, void* dst, int rows_p, int cols_p,
                       int batch, void* stream) {
    if (!src || !dst || batch <= 0) return fail(MUON_HIP_EINVAL, "null tensor or empty batch");
    if (rows <= 0 || cols <= 0 || rows > rows_p || cols > cols_p || ld < cols || cols_p % BLK_COLS || batch > 65535)
        return fail(MUON_HIP_ESHAPE, "pack: need 0 < rows <= rows_p, 0 < cols <= cols_p, ld >= cols, cols_p %% 32 == 0");
    hipError_t e = launch_pack((const bf16_t*)src, src_stride, ld, rows, cols, (bf16_t*)dst, blocked_elems(rows_p, cols_p),
                               rows_p, cols_p, batch, (hipStream_t)stream);
    return e == hipSuccess ? 0 : hip_fail(e, "pack launch");
}

int muon_hip_unpack_bf16(const void* src, int rows_p, int cols_p, void* dst, long dst_stride, int ld, int rows, int cols,
                         int batch, void* stream) {
    if (!src || !dst || batch <= 0) return fail(MUON_HIP_EINVAL, "null tensor or empty batch");
    if (rows <= 0 || cols <= 0 || rows > rows_p || cols > cols_p || ld < cols || cols_p % BLK_COLS || batch > 65535)
        return fail(MUON_HIP_ESHAPE, "unpack: need 0 < rows <= rows_p, 0 < cols <= cols_p, ld >= cols, cols_p %% 32 == 0");
    hipError_t e = launch_unpack((bf16_t*)dst, dst_stride, ld, (const bf16_t*)src, blocked_elems(rows_p, cols_p),
                                 cols_p / BLK_COLS, rows, cols, false, batch, (hipStream_t)stream);
    return e == hipSuccess ? 0 : hip_fail(e, "unpack launch");
}

int muon_hip_syrk_bf16(const void* X, void* A, int Mp, int Kp, int batch, int cfg, void* counters, void* stream) {
    const Cfg use = cfg == MUON_HIP_CFG_AUTO ? pick_cfg(Mp, EPI_SYRK) : Cfg{cfg, false};
    int tile;
    if (int rc = check_gemm(use.id, Mp, Kp, batch, tile)) return rc;
    if (!X || !A) return fail(MUON_HIP_EINVAL, "null operand");
    if (int rc = check_counters(counters)) return rc;
    const GemmItem it = syrk_item(use.id, (const bf16_t*)X, (bf16_t*)A, Mp, Kp, Kp, batch, (unsigned*)counters);
    return launch_items(MUON_HIP_K_SYRK, "syrk launch", &it, 1, use.adapt, (hipStream_t)stream);
}

// Whether the kernels read X where it lies.  They can when its rows are whole k-tiles and 16-byte pieces, a panel of 256 rows is
// addressed with 32 bits, and nothing that they write is still to be read.  They should, but
//  - where the 64 (64-tiles: 128) bytes of a row that a load instruction takes straddle two cache lines: rows are whole numbers of lines, so
//    it is the address of X that decides;
//  - on 128-tiles of an X that the L2s do not hold: those read 64 bytes of a row at a time, and rows whose pitch is a multiple of the L2
//    channels crowd into few of them.
// A small X is the better read in place in both.  Measured (profiles/mmt_packed_or_in_place.txt), packed | in place | in place on a boundary
// of 32 bytes: 64-tiles 896 x 4864 26.5 | 18.7 | 26.0 us, 896 x 32768 117 | 98 | 139; 128-tiles 2048 x 1024 18.9 | 12.0 | 13.3, 2048 x 2048
// 25.6 | 20.4 | 29.4, 2048 x 5632 44.1 | 47.7 | 70.8, 3072 x 3072 48.0 | 56.4 | 77.8; 256-tiles 4096 x 512 28.2 | 22.0 | 24.4, 4096 x 12288
// 213 | 203 | 300, 8192 x 16384 901 | 876 | 1161.  The line at 5 Mi elements is one of many shapes: on 128-tiles 2048 x 2560 would be 7 %
// faster packed, 2800 x 1920 and 2560 x 4096 13 and 7 % faster in place.
static bool mmt_reads_x(const void* X, const void* Y, int M, int K) {
    const uintptr_t x = (uintptr_t)X, y = (uintptr_t)Y;
    const bool apart = y + 2 * (size_t)M * M <= x || x + 2 * (size_t)M * K <= y;
    if (K % 128 || K > (1 << 22) || (x & 15) || !apart) return false;
    MachineShape ms;
    if (machine_shape(ms) != hipSuccess) return false;  // the launch will report it
    const long t = round_up(M, 128) / 128, t128 = t * (t + 1) / 2, t64 = t * (2 * t + 1);
    const bool small = t64 <= ms.cus, large = use_tile256(M) && t128 > 2 * ms.cus;  // as plan_gemm_nt has it
    const bool whole = x % (small ? 128 : 64) == 0;
    return (long)M * K <= (whole ? 5L : 2L) << 20 || (whole && (small || large));
}
struct MmtPlan {
    Cfg use;
    int Mp, Kp;
    bool reads_x;  // a named configuration multiplies packed operands, which every kernel takes
};
static MmtPlan mmt_plan(const void* X, const void* Y, int M, int K) {
    const int forced = g_forced_cfg.load(std::memory_order_relaxed), tile = use_tile256(M) ? 256 : 128;
    const int own = tile == 256 && M > 512 ? GEMM_CFG_256_PINGPONG : GEMM_CFG_128_PINGPONG;
    return MmtPlan{forced >= 0 ? Cfg{forced, false} : Cfg{own, true}, (int)round_up(M, tile), (int)round_up(K, tile),
                   forced < 0 && mmt_reads_x(X, Y, M, K)};
}

long muon_hip_mmt_scratch_elems(const void* X, const void* Y, int M, int K) {
    if (M <= 0 || K <= 0) return 0;
    const MmtPlan p = mmt_plan(X, Y, M, K);
    return p.reads_x ? 0 : blocked_elems(p.Mp, p.Kp);
}

int muon_hip_mmt_bf16(const void* X, void* Y, int M, int K, void* scratch, void* stream) {
    if (M <= 0 || K <= 0) return fail(MUON_HIP_EINVAL, "sizes must be positive");
    if (!X || !Y) return fail(MUON_HIP_EINVAL, "null operand");
    const MmtPlan p = mmt_plan(X, Y, M, K);
    int tile;
    if (int rc = check_gemm(p.use.id, p.Mp, p.Kp, 1, tile)) return rc;
    if (!p.reads_x) {
        if (!scratch || ((uintptr_t)scratch & 15)) return fail(MUON_HIP_EINVAL, "this X needs scratch, 16-byte aligned");
        hipError_t e = launch_pack((const bf16_t*)X, 0, K, M, K, (bf16_t*)scratch, 0, p.Mp, p.Kp, 1, (hipStream_t)stream);
        if (e != hipSuccess) return hip_fail(e, "pack launch");
    }
    GemmItem it = syrk_item(p.use.id, (const bf16_t*)(p.reads_x ? X : scratch), (bf16_t*)Y, p.Mp, (int)round_up(K, 128), p.Kp, 1, nullptr);
    it.epi = EPI_MMT;
    it.g.dense_rows = M;
    it.g.dense_pitch = p.reads_x ? K : 0;
    return launch_items(MUON_HIP_K_SYRK, "mmt launch", &it, 1, p.use.adapt, (hipStream_t)stream);
}

int muon_hip_sympoly_bf16(const void* A, void* B, int Mp, int batch, double b, double c, int cfg, void* counters,
                          void* stream) {
    const Cfg use = cfg == MUON_HIP_CFG_AUTO ? pick_cfg(Mp, EPI_SYMPOLY) : Cfg{cfg, false};
    int tile;
    if (int rc = check_gemm(use.id, Mp, Mp, batch, tile)) return rc;
    if (!A || !B || A == B) return fail(MUON_HIP_EINVAL, "null or aliased operand");
    if (int rc = check_counters(counters)) return rc;
    const GemmItem it = sympoly_item(use.id, (const bf16_t*)A, (bf16_t*)B, Mp, batch, b, c, (unsigned*)counters);
    return launch_items(MUON_HIP_K_SYMPOLY, "sympoly launch", &it, 1, use.adapt, (hipStream_t)stream);
}

int muon_hip_bx_axpy_bf16(const void* B, const void* X, void* Xout, int Mp, int Kp, int batch, double a, int cfg,
                          void* counters, void* stream) {
    const Cfg use = cfg == MUON_HIP_CFG_AUTO ? pick_cfg(Mp, EPI_BX) : Cfg{cfg, false};
    int tile;
    if (int rc = check_gemm(use.id, Mp, Kp, batch, tile)) return rc;
    if (!B || !X || !Xout) return fail(MUON_HIP_EINVAL, "null operand");
    if (Xout == X) return fail(MUON_HIP_EINVAL, "Xout must not alias X");
    if (int rc = check_counters(counters)) return rc;
    const GemmItem it = bx_item(use.id, (const bf16_t*)B, (const bf16_t*)X, (bf16_t*)Xout, Mp, Kp, Kp, batch, a, (unsigned*)counters);
    return launch_items(MUON_HIP_K_BX, "bx launch", &it, 1, use.adapt, (hipStream_t)stream);
}

int muon_hip_adamw(void* p, const void* g, void* exp_avg, void* exp_avg_sq, int dtype, long n, int step, double lr,
                   double beta1, double beta2, double eps, double weight_decay, void* stream) {
    if (!p || !g || !exp_avg || !exp_avg_sq) return fail(MUON_HIP_EINVAL, "null tensor");
    if (!dtype_ok(dtype) || n < 0 || step < 1) return fail(MUON_HIP_EINVAL, "bad dtype, size or step");
    if (n == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    Timed t(MUON_HIP_K_ADAMW, s);
    hipError_t e = launch_adamw(p, g, exp_avg, exp_avg_sq, dtype, n, step, lr, beta1, beta2, eps, weight_decay, s);
    return e == hipSuccess ? 0 : hip_fail(e, "adamw launch");
}

int muon_hip_adam_update(const void* g, void* exp_avg, void* exp_avg_sq, void* out, int dtype, long n, int step,
                         double beta1, double beta2, double eps, void* stream) {
    if (!g || !exp_avg || !exp_avg_sq || !out) return fail(MUON_HIP_EINVAL, "null tensor");
    if (!dtype_ok(dtype) || n < 0 || step < 1) return fail(MUON_HIP_EINVAL, "bad dtype, size or step");
    if (n == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    Timed t(MUON_HIP_K_ADAMW, s);
    hipError_t e = launch_adam_update(g, exp_avg, exp_avg_sq, out, dtype, n, step, beta1, beta2, eps, s);
    return e == hipSuccess ? 0 : hip_fail(e, "adam_update launch");
}

int muon_hip_scale(void* x, int dtype, long n, double scale, void* stream) {
    if (!x) return fail(MUON_HIP_EINVAL, "null tensor");
    if (!dtype_ok(dtype) || n < 0) return fail(MUON_HIP_EINVAL, "bad dtype or size");
    if (n == 0) return 0;
    hipError_t e = launch_scale(x, dtype, n, scale, (hipStream_t)stream);
    return e == hipSuccess ? 0 : hip_fail(e, "scale launch");
}

int muon_hip_decay_update(void* p, int p_dtype, const void* u, int u_dtype, long n, double lr, double weight_decay,
                          void* stream) {
    if (!p || !u) return fail(MUON_HIP_EINVAL, "null tensor");
    if (!dtype_ok(p_dtype) || !dtype_ok(u_dtype) || n < 0) return fail(MUON_HIP_EINVAL, "bad dtype or size");
    if (p_dtype == MUON_HIP_BF16 && u_dtype == MUON_HIP_F32)
        return fail(MUON_HIP_EINVAL, "an fp32 update for a bf16 parameter is not supported");
    if (n == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    Timed t(MUON_HIP_K_UPDATE, s);
    hipError_t e = launch_decay_update(p, p_dtype, u, u_dtype, n, lr, weight_decay, s);
    return e == hipSuccess ? 0 : hip_fail(e, "decay_update launch");
}

namespace {
int check_norm_type(double norm_type) {
    if (norm_type != norm_type) return fail(MUON_HIP_EINVAL, "norm_type is NaN");
    return 0;
}
int check_list(const void* ptrs, const long* numel, const long* chunk_start, int n, long chunks, int dtype) {
    if (!ptrs || !numel || !chunk_start) return fail(MUON_HIP_EINVAL, "null tensor-list array");
    if (n <= 0 || chunks <= 0) return fail(MUON_HIP_EINVAL, "a tensor list needs at least one tensor and one chunk");
    if (chunks > 0x1fffffffL) return fail(MUON_HIP_ESHAPE, "%ld chunks exceed one launch", chunks);  // at least four workgroups each
    if (!dtype_ok(dtype)) return fail(MUON_HIP_EINVAL, "unknown dtype %d", dtype);
    return 0;
}
}  // namespace

int muon_hip_adamw_multi(const void* const* p_ptrs, const void* const* g_ptrs, const void* const* exp_avg_ptrs,
                         const void* const* exp_avg_sq_ptrs, const long* numel, const long* chunk_start,
                         const double* bias1, const double* bias2, int n, long chunks, int dtype, double lr,
                         double beta1, double beta2, double eps, double weight_decay, void* stream) {
    if (int rc = check_list(p_ptrs, numel, chunk_start, n, chunks, dtype)) return rc;
    if (!g_ptrs || !exp_avg_ptrs || !exp_avg_sq_ptrs || !bias1 || !bias2) return fail(MUON_HIP_EINVAL, "null table");
    hipStream_t s = (hipStream_t)stream;
    Timed t(MUON_HIP_K_ADAMW_MULTI, s);
    const MultiTensorList l{p_ptrs, numel, chunk_start, n, chunks};
    hipError_t e = launch_adamw_multi(l, g_ptrs, exp_avg_ptrs, exp_avg_sq_ptrs, bias1, bias2, dtype, lr, beta1, beta2,
                                      eps, weight_decay, s);
    return e == hipSuccess ? 0 : hip_fail(e, "adamw_multi launch");
}

int muon_hip_grad_norms(const void* const* g_ptrs, const long* numel, const long* chunk_start, int n, long chunks,
                        int dtype, double norm_type, float* partials, float* norms, void* stream) {
    if (int rc = check_list(g_ptrs, numel, chunk_start, n, chunks, dtype)) return rc;
    if (int rc = check_norm_type(norm_type)) return rc;
    if (!partials || !norms) return fail(MUON_HIP_EINVAL, "null output");
    hipStream_t s = (hipStream_t)stream;
    Timed t(MUON_HIP_K_GRAD_NORM, s);
    const MultiTensorList l{g_ptrs, numel, chunk_start, n, chunks};
    hipError_t e = launch_tensor_norms(l, dtype, norm_type, partials, norms, s);
    return e == hipSuccess ? 0 : hip_fail(e, "grad_norms launch");
}

// ---- the entry point that allocates nothing ---------------------------------------------------
// Partial sums of muon_hip_grad_norms_static live in this array instead of a caller buffer.  Each device the
// library runs on holds its own copy at its own address, looked up once per device.
static __device__ __align__(256) float scratch[MUON_HIP_STATIC_MAX_CHUNKS];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device (0 on failure, with the error recorded).
int scratch_for_current_device(float** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
    if (dev < 0 || dev >= kMaxDevices) return fail(MUON_HIP_EINVAL, "device ordinal %d out of range", dev);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        float* ptr = nullptr;
        e = hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
        if (!ptr) return fail(MUON_HIP_EINVAL, "hipGetSymbolAddress returned a null address");
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return 0;
}
}  // namespace

int muon_hip_grad_norms_static(const void* const* g_ptrs, const long* numel, const long* chunk_start, int n,
                               long chunks, int dtype, double norm_type, float* norms, void* stream) {
    if (int rc = check_list(g_ptrs, numel, chunk_start, n, chunks, dtype)) return rc;
    if (int rc = check_norm_type(norm_type)) return rc;
    if (!norms) return fail(MUON_HIP_EINVAL, "null output");
    if (chunks > (long)MUON_HIP_STATIC_MAX_CHUNKS)
        return fail(MUON_HIP_ESHAPE, "%ld chunks exceed the %ld the built-in scratch array holds; use muon_hip_grad_norms "
                    "with a caller buffer", chunks, (long)MUON_HIP_STATIC_MAX_CHUNKS);
    float* partials = nullptr;
    if (int rc = scratch_for_current_device(&partials)) return rc;
    hipStream_t s = (hipStream_t)stream;
    Timed t(MUON_HIP_K_GRAD_NORM, s);
    const MultiTensorList l{g_ptrs, numel, chunk_start, n, chunks};
    // every partial the second kernel reads is written by the first: nothing has to start at zero
    hipError_t e = launch_tensor_norms(l, dtype, norm_type, partials, norms, s);
    return e == hipSuccess ? 0 : hip_fail(e, "grad_norms launch");
}

int muon_hip_total_norm(const float* norms, int n, int dtype, double norm_type, float* total_f32, void* total_typed,
                        void* stream) {
    if (!norms || !total_f32 || !total_typed || n <= 0 || !dtype_ok(dtype))
        return fail(MUON_HIP_EINVAL, "null pointer, empty list or unknown dtype");
    if (int rc = check_norm_type(norm_type)) return rc;
    hipError_t e = launch_total_norm(norms, n, dtype, norm_type, total_f32, total_typed,
                                     (hipStream_t)stream);
    return e == hipSuccess ? 0 : hip_fail(e, "total_norm launch");
}

int muon_hip_clip_scale(const void* const* g_ptrs, const long* numel, const long* chunk_start, int n, long chunks,
                        int dtype, const float* total_f32, int norm_dtype, double max_norm, void* stream) {
    if (int rc = check_list(g_ptrs, numel, chunk_start, n, chunks, dtype)) return rc;
    if (!total_f32 || !dtype_ok(norm_dtype)) return fail(MUON_HIP_EINVAL, "null total or unknown norm dtype");
    hipStream_t s = (hipStream_t)stream;
    Timed t(MUON_HIP_K_CLIP_SCALE, s);
    const MultiTensorList l{g_ptrs, numel, chunk_start, n, chunks};
    hipError_t e = launch_clip_scale_multi(l, dtype, total_f32, norm_dtype, max_norm, s);
    return e == hipSuccess ? 0 : hip_fail(e, "clip_scale launch");
}

int muon_hip_device_shape(int* compute_units, int* xcds) {
    MachineShape ms;
    if (hipError_t e = machine_shape(ms); e != hipSuccess) return hip_fail(e, "device attributes");
    if (compute_units) *compute_units = ms.cus;
    if (xcds) *xcds = 1 << ms.xcd_shift;
    return 0;
}

int muon_hip_timing_reserve(long launches) {
    if (launches < 0 || (size_t)launches > kMaxPool) return fail(MUON_HIP_EINVAL, "0 to %ld launches can be reserved", (long)kMaxPool);
    if (g_timing.load(std::memory_order_acquire)) return fail(MUON_HIP_EINVAL, "reserve events while timing is off");
    std::lock_guard<std::mutex> lk(g_tmu);
    return grow_pool((size_t)launches);
}

int muon_hip_timing_enable(int on) {
    std::lock_guard<std::mutex> lk(g_tmu);
    g_timing.store(false, std::memory_order_release);
    if (on) {
        if (int rc = grow_pool(kPoolChunk)) return rc;  // at least one chunk (a no-op once it exists)
        g_used.store(0, std::memory_order_relaxed);  // the pairs of the last measurement are recorded over
        g_untimed.store(0, std::memory_order_relaxed);
        g_timing.store(true, std::memory_order_release);
    }
    return 0;
}

int muon_hip_timing_read(int kernel_id, double* total_ms, long* launches) {
    if (kernel_id < 0 || kernel_id >= MUON_HIP_K_COUNT || !total_ms || !launches)
        return fail(MUON_HIP_EINVAL, "bad kernel id or null output");
    std::lock_guard<std::mutex> lk(g_tmu);
    const size_t used = std::min(g_used.load(std::memory_order_acquire), g_pool_size.load(std::memory_order_acquire));
    double tot = 0.0;
    long cnt = 0;
    for (size_t i = 0; i < used; ++i) {
        const EventPair& p = pool_at(i);
        if (p.kid != kernel_id) continue;
        hipError_t e = hipEventSynchronize(p.stop);
        if (e != hipSuccess) return hip_fail(e, "event synchronize");
        float ms = 0.f;
        e = hipEventElapsedTime(&ms, p.start, p.stop);
        if (e != hipSuccess) return hip_fail(e, "event elapsed");
        tot += ms;
        ++cnt;
    }
    *total_ms = tot;
    *launches = cnt;
    return 0;
}

long muon_hip_timing_untimed(void) { return g_untimed.load(std::memory_order_relaxed); }

}  // extern "C"
