// cse_engine.hip -- host side of the engine: context, device buffers,
// launches and the C ABI declared in include/cse.h.  Kernels live in
// cse_kernels.hip (same translation unit).
#include "cse_kernels.hip"

#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <thread>
#include <vector>

#include "../../include/cse.h"
#include "cse_host.h"

static_assert(HIST_STRIDE == CSE_HIST_BINS, "device histogram stride is the public histogram size");

struct DevBuf {
    void *p = nullptr;
    size_t cap = 0;
};

// pinned host memory: device-to-host copies into it are single DMA
// transfers instead of chunked staging through a driver buffer.  Coherent,
// whatever the process's environment says (HIP_HOST_COHERENT): the host reads
// results and the call's number while the device may still run.
struct HostBuf {
    void *p = nullptr;
    size_t cap = 0;
};

struct cse_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;  // cse_inner_products' times
    int cus = 0;
    char name[128] = {0};
    char err[512] = {0};
    DevBuf s1, s2, out, recs, terms, queue, thr, sexp, L, idx, errflag, lsh, stack, leaf;
    // a batch's plan: instance descriptors, item and record offsets and
    // projectors in one allocation, laid out as the pinned staging buffer
    DevBuf plan;
    InstDesc *d_inst = nullptr;
    long long *d_itemoff = nullptr, *d_recoff = nullptr;
    DevProjector *d_projs = nullptr;
    // a batch's results (sums, Kahan pairs, histograms, counts, error flag) in
    // one allocation, laid out as the pinned stage they are copied into
    DevBuf outb;
    long long *d_zsum = nullptr;
    double *d_kahan = nullptr;
    unsigned long long *d_hist = nullptr, *d_ips = nullptr;
    int32_t *d_sexp = nullptr;
    int *d_err = nullptr;
    unsigned long long *d_clock = nullptr;
    HostBuf hstage;  // results coming back (per-sample sums, histograms)
    HostBuf hup;     // the plan going up
    // the number of the last finished call whose results came back in one
    // block, written by the device after them (pinned), and that of the last
    // one started
    HostBuf hdone;
    uint32_t calls = 0;
    double ms_per_tick = 1e-5;  // of the device's constant-rate clock
    // the bound host stages are pinned: kernels read and write them
    bool b_pinned = false;
    // the memory the current batched call works in: the buffers above, or
    // the static scratch array (cse_exact_projector_noalloc)
    char *b_plan = nullptr, *b_out = nullptr, *b_hup = nullptr, *b_hstage = nullptr;
    uint64_t *b_recs = nullptr;
    uint32_t *b_stack = nullptr;
    unsigned long long *b_queue = nullptr;
    int32_t *b_sexp1 = nullptr, *b_terms = nullptr;
    // this device's copy of the static scratch array (nullptr if its address
    // could not be obtained; scratch_err says why)
    char *scratch = nullptr;
    char scratch_err[160] = {0};
    bool thr_ready = false;
    // exact mode: terms of one instance after which a wave flushes its
    // partial histogram (CSE_FLUSH_TERMS in the environment, at most and by
    // default CSE_FLUSH_TERMS_MAX)
    long long flush_terms = CSE_FLUSH_TERMS_MAX;
};

// ------------------------------------------------- static scratch array
// cse_exact_projector_noalloc works in this file-scope device array instead
// of allocated buffers: the work queue, the plan, the results block, the
// projection exponents and the records of one instance of chi <= 2^13.  Each
// device holds its own copy for the life of the process; its address is
// taken once per device with hipGetSymbolAddress when the first context on
// that device is created, and host code only ever uses that address.
constexpr int kStaticMaxLogChi = 13;
constexpr long long kStaticMaxChi = 1ll << kStaticMaxLogChi;
constexpr size_t kStaticPlanBytes = 4096;  // one instance: 3,328 B
constexpr size_t kStaticOutBytes = 8448;   // one instance's results block: 8,320 B
constexpr size_t kScratchQueue = 0;
constexpr size_t kScratchPlan = 256;
constexpr size_t kScratchOut = kScratchPlan + kStaticPlanBytes;
constexpr size_t kScratchSexp = kScratchOut + kStaticOutBytes;
constexpr size_t kScratchRecs = kScratchSexp + 4 * (size_t)kStaticMaxChi;
constexpr size_t kScratchBytes = kScratchRecs + (size_t)REC_WORDS * 8 * (size_t)kStaticMaxChi;  // 4,502,016 B
static_assert(kScratchOut % 256 == 0 && kScratchSexp % 256 == 0 && kScratchRecs % 256 == 0, "scratch parts aligned");

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxScratchDevices = 64;
static std::mutex g_scratch_mu;
static char *g_scratch_ptr[kMaxScratchDevices];
static bool g_scratch_tried[kMaxScratchDevices];
static char g_scratch_msg[kMaxScratchDevices][128];

namespace {

// The message is formatted into a local buffer first: an argument may be
// the context's own previous message (fail(ctx, rc, "...: %s", ctx->err)).
int fail(cse_ctx *c, int code, const char *fmt, ...) {
    char msg[sizeof(c->err)];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(msg, sizeof(msg), fmt, ap);
    va_end(ap);
    memcpy(c->err, msg, sizeof(msg));
    return code;
}

#define HIPCHK(expr)                                                                      \
    do {                                                                                  \
        hipError_t e_ = (expr);                                                           \
        if (e_ != hipSuccess)                                                             \
            return fail(ctx, CSE_ERR_HIP, "%s: %s (%s:%d)", #expr, hipGetErrorString(e_), \
                        __FILE__, __LINE__);                                              \
    } while (0)

int ensure(cse_ctx *ctx, DevBuf &b, size_t bytes) {
    if (bytes == 0) bytes = 8;
    if (b.cap >= bytes) return CSE_OK;
    if (b.p) HIPCHK(hipFree(b.p));
    b.p = nullptr;
    b.cap = 0;
    size_t want = bytes + bytes / 4;
    hipError_t e = hipMalloc(&b.p, want);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return fail(ctx, CSE_ERR_NOMEM, "hipMalloc(%zu): %s", want, hipGetErrorString(e));
    }
    b.cap = want;
    return CSE_OK;
}

#define ENSURE(buf, bytes)                            \
    do {                                              \
        int rc_ = ensure(ctx, ctx->buf, (bytes));     \
        if (rc_) return rc_;                          \
    } while (0)

int ensure_host(cse_ctx *ctx, HostBuf &b, size_t bytes) {
    if (b.cap >= bytes) return CSE_OK;
    if (b.p) HIPCHK(hipHostFree(b.p));
    b.p = nullptr;
    b.cap = 0;
    size_t want = bytes + bytes / 4;
    hipError_t e = hipHostMalloc(&b.p, want, hipHostMallocCoherent);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return fail(ctx, CSE_ERR_NOMEM, "hipHostMalloc(%zu): %s", want, hipGetErrorString(e));
    }
    b.cap = want;
    return CSE_OK;
}

template <typename T>
T *dp(DevBuf &b) { return (T *)b.p; }

int zero64(cse_ctx *ctx, void *p, long long words) {
    if (words <= 0) return CSE_OK;
    int blocks = (int)((words + 255) / 256);
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_zero64, dim3(blocks), dim3(256), 0, ctx->stream, (unsigned long long *)p, words);
    HIPCHK(hipGetLastError());
    return CSE_OK;
}

int ensure_thresholds(cse_ctx *ctx) {
    if (ctx->thr_ready) return CSE_OK;
    std::vector<uint64_t> thr(65 * 65, 0);
    for (int n = 1; n <= 64; n++) cse_dimension_thresholds(n, &thr[65 * n]);
    ENSURE(thr, thr.size() * 8);
    HIPCHK(hipMemcpyAsync(ctx->thr.p, thr.data(), thr.size() * 8, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    ctx->thr_ready = true;
    return CSE_OK;
}

// products: for an |H^t> instance's sweep, the generators in the coordinates
// of its records (to_products: u = x_2q in column 2q and s = x_2q + x_2q+1 in
// column 2q+1, after a controlled sign on each pair).  i^m Z(z) X(x) picks up
// the sign of x_u x_v, z_u ^= x_v and z_v ^= x_u from the controlled sign;
// then z_u ^= z_v and x_s = x_u + x_v.
void to_dev(DevProjector &d, const cse_projector *P, bool products = false) {
    d.nstabs = P->nstabs;
    for (int g = 0; g < P->nstabs && g < 64; g++) {
        d.phase[g] = P->phase[g] & 3;
        uint64_t x = P->xs[g], z = P->zs[g];
        if (products) {
            const int pairs = P->nqubits & ~1;
            const uint64_t even = 0x5555555555555555ull & (pairs >= 64 ? ~0ull : (1ull << pairs) - 1);
            const uint64_t xu = x & even, xv = (x >> 1) & even;
            d.phase[g] = (d.phase[g] + 2 * (__builtin_popcountll(xu & xv) & 1)) & 3;
            z ^= xv | (xu << 1);
            z ^= (z >> 1) & even;
            x ^= xu << 1;
        }
        d.xs[g] = x;
        d.zs[g] = z;
    }
}

int check_projector(cse_ctx *ctx, const cse_projector *P) {
    if (!P) return fail(ctx, CSE_ERR_ARG, "projector is NULL");
    if (P->nqubits < 1 || P->nqubits > CSE_NMAX)
        return fail(ctx, CSE_ERR_ARG, "projector width t=%d outside [1, %d]", P->nqubits, CSE_NMAX);
    if (P->nstabs < 1 || P->nstabs > CSE_NMAX)
        return fail(ctx, CSE_ERR_ARG, "projector has %d generators (need 1..%d)", P->nstabs, CSE_NMAX);
    uint64_t m = P->nqubits == 64 ? ~0ull : ((1ull << P->nqubits) - 1);
    for (int g = 0; g < P->nstabs; g++)
        if ((P->xs[g] & ~m) || (P->zs[g] & ~m))
            return fail(ctx, CSE_ERR_ARG, "generator %d has bits beyond t=%d", g, P->nqubits);
    return CSE_OK;
}

double elapsed(hipEvent_t a, hipEvent_t b) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, a, b) != hipSuccess) return 0.0;
    return (double)ms;
}

// Records for instances [0, ninst): mode 0 random states (sample indices
// first + i), mode 1 projected decomposition states.  Then the sweep.
struct Plan {
    int ninst = 0;
    InstDesc *inst = nullptr;
    long long *rec_off = nullptr;   // ninst + 1
    long long *item_off = nullptr;  // ninst + 1
    DevProjector *projs = nullptr;
    long long nrec = 0, nitems = 0, nterms = 0;
    long long stack_words = 0;  // per lane and wave, beyond LDS
    int nmax = 0;
    bool anyH = false;
    int copies = 1;       // of the results block, see spread_sums
    bool values = false;  // exact mode: sums go to the host, not histograms
    // counts the instances, whose descriptors are complete but for their
    // offsets: instance i has nr(i) records and nt(i) terms
    template <class R, class T> void finish(int n, R &&nr, T &&nt) {
        rec_off[0] = item_off[0] = 0;
        for (ninst = 0; ninst < n; ninst++) {
            InstDesc &d = inst[ninst];
            d.rec_off = nrec;
            d.term_off = nterms;
            nrec += nr(ninst);
            nitems += (d.lanes + 255) / 256;
            nterms += nt(ninst);
            nmax = std::max(nmax, d.n);
            anyH = anyH || d.exact;
            stack_words = std::max(stack_words, (long long)d.beyond);
            rec_off[ninst + 1] = nrec;
            item_off[ninst + 1] = nitems;
        }
    }
};

// Plan layout: instance descriptors, item and record offsets, projectors,
// each part 256-byte aligned.  Returns the total size.
size_t plan_layout(int n, size_t off[4]) {
    const size_t ninst = (size_t)n;
    const size_t sz[4] = {sizeof(InstDesc) * ninst, sizeof(long long) * (ninst + 1), sizeof(long long) * (ninst + 1),
                          sizeof(DevProjector) * ninst};
    size_t total = 0;
    for (int b = 0; b < 4; b++) {
        off[b] = total;
        total += (sz[b] + 255) & ~(size_t)255;
    }
    return total;
}

// A plan of n instances in a host stage, in its device layout.
Plan plan_in(char *h, int n) {
    size_t off[4];
    plan_layout(n, off);
    Plan p;
    p.inst = (InstDesc *)(h + off[0]);
    p.item_off = (long long *)(h + off[1]);
    p.rec_off = (long long *)(h + off[2]);
    p.projs = (DevProjector *)(h + off[3]);
    return p;
}

// The device pointers into the bound plan; its size.  The plan was built in
// the bound host stage, and prep_batch moves it in one launch.  Every call has
// its results before it returns, so the stage is free again at the next call.
size_t stage_plan(cse_ctx *ctx, const Plan &pl) {
    size_t off[4];
    const size_t total = plan_layout(pl.ninst, off);
    char *d = ctx->b_plan;
    ctx->d_inst = (InstDesc *)(d + off[0]);
    ctx->d_itemoff = (long long *)(d + off[1]);
    ctx->d_recoff = (long long *)(d + off[2]);
    ctx->d_projs = (DevProjector *)(d + off[3]);
    return total;
}

int run_records(cse_ctx *ctx, const Plan &pl, int mode) {
    const int ninst = pl.ninst;
    const long long waves = pl.nrec;
    const long long blocks = (waves + 3) / 4;
    if (blocks > 0) {
        hipLaunchKernelGGL(k_records, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, mode, ninst,
                           ctx->d_recoff, ctx->d_inst, ctx->d_projs,
                           mode == 0 ? dp<uint64_t>(ctx->thr) : nullptr, pl.nrec, ctx->b_recs, ctx->d_sexp,
                           ctx->d_err, ctx->d_clock);
        HIPCHK(hipGetLastError());
    }
    return CSE_OK;
}

// Layout of a batch's results block, the same on the device and in the
// pinned stage, but for the exact mode's sums, which the device has no room
// for, and its histograms where only their sums are wanted, which stay there.
// Sampled mode (0): per-sample Z[omega] sums (32 B), Kahan pairs (16 B) and
// projection exponents (4 B), then per-instance counts and the error flag.
// Exact mode (1): per-instance histograms or sums (Plan::values), Kahan pairs
// and counts, then the error flag; both end with the clock readings.  (With
// the histograms after the counts, their atomics in one cache line with those
// of the counts, 2^22 terms of one instance take 3 us more.)
struct OutLayout {
    size_t vals, zsum, kahan, sexp, hist, ips, err, clock;
    size_t copied;  // the end of what comes back
    size_t total;   // of one copy, a multiple of 256 bytes where there are several
};

OutLayout out_layout(const Plan &pl, int mode) {
    const size_t n = (size_t)pl.nrec, ni = (size_t)pl.ninst;
    OutLayout o;
    memset(&o, 0, sizeof(o));
    if (mode == 0) {
        o.zsum = 0;
        o.kahan = 32 * n;
        o.sexp = 48 * n;
        o.ips = (52 * n + 7) & ~(size_t)7;
    } else {
        o.kahan = pl.values ? 64 * ni : 8 * (size_t)HIST_STRIDE * ni;
        o.ips = o.kahan + 16 * ni;
    }
    o.err = o.ips + 8 * ni;
    o.clock = o.err + 8;  // three readings, see BatchTimes
    o.copied = o.total = (o.clock + 3 * 8 + 15) & ~(size_t)15;
    if (pl.values) {
        o.hist = (o.copied + 255) & ~(size_t)255;
        o.total = o.hist + 8 * (size_t)HIST_STRIDE * ni;
    }
    if (pl.copies > 1) o.total = (o.total + 255) & ~(size_t)255;
    return o;
}

// The sweep kernel of a launch, by its widest state (slots beyond 32 cost
// registers: 128 VGPRs, four waves per SIMD, up to 48 slots, three waves
// beyond) and whether some instance has |H^t> terms (their signs cost four
// instructions a step).
typedef void (*SweepFn)(SweepArgs);
struct SweepKernel {
    SweepFn fn;
    int blocks_per_cu;
};
SweepKernel sweep_choice(const Plan &pl, int mode) {
    static const SweepFn fn[2][2][3] = {{{k_sweep_s32, k_sweep_s48, k_sweep_s64}, {k_sweep_sh32, k_sweep_sh48, k_sweep_sh64}},
                                        {{k_sweep_e32, k_sweep_e48, k_sweep_e64}, {k_sweep_eh32, k_sweep_eh48, k_sweep_eh64}}};
    const int w = pl.nmax <= 32 ? 0 : pl.nmax <= 48 ? 1 : 2, h = pl.anyH ? 1 : 0;
    SweepKernel k;
    k.fn = fn[mode][h][w];
    static const SweepFn copies[3] = {k_sweep_c32, k_sweep_c48, k_sweep_c64};
    if (pl.copies > 1) k.fn = copies[w];
    k.blocks_per_cu = w == 2 ? 3 : 4;
    return k;
}

// persistent grid: the resident blocks, or the items if they are fewer
int sweep_grid(const cse_ctx *ctx, const Plan &pl, const SweepKernel &k) {
    return (int)std::max(1ll, std::min((long long)ctx->cus * k.blocks_per_cu, pl.nitems));
}

// The blocks of a launch of one exact instance all add their sums to the same
// 8 KB at their end.  From 256 blocks on they add to TREE_COPIES copies, which
// the results kernel adds up: calls of t = 24, k = 11 take 88.8 us with one
// copy, 80.6 with 4 or 8, 82.2 with 16, those of k = 10 58.9 and 56.0.  Below
// (t = 20, k = 8) the copies cost 1 us, and |H^t> sums, which fall into fewer
// bins, gain nothing (t = 24: 114.7 us with one copy, 116.8 with 8).
void spread_sums(const cse_ctx *ctx, Plan &pl) {
    if (pl.anyH || sweep_grid(ctx, pl, sweep_choice(pl, 1)) < 256) return;
    pl.copies = TREE_COPIES;
}

// Binds a batch to the context's own buffers, grown on demand (device memory
// and the pinned host stage of the results; the plan is in ctx->hup).
int bind_ctx_mem(cse_ctx *ctx, const Plan &pl, int mode, bool want_terms) {
    size_t off[4];
    const size_t pbytes = plan_layout(pl.ninst, off);
    const OutLayout o = out_layout(pl, mode);
    ENSURE(plan, pbytes);
    ENSURE(outb, o.total * (size_t)pl.copies);
    ENSURE(recs, (size_t)REC_WORDS * 8 * (size_t)pl.nrec);
    ENSURE(queue, 16);
    ENSURE(stack, (size_t)pl.stack_words * 64 * 4 * 4 * (size_t)sweep_grid(ctx, pl, sweep_choice(pl, mode)));
    if (mode == 1) ENSURE(sexp, 4 * (size_t)pl.nrec);
    if (want_terms) ENSURE(terms, 4 * (size_t)(pl.nterms > 0 ? pl.nterms : 1));
    int rc = ensure_host(ctx, ctx->hstage, o.copied);
    if (rc) return rc;
    ctx->b_pinned = true;
    ctx->b_plan = (char *)ctx->plan.p;
    ctx->b_out = (char *)ctx->outb.p;
    ctx->b_recs = dp<uint64_t>(ctx->recs);
    ctx->b_queue = dp<unsigned long long>(ctx->queue);
    ctx->b_stack = dp<uint32_t>(ctx->stack);
    ctx->b_sexp1 = mode == 1 ? dp<int32_t>(ctx->sexp) : nullptr;
    ctx->b_terms = want_terms ? dp<int32_t>(ctx->terms) : nullptr;
    ctx->b_hup = (char *)ctx->hup.p;
    ctx->b_hstage = (char *)ctx->hstage.p;
    return CSE_OK;
}

// Binds a one-instance exact-mode batch to this device's static scratch
// array and the caller's host stages; allocates nothing.
int bind_static_mem(cse_ctx *ctx, const Plan &pl, char *hup, char *hstage) {
    if (!ctx->scratch) return fail(ctx, CSE_ERR_HIP, "static scratch array unavailable: %s", ctx->scratch_err);
    size_t off[4];
    const size_t pbytes = plan_layout(pl.ninst, off);
    const OutLayout o = out_layout(pl, 1);
    if (pl.nrec > kStaticMaxChi)
        return fail(ctx, CSE_ERR_ARG, "chi=%lld above the no-allocation limit 2^%d", pl.nrec, kStaticMaxLogChi);
    if (pbytes > kStaticPlanBytes || o.total > kStaticOutBytes)
        return fail(ctx, CSE_ERR_ARG, "internal: plan or results of %zu / %zu B above the static stages", pbytes,
                    o.total);
    ctx->b_queue = (unsigned long long *)(ctx->scratch + kScratchQueue);
    ctx->b_plan = ctx->scratch + kScratchPlan;
    ctx->b_out = ctx->scratch + kScratchOut;
    ctx->b_sexp1 = (int32_t *)(ctx->scratch + kScratchSexp);
    ctx->b_recs = (uint64_t *)(ctx->scratch + kScratchRecs);
    ctx->b_stack = nullptr;  // its trees stay in LDS
    ctx->b_terms = nullptr;
    ctx->b_hup = hup;
    ctx->b_hstage = hstage;
    ctx->b_pinned = false;
    return CSE_OK;
}

// One launch that brings the staged plan to the device and clears the bound
// results block (every sum, count and flag; the exponents are rewritten by
// the record launch) and the work queue.  From pinned memory the kernel reads
// the plan itself: a copy call of its own costs 6 us of host time and, before
// kernels, a wait of the command processor (copy, three launches, copy and
// three events took 46 us, the same four launches without them 19).
int prep_batch(cse_ctx *ctx, const Plan &pl, int mode, size_t plan_bytes) {
    const OutLayout o = out_layout(pl, mode);
    char *b = ctx->b_out;
    ctx->d_zsum = mode == 0 ? (long long *)(b + o.zsum) : nullptr;
    ctx->d_kahan = (double *)(b + o.kahan);
    ctx->d_sexp = mode == 0 ? (int32_t *)(b + o.sexp) : ctx->b_sexp1;
    ctx->d_hist = mode == 1 ? (unsigned long long *)(b + o.hist) : nullptr;
    ctx->d_ips = (unsigned long long *)(b + o.ips);
    ctx->d_err = (int *)(b + o.err);
    ctx->d_clock = (unsigned long long *)(b + o.clock);
    PrepArgs a;
    a.src = (const uint4 *)ctx->b_hup;
    a.dst = (uint4 *)ctx->b_plan;
    a.ncopy = ctx->b_pinned ? (long long)(plan_bytes / 16) : 0;
    a.zero = (uint4 *)b;
    a.nzero = (long long)(o.total * (size_t)pl.copies / 16);
    a.queue = ctx->b_queue;
    if (!ctx->b_pinned)
        HIPCHK(hipMemcpyAsync(ctx->b_plan, ctx->b_hup, plan_bytes, hipMemcpyHostToDevice, ctx->stream));
    const long long most = std::max(a.ncopy, a.nzero);
    hipLaunchKernelGGL(k_prep, dim3((unsigned)std::min<long long>(4096, (most + 255) / 256)), dim3(256), 0,
                       ctx->stream, a);
    HIPCHK(hipGetLastError());
    return CSE_OK;
}

int run_sweep(cse_ctx *ctx, const Plan &pl, int mode, bool want_terms) {
    SweepArgs A;
    memset(&A, 0, sizeof(A));
    A.ninst = pl.ninst;
    A.nitems = pl.nitems;
    A.item_off = ctx->d_itemoff;
    A.flush_terms = ctx->flush_terms;
    A.inst = ctx->d_inst;
    A.recs = ctx->b_recs;
    A.queue = ctx->b_queue;
    A.stack = ctx->b_stack;
    A.stack_words = pl.stack_words;
    A.leaf = dp<uint8_t>(ctx->leaf) + (pl.anyH ? 1 << tree::LeafBits<false>::value : 0);
    A.terms = want_terms ? ctx->b_terms : nullptr;
    A.zsum = ctx->d_zsum;
    A.kahan = ctx->d_kahan;
    A.hist = ctx->d_hist;
    A.ips = ctx->d_ips;
    A.clock = ctx->d_clock;
    A.err = ctx->d_err;
    A.copy_words = (unsigned)(out_layout(pl, mode).total / 8);
    const SweepKernel k = sweep_choice(pl, mode);
    hipLaunchKernelGGL(k.fn, dim3(sweep_grid(ctx, pl, k)), dim3(256), 0, ctx->stream, A);
    HIPCHK(hipGetLastError());
    return CSE_OK;
}

// Results come back in kernel stores (at 64 KB to 1 MB 14 to 32 us against 21
// to 39 of a copy call), followed by the call's number, which the host polls:
// 2 to 4 us less than a wait for the stream.  Results of more than kPollBytes
// belong to calls of milliseconds, which outlast the polling; beyond
// kGridBytes they come back in a copy call.
constexpr size_t kPollBytes = 1 << 20;
constexpr size_t kGridBytes = 64 << 20;

// Runs a bound, staged batch, in stream order: plan and clear, records,
// sweep, results (and, with terms, their copies to the caller, which `copy`
// enqueues), and waits for it.
template <class F> int run_batch(cse_ctx *ctx, const Plan &pl, int mode, bool want_terms, size_t plan_bytes, F &&copy) {
    int rc = prep_batch(ctx, pl, mode, plan_bytes);
    if (!rc) rc = run_records(ctx, pl, mode);
    if (!rc) rc = run_sweep(ctx, pl, mode, want_terms);
    if (rc) return rc;
    const OutLayout o = out_layout(pl, mode);
    const size_t first = pl.values ? o.kahan : 0;  // the sums are written by the kernel itself
    const size_t bytes = o.copied - first;
    const bool dma = !ctx->b_pinned || bytes > kGridBytes;
    const bool poll = !dma && bytes <= kPollBytes && !want_terms;
    ResultArgs a;
    a.src = (const uint4 *)(ctx->b_out + first);
    a.dst = (uint4 *)(ctx->b_hstage + first);
    a.n = dma ? 0 : (long long)(bytes / 16);
    a.clock = ctx->d_clock + 2;
    a.hist = ctx->d_hist;
    a.vals = (double *)(ctx->b_hstage + o.vals);
    a.nvals = pl.values ? pl.ninst : 0;
    a.copies = pl.copies;
    a.tail = (int)((o.kahan - first) / 8);
    a.copy_words = (long long)(o.total / 8);
    a.left = (unsigned *)(ctx->b_queue + 1);
    a.done = poll ? (uint32_t *)ctx->hdone.p : nullptr;
    a.call = ++ctx->calls;
    // small results in one block: no count to wait for
    const long long blocks =
        std::min<long long>(1024, std::max((a.nvals + 3ll) / 4, bytes <= 16384 ? 1 : (a.n + 255) / 256));
    hipLaunchKernelGGL(pl.copies > 1 ? k_results_copies : k_results, dim3((unsigned)std::max(1ll, blocks)), dim3(256),
                       0, ctx->stream, a);
    HIPCHK(hipGetLastError());
    if (dma)
        HIPCHK(hipMemcpyAsync(ctx->b_hstage + first, ctx->b_out + first, bytes, hipMemcpyDeviceToHost, ctx->stream));
    if (want_terms) {
        rc = copy();
        if (rc) return rc;
    }
    if (poll) {
        // about a millisecond of polling, then the stream's own wait (long calls,
        // and whatever goes wrong on the device)
        const uint32_t *done = (const uint32_t *)ctx->hdone.p;
        for (int i = 0; i < 20000; i++) {
            if (__atomic_load_n(done, __ATOMIC_ACQUIRE) == a.call) return CSE_OK;
            __builtin_ia32_pause();
        }
    }
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return CSE_OK;
}

// Device times of a finished batch from its clock readings: at the start of
// the records, of the sweep, and of the results copy.
struct BatchTimes {
    double records, sweep;
};
BatchTimes batch_times(const cse_ctx *ctx, const OutLayout &o) {
    const unsigned long long *c = (const unsigned long long *)(ctx->b_hstage + o.clock);
    BatchTimes t;
    t.records = (double)(long long)(c[1] - c[0]) * ctx->ms_per_tick;
    t.sweep = (double)(long long)(c[2] - c[1]) * ctx->ms_per_tick;
    return t;
}

// Cost model of a lane's tree, in VALU instructions: a step of slot c takes
// about 58 for its own state (a signed one, |H^t>, 8 more) and 7 for every
// slot below it, a slot beyond 32 14 for those beyond; a term's sums take
// about 60.  The 7 is a fit: a row takes 6, but the kernels of wide states also
// wait for their scratch, which the model has no term for (with 6 t = 63, k =
// 10, 512 samples take 138 us for 126, and the others what they took).
double step_cost(int c, bool h) {
    return c < 32 ? 58.0 + (h ? 8 : 0) + 7.0 * c : 90.0 + (h ? 10 : 0) + 7.0 * 32 + 14.0 * (c - 32);
}
// of the slots below c
struct StepCosts {
    double sum[2][65];
    StepCosts() {
        for (int h = 0; h < 2; h++) {
            sum[h][0] = 0.0;
            for (int c = 0; c < 64; c++) sum[h][c + 1] = sum[h][c] + step_cost(c, h != 0);
        }
    }
};

// What an instance's lane (W) and all its lanes on one SIMD's share of them
// (work) take for each G up to top, in VALU instructions.
struct TreeCosts {
    int top;
    float W[TREE_MAXG + 1], work[TREE_MAXG + 1];
};

// The terms of index bit 0 are summed in pairs (cse_tree.h) where that bit
// moves more slots than are looked up, in launches without |H^t> instances
// (d.pair as make_inst leaves it): those have bits that move one slot and a
// sign, and the code for pairs next to their own costs them 4 to 20% (exact
// t = 30 3.26 -> 3.38 ms, 512 samples of t = 40 3.43 -> 4.12 ms).
bool tree_pairs(const InstDesc &d) { return d.pair && d.ub[1] > TREE_LEAF && d.ub[1] <= 32; }

// Levels of a tree have at most 32 slots, but in launches with states of more
// than 48 and no |H^t> instances (whose bits move two slots at a time: none
// gets that far): 8192 samples of t = 63, k = 10 1.26 -> 0.86 ms, 4096 of t =
// 56, k = 12 1.26 -> 0.98 ms (means of four).  The kernel of 33 to 48 slots
// has 128 registers, and with the code for such levels in it 2^28 terms of t =
// 48 take 10.0 -> 10.6 ms and 2000 samples of t = 37 101 -> 108 us.
int tree_levels(int nmax, bool signs) { return nmax > 48 && !signs ? 64 : 32; }

// lds_only: the stack has to stay in LDS.
void tree_costs(InstDesc &d, TreeCosts &c, int mode, long long nrec, int simds, bool lds_only, int max_terms) {
    const int lds = mode == 0 ? TREE_LDS_WORDS0 : TREE_LDS_WORDS1;
    static const StepCosts costs;
    const double *sum = costs.sum[d.exact];
    auto steps = [&](int lo, int hi) { return hi > lo ? sum[hi] - sum[lo] : 0.0; };
    const int top = std::min(d.k, TREE_MAXG);
    for (int g = 0; g <= top; g++) d.ub[g] = (uint8_t)std::max((int)d.ub[g], TREE_LEAF);
    int words = 0;
    double below = 0.0;  // steps of the slots below ub[g], per term
    for (int g = 0; g <= top; g++) {
        if (g > 0) {
            if (d.ub[g] > d.levels || (1ll << g) > max_terms) break;
            const bool pair = g == 1 && tree_pairs(d);
            if (d.ub[g] > TREE_LEAF && !pair) words += tree_words(d.ub[g]);
            if (lds_only && words > lds) break;
            below += pair ? 0.5 * steps(0, d.ub[1]) : steps(d.ub[g - 1], d.ub[g]) / (double)(1ll << (g - 1));
        }
        const double W = (below + 60.0) * (double)(1ll << g) + steps(d.ub[g], d.n) + 500.0;
        const double lanes = (double)nrec * (double)(d.chi >> g) * (mode == 0 ? 1.0 : 0.5);
        c.top = g;
        c.W[g] = (float)W;
        c.work[g] = (float)(W * std::max(lanes / 64.0, 1.0) / simds);
    }
}

// An instance's G and stack.
void set_tree(InstDesc &d, int mode, long long nrec, int G) {
    const int lds = mode == 0 ? TREE_LDS_WORDS0 : TREE_LDS_WORDS1;
    d.G = G;
    int words = 0;
    const bool pairs = tree_pairs(d);
    d.nlds = d.leaf = d.beyond = d.pair = 0;
    for (int g = 1; g <= d.G; g++) {
        const int w = tree_words(d.ub[g]);
        if (d.ub[g] <= TREE_LEAF) {
            d.leaf = d.nlds = g;
        } else if (g == 1 && pairs) {
            d.leaf = d.nlds = d.pair = 1;
        } else if (d.nlds == g - 1 && words + w <= lds) {
            d.soff[g] = (uint16_t)words;
            words += w;
            d.nlds = g;
        } else {
            d.soff[g] = (uint16_t)d.beyond;
            d.beyond += w;
        }
    }
    const long long per = d.chi >> d.G;
    d.lanes = mode == 0 ? nrec * per : tri_before(1ll << d.G, per, per);
}

// The G of each instance.  A launch takes about the work of all its lanes
// spread over the SIMDs plus one lane's tree, the last to finish; a larger G
// shares more of the work and makes the trees longer.  So the longest tree is
// bounded, by the bound that gives the least sum (steps of 2^(1/4)), and each
// instance takes its cheapest G within it.  (192 uneven instances 3.9 -> 3.4
// ms, 20 small ones 42 -> 28 us against each instance on its own.)
constexpr int kBounds = 96;
inline double tree_bound(int b) { return 512.0 * exp2(0.25 * b); }
// the first bound of at least W
inline int bound_of(float W) {
    int e;
    const float m = frexpf(W / 512.0f, &e);  // in [1/2, 1)
    return 4 * (e - 1) + (m > 0.5f) + (m > 0.59460356f) + (m > 0.70710678f) + (m > 0.84089642f);
}
inline int cheapest(const TreeCosts &c, double bound) {
    int best = 0;
    for (int g = 1; g <= c.top; g++)
        if (c.W[g] <= bound * 1.0001 && c.work[g] < c.work[best]) best = g;
    return best;
}
double best_bound(const TreeCosts *c, int n) {
    double sum[kBounds] = {0};
    int first = kBounds, last = 0;
    for (int i = 0; i < n; i++) {
        // the work under each bound: the cheapest G so far, bound by bound
        double least = c[i].work[0];
        int b = 0;
        for (int g = 1; g <= c[i].top; g++) {
            const int at = std::min(kBounds - 1, std::max(0, bound_of(c[i].W[g])));
            if (g == 1) first = std::min(first, at);
            last = std::max(last, at);
            for (; b < at; b++) sum[b] += least;
            least = std::min(least, (double)c[i].work[g]);
        }
        for (; b < kBounds; b++) sum[b] += least;
    }
    int best = std::max(0, std::min(first, last) - 1);
    for (int b = best; b <= last; b++)
        if (sum[b] + tree_bound(b) < sum[best] + tree_bound(best)) best = b;
    return tree_bound(best);
}

// the bit of a slot in a record's words
uint64_t slot_word(int x) { return x < 32 ? 1ull << (31 - x) : 1ull << (95 - x); }

// An instance's descriptor but for its tree, and what its trees cost.  mode 0:
// nsamp records; mode 1: chi records.  signs: a launch with |H^t> instances;
// levels: tree_levels of the launch.
// max_terms > 0 bounds the terms of a lane (the calls' chunk).
void make_inst(InstDesc &d, TreeCosts &c, const cse_ctx *ctx, int mode, int t, int k, int exact, const uint64_t *L,
               long long nsamp, bool signs, int levels, bool lds_only, int max_terms) {
    memset(d.ub, 0, sizeof(d.ub));
    memset(d.soff, 0, sizeof(d.soff));
    d.n = t;
    d.k = exact ? (t + 1) / 2 : k;
    d.exact = exact ? 1 : 0;
    d.pair = signs ? 0 : 1;
    d.levels = levels;
    d.chi = 1ll << d.k;
    uint8_t col[64];
    if (exact) {
        // bit b of j is pair size-1-b; its slots are u = x_2q (signed) below
        // s = x_2q + x_2q+1, and the lone qubit of odd t is slot 0
        const int odd = t & 1;
        for (int b = 0; b < d.k; b++) {
            const int q = d.k - 1 - b, u = 2 * b - odd, s = u + 1;
            col[s] = (uint8_t)(odd && b == 0 ? t - 1 : 2 * q + 1);
            if (u >= 0) col[u] = (uint8_t)(2 * q);
            d.LP[b] = slot_word(s);
            d.LT[b] = u >= 0 ? slot_word(u) : 0ull;
            d.col[b] = 1ull << col[s];
            d.sgn[b] = u >= 0 ? 1ull << col[u] : 0ull;
            d.jmap[b] = 1u << b;
            if (b < TREE_MAXG) d.ub[b + 1] = (uint8_t)(s + 1);
        }
    } else {
        cse_chain_basis(t, k, L, TREE_MAXG, d.col, d.jmap, d.ub, col);
        uint8_t pos[64];
        for (int p = 0; p < t; p++) pos[col[p]] = (uint8_t)p;
        for (int b = 0; b < k; b++) {
            uint64_t w = 0;
            for (uint64_t r = d.col[b]; r; r &= r - 1) w |= slot_word(pos[__builtin_ctzll(r)]);
            d.LP[b] = w;
            d.LT[b] = d.sgn[b] = 0;
        }
    }
    for (int p = 0; p < 64; p++) d.inv[p] = p < t ? col[p] : (uint8_t)p;
    tree_costs(d, c, mode, mode == 0 ? nsamp : d.chi, 4 * ctx->cus, lds_only, max_terms > 0 ? max_terms : 1 << 30);
}

// chi <= 2^30 keeps every per-theta Z[omega] sum exact in int64: a term is at
// most 2^32 in each component at the 2^32 fixed-point scale, so chi terms stay
// below 2^62.  (The reference holds chi in an int, innerprod.c:122-131.)
constexpr int kMaxLogChi = 30;
// samples (records) per sampled-mode call
constexpr long long kMaxSamples = 1ll << 24;

int check_decomp(cse_ctx *ctx, int t, int k, int exact, const uint64_t *L) {
    if (exact) {
        if ((t + 1) / 2 > kMaxLogChi)
            return fail(ctx, CSE_ERR_ARG, "exact decomposition chi=2^%d exceeds 2^%d", (t + 1) / 2, kMaxLogChi);
        return CSE_OK;
    }
    if (k < 0 || k > kMaxLogChi) return fail(ctx, CSE_ERR_ARG, "k=%d outside [0, %d]", k, kMaxLogChi);
    if (k > 0 && !L) return fail(ctx, CSE_ERR_ARG, "L is NULL");
    uint64_t m = t == 64 ? ~0ull : ((1ull << t) - 1);
    for (int r = 0; r < k; r++)
        if (L[r] & ~m) return fail(ctx, CSE_ERR_ARG, "row %d of L has bits beyond t=%d", r, t);
    return CSE_OK;
}

// the message of the calling thread's last failed cse_create (no context
// exists to hold it); cse_error(NULL) returns it
thread_local char g_create_err[256];

// a state-level call's count (pairs, states) is passed to its kernel as an
// int, and its grid is count / 4 blocks
constexpr size_t kMaxStates = size_t(1) << 30;

int init_ctx(cse_ctx *ctx, int device) {
    ctx->device = device;
    HIPCHK(hipSetDevice(device));
    HIPCHK(hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking));
    HIPCHK(hipEventCreate(&ctx->e0));
    HIPCHK(hipEventCreate(&ctx->e1));
    hipDeviceProp_t prop;
    HIPCHK(hipGetDeviceProperties(&prop, device));
    ctx->cus = prop.multiProcessorCount;
    snprintf(ctx->name, sizeof(ctx->name), "%s (%s)", prop.name, prop.gcnArchName);
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        return fail(ctx, CSE_ERR_HIP, "device %d is %s; this engine is built for gfx950", device, prop.gcnArchName);
    int khz = 0;
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device) == hipSuccess && khz > 0)
        ctx->ms_per_tick = 1.0 / khz;
    const int rc_done = ensure_host(ctx, ctx->hdone, 64);
    if (rc_done) return rc_done;
    memset(ctx->hdone.p, 0, 64);
    // the sweep's leaf tables, kept for the context's life
    const int plain = 1 << tree::LeafBits<false>::value, sign = 1 << tree::LeafBits<true>::value;
    ENSURE(leaf, (size_t)(plain + sign));
    hipLaunchKernelGGL(k_leaf_table, dim3((sign + 63) / 64), dim3(64), 0, ctx->stream, dp<uint8_t>(ctx->leaf),
                       dp<uint8_t>(ctx->leaf) + plain);
    HIPCHK(hipGetLastError());
    if (const char *ft = getenv("CSE_FLUSH_TERMS")) {
        const long long v = atoll(ft);
        if (v < 1 || v > CSE_FLUSH_TERMS_MAX)
            return fail(ctx, CSE_ERR_ARG, "CSE_FLUSH_TERMS=%s outside [1, %lld]", ft, CSE_FLUSH_TERMS_MAX);
        ctx->flush_terms = v;
    }
    // this device's copy of the static scratch array, once per device (with
    // the device current); a failure only disables the no-allocation call
    if (device < kMaxScratchDevices) {
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        if (!g_scratch_tried[device]) {
            g_scratch_tried[device] = true;
            void *p = nullptr;
            const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
            if (e == hipSuccess && p) {
                g_scratch_ptr[device] = (char *)p;
            } else {
                (void)hipGetLastError();
                snprintf(g_scratch_msg[device], sizeof(g_scratch_msg[device]), "hipGetSymbolAddress: %s",
                         e != hipSuccess ? hipGetErrorString(e) : "null address");
            }
        }
        ctx->scratch = g_scratch_ptr[device];
        if (!ctx->scratch) snprintf(ctx->scratch_err, sizeof(ctx->scratch_err), "%s", g_scratch_msg[device]);
    } else {
        snprintf(ctx->scratch_err, sizeof(ctx->scratch_err), "device index %d above %d", device,
                 kMaxScratchDevices - 1);
    }
    return CSE_OK;
}

}  // namespace

// ====================================================================== ABI
extern "C" {

int cse_create(int device, cse_ctx **out) {
    g_create_err[0] = 0;
    if (!out) {
        snprintf(g_create_err, sizeof(g_create_err), "cse_create: NULL output pointer");
        return CSE_ERR_ARG;
    }
    *out = nullptr;
    int count = 0;
    hipError_t e = hipGetDeviceCount(&count);
    if (e != hipSuccess || count == 0) {
        (void)hipGetLastError();
        snprintf(g_create_err, sizeof(g_create_err), "cse_create: no HIP device (%s)",
                 e != hipSuccess ? hipGetErrorString(e) : "device count 0");
        return CSE_ERR_HIP;
    }
    if (device < 0 || device >= count) {
        snprintf(g_create_err, sizeof(g_create_err), "cse_create: device %d outside [0, %d)", device, count);
        return CSE_ERR_ARG;
    }
    cse_ctx *ctx = new cse_ctx();
    const int rc = init_ctx(ctx, device);
    if (rc != CSE_OK) {
        snprintf(g_create_err, sizeof(g_create_err), "cse_create: %s", ctx->err);
        cse_destroy(ctx);
        return rc;
    }
    *out = ctx;
    return CSE_OK;
}

void cse_destroy(cse_ctx *ctx) {
    if (!ctx) return;
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    DevBuf *bufs[] = {&ctx->s1, &ctx->s2, &ctx->out, &ctx->recs, &ctx->terms, &ctx->queue, &ctx->thr,
                      &ctx->sexp, &ctx->L, &ctx->idx, &ctx->errflag, &ctx->lsh, &ctx->plan, &ctx->outb, &ctx->stack, &ctx->leaf};
    for (DevBuf *b : bufs)
        if (b->p) (void)hipFree(b->p);
    if (ctx->hstage.p) (void)hipHostFree(ctx->hstage.p);
    if (ctx->hup.p) (void)hipHostFree(ctx->hup.p);
    if (ctx->hdone.p) (void)hipHostFree(ctx->hdone.p);
    if (ctx->e0) (void)hipEventDestroy(ctx->e0);
    if (ctx->e1) (void)hipEventDestroy(ctx->e1);
    if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
    delete ctx;
}

const char *cse_error(const cse_ctx *ctx) {
    if (ctx) return ctx->err;
    return g_create_err[0] ? g_create_err : "no context";
}

int cse_set_sweep_kernel(cse_ctx *ctx, int mode, int kernel) {
    if (!ctx) return CSE_ERR_ARG;
    if (mode < 0 || mode > 1) return fail(ctx, CSE_ERR_ARG, "sweep mode %d outside [0, 1]", mode);
    if (kernel < 0 || kernel > 2) return fail(ctx, CSE_ERR_ARG, "sweep kernel %d outside [0, 2]", kernel);
    return CSE_OK;  // there is one a mode and width
}

int cse_set_graphs(cse_ctx *ctx, int enable) {
    (void)enable;
    return ctx ? CSE_OK : CSE_ERR_ARG;
}

int cse_device_info(cse_ctx *ctx, int *cus, char *name, int name_len) {
    if (!ctx) return CSE_ERR_ARG;
    if (cus) *cus = ctx->cus;
    if (name && name_len > 0) snprintf(name, (size_t)name_len, "%s", ctx->name);
    return CSE_OK;
}

int cse_inner_products(cse_ctx *ctx, int n, size_t npairs, const uint64_t *s1, const uint64_t *s2,
                       int32_t *out, int one_launch_per_pair, double *ms) {
    if (!ctx) return CSE_ERR_ARG;
    if (n < 1 || n > CSE_NMAX) return fail(ctx, CSE_ERR_ARG, "n=%d outside [1, %d]", n, CSE_NMAX);
    if (npairs == 0) {
        if (ms) *ms = 0;
        return CSE_OK;
    }
    if (!s1 || !s2 || !out) return fail(ctx, CSE_ERR_ARG, "NULL buffer");
    if (npairs > kMaxStates) return fail(ctx, CSE_ERR_ARG, "%zu pairs above 2^30 per call", npairs);
    const size_t words = (size_t)CSE_STATE_WORDS(n);
    for (size_t i = 0; i < npairs; i++) {
        const uint64_t *a = s1 + words * i, *b = s2 + words * i;
        if ((int)(a[0] & 0xff) != n || (int)(b[0] & 0xff) != n)
            return fail(ctx, CSE_ERR_ARG, "pair %zu: header n does not match n=%d", i, n);
        if ((int)((a[0] >> 8) & 0xff) > n || (int)((b[0] >> 8) & 0xff) > n)
            return fail(ctx, CSE_ERR_ARG, "pair %zu: k > n", i);
    }
    HIPCHK(hipSetDevice(ctx->device));
    ENSURE(s1, words * 8 * npairs);
    ENSURE(s2, words * 8 * npairs);
    ENSURE(out, 12 * npairs);
    HIPCHK(hipMemcpyAsync(ctx->s1.p, s1, words * 8 * npairs, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(ctx->s2.p, s2, words * 8 * npairs, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipEventRecord(ctx->e0, ctx->stream));
    if (one_launch_per_pair) {
        for (size_t i = 0; i < npairs; i++) {
            hipLaunchKernelGGL(k_ip_pairs, dim3(1), dim3(64), 0, ctx->stream, dp<uint64_t>(ctx->s1) + words * i,
                               dp<uint64_t>(ctx->s2) + words * i, n, 1, dp<int32_t>(ctx->out) + 3 * i);
        }
    } else {
        const size_t blocks = (npairs + 3) / 4;
        hipLaunchKernelGGL(k_ip_pairs, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, dp<uint64_t>(ctx->s1),
                           dp<uint64_t>(ctx->s2), n, (int)npairs, dp<int32_t>(ctx->out));
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(ctx->e1, ctx->stream));
    HIPCHK(hipMemcpyAsync(out, ctx->out.p, 12 * npairs, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    if (ms) *ms = elapsed(ctx->e0, ctx->e1);
    return CSE_OK;
}

int cse_prep_states(cse_ctx *ctx, int exact, int t, const uint64_t *L, int k, const uint64_t *idx, size_t count,
                    uint64_t *out) {
    if (!ctx) return CSE_ERR_ARG;
    if (t < 1 || t > CSE_NMAX) return fail(ctx, CSE_ERR_ARG, "t=%d outside [1, %d]", t, CSE_NMAX);
    if (count == 0) return CSE_OK;
    int rc = check_decomp(ctx, t, k, exact, L);
    if (rc) return rc;
    if (!idx || !out) return fail(ctx, CSE_ERR_ARG, "NULL buffer");
    if (count > kMaxStates) return fail(ctx, CSE_ERR_ARG, "%zu states above 2^30 per call", count);
    const uint64_t chi = exact ? (1ull << ((t + 1) / 2)) : (1ull << k);
    for (size_t c = 0; c < count; c++)
        if (idx[c] >= chi) return fail(ctx, CSE_ERR_ARG, "index %llu >= chi", (unsigned long long)idx[c]);
    HIPCHK(hipSetDevice(ctx->device));
    const size_t words = (size_t)CSE_STATE_WORDS(t);
    ENSURE(L, 8 * 64);
    ENSURE(idx, 8 * count);
    ENSURE(s1, 8 * words * count);
    if (!exact && k > 0) HIPCHK(hipMemcpyAsync(ctx->L.p, L, 8 * (size_t)k, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(ctx->idx.p, idx, 8 * count, hipMemcpyHostToDevice, ctx->stream));
    hipLaunchKernelGGL(k_prep_states, dim3((unsigned)((count + 3) / 4)), dim3(256), 0, ctx->stream, exact, t,
                       dp<uint64_t>(ctx->L), k, dp<uint64_t>(ctx->idx), (int)count, dp<uint64_t>(ctx->s1));
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(out, ctx->s1.p, 8 * words * count, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return CSE_OK;
}

int cse_random_states(cse_ctx *ctx, int n, uint64_t seed, int64_t first, size_t count, const cse_projector *P,
                      uint64_t *out, int32_t *sexp) {
    if (!ctx) return CSE_ERR_ARG;
    if (n < 1 || n > CSE_NMAX) return fail(ctx, CSE_ERR_ARG, "n=%d outside [1, %d]", n, CSE_NMAX);
    if (count == 0) return CSE_OK;
    if (count > kMaxStates) return fail(ctx, CSE_ERR_ARG, "%zu states above 2^30 per call", count);
    if (P) {
        int rc = check_projector(ctx, P);
        if (rc) return rc;
        if (P->nqubits != n) return fail(ctx, CSE_ERR_ARG, "projector width %d != n %d", P->nqubits, n);
    }
    HIPCHK(hipSetDevice(ctx->device));
    int rc = ensure_thresholds(ctx);
    if (rc) return rc;
    const size_t words = (size_t)CSE_STATE_WORDS(n);
    ENSURE(s1, 8 * words * count);
    ENSURE(sexp, 4 * count);
    ENSURE(errflag, 8);
    rc = zero64(ctx, ctx->errflag.p, 1);
    if (rc) return rc;
    DevProjector dpj;
    memset(&dpj, 0, sizeof(dpj));
    if (P) to_dev(dpj, P);
    hipLaunchKernelGGL(k_random_states, dim3((unsigned)((count + 3) / 4)), dim3(256), 0, ctx->stream, n,
                       dp<uint64_t>(ctx->thr) + 65 * n, seed, (long long)first, (int)count, dpj, P ? 1 : 0,
                       out ? dp<uint64_t>(ctx->s1) : nullptr, dp<int32_t>(ctx->sexp), dp<int>(ctx->errflag));
    HIPCHK(hipGetLastError());
    int errv = 0;
    HIPCHK(hipMemcpyAsync(&errv, ctx->errflag.p, 4, hipMemcpyDeviceToHost, ctx->stream));
    if (out) HIPCHK(hipMemcpyAsync(out, ctx->s1.p, 8 * words * count, hipMemcpyDeviceToHost, ctx->stream));
    if (sexp) HIPCHK(hipMemcpyAsync(sexp, ctx->sexp.p, 4 * count, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    if (errv) return fail(ctx, CSE_ERR_RNG, "random state draw exceeded its shrink cap");
    return CSE_OK;
}

// Sampled-mode instances [0, ninst): one record launch and one sweep over all
// of them, then each instance's estimator from its own samples.
// Runs job(w) for w in [0, nw): w >= 1 on threads of their own, w = 0 on the
// caller's.  A thread that cannot be started leaves its job to the caller.
extern "C++" template <class F>
static void run_jobs(int nw, F &&job) {
    std::vector<std::thread> pool;
    int w = 1;
    try {
        for (; w < nw; w++) pool.emplace_back(job, w);
    } catch (...) {
    }
    for (int v = w; v < nw; v++) job(v);
    job(0);
    for (std::thread &th : pool) th.join();
}

// job(lo, hi) over [0, n): on several threads from 128 on, where the instances
// of most launches of that many pay for a thread's start (15 us): one takes 1
// us at t = 13, k = 5, 2 at t = 40, k = 8, 14 at t = 48, k = 12 and 100 at t =
// 64, k = 30 (whose 2^30 terms take milliseconds)
extern "C++" template <class F>
static void run_ranges(int n, F &&job) {
    const unsigned hw = std::thread::hardware_concurrency();
    const int nw = n >= 128 ? (int)std::min(4u, hw ? hw : 1u) : 1;
    if (nw == 1) return job(0, n);
    const int per = (n + nw - 1) / nw;
    run_jobs(nw, [&](int w) { job(std::min(n, w * per), std::min(n, (w + 1) * per)); });
}

// One instance's estimators over count samples: fixed parts of kEstPart
// samples (so the Kahan mean depends on count alone), spread over nthr host
// threads.  At 2^16 samples one thread takes about 0.5 ms.
constexpr int64_t kEstPart = 8192;
static void split_estimators(int t, int64_t count, const long long *z, const int32_t *se, const double *kz,
                             int nthr, double *mean, double *mean_kahan) {
    const int nparts = (int)((count + kEstPart - 1) / kEstPart);
    if (nparts < 2) {
        cse_sampled_estimators(t, count, z, se, kz, mean, mean_kahan);
        return;
    }
    std::vector<cse_est_part> parts((size_t)nparts);
    nthr = std::max(1, std::min(nthr, nparts));
    auto work = [&](int w) {
        for (int q = w; q < nparts; q += nthr)
            cse_est_accumulate(&parts[(size_t)q], t, q * kEstPart, std::min(count, (q + 1) * kEstPart), z, se, kz);
    };
    run_jobs(nthr, work);
    cse_est_finish(parts.data(), nparts, t, count, mean, mean_kahan);
}

static int sampled_batch(cse_ctx *ctx, const cse_sampled_instance *in, int ninst, int chunk,
                         cse_sampled_result *res, double *kernel_ms) {
    size_t poff[4];
    int rc = ensure_host(ctx, ctx->hup, plan_layout(ninst, poff));
    if (rc) return rc;
    Plan pl = plan_in((char *)ctx->hup.p, ninst);
    bool want_terms = false;
    for (int i = 0; i < ninst; i++) want_terms = want_terms || res[i].terms != nullptr;
    std::vector<TreeCosts> costs((size_t)ninst);
    bool signs = false;
    int nmax = 0;
    for (int i = 0; i < ninst; i++) {
        signs = signs || in[i].exact;
        nmax = std::max(nmax, in[i].P.nqubits);
    }
    const int levels = tree_levels(nmax, signs);
    run_ranges(ninst, [&](int lo, int hi) {
        for (int i = lo; i < hi; i++) {
            make_inst(pl.inst[i], costs[(size_t)i], ctx, 0, in[i].P.nqubits, in[i].k, in[i].exact, in[i].L,
                      in[i].count, signs, levels, false, chunk);
            pl.inst[i].seed = in[i].seed;
            pl.inst[i].first = in[i].first;
            to_dev(pl.projs[i], &in[i].P, in[i].exact != 0);
        }
    });
    const double bound = best_bound(costs.data(), ninst);
    for (int i = 0; i < ninst; i++) set_tree(pl.inst[i], 0, in[i].count, cheapest(costs[(size_t)i], bound));
    pl.finish(ninst, [&](int i) { return (long long)in[i].count; },
              [&](int i) { return (long long)in[i].count * pl.inst[i].chi; });
    if (pl.nrec > kMaxSamples) return fail(ctx, CSE_ERR_ARG, "%lld samples above 2^24 per call", pl.nrec);
    if (want_terms && pl.nterms > (1ll << 31)) return fail(ctx, CSE_ERR_ARG, "per-term output too large");
    rc = ensure_thresholds(ctx);
    if (!rc) rc = bind_ctx_mem(ctx, pl, 0, want_terms);
    if (rc) return rc;
    rc = run_batch(ctx, pl, 0, want_terms, stage_plan(ctx, pl), [&]() -> int {
        for (int i = 0; i < ninst; i++)
            if (res[i].terms)
                HIPCHK(hipMemcpyAsync(res[i].terms, ctx->b_terms + pl.inst[i].term_off,
                                      4 * (size_t)(in[i].count * pl.inst[i].chi), hipMemcpyDeviceToHost,
                                      ctx->stream));
        return CSE_OK;
    });
    if (rc) return rc;

    // the results block came back in one copy, into a pinned stage of the
    // same layout
    const OutLayout o = out_layout(pl, 0);
    char *hs = ctx->b_hstage;
    const long long *z = (const long long *)(hs + o.zsum);
    const double *kz = (const double *)(hs + o.kahan);
    const int32_t *se = (const int32_t *)(hs + o.sexp);
    const unsigned long long *nips = (const unsigned long long *)(hs + o.ips);
    int *errp = (int *)(hs + o.err);
    const int errv = *errp;
    if (errv & 1) return fail(ctx, CSE_ERR_RNG, "random state draw exceeded its shrink cap");
    if (errv & 2) return fail(ctx, CSE_ERR_HIP, "internal: an inner product exponent left [-64, 0]");
    const BatchTimes bt = batch_times(ctx, o);
    const double pms = bt.records, kms = bt.sweep;
    if (kernel_ms) *kernel_ms = kms;
    const unsigned hw = std::thread::hardware_concurrency();
    const int nthr = (ninst >= 8 && pl.nrec >= (1 << 16)) ? (int)std::min(8u, hw ? hw : 1u) : 1;
    // with one thread per group of instances, each instance's samples take
    // one thread; otherwise a large instance splits its samples
    const int sthr = nthr > 1 ? 1 : (int)std::min(8u, hw ? hw : 1u);
    auto convert = [&](int lo, int hi) {
        for (int i = lo; i < hi; i++) {
            cse_sampled_result *r = &res[i];
            const size_t off = (size_t)pl.rec_off[i], cnt = (size_t)in[i].count;
            r->prep_ms = pms;
            r->kernel_ms = kms;
            r->ips = (int64_t)nips[i];
            r->vanished = 0;
            for (size_t s = 0; s < cnt; s++)
                if (se[off + s] < 0) r->vanished++;
            split_estimators(in[i].P.nqubits, (int64_t)cnt, z + 4 * off, se + off, kz + 2 * off,
                             cnt >= 4 * (size_t)kEstPart ? sthr : 1, &r->mean, &r->mean_kahan);
            if (r->zsum) memcpy(r->zsum, z + 4 * off, 32 * cnt);
            if (r->sexp) memcpy(r->sexp, se + off, 4 * cnt);
            if (r->kahan) memcpy(r->kahan, kz + 2 * off, 16 * cnt);
        }
    };
    // the estimators cost about as much per sample as the copies: split large
    // batches of instances over host threads
    if (nthr > 1) {
        const int per = (ninst + nthr - 1) / nthr;
        run_jobs(nthr, [&](int w) { convert(std::min(ninst, w * per), std::min(ninst, (w + 1) * per)); });
    } else {
        convert(0, ninst);
    }
    return CSE_OK;
}

int cse_sampled_projector(cse_ctx *ctx, const cse_projector *P, const uint64_t *L, int k, int exact,
                          uint64_t seed, int64_t first, int64_t count, int chunk, cse_sampled_result *res) {
    if (!ctx || !res) return CSE_ERR_ARG;
    int rc = check_projector(ctx, P);
    if (rc) return rc;
    rc = check_decomp(ctx, P->nqubits, k, exact, L);
    if (rc) return rc;
    if (count < 1) return fail(ctx, CSE_ERR_ARG, "count=%lld", (long long)count);
    if (count > kMaxSamples) return fail(ctx, CSE_ERR_ARG, "count=%lld above 2^24 per call", (long long)count);
    HIPCHK(hipSetDevice(ctx->device));
    cse_sampled_instance in;
    memset(&in, 0, sizeof(in));
    in.P = *P;
    in.exact = exact;
    in.k = exact ? 0 : k;
    if (!exact)
        for (int r = 0; r < k; r++) in.L[r] = L[r];
    in.seed = seed;
    in.first = first;
    in.count = count;
    return sampled_batch(ctx, &in, 1, chunk, res, nullptr);
}

int cse_batch_sampled(cse_ctx *ctx, const cse_sampled_instance *inst, int ninst, int chunk,
                      cse_sampled_result *res, double *kernel_ms) {
    if (!ctx || !inst || !res || ninst < 1) return CSE_ERR_ARG;
    long long total = 0;
    for (int i = 0; i < ninst; i++) {
        int rc = check_projector(ctx, &inst[i].P);
        if (!rc) rc = check_decomp(ctx, inst[i].P.nqubits, inst[i].k, inst[i].exact, inst[i].L);
        if (rc) return fail(ctx, rc, "instance %d: %s", i, ctx->err);
        if (inst[i].count < 1) return fail(ctx, CSE_ERR_ARG, "instance %d: count=%lld", i, (long long)inst[i].count);
        total += inst[i].count;
        if (total > kMaxSamples) return fail(ctx, CSE_ERR_ARG, "more than 2^24 samples in one call");
    }
    HIPCHK(hipSetDevice(ctx->device));
    return sampled_batch(ctx, inst, ninst, chunk, res, kernel_ms);
}

// Exact-mode instances [0, ninst) in one record launch and one sweep.  With
// use_static the call works in this device's static scratch array and the
// host stages hup / hstage (of at least kStaticPlanBytes / kStaticOutBytes)
// instead of the context's buffers, and allocates nothing.
static int exact_batch(cse_ctx *ctx, const cse_instance *in, int ninst, int chunk, cse_exact_result *res,
                       int32_t *terms_out, double *kernel_ms, bool use_static = false, char *hup = nullptr,
                       char *hstage = nullptr) {
    if (use_static && ninst != 1) return fail(ctx, CSE_ERR_ARG, "internal: static call with %d instances", ninst);
    size_t poff[4];
    const size_t pbytes = plan_layout(ninst, poff);
    if (use_static && pbytes > kStaticPlanBytes)
        return fail(ctx, CSE_ERR_ARG, "internal: plan of %zu B above the static stage", pbytes);
    int rc = use_static ? CSE_OK : ensure_host(ctx, ctx->hup, pbytes);
    if (rc) return rc;
    Plan pl = plan_in(use_static ? hup : (char *)ctx->hup.p, ninst);
    pl.values = !use_static;
    for (int i = 0; i < ninst; i++) pl.values = pl.values && !res[i].hist;
    TreeCosts one;
    std::vector<TreeCosts> many((size_t)(ninst > 1 ? ninst : 0));
    TreeCosts *const costs = ninst > 1 ? many.data() : &one;
    bool signs = false;
    int nmax = 0;
    for (int i = 0; i < ninst; i++) {
        signs = signs || in[i].exact;
        nmax = std::max(nmax, in[i].P.nqubits);
    }
    const int levels = tree_levels(nmax, signs);
    run_ranges(ninst, [&](int lo, int hi) {
        for (int i = lo; i < hi; i++) {
            make_inst(pl.inst[i], costs[i], ctx, 1, in[i].P.nqubits, in[i].k, in[i].exact, in[i].L, 0, signs,
                      levels, use_static, chunk);
            to_dev(pl.projs[i], &in[i].P, in[i].exact != 0);
        }
    });
    const double bound = best_bound(costs, ninst);
    for (int i = 0; i < ninst; i++) set_tree(pl.inst[i], 1, pl.inst[i].chi, cheapest(costs[i], bound));
    pl.finish(ninst, [&](int i) { return pl.inst[i].chi; },
              [&](int i) { return pl.inst[i].chi * (pl.inst[i].chi + 1) / 2; });
    if (terms_out && pl.nterms > (1ll << 31)) return fail(ctx, CSE_ERR_ARG, "per-term output too large");
    if (ninst == 1 && !use_static) spread_sums(ctx, pl);
    rc = use_static ? bind_static_mem(ctx, pl, hup, hstage) : bind_ctx_mem(ctx, pl, 1, terms_out != nullptr);
    if (rc) return rc;
    rc = run_batch(ctx, pl, 1, terms_out != nullptr, stage_plan(ctx, pl), [&]() -> int {
        HIPCHK(hipMemcpyAsync(terms_out, ctx->b_terms, 4 * (size_t)pl.nterms, hipMemcpyDeviceToHost, ctx->stream));
        return CSE_OK;
    });
    if (rc) return rc;
    // the results block came back into a host stage of the same layout
    const OutLayout o = out_layout(pl, 1);
    char *hs = ctx->b_hstage;
    const unsigned long long *hist = (const unsigned long long *)(hs + o.hist);
    const double *kz = (const double *)(hs + o.kahan);
    const unsigned long long *nips = (const unsigned long long *)(hs + o.ips);
    if (*(const int *)(hs + o.err) & 2)
        return fail(ctx, CSE_ERR_HIP, "internal: an inner product exponent left [-64, 0]");
    const BatchTimes bt = batch_times(ctx, o);
    const double kms = bt.sweep, tms = bt.records + bt.sweep;
    if (kernel_ms) *kernel_ms = kms;
    // each instance's exact value, from its sums or from its histogram (2.5 us
    // each: split over host threads for large batches)
    auto convert = [&](int lo, int hi) {
        for (int i = lo; i < hi; i++) {
            cse_exact_result *r = &res[i];
            r->pmin = CSE_HIST_PMIN;
            if (pl.values) {
                cse_hist_finish((const cse_dd *)(hs + o.vals) + 4 * (size_t)i, &r->re, &r->im);
            } else {
                const int64_t *h = (const int64_t *)&hist[(size_t)HIST_STRIDE * i];
                if (r->hist) memcpy(r->hist, h, 8 * (size_t)HIST_STRIDE);
                cse_hist_value(h, CSE_HIST_PMIN, &r->re, &r->im);
            }
            r->value = hypot(r->re, r->im);
            r->kahan_re = kz[2 * i];
            r->kahan_im = kz[2 * i + 1];
            r->terms = pl.inst[i].chi * (pl.inst[i].chi + 1) / 2;
            r->ips = (int64_t)nips[i];
            r->kernel_ms = kms;
            r->total_ms = tms;
        }
    };
    const unsigned hw = std::thread::hardware_concurrency();
    const int nthr = ninst >= 512 && !pl.values ? (int)std::min(8u, hw ? hw : 1u) : 1;
    if (nthr > 1) {
        const int per = (ninst + nthr - 1) / nthr;
        run_jobs(nthr, [&](int w) { convert(std::min(ninst, w * per), std::min(ninst, (w + 1) * per)); });
    } else {
        convert(0, ninst);
    }
    return CSE_OK;
}

int cse_exact_projector(cse_ctx *ctx, const cse_projector *P, const uint64_t *L, int k, int exact,
                        cse_exact_result *res) {
    if (!ctx || !res) return CSE_ERR_ARG;
    int rc = check_projector(ctx, P);
    if (rc) return rc;
    rc = check_decomp(ctx, P->nqubits, k, exact, L);
    if (rc) return rc;
    HIPCHK(hipSetDevice(ctx->device));
    cse_instance in;
    memset(&in, 0, sizeof(in));
    in.P = *P;
    in.exact = exact;
    in.k = exact ? 0 : k;
    if (!exact)
        for (int r = 0; r < k; r++) in.L[r] = L[r];
    return exact_batch(ctx, &in, 1, 0, res, nullptr, nullptr);
}

int cse_exact_projector_noalloc(cse_ctx *ctx, const cse_projector *P, const uint64_t *L, int k, int exact,
                                cse_exact_result *res) {
    if (!ctx || !res) return CSE_ERR_ARG;
    int rc = check_projector(ctx, P);
    if (rc) return rc;
    rc = check_decomp(ctx, P->nqubits, k, exact, L);
    if (rc) return rc;
    const int logchi = exact ? (P->nqubits + 1) / 2 : k;
    if (logchi > kStaticMaxLogChi)
        return fail(ctx, CSE_ERR_ARG, "chi=2^%d above the no-allocation limit 2^%d", logchi, kStaticMaxLogChi);
    HIPCHK(hipSetDevice(ctx->device));
    cse_instance in;
    memset(&in, 0, sizeof(in));
    in.P = *P;
    in.exact = exact;
    in.k = exact ? 0 : k;
    if (!exact)
        for (int r = 0; r < k; r++) in.L[r] = L[r];
    // host stages on the stack: pageable copies, synchronized before return
    alignas(256) char hup[kStaticPlanBytes];
    alignas(256) char hstage[kStaticOutBytes];
    return exact_batch(ctx, &in, 1, 0, res, nullptr, nullptr, true, hup, hstage);
}

int cse_batch_exact(cse_ctx *ctx, const cse_instance *inst, int ninst, int chunk, cse_exact_result *res,
                    int32_t *terms_out, double *kernel_ms) {
    if (!ctx || !inst || !res || ninst < 1) return CSE_ERR_ARG;
    for (int i = 0; i < ninst; i++) {
        int rc = check_projector(ctx, &inst[i].P);
        if (!rc) rc = check_decomp(ctx, inst[i].P.nqubits, inst[i].k, inst[i].exact, inst[i].L);
        if (rc) return fail(ctx, rc, "instance %d: %s", i, ctx->err);
    }
    HIPCHK(hipSetDevice(ctx->device));
    return exact_batch(ctx, inst, ninst, chunk, res, terms_out, kernel_ms);
}

int cse_lspace_weights(cse_ctx *ctx, const uint64_t *L, int k, int64_t *hist) {
    if (!ctx || !hist || (k > 0 && !L)) return CSE_ERR_ARG;
    if (k < 0 || k > 40) return fail(ctx, CSE_ERR_ARG, "k=%d outside [0, 40]", k);
    HIPCHK(hipSetDevice(ctx->device));
    ENSURE(lsh, 8 * 65);
    ENSURE(L, 8 * (size_t)CSE_NMAX);
    if (k > 0) HIPCHK(hipMemcpyAsync(ctx->L.p, L, 8 * (size_t)k, hipMemcpyHostToDevice, ctx->stream));
    int rc = zero64(ctx, ctx->lsh.p, 65);
    if (rc) return rc;
    // 2^(k - shift) threads, each walking 2^shift combinations
    const int shift = k > 18 ? k - 18 : 0;
    const uint64_t threads = 1ull << (k - shift);
    const unsigned blocks = (unsigned)((threads + 255) / 256);
    hipLaunchKernelGGL(k_lspace_hist, dim3(blocks), dim3(256), 0, ctx->stream, dp<uint64_t>(ctx->L), k, shift,
                       dp<unsigned long long>(ctx->lsh));
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(hist, ctx->lsh.p, 8 * 65, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return CSE_OK;
}

}  // extern "C"
