// Runs the sweep kernels (csrc/cse_sweep.h) on the CPU: a block is 256 fibers,
// a wave's 64 meet at every cross-lane operation, and waves run one after the
// other, in a given order, from barrier to barrier.  What a wave does is only
// seen by a wave that runs later, so a missing barrier shows.
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <ucontext.h>

#include <algorithm>
#include <vector>

#define __host__
#define __device__
#define __global__
#define __forceinline__ inline
#define __shared__ static
#define __launch_bounds__(...)
#define __align__(n) __attribute__((aligned(n)))
#define DEV inline

typedef unsigned long long u64;
struct Dim {
    unsigned x = 0;
};
static Dim threadIdx, blockIdx, blockDim, gridDim;

namespace fiber {
enum Stop { MEET, BARRIER, DONE };
constexpr size_t kStack = 256 << 10;
struct Lane {
    ucontext_t at;
    std::vector<char> stack = std::vector<char>(kStack);
    Stop stop;
    unsigned meets;
};
static Lane lane[256];
static ucontext_t host;
static u64 slot[4][2][64];
static void (*body)();
static void stop(Stop s) {
    Lane &l = lane[threadIdx.x];
    l.stop = s;
    swapcontext(&l.at, &host);
}
static void enter() {
    body();
    stop(DONE);
}
// every lane's v, after all of the wave have come here
static const u64 *meet(u64 v) {
    const unsigned t = threadIdx.x, half = lane[t].meets++ & 1u;
    slot[t >> 6][half][t & 63] = v;
    stop(MEET);
    return slot[t >> 6][half];
}
static Stop run_wave(int w) {
    while (true) {
        for (int l = 64 * w; l < 64 * w + 64; l++) {
            threadIdx.x = (unsigned)l;
            swapcontext(&host, &lane[l].at);
            if (lane[l].stop != lane[64 * w].stop) {
                fprintf(stderr, "lanes of wave %d stopped at different places\n", w);
                abort();
            }
        }
        if (lane[64 * w].stop != MEET) return lane[64 * w].stop;
    }
}
static void run_block(void (*f)(), const int *order) {
    body = f;
    for (Lane &l : lane) {
        getcontext(&l.at);
        l.at.uc_stack.ss_sp = l.stack.data();
        l.at.uc_stack.ss_size = kStack;
        l.at.uc_link = nullptr;
        l.meets = 0;
        makecontext(&l.at, enter, 0);
    }
    for (int done = 0; done < 4;) {
        done = 0;
        for (int i = 0; i < 4; i++) done += run_wave(order[i]) == DONE;
        if (done != 0 && done != 4) {
            fprintf(stderr, "%d waves of a block ended while others wait\n", done);
            abort();
        }
    }
}
}  // namespace fiber

static void __syncthreads() { fiber::stop(fiber::BARRIER); }
static int cpu_readlane(int v, int l) { return (int)fiber::meet((unsigned)v)[l & 63]; }
#define __builtin_amdgcn_readlane cpu_readlane
#define __builtin_amdgcn_readfirstlane(v) cpu_readlane((v), 0)
static double __shfl_xor(double v, int m, int) {
    u64 w;
    memcpy(&w, &v, 8);
    w = fiber::meet(w)[(threadIdx.x ^ (unsigned)m) & 63];
    memcpy(&v, &w, 8);
    return v;
}
template <class T, class V> static T atomicAdd(T *p, V v) {
    const T was = *p;
    *p = (T)(was + v);
    return was;
}
static int atomicOr(int *p, int v) {
    const int was = *p;
    *p = was | v;
    return was;
}
static unsigned long long wall_clock64() { return 0; }
static int __popc(unsigned v) { return __builtin_popcount(v); }

namespace cse {
DEV int lane_id() { return (int)(threadIdx.x & 63); }
DEV u64 lowmask(int k) { return k >= 64 ? ~0ull : (1ull << k) - 1ull; }
DEV u64 rl64(u64 v, int l) { return fiber::meet(v)[l & 63]; }
DEV u64 uniform64(u64 v) { return rl64(v, 0); }
DEV u64 shfl_xor64(u64 v, int m) { return fiber::meet(v)[lane_id() ^ m]; }
DEV u64 ballot(bool p) {
    const u64 *s = fiber::meet(p);
    u64 b = 0;
    for (int l = 0; l < 64; l++) b |= s[l] << l;
    return b;
}
// each half's bits in reverse
DEV u64 brev32x2(u64 v) {
    u64 r = 0;
    for (int b = 0; b < 64; b++)
        if (v >> b & 1) r |= 1ull << (b < 32 ? 31 - b : 95 - b);
    return r;
}
}  // namespace cse
using namespace cse;

#include "cse_internal.h"
#include "cse_tree.h"
DEV int find_instance(const long long *off, int n, long long key) {
    int i = 0;
    while (i + 1 < n && off[i + 1] <= key) i++;
    return i;
}
#include "sweep_host.h"  // cse_sweep.h without its asm statement

namespace {
std::vector<InstDesc> inst;
std::vector<long long> item_off;
std::vector<uint64_t> recs;
std::vector<uint8_t> leaf;
SweepArgs args;
void (*kernel)(SweepArgs);
void call() { kernel(args); }
long long nrec, nterms, stack_words;
}  // namespace

extern "C" {
// A new launch; then its instances, one by one.
void sweep_begin() {
    inst.clear();
    item_off.assign(1, 0);
    recs.clear();
    nrec = nterms = stack_words = 0;
}
// An instance of n slots and 2^k terms: index bit b toggles the slots LP[b] and
// the signs LT[b]; bits below g stay below slot ub[g].  G, the tree's levels
// and their stack as set_tree in cse_engine.hip lays them out, with `lds` words
// of it in LDS; pairs: the engine would let index bit 0 be summed in pairs.
int sweep_add(int mode, int n, int k, int exact, int G, const uint8_t *ub, const uint64_t *LP, const uint64_t *LT,
              int pairs, int lds, int count, const uint64_t *rec) {
    InstDesc d;
    memset(&d, 0, sizeof d);
    d.n = n;
    d.k = k;
    d.exact = exact;
    d.G = G;
    d.chi = 1ll << k;
    d.rec_off = nrec;
    d.term_off = nterms;
    for (int b = 0; b < k; b++) {
        d.LP[b] = LP[b];
        d.LT[b] = LT[b];
        d.jmap[b] = 1u << b;
    }
    for (int g = 0; g <= G; g++) d.ub[g] = (uint8_t)std::max((int)ub[g], TREE_LEAF);
    int words = 0;
    for (int g = 1; g <= G; g++) {
        const int w = tree_words(d.ub[g]);
        if (d.ub[g] <= TREE_LEAF) {
            d.leaf = d.nlds = g;
        } else if (g == 1 && pairs && d.ub[1] <= 32) {
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
    const long long per = d.chi >> G;
    d.lanes = mode == 0 ? count * per : tri_before(1ll << G, per, per);
    inst.push_back(d);
    recs.insert(recs.end(), rec, rec + (size_t)REC_WORDS * (size_t)count);
    nrec += count;
    nterms += mode == 0 ? count * d.chi : d.chi * (d.chi + 1) / 2;
    stack_words = std::max(stack_words, (long long)d.beyond);
    item_off.push_back(item_off.back() + (d.lanes + 255) / 256);
    return (int)item_off.back();
}
// Runs it with `grid` blocks whose waves run in the order given; the error flags.
int sweep_run(int mode, int nh, int ht, int copies, int grid, const int *order, long long flush_terms, int32_t *terms,
               long long *zsum, double *kahan, unsigned long long *hist, unsigned long long *ips, int copy_words) {
    static void (*const fn[2][2][3])(SweepArgs) = {
        {{k_sweep_s32, k_sweep_s48, k_sweep_s64}, {k_sweep_sh32, k_sweep_sh48, k_sweep_sh64}},
        {{k_sweep_e32, k_sweep_e48, k_sweep_e64}, {k_sweep_eh32, k_sweep_eh48, k_sweep_eh64}}};
    static void (*const cp[3])(SweepArgs) = {k_sweep_c32, k_sweep_c48, k_sweep_c64};
    const int plain = 1 << tree::LeafBits<false>::value, sign = 1 << tree::LeafBits<true>::value;
    leaf.resize((size_t)(plain + sign));
    blockDim.x = 64;
    for (blockIdx.x = 0; blockIdx.x < (unsigned)sign / 64; blockIdx.x++)
        for (threadIdx.x = 0; threadIdx.x < 64; threadIdx.x++) k_leaf_table(leaf.data(), leaf.data() + plain);
    unsigned long long queue[2] = {0, 0}, clock[3];
    int err = 0;
    std::vector<uint32_t> stack((size_t)stack_words * 256 * (size_t)grid);
    memset(&args, 0, sizeof args);
    args.ninst = (int)inst.size();
    args.nitems = item_off.back();
    args.item_off = item_off.data();
    args.flush_terms = flush_terms;
    args.inst = inst.data();
    args.recs = recs.data();
    args.queue = queue;
    args.stack = stack.data();
    args.stack_words = stack_words;
    args.leaf = leaf.data() + (ht ? plain : 0);
    args.terms = terms;
    args.zsum = zsum;
    args.kahan = kahan;
    args.hist = hist;
    args.ips = ips;
    args.clock = clock;
    args.err = &err;
    args.copy_words = (unsigned)copy_words;
    kernel = copies ? cp[nh / 16] : fn[mode][ht][nh / 16];
    blockDim.x = 256;
    gridDim.x = (unsigned)grid;
    for (int b = 0; b < grid; b++) {
        blockIdx.x = (unsigned)b;
        fiber::run_block(call, order);
    }
    return err;
}
// Adds q to the phase of record r of instance i.
void sweep_phase(int i, int r, int q) {
    uint64_t &w = recs[(size_t)REC_WORDS * (size_t)(inst[(size_t)i].rec_off + r)];
    w = (w & ~(7ull << 16)) | (uint64_t)(((int)(w >> 16) + q) & 7) << 16;
}
// The terms of record r of instance i, each by itself: (eps, p, m).
void sweep_terms(int i, int r, int *out) {
    const InstDesc &d = inst[(size_t)i];
    const uint64_t *rec = recs.data() + (size_t)REC_WORDS * (size_t)(d.rec_off + r);
    for (long long j = 0; j < d.chi; j++, out += 3) {
        uint64_t A = d.exact ? brev32x2(lowmask(d.n)) : 0ull, T = 0;
        for (int b = 0; b < d.k; b++)
            if (j >> b & 1) {
                A ^= d.LP[b];
                T ^= d.LT[b];
            }
        A ^= rec[1];
        tree::Form<32> f;
        memset(&f, 0, sizeof f);
        for (int x = 0; x < 64; x++) {
            f.lo[x] = (uint32_t)rec[REC_ROWS + x];
            if (x >= 32) f.hi[x - 32] = (uint32_t)(rec[REC_ROWS + x] >> 32);
        }
        f.A = (uint32_t)A, f.Ah = (uint32_t)(A >> 32);
        f.T = (uint32_t)T, f.Th = (uint32_t)(T >> 32);
        f.d1 = (uint32_t)rec[2], f.d1h = (uint32_t)(rec[2] >> 32);
        f.d2 = (uint32_t)rec[3], f.d2h = (uint32_t)(rec[3] >> 32);
        tree::StepsHi<32, true, 31>::run(f, d.n);
        tree::steps<32, true>(f, d.n < 32 ? d.n : 32, 0);
        int ph = (int)(rec[0] >> 16 & 7), cnt = -d.n;
        tree::fold<true>(f.d1h, f.d2h, f.Ah, f.Th, ~0u, ph, cnt);
        tree::fold<true>(f.d1, f.d2, f.A, f.T, ~0u, ph, cnt);
        out[0] = f.z >> 31 || rec[0] >> 40 & 1 ? 0 : 1;
        out[1] = cnt - (int)f.nb;
        out[2] = (ph + 2 * (int)f.q1 + 4 * __builtin_popcount(f.x2)) & 7;
    }
}
}
