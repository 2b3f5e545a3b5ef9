// cse_sweep.h -- the sweep over decomposition terms: part of cse_kernels.hip.
//
// Work: a lane takes one record (projected state) and 2^G consecutive terms
// of it, j = (jh << G) + 0 .. 2^G - 1 in the instance's own index order.  The
// slots of the form are ordered so that index bits below g toggle slots below
// ub[g] only: a lane sums out the slots from ub[G] on once, those from ub[g]
// on once per setting of the bits g .. G - 1, and a term of its own costs the
// slots below ub[1].  It walks that binary tree depth first in Gray code
// order, with the form at the last visited node of every level on a stack
// (LDS for the deepest levels, which are visited most, the device's memory
// for the others).  All lanes of a block belong to one instance, so slot
// order, levels and stack addresses are uniform, and lanes differ in masks
// only: one VALU instruction advances 64 terms.  (One wave per term, rows in
// lanes, takes 160 vector and 160 scalar instructions per term at 48 qubits;
// the tree takes 34 to 36 vector and 1.5 scalar ones.)
#pragma once

namespace {

// instance descriptors are read through the scalar cache
typedef const __attribute__((address_space(4))) InstDesc CInst;

DEV int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Record r and block c of local lane l of an exact-mode instance: block g is
// the last with tri_before(g) <= l (the root of the quadratic, then an
// integer correction of at most a step or two), then the lane within it.
DEV void tri_item(long long l, long long ch, long long nch, long long &r, long long &c) {
    const double a = 2.0 * (double)nch + 1.0;
    long long g = (long long)((a - sqrt(a * a - 8.0 * (double)l / (double)ch)) * 0.5);
    if (g < 0) g = 0;
    if (g > nch - 1) g = nch - 1;
    while (g < nch - 1 && tri_before(ch, nch, g + 1) <= l) g++;
    while (g > 0 && tri_before(ch, nch, g) > l) g--;
    const long long off = l - tri_before(ch, nch, g), per = nch - g;
    r = g * ch + off / per;
    c = g + off % per;
}

// Compensated FP32 sum s - c, plus v.  The rounding error of s + v is taken by
// Knuth's two-sum, exact whichever of the two is larger, and only summed up in
// c: what is lost is of the order of n eps^2, so a lane's sum has the error of
// its FP32 terms alone, however many it adds.  (Kahan's own step loses part of
// the error wherever a term is larger than the sum so far: over random terms
// the relative error is 3.0e-8 with runs of 4, 3.7e-8 with runs of 32, 3.9e-8
// with runs of 256; this one 3.0e-8.)
DEV void kahan1(float &s, float &c, float v) {
    const float t = s + v, b = t - s;
    c -= (s - (t - b)) + (v - b);
    s = t;
}

DEV double wave_sumf64(double v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}
DEV long long wave_sum64(long long v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += (long long)shfl_xor64((u64)v, off);
    return v;
}

// Saves the slots below c of a form (and its state words) to words 0 .. of p,
// 64 lanes apart, and reads them back.  A holds toggles of the current term
// that are not part of the node: `a` is A without them.
template <int NH, int X> DEV void rows_save(const tree::Form<NH> &f, int c, uint32_t *p) {
    if constexpr (X < 32) {
        if (c <= X) return;
        p[64 * (TREE_STATE_WORDS + X)] = f.lo[X];
        if (c > X + 1) p[64 * (TREE_STATE_WORDS + X + 1)] = f.lo[X + 1];
        rows_save<NH, X + 2>(f, c, p);
    }
}
template <int NH, int X> DEV void rows_load(tree::Form<NH> &f, int c, const uint32_t *p) {
    if constexpr (X < 32) {
        if (c <= X) return;
        f.lo[X] = p[64 * (TREE_STATE_WORDS + X)];
        if (c > X + 1) f.lo[X + 1] = p[64 * (TREE_STATE_WORDS + X + 1)];
        rows_load<NH, X + 2>(f, c, p);
    }
}
template <int NH> DEV void form_save(const tree::Form<NH> &f, unsigned a, int c, uint32_t *p) {
    p[0] = f.d1;
    p[64] = f.d2;
    p[128] = a;
    p[192] = f.x2;
    p[256] = (f.z & 0x80000000u) | (f.q1 << 8) | f.nb;
    rows_save<NH, 0>(f, c, p);
}
template <int NH> DEV void form_load(tree::Form<NH> &f, int c, const uint32_t *p) {
    f.d1 = p[0];
    f.d2 = p[64];
    f.A = p[128];
    f.x2 = p[192];
    const unsigned w = p[256];
    f.z = w & 0x80000000u;
    f.q1 = (w >> 8) & 0xffu;
    f.nb = w & 0xffu;
    rows_load<NH, 0>(f, c, p);
}
// the rest of a form on c > 32 slots, after the first 32 rows
constexpr int kHigh = TREE_STATE_WORDS + 32;
template <int NH, int X> DEV void rows_save_high(const tree::Form<NH> &f, int c, uint32_t *p) {
    if constexpr (X < NH) {
        if (c <= 32 + X) return;
        p[64 * (kHigh + TREE_HIGH_WORDS + 2 * X)] = f.lo[32 + X];
        p[64 * (kHigh + TREE_HIGH_WORDS + 2 * X + 1)] = f.hi[X];
        rows_save_high<NH, X + 1>(f, c, p);
    }
}
template <int NH> DEV void form_save_high(const tree::Form<NH> &f, unsigned a, int c, uint32_t *p) {
    p[64 * kHigh] = f.d1h;
    p[64 * (kHigh + 1)] = f.d2h;
    p[64 * (kHigh + 2)] = a;
    rows_save_high<NH, 0>(f, c, p);
}
template <int NH> DEV void form_load_high(tree::Form<NH> &f, int c, const uint32_t *p) {
    f.d1h = p[64 * kHigh];
    f.d2h = p[64 * (kHigh + 1)];
    f.Ah = p[64 * (kHigh + 2)];
#pragma unroll
    for (int x = 0; x < NH; x++) {
        // (every row gets a value, so none has to be kept from before)
        f.lo[32 + x] = f.hi[x] = 0;
        if (c > 32 + x) {
            f.lo[32 + x] = p[64 * (kHigh + TREE_HIGH_WORDS + 2 * x)];
            f.hi[x] = p[64 * (kHigh + TREE_HIGH_WORDS + 2 * x + 1)];
        }
    }
}

// What a term adds, by (p odd) 8 + m: 2^{(p odd)/2} w^m in the basis 1, w,
// w^2, w^3 and as an FP32 pair, to be scaled by 2^{p >> 1}.
struct TermTables {
    double z[16][4];
    float f[16][2];
    DEV void fill(int t) {
        if (t >= 16) return;
        const int m = t & 7;
        const float r = 0.70710678118654752f;
        for (int k = 0; k < 4; k++) {
            double v = 0.0;
            if (t < 8) {
                v = (m & 3) == k ? 1.0 : 0.0;
                if (m & 4) v = -v;
            } else {
                // sqrt2 w^m = w^{m+1} - w^{m+3}
                const int a = (m + 1) & 7, b = (m + 3) & 7;
                if ((a & 3) == k) v += a & 4 ? -1.0 : 1.0;
                if ((b & 3) == k) v -= b & 4 ? -1.0 : 1.0;
            }
            z[t][k] = v;
        }
        // the nearest FP32 numbers (sqrt2 sqrt1/2 is 1, its FP32 product is not:
        // that alone is half of the sums' error)
        const float one = t < 8 ? 1.f : 1.41421356237309505f, half = t < 8 ? r : 1.f;
        f[t][0] = m == 0 ? one : m == 4 ? -one : m == 2 || m == 6 ? 0.f : m == 1 || m == 7 ? half : -half;
        f[t][1] = m == 2 ? one : m == 6 ? -one : m == 0 || m == 4 ? 0.f : m == 1 || m == 3 ? half : -half;
    }
};

}  // namespace

// Persistent sweep, blocks of 256 lanes from a device work queue.  MODE 0
// (sampled): record r is theta_r', all j in [0, chi) contribute to per-record
// Z[w] sums.  MODE 1 (exact): record r is theta'_r of its instance, j in
// [r, chi), weight 1 on j == r and 2 Re otherwise, into the instance's (P, M)
// histogram; a block keeps its partial histogram and Kahan sums from item to
// item of one instance and adds them to the instance's global sums when it
// moves to another one and at its exit.  NH: slots beyond 32 (n <= 32 + NH).
// HT: some instance has |H^t> terms.  COPIES: one instance, its sums in copies
// (kernels of their own: the address alone cost the others 1 to 2% of a call
// of 40 us).
template <int NH, bool HT, int MODE, bool COPIES> DEV void sweep_body(const SweepArgs &A) {
    // levels beyond 32 slots: only where instances may have them (tree_levels)
    constexpr bool DEEP = NH > 16 && !HT;
    constexpr int LW = MODE == 0 ? TREE_LDS_WORDS0 : TREE_LDS_WORDS1;
    __shared__ uint32_t lstack[4][LW * 64];
    __shared__ unsigned int hist[MODE == 1 ? HIST_STRIDE : 1];
    __shared__ long long s_item;
    __shared__ double s_k[4];
    __shared__ unsigned long long s_ips[4];
    __shared__ __align__(16) TermTables s_tab;
    __shared__ uint8_t s_leaf[1 << tree::LeafBits<HT>::value];
    const int tid = (int)threadIdx.x, x = lane_id(), wv = uni(tid >> 6);
    uint32_t *const lst = &lstack[wv][x];
    uint32_t *const gst =
        A.stack + ((size_t)blockIdx.x * 4 + (size_t)wv) * (size_t)A.stack_words * 64 + (size_t)x;
    int cur = -1;
    long long pend = 0;         // MODE 1: terms counted since the last flush
    unsigned long long ips = 0; // per lane, of instance cur
    // the lane's sums: Z[w] coefficients at scale 2^32 as integers in FP64
    // (at most 2^G 2^32 <= 2^44, exact) and the compensated FP32 pair of an
    // item's terms; MODE 1 adds the items' real parts up in s_k, a wave each
    double c0 = 0.0, c1 = 0.0, c2 = 0.0, c3 = 0.0;
    float sr = 0.f, cr = 0.f, si = 0.f, ci = 0.f;
    if (blockIdx.x == 0 && tid == 0) A.clock[1] = wall_clock64();
    s_tab.fill(tid);
    for (int b = tid; b < 1 << tree::LeafBits<HT>::value; b += 256) s_leaf[b] = A.leaf[b];
    if (MODE == 1) {
        for (int b = tid; b < HIST_STRIDE; b += 256) hist[b] = 0;
        if (x == 0) s_k[wv] = 0.0;
    }
    // Other waves read the tables and add to the histogram, and no barrier of
    // the first item comes before that.
    __syncthreads();

    // adds the block's sums of instance cur to the global ones (whole block)
    auto flush = [&]() {
        const unsigned long long wi = (unsigned long long)wave_sum64((long long)ips);
        if (x == 0) s_ips[wv] = wi;
        __syncthreads();
        const unsigned copy = COPIES ? (blockIdx.x % TREE_COPIES) * A.copy_words : 0u;
        if (tid == 0) {
            atomicAdd(&(A.ips + copy)[cur], s_ips[0] + s_ips[1] + s_ips[2] + s_ips[3]);
            if (MODE == 1) atomicAdd(&(A.kahan + copy)[2 * (size_t)cur], (s_k[0] + s_k[1]) + (s_k[2] + s_k[3]));
        }
        if (MODE == 1) {
            // an off-diagonal term counts as z + conj(z): phases 0 and 4 are
            // their own conjugates (0 was counted twice already)
            for (int b = tid; b < HIST_STRIDE; b += 256) {
                const unsigned int v = hist[b];
                if (!v) continue;
                hist[b] = 0;
                const int m = b & 7;
                unsigned long long *h = A.hist + copy + (size_t)cur * HIST_STRIDE;
                atomicAdd(&h[b], (unsigned long long)v << (m == 4 ? 1 : 0));
                if (m & 3) atomicAdd(&h[(b & ~7) | (8 - m)], (unsigned long long)v);
            }
        }
        ips = 0;
        pend = 0;
        __syncthreads();
        if (MODE == 1 && x == 0) s_k[wv] = 0.0;
    };

    auto run_item = [&](long long item) {
        const int inst = A.ninst > 1 ? uni(find_instance(A.item_off, A.ninst, item)) : 0;
        if (inst != cur || (MODE == 1 && pend >= A.flush_terms)) {
            if (cur >= 0) flush();
            cur = inst;
        }
        CInst *D = (CInst *)(uintptr_t)(A.inst + inst);
        const long long item0 = A.ninst > 1 ? (long long)uniform64((u64)A.item_off[inst]) : 0ll;
        const int n = D->n, k = D->k, G = D->G;
        const long long l = (item - item0) * 256 + tid;
        bool live = l < D->lanes;
        long long r = 0, jh = 0;
        if (MODE == 0) {
            r = l >> (k - G);
            jh = l & ((1ll << (k - G)) - 1);
        } else {
            tri_item(live ? l : 0, 1ll << G, 1ll << (k - G), r, jh);
        }
        const int lg = 1 << G;
        if (MODE == 1) pend += 256ll * lg;
        if (!live) r = 0;
        const uint64_t *rec = A.recs + (size_t)REC_WORDS * (size_t)(D->rec_off + r);
        const u64 w0 = rec[0];
        const bool valid = live && !((w0 >> 40) & 1);
        const int sexp = (int)((w0 >> 24) & 0xffff);
        if (!ballot(valid) && !A.terms) return;

        // index bit b's toggles and index in lane b (read by readlane, so
        // only where all lanes are active)
        const u64 w_lp = x < TREE_MAXLOG ? A.inst[inst].LP[x] : 0ull;
        const u64 w_lt = HT && x < TREE_MAXLOG ? A.inst[inst].LT[x] : 0ull;
        const int w_jm = x < TREE_MAXLOG ? (int)A.inst[inst].jmap[x] : 0;

        tree::Form<NH> f;
        {
            const u64 F = rec[1], d1 = rec[2], d2 = rec[3];
            u64 xj = D->exact ? brev32x2(lowmask(n)) : 0ull;
            u64 T = 0;
            for (int b = G; b < k; b++) {
                const u64 on = 0ull - (u64)((jh >> (b - G)) & 1);
                xj ^= rl64(w_lp, b) & on;
                if (HT) T ^= rl64(w_lt, b) & on;
            }
            const u64 a = xj ^ F;
            f.A = (unsigned)a;
            f.Ah = (unsigned)(a >> 32);
            f.T = (unsigned)T;
            f.Th = (unsigned)(T >> 32);
            f.d1 = (unsigned)d1;
            f.d1h = (unsigned)(d1 >> 32);
            f.d2 = (unsigned)d2;
            f.d2h = (unsigned)(d2 >> 32);
        }
        f.x2 = f.z = 0;
        f.nb = f.q1 = 0;
        const uint32_t *rows = (const uint32_t *)(rec + REC_ROWS);
#pragma unroll
        for (int y = 0; y < 32 + NH; y += 4)
            if (n > y) {
#pragma unroll
                for (int z = y; z < y + 4; z++) {
                    f.lo[z] = rows[2 * z];
                    if (NH > 0 && z >= 32) f.hi[z >= 32 ? z - 32 : 0] = rows[2 * z + 1];
                }
            }
        int ph0 = (int)((w0 >> 16) & 7), cnt0 = -n;
        if (NH > 0 && !DEEP) {
            tree::StepsHi<NH, HT, NH - 1>::run(f, n);
            tree::fold<HT>(f.d1h, f.d2h, f.Ah, f.Th, ~0u, ph0, cnt0);
        }
        // by index bit g (in lane g): the slots it toggles, their signs, the
        // index j; by level: slots and place of the saved form
        const int gl = x < TREE_MAXG ? x : TREE_MAXG;
        const int v_lp = (int)(unsigned)w_lp, v_lph = (int)(unsigned)(w_lp >> 32), v_lt = (int)(unsigned)w_lt;
        const int v_lev = (int)A.inst[inst].ub[gl] | (int)A.inst[inst].soff[gl] << 8;
        const int nlds = D->nlds, leaf = D->leaf;
        const bool pair = !HT && D->pair;
        // the term within the lane (Gray code of t - 1), and what it toggles
        const unsigned T0 = f.T;
        unsigned gray = 0, ta = 0, tah = 0, tt = 0, tj = 0;
        // MODE 1: the lane's block holds the diagonal at term rl
        const int rl = MODE == 1 && jh == (r >> G) ? (int)(r & (lg - 1)) : -1;
        unsigned jhi = 0, ri = 0;
        if (A.terms)
            for (int b = G; b < k; b++)
                jhi ^= (unsigned)__builtin_amdgcn_readlane(w_jm, b) & (0u - (unsigned)((jh >> (b - G)) & 1));
        if (MODE == 1) {
            for (int b = 0; b < k; b++)
                ri ^= (unsigned)__builtin_amdgcn_readlane(w_jm, b) & (0u - (unsigned)((r >> b) & 1));
            // the record's pairs i <= j in the reference's order, counted by
            // the one lane that holds its diagonal
            if (valid && rl >= 0) ips += (unsigned long long)(D->chi - (long long)ri);
        }
        if (MODE == 0) c0 = c1 = c2 = c3 = 0.0;
        sr = cr = si = ci = 0.f;
        // adds a term: its exponent and phase, whether there is one, its place
        // within the lane and its index's low part
        auto term = [&](int p, int m, bool nz, unsigned gy, unsigned jx) {
            // an inner product has -64 <= p <= 0; another one is not added (its
            // place in the histogram may not exist) and fails the call
            const bool sum = nz && (unsigned)-p <= 64u;
            if (nz && !sum) atomicOr(A.err, 2);
            if (MODE == 0) {
                const int row = ((p & 1) << 3) | m;
                const double s = ldexp(1.0, sum ? 32 + (p >> 1) : -2000);
                c0 = fma(s_tab.z[row][0], s, c0);
                c1 = fma(s_tab.z[row][1], s, c1);
                c2 = fma(s_tab.z[row][2], s, c2);
                c3 = fma(s_tab.z[row][3], s, c3);
                const float e = ldexpf(1.f, sum ? p >> 1 : -2000);
                kahan1(sr, cr, s_tab.f[row][0] * e);
                kahan1(si, ci, s_tab.f[row][1] * e);
            } else if (sum && (int)gy >= rl) {
                const bool off = (int)gy != rl;
                const int P = p - sexp;
                kahan1(sr, cr, ldexpf(s_tab.f[((P & 1) << 3) | m][0], (P >> 1) + (off ? 1 : 0)));
                atomicAdd(&hist[m - 8 * P], off && m == 0 ? 2u : 1u);
            }
            if (A.terms && live) {
                long long j = jhi ^ jx;
                int mm = m;
                if (MODE == 0) {
                    A.terms[D->term_off + r * D->chi + j] = nz ? (-p) * 8 + mm + 1 : 0;
                } else if ((int)gy >= rl) {
                    // the pair in the reference's order i <= j, with the
                    // projection's factors of record i left out:
                    // <phi_i| Pi |phi_j> is the conjugate of <phi_j| Pi |phi_i>
                    long long i = ri;
                    int pp = p;
                    if (j < i) {
                        const long long s = i, rj = (jh << G) | (long long)gy;
                        i = j;
                        j = s;
                        mm = (8 - m) & 7;
                        pp += (int)((A.recs[(size_t)REC_WORDS * (size_t)(D->rec_off + rj)] >> 24) & 0xffff) - sexp;
                    }
                    A.terms[D->term_off + i * D->chi - i * (i - 1) / 2 + (j - i)] = nz ? (-pp) * 8 + mm + 1 : 0;
                }
            }
        };
        const int low = uni(pair ? (int)D->ub[1] : TREE_LEAF);
        int p0 = 0, m0 = 0;   // the term's exponent and phase without its last slots
        int t = 1, lev = G, top = DEEP || n < 32 ? n : 32;
        while (true) {
            if (DEEP && top > 32) {
                // the levels beyond 32 slots, and what their slots give
                while (true) {
                    const int w = __builtin_amdgcn_readlane(v_lev, lev);
                    const int c = w & 0xff;
                    tree::StepsHi<NH, HT, NH - 1>::run(f, top, c);
                    if (c <= 32) break;
                    uint32_t *const st = gst + 64 * (w >> 8);
                    form_save(f, f.A ^ ta, c, st);
                    form_save_high(f, f.Ah ^ tah, c, st);
                    top = c;
                    lev--;
                }
                ph0 = (int)((w0 >> 16) & 7);
                cnt0 = -n;
                tree::fold<HT>(f.d1h, f.d2h, f.Ah, f.Th, ~0u, ph0, cnt0);
                top = 32;
            }
            while (true) {
                if (lev >= leaf) {
                    // down from `top` to the leaf slots, saving the form at every
                    // level on the way
                    while (true) {
                        const int w = __builtin_amdgcn_readlane(v_lev, lev);
                        const int c = w & 0xff;
                        if (top > c) tree::steps<NH, HT>(f, top, c);
                        if (lev == leaf) break;
                        uint32_t *const st = lev <= nlds ? lst : gst;
                        form_save(f, f.A ^ ta, c, st + 64 * (w >> 8));
                        top = c;
                        lev--;
                    }
                    int cnt = cnt0;
                    m0 = ph0;
                    tree::fold<HT>(f.d1, f.d2, f.A, f.T, ~(~0u << (32 - low)), m0, cnt);
                    p0 = cnt - (int)f.nb;
                    m0 += 2 * (int)f.q1 + 4 * __popc(f.x2);
                }
                if (pair) {
                    tree::PairSums s;
                    int c = low;  // (out of sight of hoisting: a register a slot)
                    asm volatile("" : "+s"(c));
                    tree::pair_sums(f, c, s);
                    const bool some = valid && (int)f.z >= 0;
                    term(p0 + s.cnt[0], (m0 + s.ph[0]) & 7, some && !s.zero[0], gray, tj);
                    gray ^= 1u;
                    ta ^= (unsigned)__builtin_amdgcn_readlane(v_lp, 0);
                    if (A.terms) tj ^= D->jmap[0];
                    term(p0 + s.cnt[1], (m0 + s.ph[1]) & 7, some && !s.zero[1], gray, tj);
                    t++;
                } else {
                    // the leaf slots from the table: phase, steps of the second
                    // kind, whether the sum is 0
                    const unsigned lf = s_leaf[tree::leaf_index<HT>(f.A, f.T, f.d1, f.d2, f.lo[1])];
                    term(p0 + (int)((lf >> 3) & 7u), (m0 + (int)lf) & 7, valid && (int)f.z >= 0 && lf < 128u, gray,
                         tj);
                }
                if (t == lg) goto summed;
                const int g = __builtin_ctz(t++);
                gray ^= 1u << g;
                if (A.terms) tj ^= D->jmap[g];
                const unsigned la = (unsigned)__builtin_amdgcn_readlane(v_lp, g);
                const unsigned lt = HT ? (unsigned)__builtin_amdgcn_readlane(v_lt, g) : 0u;
                ta ^= la;
                tt ^= lt;
                if (DEEP) tah ^= (unsigned)__builtin_amdgcn_readlane(v_lph, g);
                lev = g;
                if (g < leaf) {
                    // only leaf slots change
                    f.A ^= la;
                    if (HT) f.T ^= lt;
                } else {
                    const int w = __builtin_amdgcn_readlane(v_lev, g + 1);
                    top = w & 0xff;
                    if (DEEP && top > 32) break;
                    form_load(f, top, (g + 1 <= nlds ? lst : gst) + 64 * (w >> 8));
                    f.A ^= ta;
                    if (HT) f.T = T0 ^ tt;
                }
            }
            const uint32_t *const st = gst + 64 * (__builtin_amdgcn_readlane(v_lev, lev + 1) >> 8);
            form_load(f, top, st);
            form_load_high(f, top, st);
            f.A ^= ta;
            f.Ah ^= tah;
        }
    summed:
        if (MODE == 1) {
            // (a lane's own sum across its items would take two registers that
            // the loop has not got: scratch of the 32-slot kernel 20 -> 56 bytes)
            const double wk = wave_sumf64((double)sr - (double)cr);
            if (x == 0) s_k[wv] += wk;
        }
        if (MODE == 0) {
            if (valid) ips += (unsigned long long)lg;
            // the record's sums over the lanes that share it (integers below
            // 2^50, exact in FP64): aligned groups of up to a wave, then atomics when several waves do
            const int seg = k - G < 6 ? 1 << (k - G) : 64;
            double kr = (double)sr - (double)cr, ki = (double)si - (double)ci;
            for (int o = 1; o < seg; o <<= 1) {
                c0 += __shfl_xor(c0, o, 64);
                c1 += __shfl_xor(c1, o, 64);
                c2 += __shfl_xor(c2, o, 64);
                c3 += __shfl_xor(c3, o, 64);
                kr += __shfl_xor(kr, o, 64);
                ki += __shfl_xor(ki, o, 64);
            }
            if (valid && (x & (seg - 1)) == 0) {
                unsigned long long *z = (unsigned long long *)A.zsum + 4 * (size_t)(D->rec_off + r);
                double *kz = A.kahan + 2 * (size_t)(D->rec_off + r);
                const unsigned long long z0 = (unsigned long long)(long long)c0, z1 = (unsigned long long)(long long)c1;
                const unsigned long long z2 = (unsigned long long)(long long)c2, z3 = (unsigned long long)(long long)c3;
                if (k - G <= 6) {
                    z[0] = z0;
                    z[1] = z1;
                    z[2] = z2;
                    z[3] = z3;
                    kz[0] = kr;
                    kz[1] = ki;
                } else {
                    atomicAdd(&z[0], z0);
                    atomicAdd(&z[1], z1);
                    atomicAdd(&z[2], z2);
                    atomicAdd(&z[3], z3);
                    atomicAdd(&kz[0], kr);
                    atomicAdd(&kz[1], ki);
                }
            }
        }
    };

    // The first item is the block's own; the others come from the queue, each
    // claimed when the one before is done (claimed ahead, a launch of a few
    // items a block loses 10% to its slower blocks).
    const bool more = A.nitems > (long long)gridDim.x;
    for (long long item = (long long)blockIdx.x; item < A.nitems;) {
        run_item(item);
        if (!more) break;
        __syncthreads();  // the item's sums are complete, s_item has been read
        if (tid == 0) s_item = (long long)(gridDim.x + atomicAdd(A.queue, 1ull));
        __syncthreads();
        item = (long long)uniform64((u64)s_item);
    }
    if (cur >= 0) flush();
}

// The table of the leaf slots: every form on TREE_LEAF slots taken through its
// steps.  Bits 0..2 the phase, 3..5 the steps of the second kind, 7 set when
// the sum is 0.
template <bool HT> DEV void leaf_entry(unsigned i, uint8_t *out) {
    tree::Form<0> f = {};
    tree::leaf_form<HT>(i, f);
    tree::steps<0, HT>(f, TREE_LEAF, 0);
    int ph = 0, cnt = 0;
    tree::fold<HT>(f.d1, f.d2, f.A, f.T, ~0u, ph, cnt);
    ph += 2 * (int)f.q1 + 4 * __popc(f.x2);
    out[i] = (uint8_t)((ph & 7) | ((cnt - (int)f.nb) << 3) | ((int)f.z < 0 ? 128 : 0));
}
extern "C" __global__ void k_leaf_table(uint8_t *plain, uint8_t *sign) {
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < 1u << tree::LeafBits<false>::value) leaf_entry<false>(i, plain);
    if (i < 1u << tree::LeafBits<true>::value) leaf_entry<true>(i, sign);
}

#define SWEEP_KERNEL(NAME, NH, HT, MODE, COPIES, WAVES)                                    \
    extern "C" __global__ void __launch_bounds__(256, WAVES) NAME(SweepArgs A) {           \
        sweep_body<NH, HT, MODE, COPIES>(A);                                               \
    }
SWEEP_KERNEL(k_sweep_s32, 0, false, 0, false, 4)
SWEEP_KERNEL(k_sweep_s48, 16, false, 0, false, 4)
SWEEP_KERNEL(k_sweep_s64, 32, false, 0, false, 3)
SWEEP_KERNEL(k_sweep_e32, 0, false, 1, false, 4)
SWEEP_KERNEL(k_sweep_e48, 16, false, 1, false, 4)
SWEEP_KERNEL(k_sweep_e64, 32, false, 1, false, 3)
SWEEP_KERNEL(k_sweep_sh32, 0, true, 0, false, 4)
SWEEP_KERNEL(k_sweep_sh48, 16, true, 0, false, 4)
SWEEP_KERNEL(k_sweep_sh64, 32, true, 0, false, 3)
SWEEP_KERNEL(k_sweep_eh32, 0, true, 1, false, 4)
SWEEP_KERNEL(k_sweep_eh48, 16, true, 1, false, 4)
SWEEP_KERNEL(k_sweep_eh64, 32, true, 1, false, 3)
SWEEP_KERNEL(k_sweep_c32, 0, false, 1, true, 4)
SWEEP_KERNEL(k_sweep_c48, 16, false, 1, true, 4)
SWEEP_KERNEL(k_sweep_c64, 32, false, 1, true, 3)
