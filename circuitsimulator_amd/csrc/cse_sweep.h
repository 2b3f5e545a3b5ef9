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
// the tree takes 30 vector instructions.)
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

// FP32 value of 2^{P/2} e^{i pi m/4}
DEV void term_f32(int P, int m, float &re, float &im) {
    const float r = 0.70710678118654752f;
    const int mm = m & 7;
    const float c = (mm == 0) ? 1.f : (mm == 4) ? -1.f : (mm == 2 || mm == 6) ? 0.f : (mm == 1 || mm == 7) ? r : -r;
    const float s = (mm == 2) ? 1.f : (mm == 6) ? -1.f : (mm == 0 || mm == 4) ? 0.f : (mm == 1 || mm == 3) ? r : -r;
    const float mag = ldexpf((P & 1) ? 1.41421356237309505f : 1.f, P >> 1);
    re = mag * c;
    im = mag * s;
}

// Per-lane sums of the terms.
struct LaneAcc {
    long long c0, c1, c2, c3;   // exact Z[w] partial sums, scale 2^32 (mode 0)
    float sr, cr, si, ci;       // Kahan FP32 partial sums
    DEV void clear() {
        c0 = c1 = c2 = c3 = 0;
        sr = cr = si = ci = 0.f;
    }
    DEV static void kahan1(float &s, float &c, float v) {
        const float y = v - c;
        const float t = s + y;
        c = (t - s) - y;
        s = t;
    }
    // + 2^{p/2} w^m in Z[w] coordinates (scale 2^32, -64 <= p <= 0)
    DEV void zomega(int p, int m) {
        const long long v = 1ll << (32 + (p >> 1));
        const int mm = m & 7;
        int qa, qb;
        long long sa, sb;
        if (!(p & 1)) {
            qa = mm; sa = v; qb = 0; sb = 0;
        } else {
            // sqrt2 w^m = w^{m+1} - w^{m+3}
            qa = (mm + 1) & 7; sa = v;
            qb = (mm + 3) & 7; sb = -v;
        }
        if (qa & 4) sa = -sa;
        if (qb & 4) sb = -sb;
        qa &= 3;
        qb &= 3;
        c0 += (qa == 0 ? sa : 0) + (qb == 0 ? sb : 0);
        c1 += (qa == 1 ? sa : 0) + (qb == 1 ? sb : 0);
        c2 += (qa == 2 ? sa : 0) + (qb == 2 ? sb : 0);
        c3 += (qa == 3 ? sa : 0) + (qb == 3 ? sb : 0);
    }
};

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
template <int NH> DEV void form_save(const tree::Form<NH> &f, unsigned a, int c, uint32_t *p) {
    p[0] = f.d1;
    p[64] = f.d2;
    p[128] = a;
    p[192] = f.x2;
    p[256] = (f.z & 0x80000000u) | (f.q1 << 8) | f.nb;
#pragma unroll
    for (int x = 0; x < 32; x += 2)
        if (c > x) {
            p[64 * (TREE_STATE_WORDS + x)] = f.lo[x];
            if (c > x + 1) p[64 * (TREE_STATE_WORDS + x + 1)] = f.lo[x + 1];
        }
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
#pragma unroll
    for (int x = 0; x < 32; x += 2)
        if (c > x) {
            f.lo[x] = p[64 * (TREE_STATE_WORDS + x)];
            if (c > x + 1) f.lo[x + 1] = p[64 * (TREE_STATE_WORDS + x + 1)];
        }
}

}  // namespace

// Persistent sweep, blocks of 256 lanes from a device work queue.  MODE 0
// (sampled): record r is theta_r', all j in [0, chi) contribute to per-record
// Z[w] sums.  MODE 1 (exact): record r is theta'_r of its instance, j in
// [r, chi), weight 1 on j == r and 2 Re otherwise, into the instance's (P, M)
// histogram; a block keeps its partial histogram and Kahan sums from item to
// item of one instance and adds them to the instance's global sums when it
// moves to another one and at its exit.  NH: slots beyond 32 (n <= 32 + NH).
// HT: some instance has |H^t> terms.
template <int NH, bool HT, int MODE> DEV void sweep_body(const SweepArgs &A) {
    constexpr int LW = MODE == 0 ? TREE_LDS_WORDS0 : TREE_LDS_WORDS1;
    __shared__ uint32_t lstack[4][LW * 64];
    __shared__ unsigned int hist[MODE == 1 ? HIST_STRIDE : 1];
    __shared__ long long s_item;
    __shared__ double s_k[4];
    __shared__ unsigned long long s_ips[4];
    const int tid = (int)threadIdx.x, x = lane_id(), wv = uni(tid >> 6);
    uint32_t *const lst = &lstack[wv][x];
    uint32_t *const gst =
        A.stack + ((size_t)blockIdx.x * 4 + (size_t)wv) * (size_t)A.stack_words * 64 + (size_t)x;
    int cur = -1;
    long long pend = 0;         // MODE 1: terms counted since the last flush
    unsigned long long ips = 0; // per lane, of instance cur
    LaneAcc acc;
    acc.clear();
    if (MODE == 1)
        for (int b = tid; b < HIST_STRIDE; b += 256) hist[b] = 0;

    // adds the block's sums of instance cur to the global ones (whole block)
    auto flush = [&]() {
        const unsigned long long wi = (unsigned long long)wave_sum64((long long)ips);
        double wk = 0.0;
        if (MODE == 1) wk = wave_sumf64((double)acc.sr - (double)acc.cr);
        if (x == 0) {
            s_ips[wv] = wi;
            s_k[wv] = wk;
        }
        __syncthreads();
        if (tid == 0) {
            atomicAdd(&A.ips[cur], s_ips[0] + s_ips[1] + s_ips[2] + s_ips[3]);
            if (MODE == 1) atomicAdd(&A.kahan[2 * (size_t)cur], (s_k[0] + s_k[1]) + (s_k[2] + s_k[3]));
        }
        if (MODE == 1) {
            // an off-diagonal term counts as z + conj(z): phases 0 and 4 are
            // their own conjugates (0 was counted twice already)
            for (int b = tid; b < HIST_STRIDE; b += 256) {
                const unsigned int v = hist[b];
                if (!v) continue;
                hist[b] = 0;
                const int m = b & 7;
                unsigned long long *h = A.hist + (size_t)cur * HIST_STRIDE;
                atomicAdd(&h[b], (unsigned long long)v << (m == 4 ? 1 : 0));
                if (m & 3) atomicAdd(&h[(b & ~7) | (8 - m)], (unsigned long long)v);
            }
            acc.clear();
        }
        ips = 0;
        pend = 0;
        __syncthreads();
    };

    while (true) {
        __syncthreads();
        if (tid == 0) s_item = (long long)atomicAdd(A.queue, 1ull);
        __syncthreads();
        const long long item = (long long)uniform64((u64)s_item);
        if (item >= A.nitems) break;
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
        if (!ballot(valid) && !A.terms) continue;

        tree::Form<NH> f;
        {
            const u64 F = rec[1], d1 = rec[2], d2 = rec[3];
            u64 xj = D->exact ? brev32x2(lowmask(n)) : 0ull;
            u64 T = 0;
            for (int b = G; b < k; b++) {
                const u64 on = 0ull - (u64)((jh >> (b - G)) & 1);
                xj ^= D->LP[b] & on;
                if (HT && D->exact) T ^= D->L[b] & on;
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
        if (NH > 0) {
            tree::StepsHi<NH, HT, NH - 1>::run(f, n);
            tree::fold<HT>(f.d1h, f.d2h, f.Ah, f.Th, ph0, cnt0);
        }
        // the term within the lane (Gray code of t), and what its bits toggle
        const unsigned T0 = f.T;
        unsigned gray = 0, ta = 0, tt = 0, tj = 0;
        // MODE 1: the lane's block holds the diagonal at term rl
        const int rl = MODE == 1 && jh == (r >> G) ? (int)(r & (lg - 1)) : -1;
        unsigned jhi = 0, ri = 0;
        if (A.terms)
            for (int b = G; b < k; b++)
                if ((jh >> (b - G)) & 1) jhi ^= D->jmap[b];
        if (MODE == 1) {
            for (int b = 0; b < k; b++)
                if ((r >> b) & 1) ri ^= D->jmap[b];
            // the record's pairs i <= j in the reference's order, counted by
            // the one lane that holds its diagonal
            if (valid && rl >= 0) ips += (unsigned long long)(D->chi - (long long)ri);
        }
        if (MODE == 0) acc.clear();
        int lev = G, c0 = n < 32 ? n : 32;
        for (int t = 1;; t++) {
            // down from c0 to the term, saving the form at every level
            while (true) {
                const int c1 = lev ? (int)D->ub[lev] : 0;
                tree::Steps<NH, HT, 31>::run(f, c1, (unsigned)(c0 - c1));
                if (lev == 0) break;
                if (lev <= D->nlds) form_save(f, f.A ^ ta, c1, lst + 64 * (int)D->soff[lev]);
                else form_save(f, f.A ^ ta, c1, gst + 64 * (int)D->soff[lev]);
                c0 = c1;
                lev--;
            }
            int ph = ph0, cnt = cnt0;
            tree::fold<HT>(f.d1, f.d2, f.A, f.T, ph, cnt);
            const int p = cnt - (int)f.nb;
            const int m = (ph + 2 * (int)f.q1 + 4 * __popc(f.x2)) & 7;
            const bool nz = valid && (int)f.z >= 0;
            float vr, vi;
            if (MODE == 0) {
                if (nz) {
                    acc.zomega(p, m);
                    term_f32(p, m, vr, vi);
                    LaneAcc::kahan1(acc.sr, acc.cr, vr);
                    LaneAcc::kahan1(acc.si, acc.ci, vi);
                }
            } else if (nz && (int)gray >= rl) {
                const bool off = (int)gray != rl;
                term_f32(p - sexp, m, vr, vi);
                LaneAcc::kahan1(acc.sr, acc.cr, off ? 2.f * vr : vr);
                atomicAdd(&hist[(sexp - p) * 8 + m], off && m == 0 ? 2u : 1u);
            }
            if (A.terms && live) {
                long long j = jhi ^ tj;
                int mm = m;
                if (MODE == 0) {
                    A.terms[D->term_off + r * D->chi + j] = nz ? (-p) * 8 + mm + 1 : 0;
                } else if ((int)gray >= rl) {
                    // the pair in the reference's order i <= j, with the
                    // projection's factors of record i left out:
                    // <phi_i| Pi |phi_j> is the conjugate of <phi_j| Pi |phi_i>
                    long long i = ri;
                    int pp = p;
                    if (j < i) {
                        const long long s = i, rj = (jh << G) | (long long)gray;
                        i = j;
                        j = s;
                        mm = (8 - m) & 7;
                        pp += (int)((A.recs[(size_t)REC_WORDS * (size_t)(D->rec_off + rj)] >> 24) & 0xffff) - sexp;
                    }
                    A.terms[D->term_off + i * D->chi - i * (i - 1) / 2 + (j - i)] = nz ? (-pp) * 8 + mm + 1 : 0;
                }
            }
            if (t == lg) break;
            const int g = __builtin_ctz(t);
            gray ^= 1u << g;
            ta ^= (unsigned)D->LP[g];
            if (HT && D->exact) tt ^= (unsigned)D->L[g];
            if (A.terms) tj ^= D->jmap[g];
            c0 = (int)D->ub[g + 1];
            if (g + 1 <= D->nlds) form_load(f, c0, lst + 64 * (int)D->soff[g + 1]);
            else form_load(f, c0, gst + 64 * (int)D->soff[g + 1]);
            f.A ^= ta;
            if (HT) f.T = T0 ^ tt;
            lev = g;
        }
        if (MODE == 0) {
            if (valid) ips += (unsigned long long)lg;
            // the record's sums over the lanes that share it: aligned groups
            // of up to a wave, then atomics when several waves do
            const int seg = k - G < 6 ? 1 << (k - G) : 64;
            double kr = (double)acc.sr - (double)acc.cr, ki = (double)acc.si - (double)acc.ci;
            for (int o = 1; o < seg; o <<= 1) {
                acc.c0 += (long long)shfl_xor64((u64)acc.c0, o);
                acc.c1 += (long long)shfl_xor64((u64)acc.c1, o);
                acc.c2 += (long long)shfl_xor64((u64)acc.c2, o);
                acc.c3 += (long long)shfl_xor64((u64)acc.c3, o);
                kr += __shfl_xor(kr, o, 64);
                ki += __shfl_xor(ki, o, 64);
            }
            if (valid && (x & (seg - 1)) == 0) {
                unsigned long long *z = (unsigned long long *)A.zsum + 4 * (size_t)(D->rec_off + r);
                double *kz = A.kahan + 2 * (size_t)(D->rec_off + r);
                if (k - G <= 6) {
                    z[0] = (unsigned long long)acc.c0;
                    z[1] = (unsigned long long)acc.c1;
                    z[2] = (unsigned long long)acc.c2;
                    z[3] = (unsigned long long)acc.c3;
                    kz[0] = kr;
                    kz[1] = ki;
                } else {
                    atomicAdd(&z[0], (unsigned long long)acc.c0);
                    atomicAdd(&z[1], (unsigned long long)acc.c1);
                    atomicAdd(&z[2], (unsigned long long)acc.c2);
                    atomicAdd(&z[3], (unsigned long long)acc.c3);
                    atomicAdd(&kz[0], kr);
                    atomicAdd(&kz[1], ki);
                }
            }
        }
    }
    if (cur >= 0) flush();
}

#define SWEEP_KERNEL(NAME, NH, HT, MODE, WAVES)                                            \
    extern "C" __global__ void __launch_bounds__(256, WAVES) NAME(SweepArgs A) {           \
        sweep_body<NH, HT, MODE>(A);                                                       \
    }
SWEEP_KERNEL(k_sweep_s32, 0, false, 0, 4)
SWEEP_KERNEL(k_sweep_s48, 16, false, 0, 4)
SWEEP_KERNEL(k_sweep_s64, 32, false, 0, 3)
SWEEP_KERNEL(k_sweep_e32, 0, false, 1, 4)
SWEEP_KERNEL(k_sweep_e48, 16, false, 1, 4)
SWEEP_KERNEL(k_sweep_e64, 32, false, 1, 3)
SWEEP_KERNEL(k_sweep_sh32, 0, true, 0, 4)
SWEEP_KERNEL(k_sweep_sh48, 16, true, 0, 4)
SWEEP_KERNEL(k_sweep_sh64, 32, true, 0, 3)
SWEEP_KERNEL(k_sweep_eh32, 0, true, 1, 4)
SWEEP_KERNEL(k_sweep_eh48, 16, true, 1, 4)
SWEEP_KERNEL(k_sweep_eh64, 32, true, 1, 3)
