// cse_kernels.hip -- gfx950 kernels of the stabilizer-rank inner-product
// engine.  See cse_device.h for the execution model.
//
// Kernels
//   k_ip_pairs       general <s2|s1> for packed state pairs, one wave per pair
//   k_prep_states    prepL / prepH states (reference row bookkeeping)
//   k_random_states  Philox random stabilizer states, projected by P
//   k_records        theta' = Pi phi_i or Pi theta_s, turned into a form on
//                    the instance's slots (cse_tree.h)
//   k_sweep_*        persistent, from a device work queue: every lane sums a
//                    subtree of the terms <phi_j | theta'> of one record,
//                    exactly (int64) plus a Kahan-FP32 shadow (cse_sweep.h);
//                    s / e: sampled, exact mode; h: with |H^t> instances;
//                    32, 48, 64: widest state
//   k_prep, k_results  a call's plan to the device and its results cleared;
//                    the results to pinned host memory
//   k_lspace_hist    histogram of |x| over the row space of L (decompose's
//                    fidelity)
#include "cse_device.h"
#include "cse_internal.h"
#include "cse_tree.h"

using namespace cse;

namespace {

// ------------------------------------------------------ packed state I/O
DEV void load_rstate(RState &s, const uint64_t *w) {
    const int x = lane_id();
    uint64_t hdr = w[0];
    s.n = (int)(hdr & 0xff);
    s.k = (int)((hdr >> 8) & 0xff);
    s.Q = (int)((hdr >> 16) & 7);
    s.h = w[1];
    u64 D1 = w[2], D2 = w[3];
    s.d = 2 * (int)((D1 >> x) & 1ull) + 4 * (int)((D2 >> x) & 1ull);
    const int n = s.n;
    s.G = x < n ? w[4 + x] : 0ull;
    s.Gb = x < n ? w[4 + n + x] : 0ull;
    s.J = x < n ? w[4 + 2 * n + x] : 0ull;
}

DEV void store_rstate(const RState &s, uint64_t *w) {
    const int x = lane_id();
    const int n = s.n;
    u64 D1 = ballot(x < n && (s.d & 2));
    u64 D2 = ballot(x < n && (s.d & 4));
    if (x == 0) {
        w[0] = (uint64_t)n | ((uint64_t)s.k << 8) | ((uint64_t)(s.Q & 7) << 16);
        w[1] = s.h;
        w[2] = D1;
        w[3] = D2;
    }
    if (x < n) {
        w[4 + x] = s.G;
        w[4 + n + x] = s.Gb;
        w[4 + 2 * n + x] = s.J;
    }
}

DEV void to_astate(const RState &r, AState &s) {
    const int x = lane_id();
    s.G = r.G;
    s.J = r.J;
    s.d = x < r.n ? (r.d & 6) : 0;
    s.act = lowmask(r.k);
    s.h = r.h;
    s.Q = r.Q;
}

// General alignment of innerProductExact (stabilizer.c:611-652) in the
// active-mask layout: the quadratic form of s2, rewritten in the basis of
// the restricted s1 (updateQD(y) then updateDJ(R) on a copy of s2), is
// subtracted from s1's form.
DEV void as_subtract_general(AState &s, const RState &s2) {
    const int x = lane_id();
    const int n = s2.n, k2 = s2.k;
    const u64 k2m = lowmask(k2);
    // y_b = (h + h2) . Gbar2_b
    const u64 y = ballot(x < n && par64((s.h ^ s2.h) & s2.Gb));
    // updateQD(y) on the copy of s2 (stabilizer.c:163-177)
    const bool inY = x < k2 && ((y >> x) & 1ull);
    int Q2 = s2.Q;
    Q2 += 2 * __popcll(ballot(inY && (s2.d & 2))) + 4 * __popcll(ballot(inY && (s2.d & 4)));
    Q2 += 4 * (__popcll(ballot(inY && par64(s2.J & y & k2m & ~lowmask(x + 1)))) & 1);
    Q2 &= 7;
    int d2 = s2.d;
    if (x < n && par64(s2.J & y)) d2 ^= 4;
    // R_a = (G_a . Gbar2_b)_b for the active rows a (zero beyond k2)
    u64 R = 0;
    for (int b = 0; b < k2; b++) {
        u64 g = rl64(s2.Gb, b);
        R |= (u64)par64(s.G & g) << b;
    }
    // D2'_a = sum_{b<k2} D2_b R_ab + 4 [sum_{b>c} J2_bc R_ab R_ac odd]
    const u64 M1 = ballot(x < k2 && (d2 & 2));
    const u64 M2 = ballot(x < k2 && (d2 & 4));
    int dp = 2 * __popcll(R & M1) + 4 * __popcll(R & M2);
    u64 RJ = 0;
    int cross = 0;
    for (int b = 0; b < k2; b++) {
        u64 jb = rl64(s2.J, b);
        if ((R >> b) & 1ull) {
            RJ ^= jb;
            cross ^= par64(jb & R & lowmask(b));
        }
    }
    dp = (dp + 4 * cross) & 7;
    // J2' = R J2 R^T on the active rows
    u64 J2p = 0;
    u64 act = s.act;
    while (act) {
        int a2 = __ffsll((long long)act) - 1;
        act &= act - 1;
        u64 Ra2 = rl64(R, a2);
        J2p |= (u64)par64(RJ & Ra2) << a2;
    }
    // D -= D2', J ^= J2', Q -= Q2'
    s.d = (s.d - dp + 8) & 7;
    s.J ^= J2p;
    s.Q = (s.Q - Q2 + 8) & 7;
}

// The restrictions of innerProductExact (stabilizer.c:594-607) on the packed
// layout (D_x in bits 61..63 of J_x, n <= 60), one asm block: for each row b
// of Gbar2 from k2 to n - 1, xi = that row and the right side alpha =
// h2 . xi; the column is the ballot of the parity of G & xi over the active
// rows, c = (h2 ^ h) . xi, and i = min(S) is eliminated over S: rows of S take
// J_i, D_i + 4 J_xi and G_i, the rows of M = J_i (^ S when D_i is in {2,6}) take S, and c = 1
// adds D_i to Q (bits 29..31 of s60), 4 to D on M and G_i to h.  Returns 0
// when a restriction is empty with right side 1 (the product is 0).
DEV int pk_restrict_general(unsigned &jlo, unsigned &jhi, unsigned &glo, unsigned &ghi, u64 &h, u64 &act,
                            unsigned &W, unsigned gblo, unsigned gbhi, u64 h2, unsigned bstart, unsigned bend) {
    unsigned vt0, vt1, vt2, vt3;
    int ok;
    asm volatile(
        "s_mov_b32 %[ok], 1\n\t"
        "s_mov_b32 s50, %[bstart]\n"
        "L_gb%=:\n\t"
        "s_cmp_ge_u32 s50, %[bend]\n\t"
        "s_cbranch_scc1 L_gdone%=\n\t"
        "v_readlane_b32 s52, %[gblo], s50\n\t"
        "v_readlane_b32 s53, %[gbhi], s50\n\t"
        "s_add_u32 s50, s50, 1\n\t"
        "s_xor_b64 s[66:67], %[h2], s[48:49]\n\t"
        "s_and_b64 s[66:67], s[66:67], s[52:53]\n\t"
        "s_bcnt1_i32_b64 s51, s[66:67]\n\t"
        "v_and_b32 %[vt0], s52, %[glo]\n\t"
        "v_and_b32 %[vt1], s53, %[ghi]\n\t"
        "v_bcnt_u32_b32 %[vt0], %[vt0], 0\n\t"
        "v_bcnt_u32_b32 %[vt0], %[vt1], %[vt0]\n\t"
        "v_and_b32 %[vt0], 1, %[vt0]\n\t"
        "v_cmp_ne_u32_e64 s[52:53], 0, %[vt0]\n\t"
        "s_and_b64 s[64:65], s[52:53], s[58:59]\n\t"
        "s_cbranch_scc0 L_gempty%=\n\t"
        "s_ff1_i32_b64 s56, s[64:65]\n\t"
        "s_bitset0_b64 s[58:59], s56\n\t"
        "v_readlane_b32 s66, %[jlo], s56\n\t"
        "v_readlane_b32 s67, %[jhi], s56\n\t"
        "v_readlane_b32 s46, %[glo], s56\n\t"
        "v_readlane_b32 s47, %[ghi], s56\n\t"
        "s_and_b32 s56, s67, 0xe0000000\n\t"
        "s_and_b32 s67, s67, 0x1fffffff\n\t"
        "v_cndmask_b32_e64 %[vt0], 0, -1, s[64:65]\n\t"
        "s_nop 1\n\t"
        "v_cndmask_b32_e64 %[vt3], 0, -1, s[66:67]\n\t"
        "v_bitop3_b32 %[jlo], %[jlo], s66, %[vt0] bitop3:0x78\n\t"
        "v_bitop3_b32 %[jhi], %[jhi], s67, %[vt0] bitop3:0x78\n\t"
        "v_and_b32 %[vt1], 0x80000000, %[vt3]\n\t"
        "v_bitop3_b32 %[vt2], %[vt0], s56, %[vt1] bitop3:0x60\n\t"
        "v_add_u32 %[jhi], %[jhi], %[vt2]\n\t"
        "v_bitop3_b32 %[glo], %[glo], s46, %[vt0] bitop3:0x78\n\t"
        "v_bitop3_b32 %[ghi], %[ghi], s47, %[vt0] bitop3:0x78\n\t"
        "s_bitcmp1_b32 s56, 30\n\t"
        "s_cbranch_scc0 L_gnojii%=\n\t"
        "v_xor_b32 %[vt3], %[vt3], %[vt0]\n"
        "L_gnojii%=:\n\t"
        "s_bitcmp1_b32 s51, 0\n\t"
        "s_cbranch_scc0 L_gnoc%=\n\t"
        "s_or_b32 s65, s65, 0x80000000\n\t"
        "s_add_u32 s60, s60, s56\n\t"
        "s_xor_b64 s[48:49], s[48:49], s[46:47]\n"
        "L_gnoc%=:\n\t"
        "v_bitop3_b32 %[jlo], %[jlo], s64, %[vt3] bitop3:0x78\n\t"
        "v_bitop3_b32 %[jhi], %[jhi], s65, %[vt3] bitop3:0x78\n\t"
        "s_branch L_gb%=\n"
        "L_gempty%=:\n\t"
        "s_bitcmp1_b32 s51, 0\n\t"
        "s_cbranch_scc0 L_gb%=\n\t"
        "s_mov_b32 %[ok], 0\n"
        "L_gdone%=:\n\t"
        : [ok] "=&s"(ok), [jlo] "+v"(jlo), [jhi] "+v"(jhi), [glo] "+v"(glo), [ghi] "+v"(ghi),
          "+{s[48:49]}"(h), "+{s[58:59]}"(act), "+{s60}"(W), [vt0] "=&v"(vt0), [vt1] "=&v"(vt1),
          [vt2] "=&v"(vt2), [vt3] "=&v"(vt3)
        : [gblo] "v"(gblo), [gbhi] "v"(gbhi), [h2] "s"(h2), [bstart] "s"(bstart), [bend] "s"(bend)
        : "s46", "s47", "s50", "s51", "s52", "s53", "s56", "s64", "s65", "s66", "s67", "scc");
    return ok;
}

// <s2|s1> for general packed states (stabilizer.c:589-659).  For n <= 60
// the restrictions run in pk_restrict_general and the exponential sum in
// the hand-scheduled loop (as_expsum_packed), on the packed layout.
DEV void ip_general(const RState &r1, const RState &r2, int &eps, int &p, int &m) {
    AState s;
    to_astate(r1, s);
    if (r1.n <= CSE_END_ROW) {
        const int x = lane_id();
        unsigned jlo = (unsigned)s.J, jhi = (unsigned)(s.J >> 32) | ((unsigned)s.d << 29);
        unsigned glo = (unsigned)s.G, ghi = (unsigned)(s.G >> 32);
        u64 h = uniform64(s.h), act = uniform64(s.act);
        unsigned W = (unsigned)__builtin_amdgcn_readfirstlane((int)((unsigned)s.Q << 29));
        const int ok = pk_restrict_general(jlo, jhi, glo, ghi, h, act, W, (unsigned)r2.Gb, (unsigned)(r2.Gb >> 32),
                                           uniform64(r2.h), (unsigned)__builtin_amdgcn_readfirstlane(r2.k),
                                           (unsigned)__builtin_amdgcn_readfirstlane(r2.n));
        if (!ok) {
            eps = 0; p = 0; m = 0;
            return;
        }
        s.J = ((u64)(jhi & 0x1fffffffu) << 32) | jlo;
        s.d = (int)(jhi >> 29);
        s.G = ((u64)ghi << 32) | glo;
        s.h = h;
        s.act = act;
        s.Q = (int)(W >> 29);
        as_subtract_general(s, r2);
        // packed again for the loop: D in bits 61..63, row 60 the end row
        s.J = (s.J & lowmask(CSE_END_ROW)) | ((u64)(s.d & 7) << 61);
        if (x == CSE_END_ROW) s.J = 4ull << 61;
        int pp, mm;
        eps = as_expsum_packed(s, pp, mm);
        p = eps ? pp - r1.k - r2.k : 0;
        m = mm;
        return;
    }
    for (int b = r2.k; b < r2.n; b++) {
        u64 xi = rl64(r2.Gb, b);
        int alpha = par64(r2.h & xi);
        if (!as_restrict(s, xi, alpha)) {
            eps = 0; p = 0; m = 0;
            return;
        }
    }
    as_subtract_general(s, r2);
    int pp, mm;
    eps = as_expsum(s, pp, mm);
    p = eps ? pp - r1.k - r2.k : 0;
    m = mm;
}

}  // namespace

// ======================================================================
extern "C" __global__ void __launch_bounds__(256)
k_ip_pairs(const uint64_t *__restrict__ s1, const uint64_t *__restrict__ s2, int n, int npairs,
           int32_t *__restrict__ out) {
    const int wave = (int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    if (wave >= npairs) return;
    const size_t stride = (size_t)(3 * n + 4);
    RState a, b;
    load_rstate(a, s1 + stride * wave);
    load_rstate(b, s2 + stride * wave);
    int eps, p, m;
    ip_general(a, b, eps, p, m);
    if (lane_id() == 0) {
        out[3 * wave] = eps;
        out[3 * wave + 1] = p;
        out[3 * wave + 2] = m;
    }
}

namespace {

// stateprep.c:85-120 in the reference row bookkeeping
DEV void rs_prepL(RState &s, u64 i, int t, const uint64_t *L, int k) {
    u64 xv = 0;
    for (int j = 0; j < k; j++)
        if ((i >> (k - 1 - j)) & 1ull) xv ^= L[j];
    rs_init(s, t);
    for (int q = 0; q < t; q++)
        if (!((xv >> q) & 1ull)) rs_shrink(s, bit(q), 0, false);
}

// stateprep.c:36-81 in the reference row bookkeeping
DEV void rs_prepH(RState &s, u64 i, int t) {
    const int x = lane_id();
    const int size = (t + 1) / 2;
    rs_init(s, t);
    for (int j = 0; j < size; j++) {
        int b = (int)((i >> (size - 1 - j)) & 1ull);
        if (b == 0 && !((t & 1) && j == size - 1)) {
            if (x == 2 * j) s.J |= bit(2 * j + 1);
            if (x == 2 * j + 1) s.J |= bit(2 * j);
        }
    }
    for (int j = 0; j < size; j++) {
        int b = (int)((i >> (size - 1 - j)) & 1ull);
        if ((t & 1) && j == size - 1) {
            if (b) rs_shrink(s, bit(t - 1), 0, false);
            continue;
        }
        if (b) rs_shrink(s, bit(2 * j) | bit(2 * j + 1), 0, false);
    }
}

// projection by P (innerprod.c:98-116): number of 2^-1/2 factors, -1 if 0
DEV int rs_project(RState &s, const DevProjector &P) {
    int sexp = 0;
    for (int g = 0; g < P.nstabs; g++) {
        int r = rs_measure_pauli(s, P.phase[g] & 3, P.zs[g], P.xs[g]);
        if (r == 0) return -1;
        if (r == 2) sexp++;
    }
    return sexp;
}

DEV u64 shfl64(u64 v, int lane) {
    const unsigned lo = (unsigned)__shfl((int)(unsigned)v, lane, 64);
    const unsigned hi = (unsigned)__shfl((int)(unsigned)(v >> 32), lane, 64);
    return ((u64)hi << 32) | lo;
}

// slot x at bit 31 - x of each half, as the sweep keeps its words
DEV u64 brev32x2(u64 v) { return (u64)__brev((unsigned)v) | (u64)__brev((unsigned)(v >> 32)) << 32; }

// A state as a form on all n columns (cse_tree.h): the slot of a pivot column
// is its coordinate x_a, the slot of another column the multiplier of its
// constraint.  So the state is H on the columns of F applied to the phase
// state sum_s w^{Q + D.s + 4 s J s} |s>, whatever its dimension.  Lane x holds
// row x of J, with d1 (D_x = 2 d1_x + 4 d2_x) on its diagonal; the rest is
// uniform.
struct FormState {
    u64 M;
    u64 d1, d2, F;
    int Q;
};

// The form of a state in reduced row echelon form, rows at their pivot lanes.
//  * x_a = h_a + z_a: the rows with h_a = 1 (H) are expanded about z = 1: Q +=
//    sum_H D + 4 #edges(J in H), D_a -> -D_a on H, D_x += 4 |J_x & H|;
//  * x_q = h_q + G_.q . z on another column: J_q = the column of G, D_q =
//    4 (h_q + |column & H|).  The matrix is U + U^T with U the pivot rows' part
//    of it (J below the diagonal, G at the other columns).
DEV void to_form(const AState &s, int n, FormState &f) {
    const int x = lane_id();
    const bool a = lane_in(s.act);
    const u64 H = s.act & s.h, nonact = lowmask(n) & ~s.act;
    const u64 J = a ? s.J & s.act & ~bit(x) : 0ull, Jl = J & lowmask(x);
    int d = a ? (s.d & 6) : 0;
    f.Q = (s.Q + 2 * __popcll(ballot(lane_in(H) && (d & 2))) + 4 * __popcll(ballot(lane_in(H) && (d & 4))) +
           4 * __popcll(ballot(lane_in(H) && par64(Jl & H)))) & 7;
    const u64 hq = s.h ^ wave_xor(lane_in(H) ? s.G : 0ull);
    if (lane_in(H)) d = (8 - d) & 7;
    d = (d + 4 * par64(J & H)) & 7;
    f.d1 = ballot(a && (d & 2));
    f.d2 = ballot(a && (d & 4)) | (hq & nonact);
    f.F = nonact;
    const u64 U = a ? Jl | (s.G & nonact) : 0ull;
    f.M = U ^ transpose64(U) ^ (f.d1 & bit(x));
}

// Projection of a form by P; returns the number of 2^-1/2 factors, -1 if it
// vanishes.  A generator i^m Z(zeta) X(xi) acts on the phase state as i^m'
// Z(fz) X(fx) with xi and zeta exchanged on F, and multiplies it by w^w
// (-1)^{eta.s}:
//   w = 2 m' + sum_{fx} D + 4 #edges(J in fx), eta = J fx + fz (the diagonal
//   of J is d1).
//  eta empty: nothing (w = 0) or zero (w = 4);
//  w in {2,6}: 2^-1/2 w^{+-1}, D -+= 2 on eta, J ^= eta eta^T;
//  w in {0,4}: the constraint eta . s = w/4, solved for the lowest i in eta,
//   whose slot becomes its multiplier (or its coordinate again), as in a
//   tree's step of the third kind; the updates of J keep d1 on its diagonal.
// Scalar issue bounds it: 63 scalar and 40 vector instructions a generator.
DEV int project_form(FormState &f, const DevProjector &P) {
    const int x = lane_id();
    // generator x in lane x: one load for all instead of one per step
    const u64 pz = P.zs[x], px = P.xs[x], lowx = lowmask(x);
    const int pm = P.phase[x];
    const int ng = P.nstabs;
    u64 M = f.M, d1 = f.d1, d2 = f.d2, F = f.F;
    int Q = f.Q, sexp = 0;
    for (int g = 0; g < ng; g++) {
        const u64 zeta = rl64(pz, g), xi = rl64(px, g), swap = (zeta ^ xi) & F;
        const u64 fx = xi ^ swap, in = M & fx;
        const u64 low = ballot(par64(in & lowx));
        const u64 eta = ballot(par64(in)) ^ zeta ^ swap;
        // w / 2, mod 4
        const int u = rl32(pm, g) + __popcll(d1 & fx) + 2 * (__popcll(zeta & xi & F) + __popcll((low ^ d2) & fx));
        if (eta == 0) {
            if (u & 3) return -1;
            continue;
        }
        sexp++;
        if (u & 1) {
            if (u & 2) {
                Q -= 1;
                d2 ^= eta & d1;
            } else {
                Q += 1;
                d2 ^= eta & ~d1;
            }
            d1 ^= eta;
            if (lane_in(eta)) M ^= eta;
        } else {
            const int i = __builtin_ctzll(eta);
            const u64 o = bit(i), row = rl64(M, i) & ~o, v = eta ^ o;
            const bool ti = (d2 & o) != 0;
            u64 al = row ^ o, wm = row;
            // D_x += +-D_i on v, 4 c on row, 4 on both (c = w / 4)
            if (d1 & o) {
                al ^= v;
                d2 ^= v & d1;
                d1 ^= eta;
                if (u & 2) {
                    Q += ti ? 6 : 2;
                    d2 ^= (row & ~v) ^ (ti ? 0ull : v);
                } else {
                    d2 ^= (row & v) ^ (ti ? v : 0ull);
                }
            } else {
                wm |= o;
                if (u & 2) {
                    Q += ti ? 4 : 0;
                    d2 ^= row & ~v;
                } else {
                    d2 ^= row & v;
                }
                if (ti) d2 ^= v;
            }
            d2 = u & 2 ? d2 | o : d2 & ~o;
            F ^= o;
            M ^= (lane_in(eta) ? al : 0ull) ^ (lane_in(wm) ? eta : 0ull);
        }
    }
    f.M = M;
    f.d1 = d1;
    f.d2 = d2;
    f.F = F;
    f.Q = Q & 7;
    return sexp;
}

// The record of a form: rows and, by a transpose, columns of the symmetric
// matrix move to the instance's slots.
DEV void store_form(const FormState &f, const InstDesc &D, int sexp, uint64_t *rec) {
    const int x = lane_id();
    const int src = x < D.n ? (int)D.inv[x] : x;
    const u64 M = shfl64(transpose64(shfl64(f.M & ~bit(x), src)), src);
    const u64 sx = bit(src);
    const u64 d1 = ballot(f.d1 & sx), d2 = ballot(f.d2 & sx), F = ballot(f.F & sx);
    if (x == 0) {
        rec[0] = ((uint64_t)D.n << 8) | ((uint64_t)f.Q << 16) | ((uint64_t)sexp << 24);
        rec[1] = brev32x2(F);
        rec[2] = brev32x2(d1);
        rec[3] = brev32x2(d2);
    }
    rec[REC_ROWS + x] = brev32x2(M);
}

// The coordinates in which an |H^t> instance's terms are products
// (to_dev on the host is the same change for the projector): with
// u = x_2q and s = x_2q + x_2q+1 in columns 2q and 2q+1, the term with
// coupling is the sum over u and s after a controlled sign on (x_2q, x_2q+1),
// and |00> + |11> is s = 0 with the sum over u signed (-1)^u (the same
// controlled sign undone).
DEV void to_products(AState &s, int n) {
    for (int u = 0; u + 1 < n; u += 2) {
        const u64 cu = ballot(lane_in(s.act) && ((s.G >> u) & 1ull));
        const u64 cv = ballot(lane_in(s.act) && ((s.G >> (u + 1)) & 1ull));
        const int hu = (int)((s.h >> u) & 1ull), hv = (int)((s.h >> (u + 1)) & 1ull);
        s.Q = (s.Q + 4 * (hu & hv)) & 7;
        if (lane_in((cv & allmask(hu)) ^ (cu & allmask(hv)) ^ (cu & cv))) s.d = (s.d + 4) & 7;
        if (lane_in(cu)) s.J ^= cv;
        if (lane_in(cv)) s.J ^= cu;
    }
    const u64 even = 0x5555555555555555ull & lowmask(n & ~1);
    s.G ^= (s.G & even) << 1;
    s.h ^= (s.h & even) << 1;
}

// Reduced row echelon basis of the active rows 0 .. k - 1 (basis changes of
// the form, so the state is unchanged), the rows at their pivot lanes.
DEV void to_rref(AState &s, int k) {
    const int x = lane_id();
    int src = x;
    u64 Pm = 0;
    for (int a = 0; a < k; a++) {
        const u64 Ga = rl64(s.G, a);
        const int pc = __ffsll((long long)Ga) - 1;
        if (x == pc) src = a;
        Pm |= bit(pc);
        const u64 Sp = ballot(x < k && x != a && ((s.G >> pc) & 1ull));
        int dummy;
        if (Sp) as_basis_change(s, a, Sp, true, &dummy);
    }
    // lane p's row is row src of the state, and bit p of a row is its bit src
    // (a transpose away from the same move)
    const bool piv = lane_in(Pm);
    const u64 G = shfl64(s.G, src);
    const int d = __shfl(s.d, src, 64);
    u64 J = shfl64(s.J & lowmask(k), src);
    if (!piv) J = 0;
    J = shfl64(transpose64(J), src);
    s.G = piv ? G : 0ull;
    s.J = piv ? J : 0ull;
    s.d = piv ? d & 6 : 0;
    s.act = Pm;
}

}  // namespace

extern "C" __global__ void __launch_bounds__(256)
k_prep_states(int exact, int t, const uint64_t *__restrict__ L, int k, const uint64_t *__restrict__ idx,
              int count, uint64_t *__restrict__ out) {
    const int wave = (int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    if (wave >= count) return;
    RState s;
    if (exact) rs_prepH(s, idx[wave], t);
    else rs_prepL(s, idx[wave], t, L, k);
    store_rstate(s, out + (size_t)(3 * t + 4) * wave);
}

extern "C" __global__ void __launch_bounds__(256)
k_random_states(int n, const uint64_t *__restrict__ thr, uint64_t seed, long long first, int count,
                DevProjector P, int use_proj, uint64_t *__restrict__ out, int32_t *__restrict__ sexp,
                int *__restrict__ err) {
    const int wave = (int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    if (wave >= count) return;
    RState s;
    if (!rs_random_state(s, n, thr, seed, (uint64_t)(first + wave))) {
        if (lane_id() == 0) atomicOr(err, 1);
        return;
    }
    int se = 0;
    if (use_proj) se = rs_project(s, P);
    if (out) store_rstate(s, out + (size_t)(3 * n + 4) * wave);
    if (sexp && lane_id() == 0) sexp[wave] = se;
}

// The instance that holds global index key: the largest i < n with
// off[i] <= key, for nondecreasing off with off[0] <= key.  The whole wave
// searches: each round lane x reads off[lo + x*step] and the ballot's highest
// lane narrows [lo, lo + len) to one step, so up to 4096 instances take two
// dependent loads instead of twelve.  Lane 0 reads off[lo] <= key, true by
// induction; it enters the ballot unconditionally, so no table can drive lo
// below 0.  Every lane must be active.
DEV int find_instance(const long long *__restrict__ off, int n, long long key) {
    const int x = lane_id();
    int lo = 0, len = n;
    while (len > 1) {
        const int step = (len + 63) >> 6;
        const bool ok = x * step < len && off[lo + x * step] <= key;
        const int hl = 63 - __clzll((long long)(ballot(ok) | 1ull));
        lo += hl * step;
        len = min(step, len - hl * step);
    }
    return lo;
}

// Records of projected states, one wave per record g (global index over all
// instances; instance found from the record prefix).
// mode 0: theta_s = random stabilizer state s = first + local index of the
//         instance's Philox stream (seed); |H^t> instances take it to the
//         coordinates of to_products
// mode 1: phi_i = prepH(i) (exact) or prepL(i) (|L>), i = local index
// then, as a form, Pi (innerprod.c:95-116 / :218-241) and the record.
// The state is a form from the start, so a generator needs no constraint
// solved, no G and no h.  131072 records of t = 40 with 16 generators (mode 1):
// 0.46 ms as states in echelon form (2151 vector and 1412 scalar instructions
// each), 0.249 ms as forms (687 and 1025); 4096 sampled ones of t = 40, r = 8:
// 24.4 and 19.0 us.
extern "C" __global__ void __launch_bounds__(256)
k_records(int mode, int ninst, const long long *__restrict__ rec_off, const InstDesc *__restrict__ inst,
          const DevProjector *__restrict__ projs, const uint64_t *__restrict__ thr_table, long long nrec,
          uint64_t *__restrict__ recs, int32_t *__restrict__ sexp_out, int *__restrict__ err,
          unsigned long long *__restrict__ clock) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *clock = wall_clock64();
    const long long g = (long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (g >= nrec) return;
    const int in = ninst > 1 ? find_instance(rec_off, ninst, g) : 0;
    const InstDesc &D = inst[in];
    const long long local = g - rec_off[in];
    const int n = D.n;
    uint64_t *rec = recs + (size_t)REC_WORDS * (size_t)g;
    FormState f;
    if (mode == 0) {
        RState s;
        if (!rs_random_state(s, n, thr_table + 65 * n, D.seed, (uint64_t)(D.first + local))) {
            if (lane_id() == 0) {
                atomicOr(err, 1);
                sexp_out[g] = -1;
            }
            Rec::store_vanished(rec, n);
            return;
        }
        AState a;
        to_astate(s, a);
        if (D.exact) to_products(a, n);
        to_rref(a, s.k);
        to_form(a, n, f);
    } else {
        // the decomposition state, a product of |0>, |+> and (|H^t>) |->
        const int x = lane_id();
        const bool on = x < D.k && ((local >> x) & 1);
        const u64 xv = (D.exact ? lowmask(n) : 0ull) ^ wave_xor(on ? D.col[x] : 0ull);
        f.M = 0;
        f.d1 = 0;
        f.d2 = D.exact ? wave_xor(on ? D.sgn[x] : 0ull) & xv : 0ull;
        f.F = lowmask(n) & ~xv;
        f.Q = 0;
    }
    const int se = project_form(f, projs[in]);
    if (lane_id() == 0) sexp_out[g] = se;
    if (se < 0) Rec::store_vanished(rec, n);
    else store_form(f, D, se, rec);
}

#include "cse_sweep.h"

// Histogram of the Hamming weight |x| over the 2^k combinations
// x = sum_j i_j L_j of the rows of L (decompose's Z_L, probability.c:
// 371-410).  Thread g of the grid walks the 2^shift combinations
// i = (g << shift) + (Gray code of s), s = 0 .. 2^shift - 1: bit b of i
// selects row k-1-b, as in the reference's MSB-first binrep.  The grid
// holds exactly 2^(k-shift) threads in full blocks of 256 (k - shift >= 8)
// or one block with the surplus threads idle.
extern "C" __global__ void __launch_bounds__(256)
k_lspace_hist(const uint64_t *__restrict__ L, int k, int shift, unsigned long long *__restrict__ hist) {
    __shared__ unsigned int lh[65];
    __shared__ uint64_t rows[64];
    const int tid = (int)threadIdx.x;
    if (tid < 65) lh[tid] = 0;
    if (tid < k) rows[tid] = L[tid];
    __syncthreads();
    const uint64_t g = (uint64_t)blockIdx.x * blockDim.x + (uint64_t)tid;
    if ((g >> (k - shift)) == 0) {
        const uint64_t base = g << shift;
        uint64_t x = 0;
        for (int b = shift; b < k; b++)
            if ((base >> b) & 1ull) x ^= rows[k - 1 - b];
        atomicAdd(&lh[__popcll(x)], 1u);
        const uint64_t steps = 1ull << shift;
        for (uint64_t s = 1; s < steps; s++) {
            x ^= rows[k - 1 - __builtin_ctzll(s)];
            atomicAdd(&lh[__popcll(x)], 1u);
        }
    }
    __syncthreads();
    if (tid < 65 && lh[tid]) atomicAdd(&hist[tid], (unsigned long long)lh[tid]);
}

extern "C" __global__ void k_zero64(unsigned long long *p, long long n) {
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (long long)gridDim.x * blockDim.x) p[i] = 0ull;
}

// A batch's plan copied from pinned host memory, its results block and work
// queue cleared, grid-stride.
struct PrepArgs {
    const uint4 *src;
    uint4 *dst, *zero;
    long long ncopy, nzero;  // 16-byte words
    unsigned long long *queue;  // and the count of k_results
};
extern "C" __global__ void k_prep(PrepArgs a) {
    const long long stride = (long long)gridDim.x * blockDim.x;
    const long long i0 = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    for (long long i = i0; i < a.ncopy; i += stride) a.dst[i] = a.src[i];
    for (long long i = i0; i < a.nzero; i += stride) a.zero[i] = make_uint4(0, 0, 0, 0);
    if (i0 == 0) a.queue[0] = a.queue[1] = 0;
}

// A batch's results block to pinned host memory, grid-stride; with `done`, the
// call's number after them, by the last block to finish.
//
// nvals > 0: no caller wants the histograms of the exact instances, so their
// Z[w] sums go to the host instead: 64 bytes an instance for 8,256, and what
// the host needs 2.5 us an instance for takes a wave 2 to 3.  The sums and the
// order of the additions are cse_hist_value's, so the values are the same
// bits.  (A count is at most chi^2 <= 2^60, so 64-bit integers hold every sum
// that is kept in 128 bits there.)
struct ResultArgs {
    const uint4 *src;
    uint4 *dst;
    long long n;             // 16-byte words
    unsigned long long *clock;
    const unsigned long long *hist;
    double *vals;            // 8 per instance, pinned
    int nvals;
    // one exact instance whose sums come in copies (SweepArgs): of the
    // histogram, and from word `tail` of src of the Kahan pair and the count
    int copies, tail;
    long long copy_words;
    unsigned *left;          // blocks that have finished
    uint32_t *done;
    uint32_t call;
};
namespace {

constexpr int kValueExps = (HIST_STRIDE / 8) / 2 + 2;  // powers of two: 0, -1 .. -65

struct Dd {
    double hi, lo;
};
DEV Dd dd_two_sum(double a, double b) {
    const double s = a + b, bb = s - a;
    return {s, (a - (s - bb)) + (b - bb)};
}
DEV Dd dd_quick_sum(double a, double b) {
    const double s = a + b;
    return {s, b - (s - a)};
}
DEV Dd dd_add(Dd a, Dd b) {
    Dd s = dd_two_sum(a.hi, b.hi);
    const Dd t = dd_two_sum(a.lo, b.lo);
    s.lo += t.hi;
    s = dd_quick_sum(s.hi, s.lo);
    s.lo += t.lo;
    return dd_quick_sum(s.hi, s.lo);
}
DEV Dd dd_int(long long v, int e) {
    const double hi = (double)v;
    const Dd r = dd_quick_sum(hi, (double)(v - (long long)hi));
    return {ldexp(r.hi, e), ldexp(r.lo, e)};
}

// Row P = -r of a histogram: the sums of its even phases (real, imaginary)
// and of its odd ones, the latter in units of sqrt(1/2).
struct HistRow {
    long long er = 0, ei = 0, orr = 0, oi = 0;
    DEV HistRow(const unsigned long long *h, int r) {
        if (r < 0 || r >= HIST_STRIDE / 8) return;
        const long long *b = (const long long *)h + 8 * r;
        er = b[0] - b[4];
        ei = b[2] - b[6];
        orr = (b[1] - b[3]) - (b[5] - b[7]);
        oi = (b[1] + b[3]) - (b[5] + b[7]);
    }
};

}  // namespace
template <bool COPIES> DEV void results_body(const ResultArgs &a) {
    const unsigned long long now = wall_clock64();
    __shared__ Dd s_acc[4][4][kValueExps];
    __shared__ unsigned long long s_sum[COPIES ? HIST_STRIDE + 3 : 1];
    const unsigned long long *hist = a.hist;
    if (COPIES) {
        for (int w = (int)threadIdx.x; w < HIST_STRIDE + 3; w += 256) {
            const int t = w - HIST_STRIDE;
            const unsigned long long *p = t < 0 ? a.hist + w : (const unsigned long long *)a.src + a.tail + t;
            unsigned long long v[TREE_COPIES], s = 0;
            double k = 0.0;
#pragma unroll
            for (int c = 0; c < TREE_COPIES; c++) v[c] = c < a.copies ? p[(size_t)c * (size_t)a.copy_words] : 0ull;
#pragma unroll
            for (int c = 0; c < TREE_COPIES; c++) {
                s += v[c];
                k += __longlong_as_double((long long)v[c]);
            }
            s_sum[w] = t == 0 || t == 1 ? (unsigned long long)__double_as_longlong(k) : s;
        }
        __syncthreads();
        hist = s_sum;
    }
    // an instance a wave: lane j adds up what has the power -j of two (rows
    // 2j, 2j - 1 and 2j - 2), four lanes then add the powers from the lowest
    const int x = lane_id(), wv = (int)threadIdx.x >> 6;
    for (int at = 4 * (int)blockIdx.x; at < a.nvals; at += 4 * (int)gridDim.x) {
        const int i = at + wv;
        u64 used = 0;
        if (i < a.nvals) {
            const unsigned long long *h = hist + (size_t)HIST_STRIDE * (size_t)i;
            for (int j0 = 0; j0 < kValueExps; j0 += 64) {
                const int j = j0 + x;
                const bool in = j < kValueExps;
                const HistRow r0(h, in ? 2 * j : -1), r1(h, in ? 2 * j - 1 : -1), r2(h, in ? 2 * j - 2 : -1);
                const long long v[4] = {r0.er + r1.orr, r0.ei + r1.oi, r1.er + r2.orr, r1.ei + r2.oi};
                if (in)
                    for (int q = 0; q < 4; q++) s_acc[wv][q][j] = dd_int(v[q], -j);
                const u64 some = ballot((v[0] | v[1] | v[2] | v[3]) != 0);
                if (j0 == 0) used = some;
                else if (some) used |= 1ull << 63;  // 63 stands for the rest as well
            }
        }
        __syncthreads();
        if (i < a.nvals && x < 4) {
            Dd s = {0.0, 0.0};
            if (used >> 63)
                for (int j = kValueExps - 1; j >= 63; j--) s = dd_add(s, s_acc[wv][x][j]);
            for (used &= ~(1ull << 63); used;) {
                const int j = 63 - __clzll((long long)used);
                used &= ~(1ull << j);
                s = dd_add(s, s_acc[wv][x][j]);
            }
            a.vals[8 * (size_t)i + 2 * x] = s.hi;
            a.vals[8 * (size_t)i + 2 * x + 1] = s.lo;
        }
        __syncthreads();
    }
    const long long stride = (long long)gridDim.x * blockDim.x;
    const long long i0 = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    // the clock is part of the block's last words: its 16 bytes are put
    // together by the thread that copies them
    const long long off = (const char *)a.clock - (const char *)a.src, at = off >> 4;
    const int half = (int)(off >> 3) & 1;
    if (i0 == 0 && a.n == 0) *a.clock = now;
    for (long long i = i0; i < a.n; i += stride) {
        uint4 v = a.src[i];
        if (COPIES) {
            const int w = (int)(2 * i), u = w - a.tail + HIST_STRIDE;
            unsigned long long lo = v.x | (u64)v.y << 32, hi = v.z | (u64)v.w << 32;
            if (a.nvals == 0 && w < HIST_STRIDE) lo = s_sum[w], hi = s_sum[w + 1];
            if (u >= HIST_STRIDE && u < HIST_STRIDE + 3) lo = s_sum[u];
            if (u + 1 >= HIST_STRIDE && u + 1 < HIST_STRIDE + 3) hi = s_sum[u + 1];
            v = make_uint4((unsigned)lo, (unsigned)(lo >> 32), (unsigned)hi, (unsigned)(hi >> 32));
        }
        if (i == at) {
            if (half) {
                v.z = (unsigned)now;
                v.w = (unsigned)(now >> 32);
            } else {
                v.x = (unsigned)now;
                v.y = (unsigned)(now >> 32);
            }
        }
        a.dst[i] = v;
    }
    if (a.done) {
        // a block's stores have reached the host before it counts itself (a
        // block of its own has nobody to count: the atomic costs 1 us), and
        // the last one tells the host
        __threadfence_system();
        __syncthreads();
        if (threadIdx.x == 0 &&
            (gridDim.x == 1 ||
             __hip_atomic_fetch_add(a.left, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1))
            __hip_atomic_store(a.done, a.call, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}
extern "C" __global__ void __launch_bounds__(256) k_results(ResultArgs a) { results_body<false>(a); }
extern "C" __global__ void __launch_bounds__(256) k_results_copies(ResultArgs a) { results_body<true>(a); }
