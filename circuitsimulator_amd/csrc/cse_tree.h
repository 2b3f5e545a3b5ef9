// cse_tree.h -- per-lane exponential sums of the sweep: one lane holds one
// stabilizer form and walks a binary tree of decomposition terms.
//
// The form.  A record (k_records) holds a projected state as a form on n
// slots, one per qubit, in the instance's slot order: J (symmetric, bit y of
// row x), D_x = 2 d1_x + 4 d2_x and a phase.  The slot of a pivot column q is
// the coordinate x_q itself; the slot of any other column is the multiplier y
// of its constraint, (1/2) sum_y (-1)^{y x_q}, whose value 0 stands for "x_q
// is free".  So a term <phi_j| needs, slot by slot, either the sum over the
// slot's variable or its value at 0, and a change of the term toggles the
// same slots whatever the record is: A = x_j ^ F, with bit x of A set when
// slot x is summed and F the set of slots that hold multipliers.
//
// One step sums slot c out of the form or drops it (its value is 0):
//   D_c in {2,6}: sqrt2 w^{+-1}; J ^= v v^T and D -+= 2 on v = J_c;
//   D_c in {0,4}, v empty: 2 (or 0 for D_c = 4);
//   D_c in {0,4}: sum_c gives 2 [v.z = D_c/4], which is solved for one i in v
//     and slot i then holds the multiplier of z_i (D_i = D_c, J_i = v - i):
//     "sum over z_i" is "multiplier 0" and the other way round, so bit i of A
//     is toggled, and neither the order of the slots nor the slots that
//     another term sums matter.
// Every step is the same straight-line code for all lanes, with masks where
// lanes differ.  The sum is 2^{p/2} w^m with p = (steps of the second kind)
// - n, all norms included.
//
// |H^t> terms add a sign per slot (T): a summed slot is summed with
// (-1)^{T z}, a dropped one is taken at z = T.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define TREE_DEV __device__ __forceinline__
#define TREE_BFE(v, i) ((u32)__builtin_amdgcn_sbfe((int)(v), (unsigned)(i), 1u))
// x ^ (a & b) as the one instruction that it is (left to itself the compiler
// splits the sums below into three per term)
#define TREE_XA(x, a, b) ((u32)__builtin_amdgcn_bitop3_b32((x), (a), (b), 0x78))
#define TREE_POP(v) __popc(v)
#define TREE_FFS(v) ((u32)(__ffs((int)(v)) - 1))
#else
#define TREE_DEV inline
#define TREE_BFE(v, i) ((u32)((int32_t)((uint32_t)(v) << (31 - ((i) & 31))) >> 31))
#define TREE_XA(x, a, b) ((x) ^ ((a) & (b)))
#define TREE_POP(v) __builtin_popcount(v)
#define TREE_FFS(v) ((u32)(__builtin_ffs((int)(v)) - 1))
#endif

namespace cse {
namespace tree {

typedef uint32_t u32;

// rows below slot 32 are kept as one word (the part of a row at slots >= 32
// is read from the rows of those slots), the NH rows from slot 32 on as two
template <int NH> struct Form {
    u32 lo[32 + NH];
    u32 hi[NH > 0 ? NH : 1];
    u32 d1, d2, A, T;       // slots 0..31
    u32 d1h, d2h, Ah, Th;   // slots 32..
    u32 x2;                 // parity word: 4 per set bit
    u32 z;                  // top bit set: the sum is 0
    int nb, q1;             // steps of the third kind; phase in units of 2
};

// bits of slots below c, c <= 32
TREE_DEV u32 low32(int c) { return c >= 32 ? ~0u : (1u << c) - 1u; }

// Step of slot C < 32 (all slots above it done).
template <int NH, bool HT, int C> TREE_DEV void step(Form<NH> &f) {
    const u32 below = low32(C);
    const u32 act = TREE_BFE(f.A, C);
    const u32 odd = TREE_BFE(f.d1, C);
    if (HT) {
        // a dropped slot is taken at T: D_x += 4 T J_cx
        const u32 at1 = TREE_BFE(f.T, C) & ~act;
        f.d2 ^= f.lo[C] & at1 & below;
    }
    const u32 hi = TREE_BFE(HT ? f.d2 ^ f.T : f.d2, C);
    const u32 v = f.lo[C] & act & below;
    const u32 o = v & (0u - v) & ~odd;      // the slot solved for, if any
    const u32 i = TREE_FFS(v);              // all ones when v is empty
    // second kind, in the top bit (i < 32 otherwise)
    const u32 iso = act & ~odd & i;
    f.z |= iso & hi;
    if (C == 0) return;
    const u32 oddi = TREE_BFE(f.d1, i), d2i = TREE_BFE(f.d2, i);
    const u32 e = odd | oddi;
    const u32 u = d2i ^ (hi & oddi);
    const u32 h = (odd & ~hi) | (~odd & u);
    u32 w = 0;
#pragma unroll
    for (int x = 0; x < C; x++) w = TREE_XA(w, TREE_BFE(o, x), f.lo[x]);
    w &= below & ~o;
    const u32 vp = v & ~o;
    const u32 ev = e & vp;
    const u32 al = w ^ o ^ ev;
    const u32 wm = w | (o & ~oddi);
    const u32 oh = o & hi;
    f.q1 += TREE_POP(oh & f.d1);
    f.x2 ^= oh & f.d2;
    f.nb += TREE_POP(o);
    const u32 g = h ^ (e & f.d1);
    f.d2 ^= (vp & g) ^ (w & (hi ^ vp));
    f.d1 = (f.d1 ^ ev) & ~o;
    f.d2 = (f.d2 & ~o) | oh;
#pragma unroll
    for (int x = 0; x < C; x++)
        f.lo[x] = TREE_XA(TREE_XA(f.lo[x], TREE_BFE(v, x), al), TREE_BFE(wm, x), v);
    f.A ^= o;
}

// Step of slot 32 + C.
template <int NH, bool HT, int C> TREE_DEV void step_hi(Form<NH> &f) {
    const u32 below = low32(C);
    const u32 act = TREE_BFE(f.Ah, C);
    const u32 odd = TREE_BFE(f.d1h, C);
    if (HT) {
        const u32 at1 = TREE_BFE(f.Th, C) & ~act;
        f.d2 ^= f.lo[32 + C] & at1;
        f.d2h ^= f.hi[C] & at1 & below;
    }
    const u32 hi = TREE_BFE(HT ? f.d2h ^ f.Th : f.d2h, C);
    const u32 vl = f.lo[32 + C] & act, vh = f.hi[C] & act & below;
    const u32 inl = vh ? 0u : ~0u;          // the solved slot is below 32
    const u32 ol = vl & (0u - vl) & ~odd & inl, oh = vh & (0u - vh) & ~odd;
    const u32 iso = (vl | vh) ? 0u : act & ~odd;
    f.z |= iso & hi & 0x80000000u;
    const u32 oddi = ((f.d1 & ol) | (f.d1h & oh)) ? ~0u : 0u;
    const u32 d2i = ((f.d2 & ol) | (f.d2h & oh)) ? ~0u : 0u;
    const u32 e = odd | oddi;
    const u32 u = d2i ^ (hi & oddi);
    const u32 h = (odd & ~hi) | (~odd & u);
    u32 wl = 0, wh = 0;
#pragma unroll
    for (int x = 0; x < 32; x++) wl = TREE_XA(wl, TREE_BFE(ol, x), f.lo[x]);
    const u32 il = TREE_FFS(ol);
#pragma unroll
    for (int x = 0; x < C; x++) {
        const u32 m = TREE_BFE(oh, x);
        wl = TREE_XA(wl, m, f.lo[32 + x]);
        wh = TREE_XA(wh, m, f.hi[x]);
    }
    u32 col = 0;  // column il of the rows above, when il is a slot
#pragma unroll
    for (int x = 0; x < C; x++) col |= (TREE_BFE(f.lo[32 + x], il) & 1u) << x;
    wh ^= col & (ol ? ~0u : 0u);
    wl &= ~ol;
    wh &= below & ~oh;
    const u32 vpl = vl & ~ol, vph = vh & ~oh;
    const u32 evl = e & vpl, evh = e & vph;
    const u32 all = wl ^ ol ^ evl, alh = wh ^ oh ^ evh;
    const u32 wml = wl | (ol & ~oddi), wmh = wh | (oh & ~oddi);
    const u32 ohl = ol & hi, ohh = oh & hi;
    f.q1 += TREE_POP(ohl & f.d1) + TREE_POP(ohh & f.d1h);
    f.x2 ^= (ohl & f.d2) ^ (ohh & f.d2h);
    f.nb += TREE_POP(ol) + TREE_POP(oh);
    const u32 gl = h ^ (e & f.d1), gh = h ^ (e & f.d1h);
    f.d2 ^= (vpl & gl) ^ (wl & (hi ^ vpl));
    f.d2h ^= (vph & gh) ^ (wh & (hi ^ vph));
    f.d1 = (f.d1 ^ evl) & ~ol;
    f.d1h = (f.d1h ^ evh) & ~oh;
    f.d2 = (f.d2 & ~ol) | ohl;
    f.d2h = (f.d2h & ~oh) | ohh;
#pragma unroll
    for (int x = 0; x < 32; x++)
        f.lo[x] = TREE_XA(TREE_XA(f.lo[x], TREE_BFE(vl, x), all), TREE_BFE(wml, x), vl);
#pragma unroll
    for (int x = 0; x < C; x++) {
        const u32 m1 = TREE_BFE(vh, x), m2 = TREE_BFE(wmh, x);
        f.lo[32 + x] = TREE_XA(TREE_XA(f.lo[32 + x], m1, all), m2, vl);
        f.hi[x] = TREE_XA(TREE_XA(f.hi[x], m1, alh), m2, vh);
    }
    f.A ^= ol;
    f.Ah ^= oh;
}

// Steps of the slots c1 + cn - 1 .. c1 (uniform bounds, c1 + cn <= 32).
template <int NH, bool HT, int C> struct Steps {
    static TREE_DEV void run(Form<NH> &f, int c1, u32 cn) {
        if ((u32)(C - c1) < cn) step<NH, HT, C>(f);
        Steps<NH, HT, C - 1>::run(f, c1, cn);
    }
};
template <int NH, bool HT> struct Steps<NH, HT, -1> {
    static TREE_DEV void run(Form<NH> &, int, u32) {}
};
template <int NH, bool HT, int C> struct StepsHi {
    static TREE_DEV void run(Form<NH> &f, int c0) {
        if (c0 > 32 + C) step_hi<NH, HT, C>(f);
        StepsHi<NH, HT, C - 1>::run(f, c0);
    }
};
template <int NH, bool HT> struct StepsHi<NH, HT, -1> {
    static TREE_DEV void run(Form<NH> &, int) {}
};

// What the finished slots below 32 (word arguments) or above (the h words)
// give: phase in units of 1 and the count of active slots less the steps of
// the first kind; the third kind's share (nb, q1, x2) is added at the end.
template <bool HT> TREE_DEV void fold(u32 d1, u32 d2, u32 A, u32 T, int &ph, int &cnt) {
    const u32 a1 = A & d1;
    const int na = TREE_POP(a1);
    cnt += TREE_POP(A) - na;
    ph += na - 2 * TREE_POP(a1 & (HT ? d2 ^ T : d2));
    if (HT) ph += 2 * TREE_POP(T & ~A & d1) + 4 * TREE_POP(T & ~A & d2);
}

}  // namespace tree
}  // namespace cse
