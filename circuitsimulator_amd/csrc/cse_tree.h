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
//
// Slot x < 32 is bit 31 - x of a word, slot 32 + x bit 31 - x of the next one.
//
// Instructions.  gfx950 issues and, xor, or, bitop3, add, sub, right shifts
// and fma at twice the rate of the other VALU instructions (4.4-4.6 against
// 2.2 wave instructions per ns and CU, two or more waves per SIMD), but only
// in stretches without a single one of the others: one v_bfe_i32 or v_bcnt in
// 64 brings all of them down to 2.4 until a scalar instruction shifts the
// waves' phases again.  So a step is written in the fast ones alone: a mask
// from a bit is and, sub, ashr (not v_bfe_i32), successive row masks are ashr
// and add (not v_bfe_i32 at each bit), the row of a slot that differs from
// lane to lane is picked by a tree of bitop3 selects, and counts are sums of
// masks (not v_bcnt).  With row updates through masks (rows, below, has what
// they are now) a step of slot 10 took 93 instructions at 2.4 per ns and CU
// with v_bfe_i32, 125 at 4.4 this way.
#pragma once
#include <stdint.h>

namespace cse {
namespace tree {

typedef uint32_t u32;

// truth tables of the three operands
constexpr unsigned TA = 0xF0, TB = 0xCC, TC = 0xAA;

#ifdef __HIPCC__
#define TREE_DEV __device__ __forceinline__
// the three-operand boolean function of truth table F in one instruction
#define TREE_B3(a, b, c, F) ((cse::tree::u32)__builtin_amdgcn_bitop3_b32((a), (b), (c), (F) & 0xffu))
#define TREE_POP(v) __popc(v)
// v is 0 in every lane
#define TREE_NONE(v) (__builtin_amdgcn_ballot_w64((v) != 0) == 0)
// the top n bits of v shifted in below i
#define TREE_SHIN(i, v, n) ((cse::tree::u32)__builtin_amdgcn_alignbit((i), (v), 32 - (n)))
template <u32 K> TREE_DEV u32 andk(u32 v) {
    u32 r;
    asm("v_and_b32 %0, %2, %1" : "=v"(r) : "v"(v), "n"(K));
    return r;
}
// all ones if t, a single bit or zero, is set
#define TREE_NZ(r) "v_sub_u32 " r ", 0, " r "\n\tv_ashrrev_i32 " r ", 31, " r "\n\t"
TREE_DEV u32 nz1(u32 t) {
    asm(TREE_NZ("%0") : "+&v"(t));
    return t;
}
TREE_DEV void nz2(u32 &t, u32 &u) { asm(TREE_NZ("%0") TREE_NZ("%1") : "+&v"(t), "+&v"(u)); }
// all ones if the single bit K of v is set
template <u32 K> TREE_DEV u32 bitk(u32 v) {
    u32 r;
    asm("v_and_b32 %0, %2, %1\n\t" TREE_NZ("%0") : "=v"(r) : "v"(v), "n"(K));
    return r;
}
template <u32 K> TREE_DEV void bitk2(u32 v, u32 w, u32 &r, u32 &q) {
    asm("v_and_b32 %0, %4, %2\n\tv_and_b32 %1, %4, %3\n\t" TREE_NZ("%0") TREE_NZ("%1")
        : "=&v"(r), "=&v"(q)
        : "v"(v), "v"(w), "n"(K));
}
template <u32 K> TREE_DEV void bitk4(u32 a, u32 b, u32 c, u32 d, u32 *r) {
    asm("v_and_b32 %0, %8, %4\n\tv_and_b32 %1, %8, %5\n\tv_and_b32 %2, %8, %6\n\tv_and_b32 %3, %8, %7\n\t"
        TREE_NZ("%0") TREE_NZ("%1") TREE_NZ("%2") TREE_NZ("%3")
        : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])
        : "v"(a), "v"(b), "v"(c), "v"(d), "n"(K));
}
// mask of the top bit, and the next bit moved up
TREE_DEV u32 pop_mask(u32 &t) {
    u32 m;
    asm("v_ashrrev_i32 %0, 31, %1\n\tv_add_u32 %1, %1, %1" : "=&v"(m), "+&v"(t));
    return m;
}
// the sign bit of 0 - t put in at the top of w, the others moved down (t a
// single bit or zero)
TREE_DEV u32 push_nz(u32 w, u32 t) {
    asm("v_lshrrev_b32 %0, 1, %0\n\tv_sub_u32 %1, 0, %1\n\tv_and_b32 %1, 0x80000000, %1\n\tv_or_b32 %0, %0, %1"
        : "+&v"(w), "+&v"(t));
    return w;
}
// (Operands that a block writes before its last read are early clobbers: tv
// and b start as the same value.)
// N rows r: r ^= a where tv's next bit is set, ^= b where tw's is.  One asm
// block for several rows: between blocks the compiler pads with s_nop.
//
// From four rows on a bit leaves its word as the carry of word + word, and the
// carry selects a or 0: five instructions a row.  A carry must not be read in
// the next two instructions after the one that writes it, so a row's selects
// wait behind the update of the row before.  The second carry is in a fixed
// pair below s64: with carries in s64 or above the same stream runs at 2.4
// instead of 3.7 wave instructions per ns and CU (the register allocator took
// s64 in the exact kernels, which then lost 10%).  One or two rows, where the
// wait is not filled, take masks: six a row.  2^28 terms of t = 48 with masks
// throughout 10.1 ms, with carries from eight rows on 9.5, from four 9.3.
#define TREE_CARRY "v_add_co_u32 %[tv], vcc, %[tv], %[tv]\n\tv_add_co_u32 %[tw], s[46:47], %[tw], %[tw]\n\t"
#define TREE_SEL "v_cndmask_b32 %[m], 0, %[a], vcc\n\tv_cndmask_b32 %[q], 0, %[b], s[46:47]\n\t"
#define TREE_UPD(r) "v_bitop3_b32 " r ", " r ", %[m], %[q] bitop3:0x96\n\t"
#define TREE_ROW0 TREE_CARRY "s_nop 0\n\t" TREE_SEL
#define TREE_ROW(r) TREE_CARRY TREE_UPD(r) TREE_SEL
#define TREE_ROWS_IO                                                                     \
    [tv] "+&v"(tv), [tw] "+&v"(tw), [m] "=&v"(m), [q] "=&v"(q) : [a] "v"(a), [b] "v"(b) : "vcc", "s46", "s47"
#define TREE_FEW(r)                                                                        \
    "v_ashrrev_i32 %[m], 31, %[tv]\n\tv_add_u32 %[tv], %[tv], %[tv]\n\t"                  \
    "v_bitop3_b32 " r ", " r ", %[m], %[a] bitop3:0x78\n\t"                                \
    "v_ashrrev_i32 %[m], 31, %[tw]\n\tv_add_u32 %[tw], %[tw], %[tw]\n\t"                  \
    "v_bitop3_b32 " r ", " r ", %[m], %[b] bitop3:0x78\n\t"
#define TREE_FEW_IO [tv] "+&v"(tv), [tw] "+&v"(tw), [m] "=&v"(m) : [a] "v"(a), [b] "v"(b)
template <int N> TREE_DEV void rows(u32 *r, u32 &tv, u32 &tw, u32 a, u32 b) {
    u32 m, q;
    if constexpr (N >= 8) {
        asm(TREE_ROW0 TREE_ROW("%0") TREE_ROW("%1") TREE_ROW("%2") TREE_ROW("%3") TREE_ROW("%4") TREE_ROW("%5")
                TREE_ROW("%6") TREE_UPD("%7")
            : "+&v"(r[0]), "+&v"(r[1]), "+&v"(r[2]), "+&v"(r[3]), "+&v"(r[4]), "+&v"(r[5]), "+&v"(r[6]), "+&v"(r[7]),
              TREE_ROWS_IO);
        rows<N - 8>(r + 8, tv, tw, a, b);
    } else if constexpr (N >= 4) {
        asm(TREE_ROW0 TREE_ROW("%0") TREE_ROW("%1") TREE_ROW("%2") TREE_UPD("%3")
            : "+&v"(r[0]), "+&v"(r[1]), "+&v"(r[2]), "+&v"(r[3]), TREE_ROWS_IO);
        rows<N - 4>(r + 4, tv, tw, a, b);
    } else if constexpr (N >= 2) {
        asm(TREE_FEW("%0") TREE_FEW("%1") : "+&v"(r[0]), "+&v"(r[1]), TREE_FEW_IO);
        rows<N - 2>(r + 2, tv, tw, a, b);
    } else if constexpr (N == 1) {
        asm(TREE_FEW("%0") : "+&v"(r[0]), TREE_FEW_IO);
    }
}
// the same for rows of two words
TREE_DEV void row2(u32 &r, u32 &q, u32 &tv, u32 &tw, u32 a, u32 b, u32 c, u32 d) {
    u32 m;
    asm("v_ashrrev_i32 %[m], 31, %[tv]\n\tv_add_u32 %[tv], %[tv], %[tv]\n\t"
        "v_bitop3_b32 %[r], %[r], %[m], %[a] bitop3:0x78\n\tv_bitop3_b32 %[q], %[q], %[m], %[c] bitop3:0x78\n\t"
        "v_ashrrev_i32 %[m], 31, %[tw]\n\tv_add_u32 %[tw], %[tw], %[tw]\n\t"
        "v_bitop3_b32 %[r], %[r], %[m], %[b] bitop3:0x78\n\tv_bitop3_b32 %[q], %[q], %[m], %[d] bitop3:0x78"
        : [r] "+&v"(r), [q] "+&v"(q), [tv] "+&v"(tv), [tw] "+&v"(tw), [m] "=&v"(m)
        : [a] "v"(a), [b] "v"(b), [c] "v"(c), [d] "v"(d));
}
// masks of the bits of a slot's number: w[k] starts as o with the slots that
// have bit k, and becomes all ones if that is not empty
template <int K> TREE_DEV void picked(u32 o, u32 *w) {
#define TREE_PK(i, mask) "v_and_b32 %" #i ", " #mask ", %[o]\n\t" TREE_NZ("%" #i)
    if constexpr (K == 5)
        asm(TREE_PK(0, 0x55555555) TREE_PK(1, 0x33333333) TREE_PK(2, 0x0f0f0f0f) TREE_PK(3, 0x00ff00ff)
                TREE_PK(4, 0x0000ffff)
            : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3]), "=&v"(w[4])
            : [o] "v"(o));
    if constexpr (K == 4)
        asm(TREE_PK(0, 0x55555555) TREE_PK(1, 0x33333333) TREE_PK(2, 0x0f0f0f0f) TREE_PK(3, 0x00ff00ff)
            : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3])
            : [o] "v"(o));
    if constexpr (K == 3)
        asm(TREE_PK(0, 0x55555555) TREE_PK(1, 0x33333333) TREE_PK(2, 0x0f0f0f0f)
            : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2])
            : [o] "v"(o));
    if constexpr (K == 2)
        asm(TREE_PK(0, 0x55555555) TREE_PK(1, 0x33333333) : "=&v"(w[0]), "=&v"(w[1]) : [o] "v"(o));
    if constexpr (K == 1) asm(TREE_PK(0, 0x55555555) : "=&v"(w[0]) : [o] "v"(o));
}
#else
#define TREE_DEV inline
#define TREE_POP(v) __builtin_popcount(v)
#define TREE_NONE(v) ((v) == 0)
inline u32 tree_b3(u32 a, u32 b, u32 c, unsigned F) {
    u32 r = 0;
    for (int i = 0; i < 8; i++)
        if ((F >> i) & 1) r |= ((i & 4) ? a : ~a) & ((i & 2) ? b : ~b) & ((i & 1) ? c : ~c);
    return r;
}
#define TREE_B3(a, b, c, F) (cse::tree::tree_b3((a), (b), (c), (F) & 0xffu))
#define TREE_SHIN(i, v, n) (((i) << (n)) | ((v) >> (32 - (n))))
template <u32 K> inline u32 andk(u32 v) { return v & K; }
inline u32 nz1(u32 t) { return t ? ~0u : 0u; }
inline void nz2(u32 &t, u32 &u) {
    t = nz1(t);
    u = nz1(u);
}
template <u32 K> inline u32 bitk(u32 v) { return nz1(v & K); }
template <u32 K> inline void bitk2(u32 v, u32 w, u32 &r, u32 &q) {
    r = nz1(v & K);
    q = nz1(w & K);
}
template <u32 K> inline void bitk4(u32 a, u32 b, u32 c, u32 d, u32 *r) {
    r[0] = nz1(a & K);
    r[1] = nz1(b & K);
    r[2] = nz1(c & K);
    r[3] = nz1(d & K);
}
inline u32 pop_mask(u32 &t) {
    const u32 m = nz1(t >> 31);
    t += t;
    return m;
}
inline u32 push_nz(u32 w, u32 t) { return (w >> 1) | (t ? 0x80000000u : 0u); }
template <int N> inline void rows(u32 *r, u32 &tv, u32 &tw, u32 a, u32 b) {
    for (int x = 0; x < N; x++) {
        r[x] ^= pop_mask(tv) & a;
        r[x] ^= pop_mask(tw) & b;
    }
}
inline void row2(u32 &r, u32 &q, u32 &tv, u32 &tw, u32 a, u32 b, u32 c, u32 d) {
    const u32 m = pop_mask(tv), l = pop_mask(tw);
    r ^= (m & a) ^ (l & b);
    q ^= (m & c) ^ (l & d);
}
template <int K> inline void picked(u32 o, u32 *w) {
    static const u32 with[5] = {0x55555555u, 0x33333333u, 0x0f0f0f0fu, 0x00ff00ffu, 0x0000ffffu};
    for (int k = 0; k < K; k++) w[k] = nz1(o & with[k]);
}
#endif
// x ^ (a & b)
#define TREE_XA(x, a, b) TREE_B3(x, a, b, TA ^ (TB & TC))

// rows below slot 32 are kept as one word (the part of a row at slots >= 32
// is read from the rows of those slots), the NH rows from slot 32 on as two
template <int NH> struct Form {
    u32 lo[32 + NH];
    u32 hi[NH > 0 ? NH : 1];
    u32 d1, d2, A, T;       // slots 0..31
    u32 d1h, d2h, Ah, Th;   // slots 32..
    u32 x2;                 // parity word: 4 per set bit
    u32 z;                  // top bit set: the sum is 0
    u32 nb, q1;             // steps of the third kind; phase in units of 2
};

constexpr u32 slot_bit(int x) { return 0x80000000u >> x; }
// bits of the slots below c, c < 32
constexpr u32 below(int c) { return c == 0 ? 0u : ~0u << (32 - c); }
// bits of a slot number below N
constexpr int index_bits(int N) { return N > 16 ? 5 : N > 8 ? 4 : N > 4 ? 3 : N > 2 ? 2 : N > 1 ? 1 : 0; }

// r[the slot of masks b], a tree of selects over r[LO .. LO + 2^K - 1] below N
template <int N, int K, int LO> struct Pick {
    static TREE_DEV u32 run(const u32 *r, const u32 *b) {
        const u32 lo = Pick<N, K - 1, LO>::run(r, b);
        constexpr int UP = LO + (1 << (K - 1));
        if (UP >= N) return lo;
        const u32 up = Pick<N, K - 1, (UP < N ? UP : LO)>::run(r, b);
        return TREE_B3(b[K - 1], up, lo, (TA & TB) | (~TA & TC));
    }
};
template <int N, int LO> struct Pick<N, 0, LO> {
    static TREE_DEV u32 run(const u32 *r, const u32 *) { return r[LO]; }
};
template <int N> TREE_DEV u32 pick(const u32 *r, const u32 *b) { return Pick<N, index_bits(N), 0>::run(r, b); }

// Step of slot C < 32 (all slots above it done).
template <int NH, bool HT, int C> TREE_DEV void step(Form<NH> &f) {
    u32 act, odd;
    bitk2<slot_bit(C)>(f.A, f.d1, act, odd);
    const u32 row = andk<below(C)>(f.lo[C]);
    // a dropped slot is taken at T: D_x += 4 T J_cx
    if (HT) f.d2 = TREE_XA(f.d2, row, TREE_B3(bitk<slot_bit(C)>(f.T), act, act, TA & ~TB));
    const u32 hi = bitk<slot_bit(C)>(HT ? f.d2 ^ f.T : f.d2);
    const u32 v = row & act, neg = 0u - v;
    // second kind (v empty), in the top bit
    const u32 iso = TREE_B3(act, odd, v | neg, TA & ~TB & ~TC);
    f.z = TREE_B3(f.z, iso, hi, TA | (TB & TC));
    if (C == 0) return;
    const u32 o = TREE_B3(v, neg, odd, TA & TB & ~TC);  // the slot solved for, if any
    const u32 bm = nz1(o);
    f.nb -= bm;
    u32 oddi = f.d1 & o, d2i = f.d2 & o;
    nz2(oddi, d2i);
    const u32 e = odd | oddi;
    const u32 u = TREE_XA(d2i, hi, oddi);
    const u32 h = TREE_B3(odd, hi, u, (TA & ~TB) | (~TA & TC));
    u32 p[5];
    picked<index_bits(C)>(o, p);
    const u32 w = TREE_B3(pick<C>(f.lo, p), andk<below(C)>(bm), o, TA & TB & ~TC);
    const u32 vp = TREE_B3(v, o, o, TA & ~TB);
    const u32 ev = e & vp;
    const u32 al = TREE_B3(w, o, ev, TA ^ TB ^ TC);
    u32 wm = TREE_B3(w, o, oddi, TA | (TB & ~TC));
    const u32 oh = o & hi;
    f.q1 -= TREE_B3(hi, oddi, bm, TA & TB & TC);
    f.x2 = TREE_XA(f.x2, oh, f.d2);
    const u32 g = TREE_XA(h, e, f.d1);
    f.d2 = TREE_XA(f.d2, vp, g);
    f.d2 ^= TREE_B3(w, hi, vp, TA & (TB ^ TC));
    f.d2 = TREE_B3(f.d2, o, oh, (TA & ~TB) | TC);
    f.d1 = TREE_B3(f.d1, ev, o, (TA ^ TB) & ~TC);
    u32 tv = v;
    rows<C>(f.lo, tv, wm, al, v);
    f.A ^= o;
}

// Step of slot 32 + C.
template <int NH, bool HT, int C> TREE_DEV void step_hi(Form<NH> &f) {
    u32 act, odd;
    bitk2<slot_bit(C)>(f.Ah, f.d1h, act, odd);
    const u32 rowl = f.lo[32 + C], rowh = andk<below(C)>(f.hi[C]);
    if (HT) {
        const u32 at1 = TREE_B3(bitk<slot_bit(C)>(f.Th), act, act, TA & ~TB);
        f.d2 = TREE_XA(f.d2, rowl, at1);
        f.d2h = TREE_XA(f.d2h, rowh, at1);
    }
    const u32 hi = bitk<slot_bit(C)>(HT ? f.d2h ^ f.Th : f.d2h);
    const u32 vl = rowl & act, vh = rowh & act, negl = 0u - vl, negh = 0u - vh;
    const u32 nh = vh | negh;               // top bit: vh is not empty
    const u32 iso = TREE_B3(act, odd, TREE_B3(nh, vl, negl, TA | TB | TC), TA & ~TB & ~TC);
    f.z = TREE_B3(f.z, iso, hi, TA | (TB & TC));
    // Slots without a row in any lane have no more to do.  The chain of 64 steps
    // is all that a launch of few terms takes: exact t = 64, k = 0, 5 generators
    // 72 -> 48 us (one wave a term, rows in lanes: 50 to 58), 20 generators 77 ->
    // 64 (58 to 62), and 2^28 terms of t = 48 take what they took.  (Below slot
    // 32 the test gains 3 us more there and costs |H^t> calls 1%.)
    if (TREE_NONE(vl | vh)) return;
    // the slot solved for, among those from 32 on if there is one
    u32 nhm = nh;
    const u32 ol = TREE_B3(TREE_B3(vl, negl, odd, TA & TB & ~TC), pop_mask(nhm), odd, TA & ~TB);
    const u32 oh = TREE_B3(vh, negh, odd, TA & TB & ~TC);
    u32 bl = ol, bh = oh;
    nz2(bl, bh);
    f.nb -= bl;
    f.nb -= bh;
    u32 oddi = TREE_B3(f.d1 & ol, f.d1h, oh, TA | (TB & TC));
    u32 d2i = TREE_B3(f.d2 & ol, f.d2h, oh, TA | (TB & TC));
    nz2(oddi, d2i);
    const u32 e = odd | oddi;
    const u32 u = TREE_XA(d2i, hi, oddi);
    const u32 h = TREE_B3(odd, hi, u, (TA & ~TB) | (~TA & TC));
    // the row of that slot
    u32 pl[5];
    picked<5>(ol, pl);
    u32 wl = pick<32>(f.lo, pl) & bl, wh = 0;
    if (C > 0) {
        u32 ph[5];
        picked<index_bits(C)>(oh, ph);
        wl = TREE_B3(wl, pick<(C > 0 ? C : 1)>(f.lo + 32, ph), bh, TA | (TB & TC));
        // its slots from 32 on: of a row below 32, one bit of each of theirs
#pragma unroll
        for (int x = C - 1; x >= 0; x--) wh = push_nz(wh, f.lo[32 + x] & ol);
        wh = TREE_B3(wh, pick<(C > 0 ? C : 1)>(f.hi, ph), bh, TA | (TB & TC));
    }
    wl = TREE_B3(wl, ol, ol, TA & ~TB);
    wh = TREE_B3(andk<below(C)>(wh), oh, oh, TA & ~TB);
    const u32 vpl = TREE_B3(vl, ol, ol, TA & ~TB), vph = TREE_B3(vh, oh, oh, TA & ~TB);
    const u32 evl = e & vpl, evh = e & vph;
    const u32 all = TREE_B3(wl, ol, evl, TA ^ TB ^ TC), alh = TREE_B3(wh, oh, evh, TA ^ TB ^ TC);
    u32 wml = TREE_B3(wl, ol, oddi, TA | (TB & ~TC)), wmh = TREE_B3(wh, oh, oddi, TA | (TB & ~TC));
    const u32 ohl = ol & hi, ohh = oh & hi;
    f.q1 -= TREE_B3(hi, oddi, bl | bh, TA & TB & TC);
    f.x2 = TREE_XA(f.x2, ohl, f.d2);
    f.x2 = TREE_XA(f.x2, ohh, f.d2h);
    const u32 gl = TREE_XA(h, e, f.d1), gh = TREE_XA(h, e, f.d1h);
    f.d2 = TREE_XA(f.d2, vpl, gl);
    f.d2 ^= TREE_B3(wl, hi, vpl, TA & (TB ^ TC));
    f.d2 = TREE_B3(f.d2, ol, ohl, (TA & ~TB) | TC);
    f.d2h = TREE_XA(f.d2h, vph, gh);
    f.d2h ^= TREE_B3(wh, hi, vph, TA & (TB ^ TC));
    f.d2h = TREE_B3(f.d2h, oh, ohh, (TA & ~TB) | TC);
    f.d1 = TREE_B3(f.d1, evl, ol, (TA ^ TB) & ~TC);
    f.d1h = TREE_B3(f.d1h, evh, oh, (TA ^ TB) & ~TC);
    u32 tv = vl;
    rows<32>(f.lo, tv, wml, all, vl);
    tv = vh;
#pragma unroll
    for (int x = 0; x < C; x++) row2(f.lo[32 + x], f.hi[x], tv, wmh, all, vl, alh, vh);
    f.A ^= ol;
    f.Ah ^= oh;
}

// Steps of the slots whose bits are set in `todo` (uniform; bit C for slot C),
// the highest first.  A stretch tests a bit a slot, in groups of 16, 8 and 4
// behind one test each: the |H^t> sweep takes two steps a stretch, and with
// two comparisons for each of the 32 slots its scalar instructions, one a
// cycle and CU, outlasted the vector ones.
template <int NH, bool HT, int C, int N> struct Steps {
    static TREE_DEV void run(Form<NH> &f, u32 todo) {
        if (N <= 2 || (todo & (((1u << N) - 1u) << C))) {
            Steps<NH, HT, C + N / 2, N / 2>::run(f, todo);
            Steps<NH, HT, C, N / 2>::run(f, todo);
        }
    }
};
template <int NH, bool HT, int C> struct Steps<NH, HT, C, 1> {
    static TREE_DEV void run(Form<NH> &f, u32 todo) {
        if (todo & (1u << C)) step<NH, HT, C>(f);
    }
};
// Steps of the slots c0 - 1 .. c1, 32 >= c0 > c1.
template <int NH, bool HT> TREE_DEV void steps(Form<NH> &f, int c0, int c1) {
    const u32 todo = (~0u >> (32 - c0)) & (~0u << c1);
    Steps<NH, HT, 16, 16>::run(f, todo);
    Steps<NH, HT, 0, 16>::run(f, todo);
}
// Steps of the slots c0 - 1 .. c1 that are 32 or more.
template <int NH, bool HT, int C> struct StepsHi {
    static TREE_DEV void run(Form<NH> &f, int c0, int c1 = 32) {
        if (c0 > 32 + C && c1 <= 32 + C) step_hi<NH, HT, C>(f);
        StepsHi<NH, HT, C - 1>::run(f, c0, c1);
    }
};
template <int NH, bool HT> struct StepsHi<NH, HT, -1> {
    static TREE_DEV void run(Form<NH> &, int, int = 32) {}
};

// Two terms that differ in every slot left (the lowest index bit moves just
// these slots): the slots one of them sums are those the other drops, and a
// dropped slot is at 0, so neither sees the other's part of J.  With J taken
// as block diagonal, the slots of A and the others, one pass over the slots
// gives both sums, each step being one of the term that sums its slot.  There
// is nothing after it, so a slot that is solved for just leaves (`lv` holds
// the slots still there, `gone` the ones that left); its D stays where the
// constraint adds it to the phase, and the d2 of a slot of the third kind is
// cleared, so that d2 without d1 means a sum that is 0.
template <int NH, int C> TREE_DEV void pair_step(Form<NH> &f, u32 &lv, u32 &gone) {
    u32 b[4];
    bitk4<slot_bit(C)>(lv, f.d1, f.d2, f.A, b);
    const u32 act = b[0], odd = b[1], hi = b[2];
    lv = andk<~slot_bit(C)>(lv);
    const u32 own = TREE_B3(lv, f.A, b[3], TA & ~(TB ^ TC));
    const u32 v = TREE_B3(f.lo[C], own, act, TA & TB & TC), neg = 0u - v;
    const u32 o = TREE_B3(v, neg, odd, TA & TB & ~TC);
    const u32 bm = nz1(o);
    u32 oddi = f.d1 & o, d2i = f.d2 & o;
    nz2(oddi, d2i);
    const u32 e = odd | oddi;
    const u32 u = TREE_XA(d2i, hi, oddi);
    const u32 h = TREE_B3(odd, hi, u, (TA & ~TB) | (~TA & TC));
    u32 p[5];
    picked<index_bits(C)>(o, p);
    const u32 w = pick<C>(f.lo, p) & TREE_B3(own, bm, o, TA & TB & ~TC);
    lv = TREE_B3(lv, o, o, TA & ~TB);
    gone |= o;
    const u32 vp = TREE_B3(v, o, o, TA & ~TB);
    const u32 ev = e & vp;
    const u32 al = w ^ ev;
    const u32 g = TREE_XA(h, e, f.d1);
    f.d2 = TREE_XA(f.d2, vp, g);
    f.d2 ^= TREE_B3(w, hi, vp, TA & (TB ^ TC));
    f.d2 = TREE_B3(f.d2, o, hi, TA & (~TB | TC));
    const u32 third = andk<slot_bit(C)>(bm);
    f.d2 = TREE_B3(f.d2, third, third, TA & ~TB);
    f.d1 ^= ev;
    f.d1 = TREE_B3(f.d1, o, hi, TA & (~TB | TC));
    u32 tv = vp, tw = w;
    rows<C>(f.lo, tv, tw, al, vp);
}
template <int NH, int C, int N> struct PairSteps {
    static TREE_DEV void run(Form<NH> &f, u32 todo, u32 &lv, u32 &gone) {
        if (N <= 2 || (todo & (((1u << N) - 1u) << C))) {
            PairSteps<NH, C + N / 2, N / 2>::run(f, todo, lv, gone);
            PairSteps<NH, C, N / 2>::run(f, todo, lv, gone);
        }
    }
};
template <int NH, int C> struct PairSteps<NH, C, 1> {
    static TREE_DEV void run(Form<NH> &f, u32 todo, u32 &lv, u32 &gone) {
        if (C > 0 && (todo & (1u << C))) pair_step<NH, (C > 0 ? C : 1)>(f, lv, gone);
    }
};
// The slots below c, 1 <= c <= 32, of both terms: phases and counts as in
// fold, without a sum where zero is not 0; [0] of the term that sums A.
struct PairSums {
    int ph[2], cnt[2];
    u32 zero[2];
};
template <int NH> TREE_DEV void pair_sums(Form<NH> &f, int c, PairSums &s) {
    const u32 todo = ~0u >> (32 - c), in = ~0u << (32 - c);
    u32 lv = in, gone = 0;
    PairSteps<NH, 16, 16>::run(f, todo, lv, gone);
    PairSteps<NH, 0, 16>::run(f, todo, lv, gone);
    const u32 odd = TREE_B3(in & f.d1, gone, gone, TA & ~TB);        // first kind
    const u32 two = in & TREE_B3(f.d1, f.d2, gone, TA & (TB | TC));  // 2 each
    const u32 four = in & TREE_B3(f.d2, f.d1, gone, TA & (TB | TC)); // 4 each
    const u32 none = TREE_B3(in & f.d2, f.d1, gone, TA & ~TB & ~TC); // sums that are 0
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const u32 m = in & (k ? ~f.A : f.A);
        const int na = TREE_POP(odd & m);
        s.cnt[k] = TREE_POP(m) - na - 2 * TREE_POP(gone & m);
        s.ph[k] = na + 2 * TREE_POP(two & m) + 4 * TREE_POP(four & m);
        s.zero[k] = none & m;
    }
}

// What finished slots give, those of `in` of a word's 32: phase in units of 1
// and the count of active slots less the steps of the first kind; the third
// kind's share (nb, q1, x2) is added at the end.
template <bool HT> TREE_DEV void fold(u32 d1, u32 d2, u32 A, u32 T, u32 in, int &ph, int &cnt) {
    const u32 a1 = A & d1 & in;
    const int na = TREE_POP(a1);
    cnt += TREE_POP(A & in) - na;
    ph += na - 2 * TREE_POP(a1 & (HT ? d2 ^ T : d2));
    if (HT) {
        const u32 t = T & ~A & in;
        ph += 2 * TREE_POP(t & d1) + 4 * TREE_POP(t & d2);
    }
}

// The last TREE_LEAF slots are looked up: the index of their form is the top
// bits of A, d1, d2 and J_10 (and T).
#define TREE_LEAF 2
template <bool HT> struct LeafBits {
    static constexpr int value = HT ? 9 : 7;
};
template <bool HT> TREE_DEV u32 leaf_index(u32 A, u32 T, u32 d1, u32 d2, u32 row1) {
    u32 i = A >> 30;
    i = TREE_SHIN(i, d1, 2);
    i = TREE_SHIN(i, d2, 2);
    i = TREE_SHIN(i, row1, 1);
    return HT ? TREE_SHIN(i, T, 2) : i;
}
template <bool HT> TREE_DEV void leaf_form(u32 i, Form<0> &f) {
    if (HT) {
        f.T = i << 30;
        i >>= 2;
    }
    f.lo[1] = i << 31;
    f.lo[0] = (i & 1u) << 30;
    f.d2 = (i >> 1) << 30;
    f.d1 = (i >> 3) << 30;
    f.A = (i >> 5) << 30;
}

}  // namespace tree
}  // namespace cse
