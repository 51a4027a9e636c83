// XYZZ points held by four lanes, one coordinate each, for the parts of an
// MSM that are chains of point additions with too few points to fill the
// device (merging the partial sums of a bucket, summing the buckets of a
// window).
//
// Why: one lane's XYZZ addition is about 3500 dependent-ish instructions
// (14 products), 6.7 us when a wave has a SIMD to itself, and a small MSM
// is a few dozen of them in a row.  Four of the products are independent at
// every stage, so a quad of lanes does the addition in four product steps:
//   1. U1, S1, U2, S2        lanes 0..3: own coordinate x the partner's
//   2. PP, RR, ZZ12, ZZZ12
//   3. Q, PPP, ZZ3, -
//   4. R (Q - X3), S1 PPP, -, ZZZ3
// with operands moved by DPP quad permutations (no LDS): about 1300
// instructions per addition, 2.7 times less latency at 1.5 times the lane
// work.  A lane holds 9 limbs instead of 36, so the kernels also keep eight
// waves per SIMD.  All four lanes of a quad must be active together.
#pragma once
#include "ff29.h"

namespace zk {

// lane q of a quad: coordinate q of (x, y, zz, zzz), each < 2p
struct Q29 {
    F29 c;
};

// every lane's value from lane CTRL[q] of its quad (DPP quad permutation)
template <int CTRL>
__device__ __forceinline__ F29 f29_quad(const F29 &a) {
    F29 r;
#pragma unroll
    for (int i = 0; i < 9; i++)
        r.l[i] = (uint32_t)__builtin_amdgcn_mov_dpp((int)a.l[i], CTRL, 0xF, 0xF, false);
    return r;
}
constexpr int kQuad0 = 0x00, kQuad1 = 0x55, kQuad3 = 0xFF;  // broadcast of lane 0, 1, 3
constexpr int kQuadXor2 = 0x4E;                             // lane ^ 2

template <int CTRL>
__device__ __forceinline__ bool flag_quad(bool f) {
    return __builtin_amdgcn_mov_dpp(f ? 1 : 0, CTRL, 0xF, 0xF, false) != 0;
}
__device__ __forceinline__ F29 f29_pick(bool c, const F29 &a, const F29 &b) {
    F29 r;
#pragma unroll
    for (int i = 0; i < 9; i++) r.l[i] = c ? a.l[i] : b.l[i];
    return r;
}

// p <- 2p (dbl-2008-s-1, a = 0) in three product steps
__device__ __forceinline__ void q29_dbl(Q29 &p, uint32_t q) {
    const bool l0 = q == 0, l1 = q == 1, l2 = q == 2;
    const F29 y = f29_quad<kQuad1>(p.c);
    const F29 U = f29_dbl(y);
    // lane 0: X^2; lane 1: V = U^2 (lanes 2, 3 unused)
    const F29 a1 = f29_pick(l0, p.c, U);
    const F29 r1 = f29_mul(a1, a1);
    const F29 V = f29_quad<kQuad1>(r1), X2 = f29_quad<kQuad0>(r1);
    const F29 M = f29_add(f29_dbl(X2), X2);
    // lane 0: S = X V; lane 1: W = U V; lane 2: ZZ3 = ZZ V; lane 3: M^2
    const F29 a2 = f29_pick(l1, U, f29_pick(q == 3, M, p.c));
    const F29 r2 = f29_mul(a2, f29_pick(q == 3, M, V));
    const F29 S = f29_quad<kQuad0>(r2), W = f29_quad<kQuad1>(r2), MM = f29_quad<kQuad3>(r2);
    const F29 X3 = f29_sub(MM, f29_dbl(S));
    // lane 0: M (S - X3); lane 1: W Y; lane 3: ZZZ3 = W ZZZ
    const F29 r3 = f29_mul(f29_pick(l0, M, W), f29_pick(l0, f29_sub(S, X3), p.c));
    const F29 Y3 = f29_sub(f29_quad<kQuad0>(r3), r3);
    p.c = f29_pick(l0, X3, f29_pick(l1, Y3, f29_pick(l2, r2, r3)));
}

// p += r (add-2008-s); the flags, the same in all four lanes, mark the
// identity.  q: lane & 3.
__device__ __forceinline__ void q29_add(Q29 &p, bool &pe, const Q29 &r, bool re, uint32_t q) {
    if (re) return;
    if (pe) {
        p = r;
        pe = false;
        return;
    }
    const bool l0 = q == 0, l1 = q == 1, lo = q < 2;
    // 1. X1 ZZ2, Y1 ZZZ2, ZZ1 X2, ZZZ1 Y2: U1, S1, U2, S2
    const F29 A = f29_mul(p.c, f29_quad<kQuadXor2>(r.c));
    // lanes 0, 1: P = U2 - U1, R = S2 - S1 (+ 2p, < 4p: only multiplied)
    const F29 D = f29_sub_nr<2>(f29_quad<kQuadXor2>(A), A);
    // 2. P^2, R^2, ZZ1 ZZ2, ZZZ1 ZZZ2; a square is zero exactly when P, R is
    const F29 C = f29_mul(f29_pick(lo, D, p.c), f29_pick(lo, D, r.c));
    const bool zero = f29_is_zero(C);
    if (flag_quad<kQuad0>(zero)) {
        if (flag_quad<kQuad1>(zero))
            q29_dbl(p, q);  // the same point twice
        else
            pe = true;
        return;
    }
    // 3. Q = U1 PP, PPP = P PP, ZZ3 = ZZ12 PP, PPP again
    const F29 E = f29_mul(f29_pick(l0, A, f29_pick(q == 2, C, f29_quad<kQuad0>(D))), f29_quad<kQuad0>(C));
    // lane 0: X3 = RR - PPP - 2Q + 6p (< 8p)
    const F29 X3 = f29_sub_sub2_nr(f29_quad<kQuad1>(C), f29_quad<kQuad1>(E), E);
    // 4. R (Q - X3 + 8p), S1 PPP, -, ZZZ12 PPP (operands < 4p, < 10p)
    const F29 H = f29_mul(f29_pick(l0, f29_quad<kQuad1>(D), f29_pick(l1, A, C)),
                          f29_pick(l0, f29_sub_nr<8>(E, X3), E));
    // lane 1: Y3 = R (Q - X3) - S1 PPP + 2p (< 4p)
    const F29 Y3 = f29_sub_nr<2>(f29_quad<kQuad0>(H), H);
    const F29 xy = f29_reduce8(f29_pick(l0, X3, Y3));
    p.c = f29_pick(lo, xy, f29_pick(q == 2, E, H));
}

// lane q's nine limbs of a stored point (X29S: 36 words, zz = 0 marks the
// identity); a quad reads or writes 144 consecutive bytes
__device__ __forceinline__ Q29 q29_load(const X29S *s, bool &empty, uint32_t q) {
    const uint32_t *w = reinterpret_cast<const uint32_t *>(s) + 9 * q;
    Q29 p;
    uint32_t z = 0;
#pragma unroll
    for (int i = 0; i < 9; i++) {
        p.c.l[i] = w[i];
        z |= w[i];
    }
    empty = __builtin_amdgcn_mov_dpp((int)z, 0xAA, 0xF, 0xF, false) == 0;  // lane 2: zz
    return p;
}
__device__ __forceinline__ void q29_store(X29S *d, const Q29 &p, bool empty, uint32_t q) {
    uint32_t *w = reinterpret_cast<uint32_t *>(d) + 9 * q;
#pragma unroll
    for (int i = 0; i < 9; i++) w[i] = empty ? 0u : p.c.l[i];
}
// the point of the quad 2^B lanes away (B >= 2: another quad)
__device__ __forceinline__ Q29 q29_shfl_xor(const Q29 &p, bool pe, bool &oe, int m) {
    Q29 o;
#pragma unroll
    for (int i = 0; i < 9; i++) o.c.l[i] = (uint32_t)__shfl_xor((int)p.c.l[i], m);
    oe = __shfl_xor((int)pe, m) != 0;
    return o;
}

}  // namespace zk
