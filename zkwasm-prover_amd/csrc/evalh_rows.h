// Row arithmetic of the eval_h folds in lazy 29-bit limbs (kernels in
// evalh.hip).  With 32-bit products the folds were bound by VALU issue; here
// a fold t y + a b is one f29_mul2, two products under one reduction, and
// nothing is reduced below r before the store.  2^22 rows: logup fold 358 ->
// 291 us, shuffle 360 -> 267, first permutation fold 209 -> 169 (273, 210 and
// 157 us of traffic), permutation product of four columns 723 -> 660 (18
// products a row, still VALU-bound).  The term list of k_batch_mul_sum stays
// in 32-bit products: it is bound by its loads (384 us, 400 with these).
//
// An operand of a product enters as it is (lo) or times 2^5 (hi): lo x hi
// stays in the stored 2^256 domain, hi x hi in the 2^261 domain.  Stored
// values are below r.  A product of operands below a r and b r is below (1 + a
// b / 169.3) r and a mul2 below (1 + (a b + c d) / 169.3) r (2^261 = 169.3 r).
// What a row stores must be below 2 r, which f29_to_fr brings below r; the
// bounds, in units of r, stand at each function.  One operand of a product
// may have limbs up to 2^30.6 (sums without carries).
//
// The functions also compile for the host.
#pragma once
#include "ff29.h"

namespace zk {

__device__ __forceinline__ F29 lo(const Fr &x) { return f29_repack(x.v); }
__device__ __forceinline__ F29 hi(const Fr &x) { return f29_from32(x); }
__device__ __forceinline__ F29 mul(const F29 &a, const F29 &b) { return f29_mul<Fr29Mod>(a, b); }
__device__ __forceinline__ F29 mul2(const F29 &a, const F29 &b, const F29 &c, const F29 &d) {
    return f29_mul2<Fr29Mod>(a, b, c, d);
}
__device__ __forceinline__ F29 add_nc(const F29 &a, const F29 &b) {
    F29 r;
#pragma unroll
    for (int i = 0; i < 9; i++) r.l[i] = a.l[i] + b.l[i];
    return r;
}
// 2 r, every limb but the top raised by 2^29 that is taken from the next: no
// limb of a difference is negative
constexpr uint32_t kR2x29[9] = {0x20000002u, 0x3e1f593eu, 0x3cb848a0u, 0x2fa121e5u, 0x2b0ba505u,
                                0x25b68180u, 0x214dc281u, 0x3cb84c67u, 0x0060c89bu};
__device__ __forceinline__ F29 sub_nc(const F29 &a, const F29 &b) {  // a + 2 r - b, b < 1.9 r
    F29 r;
#pragma unroll
    for (int i = 0; i < 9; i++) r.l[i] = a.l[i] + kR2x29[i] - b.l[i];
    return r;
}
// a + r - b (< 2 r) and r - b
__device__ __forceinline__ Fr sub_lazy(const Fr &a, const Fr &b) {
    Fr t;
    uint32_t c = 0, br = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) t.v[i] = add_cc(a.v[i], FrParams::M[i], c);
#pragma unroll
    for (int i = 0; i < 8; i++) t.v[i] = sub_bb(t.v[i], b.v[i], br);
    return t;
}
__device__ __forceinline__ Fr neg_lazy(const Fr &b) {
    Fr t;
    uint32_t br = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) t.v[i] = sub_bb(FrParams::M[i], b.v[i], br);
    return t;
}

// In all of these y is hi(the challenge).  Rows of many operands take the columns
// and the row's index i (rn: the rotated row) and load each operand where it is
// used: loaded first, they cost a wave per SIMD and the folds of 2^22 rows 4 %.
__device__ __forceinline__ Fr ld(const Fr *p) { return fe_load<FrParams>(p); }

// permutation: (res y + (1 - first) l0) y + (last^2 - last) l_last
__device__ __forceinline__ Fr perm_p1_row(const Fr *res, const Fr *__restrict__ first, const Fr *__restrict__ last,
                                          const Fr *__restrict__ l0, const Fr *__restrict__ l_last, uint32_t i,
                                          const Fr &one, const F29 &y) {
    F29 t = mul2(lo(ld(&res[i])), y, lo(sub_lazy(one, ld(&first[i]))), hi(ld(&l0[i])));  // 1 + (32 + 64) / 169.3 = 1.57
    const Fr ls = ld(&last[i]);
    // the second factor: 1 + 64 / 169.3 = 1.38; the sum: 1 + (50.2 + 44.1) / 169.3 = 1.56
    t = mul2(t, y, mul(lo(ls), hi(sub_lazy(ls, one))), hi(ld(&l_last[i])));
    return f29_to_fr(t);
}

// t y + (z_j - z_prev) l, l = hi(l0): below 1.70 for t below 1.70
// (1 + (54.4 + 64) / 169.3)
__device__ __forceinline__ F29 perm_p2_step(const F29 &t, const Fr &zj, const Fr &zprev, const F29 &l, const F29 &y) {
    return mul2(t, y, lo(sub_lazy(zj, zprev)), l);
}

// logup: ((res y + l0 z) y + l_last zl) y + l_active (ip ((zn - z) table + m) - table ips)
__device__ __forceinline__ Fr logup_row(const Fr *res, const Fr *__restrict__ ip, const Fr *__restrict__ ips,
                                        const Fr *__restrict__ table, const Fr *__restrict__ m,
                                        const Fr *__restrict__ zf, const Fr *__restrict__ zl,
                                        const Fr *__restrict__ l0, const Fr *__restrict__ l_last,
                                        const Fr *__restrict__ l_active, uint32_t i, uint32_t rn, const F29 &y) {
    const Fr z = ld(&zf[i]);
    F29 t = mul2(lo(ld(&res[i])), y, lo(ld(&l0[i])), hi(z));  // 1 + 64 / 169.3 = 1.38
    t = mul2(t, y, lo(ld(&l_last[i])), hi(ld(&zl[i])));       // 1 + (44.1 + 32) / 169.3 = 1.45
    const F29 tb = lo(ld(&table[i]));
    F29 u = add_nc(mul(lo(sub_lazy(ld(&zf[rn]), z)), f29_shl5(tb)), lo(ld(&m[i])));  // 1 + 64 / 169.3 + 1 = 2.38
    u = mul2(u, hi(ld(&ip[i])), tb, hi(neg_lazy(ld(&ips[i]))));                      // 1 + (76.1 + 32) / 169.3 = 1.64
    return f29_to_fr(mul2(t, y, u, hi(ld(&l_active[i]))));                           // 1 + (46.4 + 52.5) / 169.3 = 1.59
}

// res y + l_active ((zn - z) ip - ips)
__device__ __forceinline__ Fr logup_extra_row(const Fr *res, const Fr *__restrict__ ip, const Fr *__restrict__ ips,
                                              const Fr *__restrict__ zp, const Fr *__restrict__ l_active, uint32_t i,
                                              uint32_t rn, const F29 &y) {
    // 1 + 64 / 169.3 + 1 = 2.38
    const F29 u = add_nc(mul(lo(sub_lazy(ld(&zp[rn]), ld(&zp[i]))), hi(ld(&ip[i]))), lo(neg_lazy(ld(&ips[i]))));
    return f29_to_fr(mul2(u, hi(ld(&l_active[i])), lo(ld(&res[i])), y));  // 1 + (76.1 + 32) / 169.3 = 1.64
}

// acc (v + beta), beta = hi: below 1.61 for acc below 1.61 (1 + 64 * 1.61 / 169.3)
__device__ __forceinline__ F29 shuffle_factor(const F29 &acc, const Fr &v, const F29 &beta) {
    return mul(add_nc(hi(v), beta), acc);
}
// shared tail of the two shuffle kernels (cuda/bn254.cu:990-1013, :1049-1068):
// ((res y + l0 (1 - z)) y + l_last (z^2 - z)) y + l_active (rhs zn - lhs z)
__device__ __forceinline__ Fr shuffle_fold(const Fr &res, const F29 &lhs, const F29 &rhs, const Fr &z, const Fr &zn,
                                           const Fr &l0, const Fr &l_last, const Fr &l_active, const F29 &y) {
    const Fr one = fe_one<FrParams>();
    F29 t = mul2(lo(res), y, lo(l0), hi(sub_lazy(one, z)));           // 1 + (32 + 64) / 169.3 = 1.57
    t = mul2(t, y, mul(lo(z), hi(sub_lazy(z, one))), hi(l_last));     // 1 + (50.2 + 44.1) / 169.3 = 1.56
    const F29 u = mul2(rhs, hi(zn), lhs, hi(neg_lazy(z)));            // 1 + 2 * 1.61 * 32 / 169.3 = 1.61
    return f29_to_fr(mul2(t, y, u, hi(l_active)));                    // 1 + (49.9 + 51.5) / 169.3 = 1.60
}

// acc (v + gamma + b s), vg = hi(v + gamma), b and s hi: the factor, in the
// 2^261 domain, is below 32 + 1 + 1024 / 169.3 = 39.1, the product below 1.31
// for acc below 1.31
__device__ __forceinline__ F29 perm_set_factor(const F29 &acc, const F29 &vg, const F29 &b, const F29 &s) {
    return mul(add_nc(vg, mul(b, s)), acc);
}
// h y + l_active (l - r): 1 + (3.31 * 32 + 32) / 169.3 = 1.82
__device__ __forceinline__ Fr perm_set_fold(const Fr &h, const F29 &l, const F29 &r, const Fr &l_active, const F29 &y) {
    return f29_to_fr(mul2(sub_nc(l, r), hi(l_active), lo(h), y));
}

// gates: q (y^G (a b + c - d) + sum_g y^(G-1-g) (f_g a - e_g)), a = hi; the sum
// is below 1 + 32 / 169.3 + 2 = 3.19 after the first step and stays so (1 +
// (102.1 + 32) / 169.3 + 1 = 2.80), the product with q below 1.61
__device__ __forceinline__ F29 gate_first(const F29 &a, const Fr &b, const Fr &c, const Fr &d) {
    return add_nc(mul(lo(b), a), lo(sub_lazy(c, d)));
}
__device__ __forceinline__ F29 gate_step(const F29 &acc, const F29 &a, const Fr &f, const Fr &e, const F29 &y) {
    return add_nc(mul2(acc, y, lo(f), a), lo(neg_lazy(e)));
}
__device__ __forceinline__ Fr gate_last(const F29 &acc, const Fr &q) { return f29_to_fr(mul(acc, hi(q))); }

}  // namespace zk
