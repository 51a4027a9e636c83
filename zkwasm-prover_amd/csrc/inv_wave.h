// One modular inversion by a whole wave: the optimized binary GCD of
// inv_bingcd.h (T. Pornin, 2020; same invariant, same kBits and final
// constant) laid out for the latency of a single chain, since a batch
// inversion waits for one inversion per tile.
//
//  - The inner steps work on two 64-bit approximations and 2 x 2 factors, the
//    same for every lane, so they run on the scalar unit: 64-bit shifts,
//    subtractions with borrow and count-trailing-zeros are one or two
//    instructions there (4.9 cycles each, as VALU ones, but no carry-mask
//    waits and real branches), and runs of zero bits are shifted out at once.
//    A factor pair (f, g) is one 64-bit f + g 2^32.
//  - The full-length updates run on the vector unit with even lanes taking the
//    first row (a, u) and odd lanes the second (b, v), exchanged by DPP.  The
//    factors of a row have opposite signs, so a f + b g is plus or minus
//    a |f| - b |g|, formed from unsigned products alone (-b |g| = ~b |g| + |g| -
//    2^256 |g|), and its absolute value is what is kept.
//  - Random inputs reach a = 0 after 12 or 13 of the 18 steps; the factors
//    2^-2 of v that the others would bring come from a short loop.
// Measured for the inversion alone: 57 us with one lane per inversion, 21 us.
// The functions also compile for the host, where the two rows are computed
// one after the other.
#pragma once
#include "inv_bingcd.h"

namespace zkinv {

// kBits steps on the approximations (ab, bb), bb odd: factors of the two rows
ZK_HD void gcd_inner(uint64_t ab, uint64_t bb, uint32_t fg0[2], uint32_t fg1[2]) {
#if defined(__HIP_DEVICE_COMPILE__)
    // every operand is wave-uniform; the loop ends after kBits shifts in all
    // (each round shifts at least one bit: the difference of two odd numbers
    // is even, and a zero ab shifts out all the bits left)
    asm volatile(
        "s_mov_b32 s84, %4\n s_mov_b32 s85, %5\n s_mov_b32 s86, %6\n s_mov_b32 s87, %7\n"
        "s_mov_b64 s[88:89], 1\n s_mov_b32 s90, 0\n s_mov_b32 s91, 1\n s_mov_b32 s95, %8\n"
        "1:\n"
        "s_ff1_i32_b64 s94, s[84:85]\n"  // -1 for zero
        "s_min_u32 s94, s94, s95\n"
        "s_lshr_b64 s[84:85], s[84:85], s94\n"
        "s_lshl_b64 s[90:91], s[90:91], s94\n"
        "s_sub_u32 s95, s95, s94\n"
        "s_cmp_eq_u32 s95, 0\n"
        "s_cbranch_scc1 3f\n"
        "s_sub_u32 s92, s84, s86\n s_subb_u32 s93, s85, s87\n"
        "s_cbranch_scc1 2f\n"
        "s_mov_b64 s[84:85], s[92:93]\n"
        "s_sub_u32 s88, s88, s90\n s_subb_u32 s89, s89, s91\n"
        "s_branch 1b\n"
        "2:\n"
        "s_sub_u32 s92, s86, s84\n s_subb_u32 s93, s87, s85\n"
        "s_mov_b64 s[86:87], s[84:85]\n s_mov_b64 s[84:85], s[92:93]\n"
        "s_sub_u32 s92, s90, s88\n s_subb_u32 s93, s91, s89\n"
        "s_mov_b64 s[90:91], s[88:89]\n s_mov_b64 s[88:89], s[92:93]\n"
        "s_branch 1b\n"
        "3:\n"
        "s_mov_b32 %0, s88\n s_mov_b32 %1, s89\n s_mov_b32 %2, s90\n s_mov_b32 %3, s91\n"
        : "=&s"(fg0[0]), "=&s"(fg0[1]), "=&s"(fg1[0]), "=&s"(fg1[1])
        : "s"((uint32_t)ab), "s"((uint32_t)(ab >> 32)), "s"((uint32_t)bb), "s"((uint32_t)(bb >> 32)), "n"(kBits)
        : "s84", "s85", "s86", "s87", "s88", "s89", "s90", "s91", "s92", "s93", "s94", "s95", "scc");
#else
    uint64_t p0 = 1, p1 = 1ull << 32;
    for (uint32_t rem = kBits;;) {
        uint32_t k = ab ? (uint32_t)__builtin_ctzll(ab) : rem;
        if (k > rem) k = rem;
        ab >>= k;
        p1 <<= k;
        rem -= k;
        if (!rem) break;
        if (ab < bb) {
            const uint64_t t = ab, tp = p0;
            ab = bb - ab;
            bb = t;
            p0 = p1 - p0;
            p1 = tp;
        } else {
            ab -= bb;
            p0 -= p1;
        }
    }
    fg0[0] = (uint32_t)p0;
    fg0[1] = (uint32_t)(p0 >> 32);
    fg1[0] = (uint32_t)p1;
    fg1[1] = (uint32_t)(p1 >> 32);
#endif
}

// |f| and |g| of a packed pair f + g 2^32 (both at most 2^30 in size)
ZK_HD void unpack_abs(const uint32_t fg[2], uint32_t &f, uint32_t &g) {
    const int32_t lo = (int32_t)fg[0], hi = (int32_t)(fg[1] + (uint32_t)(lo < 0));
    f = (uint32_t)(lo < 0 ? -lo : lo);
    g = (uint32_t)(hi < 0 ? -hi : hi);
}

// words of x f - y g, returning the signed word above them
ZK_HD int64_t diff_row(uint32_t r[8], const uint32_t x[8], const uint32_t y[8], uint32_t f, uint32_t g) {
    uint64_t acc = g;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        acc += (uint64_t)x[i] * f;  // f, g <= 2^30: the sum stays below 2^64
        acc += (uint64_t)(~y[i]) * g;
        r[i] = (uint32_t)acc;
        acc >>= 32;
    }
    return (int64_t)acc - (int64_t)(uint64_t)g;
}

// a row of the update: na = |a f - b g| >> kBits (exact), nu = (u f - v g)
// 2^-32 mod M with the sign that made na positive; M below 2^254, minv =
// -M^-1 mod 2^32
ZK_HD void gcd_row(uint32_t na[8], uint32_t nu[8], const uint32_t a[8], const uint32_t b[8], const uint32_t u[8],
                   const uint32_t v[8], uint32_t f, uint32_t g, const uint32_t M[8], uint32_t minv) {
    uint32_t r[9];
    const int64_t top = diff_row(r, a, b, f, g);
    r[8] = (uint32_t)top;
    const uint32_t neg = (uint32_t)(top >> 63);  // all ones or zero
    uint32_t c = neg & 1u;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint64_t t = (uint64_t)(((r[i] >> kBits) | (r[i + 1] << (32 - kBits))) ^ neg) + c;
        na[i] = (uint32_t)t;
        c = (uint32_t)(t >> 32);
    }
    uint32_t s[8];
    const int64_t utop = diff_row(r, u, v, f, g);
    // t' = (t + q M) 2^-32 with |t| <= 2^30 M and q < 2^32: in (-M/4, 5M/4)
    const uint32_t q = r[0] * minv;
    uint64_t cc = ((uint64_t)q * M[0] + r[0]) >> 32;
#pragma unroll
    for (int i = 1; i < 8; i++) {
        cc += (uint64_t)q * M[i] + r[i];  // below 2^64: (2^32-1)^2 + 2 (2^32-1)
        s[i - 1] = (uint32_t)cc;
        cc >>= 32;
    }
    const int64_t t7 = (int64_t)cc + utop;
    s[7] = (uint32_t)t7;
    // into [0, M): + M if negative, then - M unless that borrows
    const uint32_t low = (uint32_t)(t7 >> 63);
    uint32_t d[8], ca = 0, br = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint64_t t = (uint64_t)s[i] + (M[i] & low) + ca;
        s[i] = (uint32_t)t;
        ca = (uint32_t)(t >> 32);
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint64_t t = (uint64_t)s[i] - M[i] - br;
        d[i] = (uint32_t)t;
        br = (uint32_t)(t >> 63);
    }
    // s or d, or M minus it where the row was negated
    const uint32_t keep = 0u - br;
    uint32_t bo = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t w = (s[i] & keep) | (d[i] & ~keep);
        const uint64_t t = (uint64_t)(M[i] & neg) - bo - (w ^ (w & ~neg));
        bo = (uint32_t)(t >> 63);
        nu[i] = (w & ~neg) | ((uint32_t)t & neg);
    }
}

// y^-1 = v 2^((32 - kBits) kSteps) mod M for 0 < y < M, y and v the same in
// all lanes of the (fully active) wave; false when b did not end at 1
ZK_HD bool bingcd_wave(uint32_t v_out[8], const uint32_t y[8], const uint32_t M[8], uint32_t minv) {
    uint32_t a[8], b[8], u[8], v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        a[i] = y[i];
        b[i] = M[i];
        u[i] = i == 0;
        v[i] = 0;
    }
    int step = 0;
    for (; step < kSteps; step++) {
        // the two words of a and b from the top one of the longer
        uint32_t ha = a[1], la = a[0], hb = b[1], lb = b[0], nz = 0, any = a[0] | a[1];
#pragma unroll
        for (int i = 2; i < 8; i++) {
            const bool c = (a[i] | b[i]) != 0;
            ha = c ? a[i] : ha;
            la = c ? a[i - 1] : la;
            hb = c ? b[i] : hb;
            lb = c ? b[i - 1] : lb;
            nz |= a[i] | b[i];
            any |= a[i];
        }
        uint32_t a0 = a[0], b0 = b[0];
#if defined(__HIP_DEVICE_COMPILE__)
        any = __builtin_amdgcn_readfirstlane(any);
        nz = __builtin_amdgcn_readfirstlane(nz);
        ha = __builtin_amdgcn_readfirstlane(ha);
        la = __builtin_amdgcn_readfirstlane(la);
        hb = __builtin_amdgcn_readfirstlane(hb);
        lb = __builtin_amdgcn_readfirstlane(lb);
        a0 = __builtin_amdgcn_readfirstlane(a0);
        b0 = __builtin_amdgcn_readfirstlane(b0);
#endif
        if (!any) break;  // b is the gcd
        // low kBits bits exact, 33 bits from the longer one's top (at least
        // kBits + 2 are needed); values below 2^64 are exact
        uint64_t ab = ((uint64_t)ha << 32) | la, bb = ((uint64_t)hb << 32) | lb;
        if (nz) {
            const int z = __builtin_clz(ha | hb);
            const uint32_t low = (1u << kBits) - 1;
            ab = ((ab << z) >> 31 << kBits) | (a0 & low);
            bb = ((bb << z) >> 31 << kBits) | (b0 & low);
        }
        uint32_t p0[2], p1[2], f, g;
        gcd_inner(ab, bb, p0, p1);
        uint32_t na[8], nu[8];
#if defined(__HIP_DEVICE_COMPILE__)
        const bool odd = threadIdx.x & 1;
        const uint32_t pl[2] = {odd ? p1[0] : p0[0], odd ? p1[1] : p0[1]};
        unpack_abs(pl, f, g);
        gcd_row(na, nu, a, b, u, v, f, g, M, minv);
#pragma unroll
        for (int i = 0; i < 8; i++) {  // even lanes' rows, odd lanes' rows
            a[i] = (uint32_t)__builtin_amdgcn_mov_dpp((int)na[i], 0xA0, 0xF, 0xF, false);
            b[i] = (uint32_t)__builtin_amdgcn_mov_dpp((int)na[i], 0xF5, 0xF, 0xF, false);
            u[i] = (uint32_t)__builtin_amdgcn_mov_dpp((int)nu[i], 0xA0, 0xF, 0xF, false);
            v[i] = (uint32_t)__builtin_amdgcn_mov_dpp((int)nu[i], 0xF5, 0xF, 0xF, false);
        }
#else
        uint32_t nb[8], nv[8];
        unpack_abs(p0, f, g);
        gcd_row(na, nu, a, b, u, v, f, g, M, minv);
        unpack_abs(p1, f, g);
        gcd_row(nb, nv, a, b, u, v, f, g, M, minv);
        for (int i = 0; i < 8; i++) {
            a[i] = na[i];
            b[i] = nb[i];
            u[i] = nu[i];
            v[i] = nv[i];
        }
#endif
    }
    // the steps left out: v <- v 2^(kBits - 32) each
    for (; step < kSteps; step++) {
        uint32_t na[8], nu[8];
        gcd_row(na, nu, b, a, v, u, 1u << kBits, 0, M, minv);
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = nu[i];
    }
    uint32_t one = b[0] ^ 1u;
#pragma unroll
    for (int i = 1; i < 8; i++) one |= b[i];
#pragma unroll
    for (int i = 0; i < 8; i++) v_out[i] = v[i];
    return one == 0;
}

}  // namespace zkinv
