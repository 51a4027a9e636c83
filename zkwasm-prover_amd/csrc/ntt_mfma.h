// NTT passes of radix 2^6 .. 2^8 on the matrix cores.
//
// A pass of radix D = SA SB (SA, SB in {8, 16}) is, per column, a DFT of size
// SA over j2, a twiddle product, and a DFT of size SB over j1:
//   X[k1 + SA k2] = sum_j1 w_SB^(j1 k2) w_D^(j1 k1) sum_j2 w_SA^(j2 k1) x[j2 SB + j1].
// The small DFTs are contractions with a constant matrix that every column
// shares, so they go to v_mfma_i32_16x16x64_i8: an element is 32 bytes, the
// matrix entry for (k, i, byte b) is w^(k i) 2^(8 b) mod r in balanced bytes, and
// the sum over i and b of byte products gives the 32 byte columns of
// sum_i w^(k i) x_i already reduced to 14 bits over r: no carries, no
// Montgomery reduction, one small quotient per output.  VALU work is
// left for the twiddles (one product per element instead of four levels of
// half a product each) and for folding the columns.
//
//  - Bytes are signed in the matrix product.  Adding 0x80 to every byte (with
//    carries) and flipping the top bits turns a 256-bit two's-complement
//    number into balanced bytes of the same value, so no bias terms arise.
//  - One radix-2 step comes first: the even outputs are a DFT of half the size
//    of u_i = x_i + x_{i+S/2}, the odd ones the odd rows applied to v_i = x_i -
//    x_{i+S/2}.  It halves the matrix work for 20 instructions per element; a
//    second step would need values beyond 2^255.
//  - Fragments need no lane movement: lane (n, h) of a wave (n < 16, h < 4)
//    holds whole elements of DFT n, supplying 16 bytes of one per instruction
//    as column n's quarter h of K; the matrix rows are ordered so that the
//    accumulators of outputs (k_0 .. k_3) leave lane (n, h) with all 32
//    columns of output k_h.
//  - At S = 16 a lane's elements of one half are an even and an odd i: their
//    products are summed apart, and sum and difference of the folded pairs are
//    outputs k and k + 8.  At S = 8 two groups of DFTs share the matrix reads.
//    Both halve the LDS traffic of the matrix (one 16-byte read per lane and
//    instruction), which bounded the plain form.
//  - The exchange between the two DFTs stays inside the wave (its 256
//    elements are whole columns): through LDS, 16 bytes of each element at a
//    time, rows padded by one element.
//
// Bounds: matrix entries are at most r / 2 in size and bytes 2^7, so a column
// sum of 8 x 32 terms is at most 2^22 and a value 2^14 r; the fold returns
// values in (0, 1.001 r), the twiddle product (reduced twiddle, 2^261 >
// 169 r) 1.01 r, inter-pass twiddled input 1.2 r: u stays below 2.4 r < 2^255.
#pragma once
#include "ff29.h"
#include "zkcore.h"

namespace zk {

typedef int nv4i __attribute__((ext_vector_type(4)));

constexpr int kMfmaThreads = 1024;
constexpr int kMfmaTile = 256;    // elements of a wave's tile, 4 per lane
constexpr int kMfmaTwWords = 12;  // a 29-bit twiddle padded to 48 bytes (aligned 16-byte LDS reads)

// LDS of a workgroup: matrix bytes [16 exponents][byte half][32 columns][16]
// with exponent rows shifted by 64 bytes per mfma_matrix_at, twiddles w_D^e
// (times n^-1 in an iNTT's last pass), and the exchange
struct MfmaLds {
    static constexpr int kMat = 16 * 1024 + 512;
    static constexpr int twiddles(int deg) { return (1 << deg) * kMfmaTwWords * 4; }
    // SB rows x columns x (SA + 1) x 16 B
    static constexpr int exchange(int la, int lb) { return (kMfmaTile >> la) * ((1 << la) + 1) * 16; }
    static constexpr int bytes(int la, int lb) { return kMat + twiddles(la + lb) + kMfmaThreads / 64 * exchange(la, lb); }
};

// start of exponent e's rows: lanes of one LDS access read exponents that
// differ by an even number
__device__ __forceinline__ uint32_t mfma_matrix_at(uint32_t e) { return e * 1024 + (e >> 1) * 64; }

// r in signed 32-bit digits (r = sum rho_j 2^(32 j))
__device__ constexpr int32_t kRho[8] = {(int32_t)0xf0000001u, 0x43e1f594, 0x79b97091, 0x2833e848,
                                        (int32_t)0x8181585du, (int32_t)0xb85045b7u, (int32_t)0xe131a02au, 0x30644e73};

// byte columns of w 2^(8 b) for the matrix: w in Montgomery form, b < 32
__device__ __forceinline__ void mfma_matrix_entry(uint8_t *mat, uint32_t e, uint32_t b, const Fr &w) {
    // the product with the plain number 2^(8b + 5) (< r) less 2^261 is w 2^(8b) itself
    F29 f;
    const uint32_t bit = 8 * b + 5, limb = bit / 29;
#pragma clang loop unroll(full)
    for (uint32_t i = 0; i < 9; i++) f.l[i] = i == limb ? 1u << (bit - 29 * limb) : 0u;
    const Fr v = fr_mul_w29(w, f);
    // the representative in (-r/2, r/2): v - r when v > r/2, i.e. when 2v >= r
    Fr d;
    uint32_t br = 0;
#pragma clang loop unroll(full)
    for (int i = 0; i < 8; i++) {
        const uint32_t x = (v.v[i] << 1) | (i ? v.v[i - 1] >> 31 : 0u);
        (void)sub_bb(x, FrParams::M[i], br);
    }
    const uint32_t low = 0u - br;  // all ones: 2v < r
    br = 0;
#pragma clang loop unroll(full)
    for (int i = 0; i < 8; i++) d.v[i] = sub_bb(v.v[i], FrParams::M[i] & ~low, br);
    // balanced bytes: add 0x80..80 with carries, flip the top bits
    uint32_t c = 0;
    uint8_t *p = mat + mfma_matrix_at(e) + (b >> 4) * 512 + (b & 15);
#pragma clang loop unroll(full)
    for (int i = 0; i < 8; i++) {
        const uint32_t x = add_cc(d.v[i], 0x80808080u, c) ^ 0x80808080u;
#pragma clang loop unroll(full)
        for (int q = 0; q < 4; q++) p[(4 * i + q) * 16] = (uint8_t)(x >> (8 * q));
    }
}

// One output from its 32 byte columns, added in pairs (z_j = y_2j + 2^8
// y_2j+1, |y| <= 2^22): V = sum z_j 2^(16j) less q r, in (0, 1.001 r).  The
// quotient comes from the top two pairs: with T = z15 2^16 + z14 in units of
// 2^224, m = floor(floor(T / 2^15) 2^60 / (r / 2^224) / 2^32) is 2^13 V / r to
// within (-0.3, 1.6) (the pairs below add 0.2, the two floors 0.4 and 1, the
// constant 0.1), so q = floor((m - 2) / 2^13) never exceeds V / r.
__device__ __forceinline__ void mfma_fold(uint32_t out[8], const int32_t (&z)[16]) {
    const int32_t t15 = (int32_t)((uint32_t)z[15] << 1) + (z[14] >> 15);
    // 2^60 / 811880050.88 = 1420063842.4
    const int32_t nq = -((__mulhi(t15, 1420063842) - 2) >> 13);
    int32_t carry = 0;  // below 2^16 in size: fits beside an even pair
#pragma clang loop unroll(full)
    for (int j = 0; j < 8; j++) {
        int64_t acc = z[2 * j] + carry;
        acc += (int64_t)z[2 * j + 1] * 65536;
        acc += (int64_t)nq * kRho[j];
        out[j] = (uint32_t)acc;
        carry = (int32_t)(acc >> 32);
    }
}

// u = x + y and v = x - y as balanced bytes (x, y < 1.2 r and the like)
__device__ __forceinline__ void mfma_split(uint32_t u[8], uint32_t v[8]) {
    uint32_t x[8], c = 0;
#pragma clang loop unroll(full)
    for (int i = 0; i < 8; i++) x[i] = add_cc(u[i], 0x80808080u, c);
    uint32_t cu = 0, bv = 0;
#pragma clang loop unroll(full)
    for (int i = 0; i < 8; i++) {
        const uint32_t y = v[i];
        u[i] = add_cc(x[i], y, cu) ^ 0x80808080u;
        v[i] = sub_bb(x[i], y, bv) ^ 0x80808080u;
    }
}

// The DFTs of size S = 2^LS of the wave's 256 elements, in place: x[s] is slot
// s of lane (n, h), input mfma_in(s, h) and afterwards output mfma_out(s, h) of
// its DFT.  S = 16: one group of 16 DFTs; the odd and the even i are summed
// apart, their sum and difference are outputs k and k + 8.  S = 8: two groups
// that share the matrix reads.
template <int LS>
__device__ __forceinline__ void mfma_dft(uint32_t (&x)[4][8], const uint8_t *mat, uint32_t lane) {
    static_assert(LS == 3 || LS == 4, "sizes 8 and 16");
    const uint32_t row = lane & 15, kh = lane >> 4, hrow = row >> 2;
    mat += (row & 3) * 16;
    if constexpr (LS == 4) {
        mfma_split(x[0], x[2]);
        mfma_split(x[1], x[3]);
    } else {
        mfma_split(x[0], x[1]);
        mfma_split(x[2], x[3]);
    }
#pragma clang loop unroll(full)
    for (int part = 0; part < 2; part++) {
        // exponents of (k, i) in units of w_16 for this lane's rows (outputs
        // k = 2 hrow + part) and quarter of K (elements i)
        const uint32_t k = 2 * hrow + part;
        const uint8_t *m0 = mat + mfma_matrix_at((LS == 4 ? k * 2 * kh : 2 * k * kh) & 15);
        const uint8_t *m1 = LS == 4 ? mat + mfma_matrix_at((k * (2 * kh + 1)) & 15) : m0;
        uint32_t *s0 = x[LS == 4 ? 2 * part : part], *s1 = x[LS == 4 ? 2 * part + 1 : 2 + part];
        nv4i b0[2], b1[2];
#pragma clang loop unroll(full)
        for (int i = 0; i < 4; i++) {
            b0[0][i] = (int)s0[i], b0[1][i] = (int)s0[4 + i];
            b1[0][i] = (int)s1[i], b1[1][i] = (int)s1[4 + i];
        }
        int32_t z0[16], z1[16];
#pragma clang loop unroll(full)
        for (int t = 0; t < 8; t++) {
            nv4i y0 = {0, 0, 0, 0}, y1 = {0, 0, 0, 0};
#pragma clang loop unroll(full)
            for (int b = 0; b < 2; b++) {
                const nv4i a0 = *reinterpret_cast<const nv4i *>(m0 + b * 512 + t * 64);
                const nv4i a1 = LS == 4 ? *reinterpret_cast<const nv4i *>(m1 + b * 512 + t * 64) : a0;
                y0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, b0[b], y0, 0, 0, 0);
                y1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, b1[b], y1, 0, 0, 0);
            }
#pragma clang loop unroll(full)
            for (int j = 0; j < 2; j++) {
                const int32_t c0 = y0[2 * j] + (int32_t)((uint32_t)y0[2 * j + 1] << 8);
                const int32_t c1 = y1[2 * j] + (int32_t)((uint32_t)y1[2 * j + 1] << 8);
                z0[2 * t + j] = LS == 4 ? c0 + c1 : c0;
                z1[2 * t + j] = LS == 4 ? c0 - c1 : c1;
            }
        }
        mfma_fold(s0, z0);
        mfma_fold(s1, z1);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// slot s of a DFT of size 2^LS: DFT index within the tile, input i, output k
template <int LS>
__device__ __forceinline__ constexpr uint32_t mfma_dft_index(int s, uint32_t n) {
    return (uint32_t)(s >> (LS - 2)) * 16 + n;
}
template <int LS>
__device__ __forceinline__ constexpr uint32_t mfma_in(int s, uint32_t h) {
    return LS == 4 ? 8 * (uint32_t)(s >> 1) + 2 * h + (uint32_t)(s & 1) : 4 * (uint32_t)(s & 1) + h;
}
template <int LS>
__device__ __forceinline__ constexpr uint32_t mfma_out(int s, uint32_t h) {
    return LS == 4 ? 8 * (uint32_t)(s & 1) + 2 * h + (uint32_t)(s >> 1) : 2 * h + (uint32_t)(s & 1);
}

// v - r when that is not negative
__device__ __forceinline__ void fr_cond_sub(uint32_t v[8]) {
    Fr t;
#pragma clang loop unroll(full)
    for (int i = 0; i < 8; i++) t.v[i] = v[i];
    t = fe_reduce_once<FrParams>(t);
#pragma clang loop unroll(full)
    for (int i = 0; i < 8; i++) v[i] = t.v[i];
}

}  // namespace zk
