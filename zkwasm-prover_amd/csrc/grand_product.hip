// Permutation and shuffle grand products on the device.
//
// The reference computes these on host cores (src/permutation.rs:16-150,
// src/shuffle.rs:16-215) while the GPU runs the logup work.  Here
//   z[i] = prod_{j < i} num_j / den_j = N_i S_i / D,
// N_i the product of the numerators before row i, S_i that of the denominators
// from row i on and D = S_0: one inversion in all instead of one per row
// (batched: three products per row and the inversions' latency), in three
// launches:
//   1. tiles    num_i and den_i of 1024 rows from the columns, their in-tile
//               inclusive prefix products (num, into z) and suffix products
//               (den, into temp);
//   2. top      one workgroup: the tiles' factors K_b = (numerators before the
//               tile) (denominators after it) / D, into z at the tile's last
//               row, whose prefix product no row of the tile needs;
//   3. combine  z[i] = prefix[i - 1] suffix[i] K_b.
// The numerators and the denominators of a tile go to workgroups of their own:
// the pass is bound by the chain of products of a wave, and twice the waves
// with half of it each overlap better (300007 rows, four columns: 155 -> 107 us).
// A zero denominator counts as 1 and z is 0 after its row, which is what
// inverting it to zero (halo2's BatchInvert) gives; the free top bits of the
// suffix products mark such rows and their tiles.  The
// reference splits the product into chunks with carried tails; field
// multiplication is exact, so every z[i] equals the sequential quotient bit
// for bit.  Rows after the last usable row are filled with blinding values by
// the caller, as fill_random does in the reference.
// Three sets of four columns over 300007 rows: 1147 -> 524 us.
#include "ff29.h"
#include "inv_dev.h"
#include "zkcore.h"

using namespace zk;

namespace {

constexpr uint32_t kThreads = 256;
constexpr uint32_t kRows = 4;  // consecutive rows per thread in the tile and combine passes
constexpr uint32_t kTile = kThreads * kRows;

// Products are 29-bit ones (ff29.h): shorter dependent chains than the 32-bit
// product's, which is what these passes wait for.  Running products stay in
// the 2^256 Montgomery domain and below 2r unless noted; one operand of each
// product is moved to the 2^261 domain.
__device__ __forceinline__ F29 mul_run(const F29 &a, const F29 &b) { return f29_mul<Fr29Mod>(a, f29_shl5(b)); }
__device__ __forceinline__ F29 f29_one_mont() { return f29_repack(FrParams::ONE); }

// v from `d` lanes below (up) or above (down) in the wave
template <bool UP>
__device__ __forceinline__ F29 f29_shfl(const F29 &v, int d) {
    F29 o;
#pragma clang loop unroll(full)
    for (int i = 0; i < 9; i++)
        o.l[i] = (uint32_t)(UP ? __shfl_up((int)v.l[i], d, 64) : __shfl_down((int)v.l[i], d, 64));
    return o;
}

// Products over the 256 threads of a workgroup: UP, of the earlier threads'
// values, else of the later ones' (exclusive).  Inside a wave by shuffles, the
// four wave products through sh[4].
template <bool UP>
__device__ __forceinline__ F29 block_scan_mul(F29 p, F29 *sh) {
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const uint32_t ahead = UP ? lane : 63 - lane;  // lanes on the side the product comes from
#pragma unroll 1
    for (int d = 1; d < 64; d <<= 1) {
        const F29 a = f29_shfl<UP>(p, d);
        if (ahead >= (uint32_t)d) p = mul_run(p, a);
    }
    if (ahead == 63) sh[wv] = p;
    __syncthreads();
    F29 other = f29_one_mont();
#pragma unroll 1
    for (uint32_t w = 0; w < 4; w++)
        if (UP ? w < wv : w > wv) other = mul_run(other, sh[w]);
    p = f29_shfl<UP>(p, 1);
    __syncthreads();
    return ahead ? mul_run(other, p) : other;
}

constexpr uint32_t kRowZero = 1u << 30, kTileZero = 1u << 31;  // marks in a suffix product's top word

// Tile pass, last part: the thread's kRows consecutive rows from row i0 (rows
// past n: 1; below 2r) -> the tile's inclusive prefix products into z (UP) or
// suffix products into temp, with the marks of zero denominators.
template <bool UP>
__device__ __forceinline__ void store_tile(F29 (&v)[kRows], uint64_t i0, uint32_t n, Fr *__restrict__ out, F29 *sh,
                                           uint32_t *any) {
    uint32_t zero = 0;
    if (!UP) {
        if (threadIdx.x == 0) *any = 0;
        __syncthreads();
#pragma clang loop unroll(full)
        for (uint32_t k = 0; k < kRows; k++) {
            if (fe_is_zero<FrParams>(f29_to_fr(v[k]))) {
                v[k] = f29_one_mont();
                zero |= 1u << k;
                *any = 1;
            }
        }
    }
#pragma clang loop unroll(full)
    for (uint32_t k = 1; k < kRows; k++) {
        if (UP)
            v[k] = mul_run(v[k - 1], v[k]);
        else
            v[kRows - 1 - k] = mul_run(v[kRows - 1 - k], v[kRows - k]);
    }
    const F29 p = f29_shl5(block_scan_mul<UP>(UP ? v[kRows - 1] : v[0], sh));
#pragma clang loop unroll(full)
    for (uint32_t k = 0; k < kRows; k++) {
        if (i0 + k >= n) continue;
        Fr r = f29_to_fr(f29_mul<Fr29Mod>(v[k], p));
        if (!UP) {
            if ((zero >> k) & 1u) r.v[7] |= kRowZero;
            if (k == 0 && threadIdx.x == 0 && *any) r.v[7] |= kTileZero;
        }
        fe_store<FrParams>(&out[i0 + k], r);
    }
}

// the kRows rows of a column from i0 (rows past n read as row n - 1)
__device__ __forceinline__ void load_rows(Fr (&v)[kRows], const Fr *__restrict__ col, uint64_t i0, uint32_t n) {
#pragma clang loop unroll(full)
    for (uint32_t k = 0; k < kRows; k++) v[k] = fe_load<FrParams>(&col[i0 + k < n ? i0 + k : n - 1]);
}

// 32 a mod r: a constant whose 29-bit form (f29_from32) then carries 2^266, so
// that a product with it lands in the 2^261 domain
__device__ __forceinline__ Fr fr_times32(Fr a) {
#pragma unroll 1
    for (int k = 0; k < 5; k++) a = a + a;
    return a;
}
// a + b + c, limbs normalised (value below 2^261)
__device__ __forceinline__ F29 f29_add3(const F29 &a, const F29 &b, const F29 &c) {
    F29 r;
    uint32_t cy = 0;
#pragma clang loop unroll(full)
    for (int i = 0; i < 9; i++) {
        const uint32_t s = a.l[i] + b.l[i] + c.l[i] + cy;
        r.l[i] = s & kM29;
        cy = s >> 29;
    }
    return r;
}
// acc[k] *= m[k] c + v[k] + g with m below r (2^256 domain), c29 carrying
// 2^266, g29 below r in the 2^261 domain: the factor is below 2r + 32r + r and
// the product below (35 / 169) 1.3 r + r < 1.3 r for acc below 1.3 r (2^261 >
// 169 r).  The first factor is taken times 1.
__device__ __forceinline__ void fold_rows(F29 (&acc)[kRows], const F29 (&m)[kRows], const F29 &c29,
                                          const Fr (&v)[kRows], const F29 &g29) {
#pragma clang loop unroll(full)
    for (uint32_t k = 0; k < kRows; k++) {
        const F29 t = f29_add3(f29_mul<Fr29Mod>(m[k], c29), f29_from32(v[k]), g29);
        acc[k] = f29_mul<Fr29Mod>(acc[k], t);
    }
}

// grid (tiles, 2): y = 0, num = prod_j (v_j + beta delta_start delta^j omega^i
// + gamma) (src/permutation.rs:79-95); y = 1, den = prod_j (v_j + beta sigma_j
// + gamma) (:53-70).  The first wave squares omega up to the tile's bits and
// makes two 16-entry tables, omega^(64 a + tile's first row) and omega^(4 b), so
// that thread 16 a + b's first power is one product.
__global__ __launch_bounds__(kThreads, 3) void k_perm_tiles(Fr *__restrict__ z, Fr *__restrict__ temp,
                                                         const Fr *const *__restrict__ vals,
                                                         const Fr *const *__restrict__ sig, int ncols,
                                                         const Fr *__restrict__ beta, const Fr *__restrict__ gamma,
                                                         const Fr *__restrict__ delta_start,
                                                         const Fr *__restrict__ delta,
                                                         const Fr *__restrict__ omega, uint32_t n) {
    static_assert(kRows == 4 && kThreads == 256, "rows 4 (16 a + b) in the tile");
    __shared__ F29 sh[4], pw[10], tab[32];  // pw[k] = omega^(2^k), tab: the two tables
    __shared__ uint32_t any;
    const uint32_t t = threadIdx.x, tile0 = blockIdx.x * kTile;
    const uint64_t i0 = (uint64_t)tile0 + t * kRows;
    const F29 g = f29_repack(fr_times32(fe_load<FrParams>(gamma)).v);
    F29 acc[kRows], m[kRows];
    Fr v[kRows];
#pragma clang loop unroll(full)
    for (uint32_t k = 0; k < kRows; k++) acc[k] = f29_one_mont();
    if (blockIdx.y) {
        const F29 b = f29_from32(fr_times32(fe_load<FrParams>(beta)));
#pragma unroll 1
        for (int j = 0; j < ncols; j++) {
            load_rows(v, sig[j], i0, n);
#pragma clang loop unroll(full)
            for (uint32_t k = 0; k < kRows; k++) m[k] = f29_repack(v[k].v);
            load_rows(v, vals[j], i0, n);
            fold_rows(acc, m, b, v, g);
        }
#pragma clang loop unroll(full)
        for (uint32_t k = 0; k < kRows; k++)
            if (i0 + k >= n) acc[k] = f29_one_mont();
        store_tile<false>(acc, i0, n, temp, sh, &any);
        return;
    }
    if (t < 64) {
        F29 w = f29_repack(fe_load<FrParams>(omega).v), base = f29_one_mont();
#pragma unroll 1
        for (uint32_t k = 0; (1u << k) <= (tile0 | (kTile - 1)); k++) {
            if (k < 10 && t == 0) pw[k] = w;
            const F29 ws = f29_shl5(w);
            if ((tile0 >> k) & 1u) base = f29_mul<Fr29Mod>(base, ws);
            if (k == 31) break;
            w = f29_mul<Fr29Mod>(w, ws);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        __builtin_amdgcn_wave_barrier();
        // lanes 0..15: powers 4 b; 16..31: powers 64 a times the tile's
        F29 e = t & 16 ? base : f29_one_mont();
#pragma unroll 1
        for (uint32_t k = 0; k < 4; k++) {
            const F29 f = pw[k + (t & 16 ? 6 : 2)];
            if ((t >> k) & 1u) e = mul_run(e, f);
        }
        if (t < 32) tab[t] = e;
    }
    __syncthreads();
    // m[k] = omega^(i0 + k)
    const F29 w = f29_shl5(pw[0]), d = f29_from32(fe_load<FrParams>(delta));
    m[0] = mul_run(tab[t & 15], tab[16 + (t >> 4)]);
#pragma clang loop unroll(full)
    for (uint32_t k = 1; k < kRows; k++) m[k] = f29_mul<Fr29Mod>(m[k - 1], w);
    // 32 beta delta_start delta^j
    Fr bd = fr_times32(fe_load<FrParams>(beta)) * fe_load<FrParams>(delta_start);
#pragma unroll 1
    for (int j = 0; j < ncols; j++) {
        load_rows(v, vals[j], i0, n);
        fold_rows(acc, m, f29_from32(bd), v, g);
        bd = fr_mul_w29(bd, d);
    }
#pragma clang loop unroll(full)
    for (uint32_t k = 0; k < kRows; k++)
        if (i0 + k >= n) acc[k] = f29_one_mont();
    store_tile<true>(acc, i0, n, z, sh, &any);
}

// grid (tiles, 2): y = 0, num = prod_j (input_j + betas[j]) (src/shuffle.rs:
// 167-176); y = 1, den = prod_j (shuffle_j + betas[j]) (:148-161)
__global__ __launch_bounds__(kThreads, 4) void k_shuffle_tiles(Fr *__restrict__ z, Fr *__restrict__ temp,
                                                            const Fr *const *__restrict__ inputs,
                                                            const Fr *const *__restrict__ shuffles,
                                                            const Fr *__restrict__ betas, int group_len, uint32_t n) {
    __shared__ F29 sh[4];
    __shared__ uint32_t any;
    const uint64_t i0 = (uint64_t)blockIdx.x * kTile + threadIdx.x * kRows;
    const Fr *const *cols = blockIdx.y ? shuffles : inputs;
    F29 acc[kRows];
    Fr v[kRows];
#pragma clang loop unroll(full)
    for (uint32_t k = 0; k < kRows; k++) acc[k] = f29_one_mont();
#pragma unroll 1
    for (int j = 0; j < group_len; j++) {
        const Fr b = fe_load<FrParams>(&betas[j]);
        load_rows(v, cols[j], i0, n);
#pragma clang loop unroll(full)
        for (uint32_t k = 0; k < kRows; k++) acc[k] = f29_mul<Fr29Mod>(acc[k], f29_from32(v[k] + b));
    }
#pragma clang loop unroll(full)
    for (uint32_t k = 0; k < kRows; k++)
        if (i0 + k >= n) acc[k] = f29_one_mont();
    if (blockIdx.y)
        store_tile<false>(acc, i0, n, temp, sh, &any);
    else
        store_tile<true>(acc, i0, n, z, sh, &any);
}

__device__ __forceinline__ uint64_t tile_last(uint32_t b, uint32_t n) {
    const uint64_t e = ((uint64_t)b + 1) * kTile;
    return (e < n ? e : n) - 1;
}

// One workgroup: tile b's products are z[tile_last(b)] (num) and temp[b *
// kTile] (den); z[tile_last(b)] becomes K_b.  Thread t < 256 owns `per`
// consecutive tiles; a fifth wave inverts the denominators' product while the
// others scan.  Up to kKeep tiles per thread stay in registers (n <= 2^20), so
// that only the product with the inverse is left to do after it.  A tile with
// a zero denominator makes every later K_b zero.
constexpr uint32_t kTopThreads = kThreads + 64, kKeep = 4;
__global__ __launch_bounds__(kTopThreads) void k_product_top(Fr *__restrict__ z, const Fr *__restrict__ temp,
                                                             uint32_t n, uint32_t nb) {
    __shared__ F29 sp[4], sq[4], waves[4], inv;
    const uint32_t t = threadIdx.x, lane = t & 63, wv = t >> 6, per = (nb + kThreads - 1) / kThreads;
    const bool data = t < kThreads;
    const uint32_t b0 = !data || t * per > nb ? nb : t * per, b1 = b0 + per < nb ? b0 + per : nb;
    auto num_of = [&](uint32_t b) {
        const Fr v = fe_load<FrParams>(&z[tile_last(b, n)]);
        return f29_repack((temp[(uint64_t)b * kTile].v[7] & kTileZero ? fe_zero<FrParams>() : v).v);
    };
    auto den_of = [&](uint32_t b) {
        Fr v = fe_load<FrParams>(&temp[(uint64_t)b * kTile]);
        v.v[7] &= ~(kRowZero | kTileZero);
        return f29_repack(v.v);
    };
    const bool keep = per <= kKeep;
    F29 p = f29_one_mont(), q = p, nv[kKeep], dq[kKeep];
    if (keep) {
#pragma clang loop unroll(full)
        for (uint32_t k = 0; k < kKeep; k++) {
            nv[k] = dq[k] = f29_one_mont();
            if (b0 + k < b1) {
                nv[k] = num_of(b0 + k);
                dq[k] = den_of(b0 + k);
            }
        }
        p = nv[0];
        q = dq[0];
#pragma clang loop unroll(full)
        for (uint32_t k = 1; k < kKeep; k++) {
            if (k < per) {  // uniform
                p = mul_run(p, nv[k]);
                q = mul_run(q, dq[k]);
            }
        }
    } else {
#pragma unroll 1
        for (uint32_t b = b0; b < b1; b++) {
            p = mul_run(p, num_of(b));
            q = mul_run(q, den_of(b));
        }
    }
    if (data) {
        F29 all = q;
#pragma unroll 1
        for (int d = 1; d < 64; d <<= 1) {
            F29 o;
#pragma clang loop unroll(full)
            for (int i = 0; i < 9; i++) o.l[i] = (uint32_t)__shfl_xor((int)all.l[i], d);
            all = mul_run(all, o);
        }
        if (lane == 0) waves[wv] = all;
    }
    __syncthreads();
    if (!data) {
        const F29 all = mul_run(mul_run(waves[0], waves[1]), mul_run(waves[2], waves[3]));
        const Fr r = fr_inv_wave(f29_to_fr(all));
        if (lane == 0) inv = f29_from32(r);
        for (int k = 0; k < 4; k++) __syncthreads();  // block_scan_mul's, twice
    } else {
        p = block_scan_mul<true>(p, sp);
        q = block_scan_mul<false>(q, sq);
        if (keep) {
            // nv[k] <- the numerators before tile k times the denominators after it
#pragma clang loop unroll(full)
            for (uint32_t k = 0; k < kKeep; k++) {
                if (k < per) {
                    const F29 v = nv[k];
                    nv[k] = p;
                    p = mul_run(p, v);
                }
            }
#pragma clang loop unroll(full)
            for (int k = (int)kKeep - 1; k >= 0; k--) {
                if ((uint32_t)k < per) {
                    nv[k] = mul_run(nv[k], q);
                    q = mul_run(q, dq[k]);
                }
            }
        }
    }
    __syncthreads();
    const F29 w = inv;
    if (keep) {
#pragma clang loop unroll(full)
        for (uint32_t k = 0; k < kKeep; k++)
            if (b0 + k < b1) fe_store<FrParams>(&z[tile_last(b0 + k, n)], f29_to_fr(f29_mul<Fr29Mod>(nv[k], w)));
        return;
    }
    // forward: the numerators before each tile; backward: times the
    // denominators after it and the inverse
#pragma unroll 1
    for (uint32_t b = b0; b < b1; b++) {
        const F29 v = num_of(b);
        fe_store<FrParams>(&z[tile_last(b, n)], f29_to_fr(p));
        p = mul_run(p, v);
    }
    q = f29_mul<Fr29Mod>(q, w);
#pragma unroll 1
    for (uint32_t b = b1; b-- > b0;) {
        const uint64_t l = tile_last(b, n);
        fe_store<FrParams>(&z[l], f29_to_fr(mul_run(f29_repack(fe_load<FrParams>(&z[l]).v), q)));
        q = mul_run(q, den_of(b));
    }
}

// z[i] = prefix[i - 1] suffix[i] K_b, in place: a tile's rows are read before
// any is written
__global__ __launch_bounds__(kThreads) void k_product_combine(Fr *z, const Fr *__restrict__ temp, uint32_t n) {
    __shared__ uint32_t first_zero;  // the tile's first row with a zero denominator
    const uint32_t b = blockIdx.x, t = threadIdx.x;
    const uint64_t base = (uint64_t)b * kTile;
    const F29 kb = f29_from32(fe_load<FrParams>(&z[tile_last(b, n)]));
    const bool zeros = temp[base].v[7] & kTileZero;
    if (t == 0) first_zero = kTile;
    __syncthreads();
    Fr r[kRows];
#pragma clang loop unroll(full)
    for (uint32_t k = 0; k < kRows; k++) {
        const uint32_t e = k * kThreads + t;
        const uint64_t i = base + e;
        if (i < n) {
            r[k] = fe_load<FrParams>(&temp[i]);
            if (r[k].v[7] & kRowZero) atomicMin(&first_zero, e);
            r[k].v[7] &= ~(kRowZero | kTileZero);
            if (e) r[k] = fr_mul_w29(r[k], f29_from32(fe_load<FrParams>(&z[i - 1])));
            r[k] = fr_mul_w29(r[k], kb);
        }
    }
    __syncthreads();
#pragma clang loop unroll(full)
    for (uint32_t k = 0; k < kRows; k++) {
        const uint32_t e = k * kThreads + t;
        if (base + e >= n) continue;
        if (zeros && e > first_zero) r[k] = fe_zero<FrParams>();
        fe_store<FrParams>(&z[base + e], r[k]);
    }
}

// launches 2 and 3 after a tile pass
hipError_t product_finish(Fr *z, Fr *temp, uint32_t n, hipStream_t stream) {
    ZK_CHECK(hipGetLastError());
    const uint32_t nb = (n + kTile - 1) / kTile;
    k_product_top<<<1, kTopThreads, 0, stream>>>(z, temp, n, nb);
    ZK_CHECK(hipGetLastError());
    k_product_combine<<<nb, kThreads, 0, stream>>>(z, temp, n);
    return hipGetLastError();
}

// tails[s] = prod_{s' < s} z_{s'}[u]   (src/permutation.rs:131-145); one thread
__global__ void k_perm_tails(const Fr *const *__restrict__ zs, int nsets, uint32_t u, Fr *__restrict__ tails) {
    if (threadIdx.x || blockIdx.x) return;
    Fr acc = fe_one<FrParams>();
    for (int s = 0; s < nsets; s++) {
        fe_store<FrParams>(&tails[s], acc);
        acc = acc * fe_load<FrParams>(&zs[s][u]);
    }
}
// z_s[i] *= tails[s] for i <= u, s >= 1
__global__ void k_perm_chain(Fr *const *__restrict__ zs, int nsets, uint32_t u, const Fr *__restrict__ tails) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t s = blockIdx.y + 1;
    if (i > u || s >= (uint32_t)nsets) return;
    fe_store<FrParams>(&zs[s][i], fe_load<FrParams>(&zs[s][i]) * fe_load<FrParams>(&tails[s]));
}

}  // namespace

extern "C" {

hipError_t zk_permutation_z_set(void *z, const void *values, const void *sigmas, int ncols, const void *beta,
                                const void *gamma, const void *delta_start, const void *delta, const void *omega,
                                void *temp, int n, hipStream_t stream) {
    if (n <= 0 || ncols <= 0 || !z || !values || !sigmas || !beta || !gamma || !delta_start || !delta || !omega ||
        !temp)
        return hipErrorInvalidValue;
    Fr *zz = (Fr *)z;
    Fr *tmp = (Fr *)temp;
    const uint32_t un = (uint32_t)n;
    k_perm_tiles<<<dim3((un + kTile - 1) / kTile, 2), kThreads, 0, stream>>>(
        zz, tmp, (const Fr *const *)values, (const Fr *const *)sigmas, ncols, (const Fr *)beta, (const Fr *)gamma,
        (const Fr *)delta_start, (const Fr *)delta, (const Fr *)omega, un);
    return product_finish(zz, tmp, un, stream);
}

hipError_t zk_permutation_chain(void *zs, int nsets, int u, int n, void *tails, hipStream_t stream) {
    if (nsets <= 0 || n <= 0 || u < 0 || u >= n || !zs || !tails) return hipErrorInvalidValue;
    k_perm_tails<<<1, 64, 0, stream>>>((const Fr *const *)zs, nsets, (uint32_t)u, (Fr *)tails);
    ZK_CHECK(hipGetLastError());
    if (nsets > 1) {
        dim3 grid(((uint32_t)u + 1 + kThreads - 1) / kThreads, (uint32_t)nsets - 1);
        k_perm_chain<<<grid, kThreads, 0, stream>>>((Fr *const *)zs, nsets, (uint32_t)u, (const Fr *)tails);
        ZK_CHECK(hipGetLastError());
    }
    return hipSuccess;
}

hipError_t zk_shuffle_z(void *z, const void *inputs, const void *shuffles, int group_len, const void *betas, void *temp,
                        int n, hipStream_t stream) {
    if (n <= 0 || group_len <= 0 || !z || !inputs || !shuffles || !betas || !temp) return hipErrorInvalidValue;
    Fr *zz = (Fr *)z;
    Fr *tmp = (Fr *)temp;
    const uint32_t un = (uint32_t)n;
    k_shuffle_tiles<<<dim3((un + kTile - 1) / kTile, 2), kThreads, 0, stream>>>(
        zz, tmp, (const Fr *const *)inputs, (const Fr *const *)shuffles, (const Fr *)betas, group_len, un);
    return product_finish(zz, tmp, un, stream);
}

}  // extern "C"
