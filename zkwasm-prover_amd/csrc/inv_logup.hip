// Batch inversion, logup grand sums and field prefix scans for gfx950.
//
// Drop-in for `logup_sum_input_inv`, `eval_logup_z_compose` and
// `eval_logup_z_pure` (cuda/bn254.cu:19-220, :1914-1993; caller
// src/lib.rs:590-745), plus zk_batch_invert.
//
// Batch inversion is Montgomery's trick in one launch over tiles of 256 E
// elements (details at k_binv below); the logup's z[i] = s[i] - m[i] / (t[i] +
// beta) and its tile sums come out of the same pass.
// A zero input stays zero and does not disturb the others (halo2
// BatchInvert semantics); the reference's chunked kernel would zero its chunk
// instead, a case its callers never produce (beta is random).
//
// The logup z scan (exclusive prefix sum with a carried start value) is a
// three-kernel block scan: block totals (from k_binv where that wrote z), a
// one-block scan of the totals with the carry, then the in-block exclusive
// scan plus offset.
#include "ff29.h"
#include "inv_dev.h"
#include "zkcore.h"

using namespace zk;

namespace {

constexpr uint32_t kScanBlock = 2048;  // elements per scan block (256 threads x 8)

enum BinvMode {
    OUT_SET = 0,   // out[i] = 1 / x'[i]
    OUT_ADD = 1,   // out[i] += 1 / x'[i]
    OUT_LOGUP = 2  // out[i] = s[i] - m[i] / x'[i], and x[tile start] = the tile's sum of out
};

// ---- batch inversion ------------------------------------------------------
// One workgroup per tile of 256 E elements, thread t owning the elements k *
// 256 + t (k < E), so every access is coalesced.  Each thread forms its prefix
// products in registers; the 256 thread products go through a product tree in
// LDS; the first wave inverts the tile's product (inv_wave.h); the tree is
// walked down, and each thread emits its elements' inverses backwards.  Three
// products per element and one read (two of x, the second from cache) and one
// write of each array.
//
// Why one launch: with the prefix products through memory and the tiles'
// products inverted by a launch of their own it moved 5 x 32 B per element and
// waited 70 us for the inversions with the device idle; here other tiles'
// products run meanwhile (2^22 elements: 264 -> 191 us; 2^18: 160 -> 50).
// The products are the 29-bit ones (ff29.h): running products stay in the
// 256-bit Montgomery domain below 2r, and one operand of each product is
// shifted into the 2^261 domain (f29_from32 of an element, f29_shl5 of a
// product).  Four waves per SIMD measured best: 2^22 elements 225 us with
// three, 191 with four, 208 with five, although the prefixes of eight elements
// (nine registers each) don't fit its 128 registers: 88 B per lane go to
// scratch (none with two or four elements).
constexpr uint32_t kBT = 256;

struct BinvNode {
    uint32_t l[9];  // stride of nine words: no bank conflicts
};
__device__ __forceinline__ F29 node_load(const BinvNode &n) {
    F29 r;
#pragma unroll
    for (int i = 0; i < 9; i++) r.l[i] = n.l[i];
    return r;
}
__device__ __forceinline__ void node_store(BinvNode &n, const F29 &v) {
#pragma unroll
    for (int i = 0; i < 9; i++) n.l[i] = v.l[i];
}

template <int MODE, int E>
__global__ __launch_bounds__(kBT, 4) void k_binv(Fr *x, const Fr *__restrict__ beta, Fr *out, uint32_t n, const Fr *s,
                                                 const Fr *__restrict__ m) {
    __shared__ BinvNode tree[2 * kBT];
    __shared__ Fr part[kBT / 64];
    const uint32_t t = threadIdx.x;
    const uint64_t base = (uint64_t)blockIdx.x * (kBT * E) + t;
    const bool hb = beta != nullptr;
    const Fr b = hb ? fe_load<FrParams>(beta) : fe_zero<FrParams>();
    F29 pre[E], acc = f29_repack(FrParams::ONE);
    uint32_t live = 0;  // bit k: element k exists and is not zero
#pragma clang loop unroll(full)
    for (int k = 0; k < E; k++) {
        const uint64_t i = base + (uint32_t)k * kBT;
        pre[k] = acc;
        if (i < n) {
            Fr v = fe_load<FrParams>(&x[i]);
            if (hb) v = v + b;
            if (!fe_is_zero<FrParams>(v)) {
                live |= 1u << k;
                acc = f29_mul<Fr29Mod>(acc, f29_from32(v));
            }
        }
    }
    node_store(tree[kBT + t], acc);
    __syncthreads();
    for (uint32_t w = kBT / 2; w >= 1; w >>= 1) {
        if (t < w) {
            const uint32_t p = w + t;
            node_store(tree[p], f29_mul<Fr29Mod>(node_load(tree[2 * p]), f29_shl5(node_load(tree[2 * p + 1]))));
        }
        __syncthreads();
    }
    if (t < 64) {
        const Fr inv = fr_inv_wave(f29_to_fr(node_load(tree[1])));
        if (t == 0) node_store(tree[1], f29_repack(inv.v));
    }
    __syncthreads();
    for (uint32_t w = 1; w < kBT; w <<= 1) {
        if (t < w) {
            const uint32_t p = w + t;
            const F29 ip = f29_shl5(node_load(tree[p]));
            const F29 l = node_load(tree[2 * p]), r = node_load(tree[2 * p + 1]);
            node_store(tree[2 * p], f29_mul<Fr29Mod>(ip, r));
            node_store(tree[2 * p + 1], f29_mul<Fr29Mod>(ip, l));
        }
        __syncthreads();
    }
    acc = node_load(tree[kBT + t]);
    Fr sum = fe_zero<FrParams>();
    // fully unrolled: an indexed array would go to scratch whole
#pragma clang loop unroll(full)
    for (int k = E - 1; k >= 0; k--) {
        const uint64_t i = base + (uint32_t)k * kBT;
        if (i < n) {
            Fr r = fe_zero<FrParams>();
            if ((live >> k) & 1u) {
                r = f29_to_fr(k ? f29_mul<Fr29Mod>(f29_shl5(acc), pre[k]) : acc);
                if (k) {
                    Fr v = fe_load<FrParams>(&x[i]);
                    if (hb) v = v + b;
                    acc = f29_mul<Fr29Mod>(acc, f29_from32(v));
                }
            }
            if (MODE == OUT_ADD) r = fe_load<FrParams>(&out[i]) + r;
            if (MODE == OUT_LOGUP) {
                r = fe_load<FrParams>(&s[i]) - fr_mul_w29(fe_load<FrParams>(&m[i]), f29_from32(r));
                sum = sum + r;
            }
            fe_store<FrParams>(&out[i], r);
        }
    }
    if (MODE == OUT_LOGUP) {
        // the tile's sum into x's slot of its first element, which only this
        // workgroup has read
#pragma unroll
        for (int d = 32; d; d >>= 1) {
            Fr o;
#pragma unroll
            for (int i = 0; i < 8; i++) o.v[i] = (uint32_t)__shfl_xor((int)sum.v[i], d);
            sum = sum + o;
        }
        if ((t & 63) == 0) part[t >> 6] = sum;
        __syncthreads();  // also: every read of x in this tile is done
        if (t == 0) {
            for (uint32_t w = 1; w < kBT / 64; w++) sum = sum + part[w];
            fe_store<FrParams>(&x[base], sum);
        }
    }
}

// Elements per thread.  A tile costs a tree (about 27 wave products) and an
// inversion's latency whatever its size, which eight elements per thread
// amortise; small inputs take fewer so that more workgroups share the products
// (2 / 4 / 8 per thread: 2^16 elements 44 / 49 / 60 us, 2^18 50 / 50 / 60, 2^20
// 107 / 73 / 77, 2^22 370 / 257 / 191).
int binv_elems(uint32_t n) { return n <= (1u << 17) ? 2 : n <= (1u << 20) ? 4 : 8; }
template <int MODE>
hipError_t binv_launch(Fr *x, const Fr *beta, Fr *out, uint32_t n, const Fr *s, const Fr *m, hipStream_t stream) {
    const int e = binv_elems(n);
    const uint32_t tiles = (uint32_t)(((uint64_t)n + (uint64_t)kBT * e - 1) / ((uint64_t)kBT * e));
    if (e == 2)
        k_binv<MODE, 2><<<tiles, kBT, 0, stream>>>(x, beta, out, n, s, m);
    else if (e == 4)
        k_binv<MODE, 4><<<tiles, kBT, 0, stream>>>(x, beta, out, n, s, m);
    else
        k_binv<MODE, 8><<<tiles, kBT, 0, stream>>>(x, beta, out, n, s, m);
    return hipGetLastError();
}

__global__ void k_logup_step2(Fr *__restrict__ z, const Fr *__restrict__ s, const Fr *__restrict__ tinv,
                              const Fr *__restrict__ m, uint32_t n) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t stride = gridDim.x * blockDim.x;
    for (; i < n; i += stride)
        fe_store<FrParams>(&z[i], fe_load<FrParams>(&s[i]) - fe_load<FrParams>(&m[i]) * fe_load<FrParams>(&tinv[i]));
}

// ---- additive prefix scan ---------------------------------------------------
// block totals: 256 threads x 8 contiguous elements
__global__ __launch_bounds__(256) void k_fscan_totals(const Fr *__restrict__ z, uint32_t n, Fr *__restrict__ tot) {
    __shared__ Fr sh[256];
    uint32_t base = blockIdx.x * kScanBlock + threadIdx.x * 8;
    Fr acc = fe_zero<FrParams>();
    for (uint32_t k = 0; k < 8; k++)
        if (base + k < n) acc = acc + fe_load<FrParams>(&z[base + k]);
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (uint32_t s = 128; s; s >>= 1) {
        if (threadIdx.x < s) sh[threadIdx.x] = sh[threadIdx.x] + sh[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) fe_store<FrParams>(&tot[blockIdx.x], sh[0]);
}

// exclusive scan over a workgroup of 256 threads: shuffles inside each wave,
// the wave totals through LDS.  Returns the sum of the earlier threads'
// values; total (every thread): the workgroup's.
__device__ __forceinline__ Fr block_scan_add(const Fr &v, Fr *sh, Fr &total) {
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    Fr inc = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        Fr o;
#pragma unroll
        for (int i = 0; i < 8; i++) o.v[i] = (uint32_t)__shfl_up((int)inc.v[i], d, 64);
        if (lane >= (uint32_t)d) inc = inc + o;
    }
    if (lane == 63) sh[wv] = inc;
    __syncthreads();
    Fr off = fe_zero<FrParams>();
    total = fe_zero<FrParams>();
    for (uint32_t w = 0; w < 4; w++) {
        if (w < wv) off = off + sh[w];
        total = total + sh[w];
    }
    __syncthreads();
    return off + (inc - v);
}

// one block: exclusive scan of the nb totals at tot[b * stride] in place,
// starting from *carry (zero when carry == null)
__global__ __launch_bounds__(256) void k_fscan_top(Fr *tot, uint32_t nb, size_t stride, const Fr *__restrict__ carry) {
    __shared__ Fr sh[4];
    Fr run = carry ? fe_load<FrParams>(carry) : fe_zero<FrParams>();
    // each round covers 256 * 8 totals: thread-local serial part + block scan
    for (uint32_t base = 0; base < nb; base += 256 * 8) {
        uint32_t b0 = base + threadIdx.x * 8;
        Fr loc[8];
        Fr acc = fe_zero<FrParams>(), total;
#pragma unroll
        for (uint32_t k = 0; k < 8; k++) {
            loc[k] = b0 + k < nb ? fe_load<FrParams>(&tot[(b0 + k) * stride]) : fe_zero<FrParams>();
            acc = acc + loc[k];
        }
        Fr pre = run + block_scan_add(acc, sh, total);
#pragma unroll
        for (uint32_t k = 0; k < 8; k++) {
            if (b0 + k < nb) fe_store<FrParams>(&tot[(b0 + k) * stride], pre);
            pre = pre + loc[k];
        }
        run = run + total;
    }
}

// z[i] = offset of the block + exclusive in-block prefix; last_z gets
// z[last_index].  Blocks of 256 E elements, thread t owning E consecutive
// ones; block b's offset is at tot[b * stride].
template <int E>
__global__ __launch_bounds__(256) void k_fscan_apply(Fr *z, uint32_t n, const Fr *__restrict__ tot, size_t stride,
                                                     Fr *last_z, int64_t last_index) {
    __shared__ Fr sh[4];
    const uint64_t base = (uint64_t)blockIdx.x * (256 * E) + threadIdx.x * E;
    Fr loc[E];
    Fr acc = fe_zero<FrParams>(), total;
#pragma unroll
    for (uint32_t k = 0; k < E; k++) {
        loc[k] = base + k < n ? fe_load<FrParams>(&z[base + k]) : fe_zero<FrParams>();
        acc = acc + loc[k];
    }
    Fr pre = fe_load<FrParams>(&tot[blockIdx.x * stride]) + block_scan_add(acc, sh, total);
#pragma unroll
    for (uint32_t k = 0; k < E; k++) {
        const uint64_t i = base + k;
        if (i < n) {
            fe_store<FrParams>(&z[i], pre);
            if (last_z && (int64_t)i == last_index) fe_store<FrParams>(last_z, pre);
        }
        pre = pre + loc[k];
    }
}

// the wave-wide inversion's cofactor and whether its GCD ended, unchecked: one
// wave per element
__global__ __launch_bounds__(64) void k_fr_inv_wave(Fr *__restrict__ out, uint32_t *__restrict__ ok,
                                                    const Fr *__restrict__ a) {
    const Fr y = fe_load<FrParams>(&a[blockIdx.x]);
    uint32_t v[8];
    const bool good = zkinv::bingcd_wave(v, y.v, FrParams::M, FrParams::INV);
    if (threadIdx.x) return;
    fe_store<FrParams>(&out[blockIdx.x], fe_from_raw<FrParams>(v));
    ok[blockIdx.x] = good ? 1u : 0u;
}

}  // namespace

namespace zk {

// out[i] = 1/(x[i] (+ beta)) (mode OUT_SET) or out[i] += that (OUT_ADD).
// out may alias x.
hipError_t batch_invert_ex(const Fr *x, const Fr *beta, Fr *out, int mode, uint32_t n, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    Fr *xx = const_cast<Fr *>(x);  // written in OUT_LOGUP only
    return mode == OUT_ADD ? binv_launch<OUT_ADD>(xx, beta, out, n, nullptr, nullptr, stream)
                           : binv_launch<OUT_SET>(xx, beta, out, n, nullptr, nullptr, stream);
}

// exclusive sum scan in place; carry (device) = start value or null for
// zero; last_z (device, may be null) receives z[last_index].  tot: one Fr per
// kScanBlock elements.
static hipError_t field_scan(Fr *z, uint32_t n, const Fr *carry, Fr *last_z, int64_t last_index, Fr *tot,
                             hipStream_t stream) {
    if (n == 0) return hipSuccess;
    uint32_t nb = (n + kScanBlock - 1) / kScanBlock;
    k_fscan_totals<<<nb, 256, 0, stream>>>(z, n, tot);
    ZK_CHECK(hipGetLastError());
    k_fscan_top<<<1, 256, 0, stream>>>(tot, nb, 1, carry);
    ZK_CHECK(hipGetLastError());
    k_fscan_apply<8><<<nb, 256, 0, stream>>>(z, n, tot, 1, last_z, last_index);
    return hipGetLastError();
}

}  // namespace zk

namespace zk {

// out = (x + beta)^-1 element-wise (zeros stay zero); temp: n Fr
hipError_t batch_invert_shifted(void *out, const void *x, const void *beta, void *temp, int n, hipStream_t stream) {
    if (n <= 0 || !out || !x || !beta || !temp) return hipErrorInvalidValue;
    return batch_invert_ex((const Fr *)x, (const Fr *)beta, (Fr *)out, OUT_SET, (uint32_t)n, stream);
}

// eval_logup_z_compose after its table inversion: z from the logup sum
// `input` (clobbered as scan scratch), the inverted table (t + beta)^-1 and
// the multiplicities; the same steps and bytes as the drop-in
hipError_t logup_z_inverted(void *z, void *input, const void *table_inv, const void *multiplicity, void *last_z,
                            int last_z_index, int n, hipStream_t stream) {
    if (n <= 0 || !z || !input || !table_inv || !multiplicity || !last_z || last_z_index < 0 || last_z_index >= n)
        return hipErrorInvalidValue;
    uint32_t blocks = ((uint32_t)n + 255) / 256;
    if (blocks > 16384) blocks = 16384;
    k_logup_step2<<<blocks, 256, 0, stream>>>((Fr *)z, (const Fr *)input, (const Fr *)table_inv,
                                               (const Fr *)multiplicity, (uint32_t)n);
    ZK_CHECK(hipGetLastError());
    return field_scan((Fr *)z, (uint32_t)n, (const Fr *)last_z, (Fr *)last_z, last_z_index, (Fr *)input,
                      stream);
}

}  // namespace zk

extern "C" {

// In-place batch inversion; temp (n Fr) is not needed by this implementation.
hipError_t zk_batch_invert(void *a, void *temp, int n, hipStream_t stream) {
    if (n < 0 || (n > 0 && (!a || !temp))) return hipErrorInvalidValue;
    return batch_invert_ex((const Fr *)a, nullptr, (Fr *)a, OUT_SET, (uint32_t)n, stream);
}

// Test entry: v with y^-1 = v 2^36 mod r for y = a[i] as a plain number, and
// ok[i] = 1 unless the GCD did not end at 1 (y = 0).
hipError_t zk_fr_inv_wave(void *out, void *ok, const void *a, int n, hipStream_t stream) {
    if (n <= 0 || !out || !ok || !a) return hipErrorInvalidValue;
    k_fr_inv_wave<<<(uint32_t)n, 64, 0, stream>>>((Fr *)out, (uint32_t *)ok, (const Fr *)a);
    return hipGetLastError();
}

// cuda/bn254.cu:1914-1934: sum[i] (=, or += when init != 0) 1/(input[i] + beta).
// temp (n Fr) is not needed by this implementation.
hipError_t logup_sum_input_inv(void *sum, const void *input, void *temp, const void *beta, int init, int n,
                               hipStream_t stream) {
    if (n <= 0 || !sum || !input || !beta || !temp) return hipErrorInvalidValue;
    return batch_invert_ex((const Fr *)input, (const Fr *)beta, (Fr *)sum, init ? OUT_ADD : OUT_SET, (uint32_t)n,
                           stream);
}

// cuda/bn254.cu:1936-1966: z in place; input (n Fr) is scratch for the scan.
hipError_t eval_logup_z_pure(void *z, void *input, void *table, void *last_z, int last_z_index, int n,
                             hipStream_t stream) {
    (void)table;
    if (n <= 0 || !z || !input || !last_z || last_z_index < 0 || last_z_index >= n) return hipErrorInvalidValue;
    return field_scan((Fr *)z, (uint32_t)n, (const Fr *)last_z, (Fr *)last_z, last_z_index, (Fr *)input,
                      stream);
}

// cuda/bn254.cu:1968-1993.  z[i] = input[i] - m[i] / (table[i] + beta), then
// the exclusive scan with carry last_z[0]; last_z[0] = z[last_z_index] at the
// end.  The inversion's pass writes z and its tiles' sums, the latter into
// table (scratch, as input is: the reference inverts table in place with z as
// temporary storage).
hipError_t eval_logup_z_compose(void *z, void *input, void *table, const void *multiplicity, const void *beta,
                                void *last_z, int last_z_index, int n, hipStream_t stream) {
    if (n <= 0 || !z || !input || !table || !multiplicity || !beta || !last_z || last_z_index < 0 ||
        last_z_index >= n)
        return hipErrorInvalidValue;
    const uint32_t un = (uint32_t)n;
    const int e = binv_elems(un);
    const size_t tile = (size_t)kBT * e;
    const uint32_t nb = (uint32_t)((un + tile - 1) / tile);
    Fr *zz = (Fr *)z, *tab = (Fr *)table, *lz = (Fr *)last_z;
    ZK_CHECK(binv_launch<OUT_LOGUP>(tab, (const Fr *)beta, zz, un, (const Fr *)input, (const Fr *)multiplicity,
                                    stream));
    k_fscan_top<<<1, 256, 0, stream>>>(tab, nb, tile, lz);
    ZK_CHECK(hipGetLastError());
    if (e == 2)
        k_fscan_apply<2><<<nb, 256, 0, stream>>>(zz, un, tab, tile, lz, last_z_index);
    else if (e == 4)
        k_fscan_apply<4><<<nb, 256, 0, stream>>>(zz, un, tab, tile, lz, last_z_index);
    else
        k_fscan_apply<8><<<nb, 256, 0, stream>>>(zz, un, tab, tile, lz, last_z_index);
    return hipGetLastError();
}

}  // extern "C"
