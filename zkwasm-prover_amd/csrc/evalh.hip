// eval_h expression evaluator and constraint kernels for gfx950.
//
// Drop-in for field_op, field_op_batch_mul_sum, field_mul_zip, the
// permutation / logup / shuffle eval_h kernels and
// logup_eval_h_inputs_product_sum (cuda/bn254.cu:542-1213 and the wrappers at
// :1215-1635; callers src/eval_h.rs, src/expr.rs, src/cuda/bn254.rs).
//
// Every kernel is element-wise over the (extended) domain: grid-stride loops
// with 256-thread workgroups, each row reading its operands once (rotations
// are constant index shifts, so loads stay coalesced).  The per-row formulas
// and the order of the `t = t*y + ...` folds are exactly the reference's,
// which fixes h(X) bit for bit.  The term list of field_op_batch_mul_sum is
// staged once per workgroup in LDS instead of being re-read per row.
#include <string.h>

#include "evalh_rows.h"
#include "zkcore.h"

using namespace zk;

namespace {

constexpr uint32_t kThreads = 256;
constexpr int kMaxLdsTerms = 2048;

uint32_t grid_for(uint32_t n) {
    uint32_t b = (n + kThreads - 1) / kThreads;
    return b > 32768 ? 32768 : (b ? b : 1);
}

__device__ __forceinline__ void st(Fr *p, const Fr &v) { fe_store<FrParams>(p, v); }

#define GRID_LOOP(i, n)                                                \
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < (n); \
         i += gridDim.x * blockDim.x)

__device__ __forceinline__ uint32_t rot_mod(uint32_t i, int rot, uint32_t n) {
    int64_t v = ((int64_t)i + rot) % (int64_t)n;
    return (uint32_t)(v < 0 ? v + n : v);
}

// cuda/bn254.cu:585-639
__global__ void k_field_op(Fr *res, const Fr *l, int l_rot, const Fr *l_c, const Fr *r, int r_rot, const Fr *r_c,
                           uint32_t n, int op) {
    Fr lc = l_c ? ld(l_c) : fe_zero<FrParams>();
    Fr rc = r_c ? ld(r_c) : fe_zero<FrParams>();
    GRID_LOOP(i, n) {
        Fr fl, fr = fe_zero<FrParams>();
        if (l) {
            fl = ld(&l[rot_mod(i, l_rot, n)]);
            if (l_c) fl = fl * lc;
        } else {
            fl = lc;
        }
        if (r) {
            fr = ld(&r[rot_mod(i, r_rot, n)]);
            if (r_c) fr = fr * rc;
        } else if (r_c) {
            fr = rc;
        }
        Fr o;
        if (op == 0) o = fl + fr;
        else if (op == 1) o = fl * fr;
        else if (op == 2) o = fl;
        else o = fl - fr;
        // res may alias l or r with a rotation: every row reads its operands
        // before the (same-row) write, as in the reference
        st(&res[i], o);
    }
}

// cuda/bn254.cu:542-572: res[i] += sum_t c_t * prod_j v_tj[(i + rot_tj) & (n-1)]
// v = [c0, a00, a01, NULL, c1, a10, NULL, ...]; rot has one entry per column
// pointer (the non-NULL entries that are not coefficients).
__global__ __launch_bounds__(kThreads) void k_batch_mul_sum(Fr *res, const Fr *const *__restrict__ v,
                                                            const int *__restrict__ rot, int v_n, uint32_t n) {
    __shared__ const Fr *sv[kMaxLdsTerms];
    __shared__ int sr[kMaxLdsTerms];
    __shared__ int n_cols;
    const bool in_lds = v_n <= kMaxLdsTerms;
    if (in_lds) {
        for (int k = threadIdx.x; k < v_n; k += blockDim.x) sv[k] = v[k];
        __syncthreads();
        if (threadIdx.x == 0) {
            int vi = 0, cols = 0;
            while (vi < v_n) {
                vi++;  // coefficient
                while (vi < v_n && sv[vi]) { vi++; cols++; }
                vi++;  // separator
            }
            n_cols = cols;
        }
        __syncthreads();
        for (int k = threadIdx.x; k < n_cols; k += blockDim.x) sr[k] = rot[k];
    }
    __syncthreads();
    const Fr *const *V = in_lds ? (const Fr *const *)sv : v;
    const int *Rt = in_lds ? (const int *)sr : rot;
    const uint32_t mask = n - 1;
    GRID_LOOP(i, n) {
        Fr acc = fe_zero<FrParams>();
        int vi = 0, ri = 0;
        while (vi < v_n) {
            Fr term = ld(V[vi++]);  // coefficient
            while (vi < v_n && V[vi]) {
                term = term * ld(&V[vi][(i + (uint32_t)Rt[ri]) & mask]);
                vi++;
                ri++;
            }
            acc = acc + term;
            vi++;  // NULL separator
        }
        st(&res[i], ld(&res[i]) + acc);
    }
}

// cuda/bn254.cu:1121-1131
__global__ void k_field_mul_zip(Fr *buf, const Fr *__restrict__ coeff, uint32_t coeff_n, uint32_t n) {
    GRID_LOOP(i, n) st(&buf[i], ld(&buf[i]) * ld(&coeff[i % coeff_n]));
}

// cuda/bn254.cu:664-702
__global__ void k_perm_p1(Fr *res, const Fr *__restrict__ first, const Fr *__restrict__ last,
                          const Fr *__restrict__ l0, const Fr *__restrict__ l_last, const Fr *__restrict__ yp,
                          uint32_t n) {
    const F29 y = hi(ld(yp));
    const Fr one = fe_one<FrParams>();
    GRID_LOOP(i, n) st(&res[i], perm_p1_row(res, first, last, l0, l_last, i, one, y));
}

// cuda/bn254.cu:704-739 (also logup_eval_h_z_set)
__global__ void k_perm_p2(Fr *res, const Fr *const *__restrict__ set, const Fr *__restrict__ l0,
                          const Fr *__restrict__ yp, int n_set, int rot, uint32_t n) {
    const F29 y = hi(ld(yp));
    GRID_LOOP(i, n) {
        uint32_t rp = (i + n + (uint32_t)rot) & (n - 1);
        F29 t = lo(ld(&res[i]));
        const F29 l = hi(ld(&l0[i]));
        for (int j = 1; j < n_set; j++) t = perm_p2_step(t, ld(&set[j][i]), ld(&set[j - 1][rp]), l, y);
        st(&res[i], f29_to_fr(t));
    }
}

// cuda/bn254.cu:741-765
__global__ void k_perm_l(Fr *res, const Fr *__restrict__ beta, const Fr *__restrict__ gamma, const Fr *__restrict__ p,
                         uint32_t n) {
    Fr b = ld(beta), g = ld(gamma);
    GRID_LOOP(i, n) {
        Fr t = ld(&p[i]) * b;
        if (i == 0) t = t + g;
        st(&res[i], ld(&res[i]) + t);
    }
}

// cuda/bn254.cu:867-918
__global__ void k_logup_eval_h(Fr *res, const Fr *__restrict__ ip, const Fr *__restrict__ ips,
                               const Fr *__restrict__ table, const Fr *__restrict__ m, const Fr *__restrict__ zf,
                               const Fr *__restrict__ zl, const Fr *__restrict__ l0, const Fr *__restrict__ l_last,
                               const Fr *__restrict__ l_active, const Fr *__restrict__ yp, int rot, uint32_t n) {
    const F29 y = hi(ld(yp));
    GRID_LOOP(i, n) {
        uint32_t rn = (i + (uint32_t)rot) & (n - 1);
        st(&res[i], logup_row(res, ip, ips, table, m, zf, zl, l0, l_last, l_active, i, rn, y));
    }
}

// cuda/bn254.cu:920-949
__global__ void k_logup_extra(Fr *res, const Fr *__restrict__ ip, const Fr *__restrict__ ips, const Fr *__restrict__ zp,
                              const Fr *__restrict__ l_active, const Fr *__restrict__ yp, int rot, uint32_t n) {
    const F29 y = hi(ld(yp));
    GRID_LOOP(i, n) {
        uint32_t rn = (i + (uint32_t)rot) & (n - 1);
        st(&res[i], logup_extra_row(res, ip, ips, zp, l_active, i, rn, y));
    }
}

// cuda/bn254.cu:1172-1213 (the product-sum rebuilt per j like the reference,
// which costs n_set^2 multiplies; n_set is small)
__global__ void k_inputs_product_sum(Fr *__restrict__ prod, Fr *__restrict__ psum, const Fr *const *__restrict__ set,
                                     int n_set, uint32_t n) {
    GRID_LOOP(i, n) {
        Fr p = fe_one<FrParams>();
        for (int j = 0; j < n_set; j++) p = p * ld(&set[j][i]);
        st(&prod[i], p);
        Fr sum = fe_zero<FrParams>();
        for (int j = 0; j < n_set; j++) {
            Fr u = fe_one<FrParams>();
            for (int k = 0; k < n_set; k++)
                if (k != j) u = u * ld(&set[k][i]);
            sum = sum + u;
        }
        st(&psum[i], sum);
    }
}

__global__ void k_shuffle(Fr *res, const Fr *__restrict__ input, const Fr *__restrict__ table, const Fr *__restrict__ zp,
                          const Fr *__restrict__ l0, const Fr *__restrict__ l_last, const Fr *__restrict__ l_active,
                          const Fr *__restrict__ yp, int rot, uint32_t n) {
    const F29 y = hi(ld(yp));
    GRID_LOOP(i, n) {
        uint32_t rn = (i + (uint32_t)rot) & (n - 1);
        st(&res[i], shuffle_fold(ld(&res[i]), lo(ld(&input[i])), lo(ld(&table[i])), ld(&zp[i]), ld(&zp[rn]), ld(&l0[i]),
                                 ld(&l_last[i]), ld(&l_active[i]), y));
    }
}

__global__ void k_shuffle_v2(Fr *res, const Fr *const *__restrict__ inputs, const Fr *const *__restrict__ tables,
                             const Fr *__restrict__ betas, int group_len, const Fr *__restrict__ zp,
                             const Fr *__restrict__ l0, const Fr *__restrict__ l_last, const Fr *__restrict__ l_active,
                             const Fr *__restrict__ yp, int rot, uint32_t n) {
    const F29 y = hi(ld(yp));
    GRID_LOOP(i, n) {
        uint32_t rn = (i + (uint32_t)rot) & (n - 1);
        Fr b0 = ld(&betas[0]);
        F29 l = lo(ld(&inputs[0][i]) + b0);
        F29 r = lo(ld(&tables[0][i]) + b0);
        for (int j = 1; j < group_len; j++) {
            const F29 bj = hi(ld(&betas[j]));
            l = shuffle_factor(l, ld(&inputs[j][i]), bj);
            r = shuffle_factor(r, ld(&tables[j][i]), bj);
        }
        st(&res[i], shuffle_fold(ld(&res[i]), l, r, ld(&zp[i]), ld(&zp[rn]), ld(&l0[i]), ld(&l_last[i]),
                                 ld(&l_active[i]), y));
    }
}

bool bad_n(int n) { return n <= 0 || (n & (n - 1)); }

// cuda/bn254.cu:496-540: res[i] = sum_j v_j[i] * w^(rot_j * i) (* c_j when
// v_c[j] is set), the sum of coefficient vectors each rotated by w^rot_j.
// The term pointers are staged in LDS once per workgroup.  The exponent is
// taken mod n with 32-bit wrap-around, as the reference's int arithmetic
// gives for every rotation (n divides 2^32).
constexpr int kMaxSumTerms = 256;
__global__ __launch_bounds__(kThreads) void k_field_sum(Fr *res, const Fr *const *__restrict__ v,
                                                        const Fr *const *__restrict__ v_c,
                                                        const int *__restrict__ v_rot,
                                                        const Fr *__restrict__ omegas, int v_n, uint32_t n) {
    __shared__ const Fr *sv[kMaxSumTerms];
    __shared__ const Fr *sc[kMaxSumTerms];
    __shared__ uint32_t sr[kMaxSumTerms];
    for (int k = threadIdx.x; k < v_n; k += blockDim.x) {
        sv[k] = v[k];
        sc[k] = v_c[k];
        sr[k] = (uint32_t)v_rot[k];
    }
    __syncthreads();
    GRID_LOOP(i, n) {
        Fr acc = fe_zero<FrParams>();
        for (int j = 0; j < v_n; j++) {
            Fr t = ld(&sv[j][i]) * ld(&omegas[(sr[j] * i) & (n - 1)]);
            if (sc[j]) t = t * ld(sc[j]);
            acc = j ? acc + t : t;
        }
        st(&res[i], acc);
    }
}

// cuda/bn254.cu:798-866: the permuted-column lookup's five folds
//   l0 (1 - z); l_last (z^2 - z);
//   l_active (z(wX) (a' + beta)(s' + gamma) - z(X) input * table);
//   l0 (a' - s'); l_active (a' - s')(a' - a'(w^-1 X))
// where input and table are the compressed expressions with beta and gamma
// already added.
__global__ void k_lookup_eval_h(Fr *res, const Fr *__restrict__ input, const Fr *__restrict__ table,
                                const Fr *__restrict__ pin, const Fr *__restrict__ ptab, const Fr *__restrict__ z,
                                const Fr *__restrict__ l0, const Fr *__restrict__ l_last,
                                const Fr *__restrict__ l_active, const Fr *__restrict__ yp,
                                const Fr *__restrict__ betap, const Fr *__restrict__ gammap, int rot, uint32_t n) {
    const Fr y = ld(yp), beta = ld(betap), gamma = ld(gammap), one = fe_one<FrParams>();
    GRID_LOOP(i, n) {
        const uint32_t rn = (i + (uint32_t)rot) & (n - 1);
        const uint32_t rp = (i + n - (uint32_t)rot) & (n - 1);
        const Fr zi = ld(&z[i]), a = ld(&pin[i]), sp = ld(&ptab[i]);
        Fr t = ld(&res[i]) * y;
        t = t + ld(&l0[i]) * (one - zi);
        t = t * y;
        t = t + ld(&l_last[i]) * (fe_sqr<FrParams>(zi) - zi);
        t = t * y;
        const Fr la = ld(&l_active[i]);
        Fr u = (a + beta) * (sp + gamma) * ld(&z[rn]) - zi * (ld(&input[i]) * ld(&table[i]));
        t = t + u * la;
        t = t * y;
        const Fr d = a - sp;
        t = t + ld(&l0[i]) * d;
        t = t * y;
        t = t + (a - ld(&pin[rp])) * d * la;
        st(&res[i], t);
    }
}

// One permutation set's product term on the extended coset, fused:
// h = h*y + l_active * ( z(wX) * prod_c (v_c + beta*sigma_c + gamma)
//                      - z(X)  * prod_c (v_c + gamma + bd_c * X) )
// with bd_c = beta * delta^c and X the coset points.  The reference builds the
// same term from field_op / permutation_eval_h_l and one extended NTT per
// side and column (src/eval_h.rs:700-840); here sigma_c and X stay resident as
// coset evaluations and one pass reads each operand once.
// Five waves per SIMD asked for: 97 registers without it, one too many.
constexpr int kMaxPermCols = 16;
__global__ __launch_bounds__(kThreads, 5) void k_perm_set_eval(Fr *h, const Fr *__restrict__ z, const Fr *const *__restrict__ v,
                                const Fr *const *__restrict__ sig, int nc, const Fr *__restrict__ beta,
                                const Fr *__restrict__ gamma, const Fr *__restrict__ bd, const Fr *__restrict__ X,
                                const Fr *__restrict__ l_active, const Fr *__restrict__ yp, int rot, uint32_t n) {
    __shared__ const Fr *sv[kMaxPermCols], *ss[kMaxPermCols];
    __shared__ F29 sb[kMaxPermCols];
    if (threadIdx.x < (unsigned)nc) {
        sv[threadIdx.x] = v[threadIdx.x];
        ss[threadIdx.x] = sig[threadIdx.x];
        sb[threadIdx.x] = hi(ld(&bd[threadIdx.x]));
    }
    __syncthreads();
    const F29 b = hi(ld(beta)), y = hi(ld(yp));
    const Fr g = ld(gamma);
    GRID_LOOP(i, n) {
        const uint32_t rn = (i + (uint32_t)rot) & (n - 1);
        const F29 x = hi(ld(&X[i]));
        F29 l = lo(ld(&z[rn])), r = lo(ld(&z[i]));
        for (int c = 0; c < nc; c++) {
            const F29 vg = hi(ld(&sv[c][i]) + g);
            l = perm_set_factor(l, vg, b, hi(ld(&ss[c][i])));
            r = perm_set_factor(r, vg, sb[c], x);
        }
        st(&h[i], perm_set_fold(ld(&h[i]), l, r, ld(&l_active[i]), y));
    }
}

// The benchmark circuit's gates folded into h in one pass (no reference
// entry: the prover core's replacement for its field_op_batch_mul_sum term
// list, which spells the same polynomial as 3 + 2G terms):
//   h[i] = q (y^G (a b + c - d) + sum_g y^(G-1-g) (f_g a - e_g)),
// evaluated by Horner in y with q factored out: 2 + 2G products per row
// instead of 7 + 5G.  Field arithmetic is exact, so the value (and its
// canonical bytes) is the term list's.  h is written, not accumulated.
constexpr int kMaxGates = 32;
struct GateArgs {
    const Fr *q, *a, *b, *c, *d;
    const Fr *f[kMaxGates];
    const Fr *e[kMaxGates];
    int ng;
};
__global__ __launch_bounds__(kThreads) void k_gate_eval(Fr *__restrict__ h, const GateArgs g,
                                                        const Fr *__restrict__ yp, uint32_t n) {
    const F29 y = hi(ld(yp));
    GRID_LOOP(i, n) {
        const F29 a = hi(ld(&g.a[i]));
        F29 acc = gate_first(a, ld(&g.b[i]), ld(&g.c[i]), ld(&g.d[i]));
        for (int k = 0; k < g.ng; k++) acc = gate_step(acc, a, ld(&g.f[k][i]), ld(&g.e[k][i]), y);
        st(&h[i], gate_last(acc, ld(&g.q[i])));
    }
}

}  // namespace

namespace zk {

hipError_t gate_eval_h(void *h, const void *q, const void *a, const void *b, const void *c, const void *d,
                       const void *const *f, const void *const *e, int ng, const void *y, int n, hipStream_t stream) {
    if (bad_n(n) || !h || !q || !a || !b || !c || !d || !y || ng < 0 || ng > kMaxGates || (ng && (!f || !e)))
        return hipErrorInvalidValue;
    GateArgs g;
    memset(&g, 0, sizeof(g));
    g.q = (const Fr *)q;
    g.a = (const Fr *)a;
    g.b = (const Fr *)b;
    g.c = (const Fr *)c;
    g.d = (const Fr *)d;
    for (int k = 0; k < ng; k++) {
        if (!f[k] || !e[k]) return hipErrorInvalidValue;
        g.f[k] = (const Fr *)f[k];
        g.e[k] = (const Fr *)e[k];
    }
    g.ng = ng;
    k_gate_eval<<<grid_for((uint32_t)n), kThreads, 0, stream>>>((Fr *)h, g, (const Fr *)y, (uint32_t)n);
    return hipGetLastError();
}

}  // namespace zk

extern "C" {

// cuda/bn254.cu:1269-1286 (the reference asserts 64 | n; any n >= 1 works here)
hipError_t field_op(void *res, const void *l, int l_rot, const void *l_c, const void *r, int r_rot, const void *r_c,
                    int size, int op, hipStream_t stream) {
    if (size <= 0 || !res || op < 0 || op > 3 || (!l && !l_c)) return hipErrorInvalidValue;
    k_field_op<<<grid_for(size), kThreads, 0, stream>>>((Fr *)res, (const Fr *)l, l_rot, (const Fr *)l_c,
                                                        (const Fr *)r, r_rot, (const Fr *)r_c, (uint32_t)size, op);
    return hipGetLastError();
}

// cuda/bn254.cu:1255-1267.  rot holds one entry per column pointer; the
// number of entries is v_n minus the coefficient and separator slots.
hipError_t field_op_batch_mul_sum(void *res, const void *v, const void *rot, int v_n, int n, hipStream_t stream) {
    if (bad_n(n) || !res || v_n < 0 || (v_n && !v)) return hipErrorInvalidValue;
    if (v_n == 0) return hipSuccess;
    k_batch_mul_sum<<<grid_for(n), kThreads, 0, stream>>>((Fr *)res, (const Fr *const *)v, (const int *)rot, v_n,
                                                          (uint32_t)n);
    return hipGetLastError();
}

hipError_t zk_field_mul_zip_on(void *buf, const void *coeff, int coeff_n, int n, hipStream_t stream) {
    if (n <= 0 || coeff_n <= 0 || !buf || !coeff) return hipErrorInvalidValue;
    k_field_mul_zip<<<grid_for(n), kThreads, 0, stream>>>((Fr *)buf, (const Fr *)coeff, (uint32_t)coeff_n, (uint32_t)n);
    return hipGetLastError();
}

hipError_t field_mul_zip(void *buf, const void *coeff, int coeff_n, int n) {
    return zk_field_mul_zip_on(buf, coeff, coeff_n, n, 0);
}

hipError_t zk_permutation_eval_h_p1_on(void *res, const void *first_set, const void *last_set, const void *l0,
                                 const void *l_last, const void *y, int n, hipStream_t stream) {
    if (n <= 0 || !res || !first_set || !last_set || !l0 || !l_last || !y) return hipErrorInvalidValue;
    k_perm_p1<<<grid_for(n), kThreads, 0, stream>>>((Fr *)res, (const Fr *)first_set, (const Fr *)last_set, (const Fr *)l0,
                                               (const Fr *)l_last, (const Fr *)y, (uint32_t)n);
    return hipGetLastError();
}

hipError_t permutation_eval_h_p1(void *res, const void *first_set, const void *last_set, const void *l0,
                                 const void *l_last, const void *y, int n) {
    return zk_permutation_eval_h_p1_on(res, first_set, last_set, l0, l_last, y, n, 0);
}

hipError_t zk_permutation_eval_h_p2_on(void *res, const void *set, const void *l0, const void *l_last, const void *y,
                                 int n_set, int rot, int n, hipStream_t stream) {
    (void)l_last;
    if (bad_n(n) || !res || n_set < 0 || (n_set > 1 && !set) || !l0 || !y) return hipErrorInvalidValue;
    k_perm_p2<<<grid_for(n), kThreads, 0, stream>>>((Fr *)res, (const Fr *const *)set, (const Fr *)l0, (const Fr *)y, n_set,
                                               rot, (uint32_t)n);
    return hipGetLastError();
}

hipError_t permutation_eval_h_p2(void *res, const void *set, const void *l0, const void *l_last, const void *y,
                                 int n_set, int rot, int n) {
    return zk_permutation_eval_h_p2_on(res, set, l0, l_last, y, n_set, rot, n, 0);
}

hipError_t permutation_eval_h_l(void *res, const void *beta, const void *gamma, const void *p, int n,
                                hipStream_t stream) {
    if (n <= 0 || !res || !beta || !gamma || !p) return hipErrorInvalidValue;
    k_perm_l<<<grid_for(n), kThreads, 0, stream>>>((Fr *)res, (const Fr *)beta, (const Fr *)gamma, (const Fr *)p,
                                                   (uint32_t)n);
    return hipGetLastError();
}

hipError_t logup_eval_h(void *res, const void *input_product, const void *input_product_sum, const void *table,
                        const void *multiplicity, const void *z_first, const void *z_last, const void *l0,
                        const void *l_last, const void *l_active_row, const void *y, int rot, int n,
                        hipStream_t stream) {
    if (bad_n(n) || !res || !input_product || !input_product_sum || !table || !multiplicity || !z_first || !z_last ||
        !l0 || !l_last || !l_active_row || !y)
        return hipErrorInvalidValue;
    k_logup_eval_h<<<grid_for(n), kThreads, 0, stream>>>(
        (Fr *)res, (const Fr *)input_product, (const Fr *)input_product_sum, (const Fr *)table,
        (const Fr *)multiplicity, (const Fr *)z_first, (const Fr *)z_last, (const Fr *)l0, (const Fr *)l_last,
        (const Fr *)l_active_row, (const Fr *)y, rot, (uint32_t)n);
    return hipGetLastError();
}

hipError_t logup_eval_h_extra_inputs(void *res, const void *input_product, const void *input_product_sum,
                                     const void *z, const void *l_active_row, const void *y, int rot, int n,
                                     hipStream_t stream) {
    if (bad_n(n) || !res || !input_product || !input_product_sum || !z || !l_active_row || !y)
        return hipErrorInvalidValue;
    k_logup_extra<<<grid_for(n), kThreads, 0, stream>>>((Fr *)res, (const Fr *)input_product,
                                                        (const Fr *)input_product_sum, (const Fr *)z,
                                                        (const Fr *)l_active_row, (const Fr *)y, rot, (uint32_t)n);
    return hipGetLastError();
}

hipError_t logup_eval_h_z_set(void *res, const void *set, const void *l0, const void *l_last, const void *y, int n_set,
                              int rot, int n, hipStream_t stream) {
    (void)l_last;
    if (bad_n(n) || !res || n_set < 0 || (n_set > 1 && !set) || !l0 || !y) return hipErrorInvalidValue;
    k_perm_p2<<<grid_for(n), kThreads, 0, stream>>>((Fr *)res, (const Fr *const *)set, (const Fr *)l0, (const Fr *)y,
                                                    n_set, rot, (uint32_t)n);
    return hipGetLastError();
}

hipError_t logup_eval_h_inputs_product_sum(void *product, void *product_sum, const void *sets, int n_set, int n,
                                           hipStream_t stream) {
    if (n <= 0 || n_set <= 0 || !product || !product_sum || !sets) return hipErrorInvalidValue;
    k_inputs_product_sum<<<grid_for(n), kThreads, 0, stream>>>((Fr *)product, (Fr *)product_sum,
                                                               (const Fr *const *)sets, n_set, (uint32_t)n);
    return hipGetLastError();
}

hipError_t zk_shuffle_eval_h_on(void *res, const void *input, const void *table, const void *z, const void *l0,
                          const void *l_last, const void *l_active_row, const void *y, int rot, int n, hipStream_t stream) {
    if (bad_n(n) || !res || !input || !table || !z || !l0 || !l_last || !l_active_row || !y) return hipErrorInvalidValue;
    k_shuffle<<<grid_for(n), kThreads, 0, stream>>>((Fr *)res, (const Fr *)input, (const Fr *)table, (const Fr *)z,
                                               (const Fr *)l0, (const Fr *)l_last, (const Fr *)l_active_row,
                                               (const Fr *)y, rot, (uint32_t)n);
    return hipGetLastError();
}

hipError_t shuffle_eval_h(void *res, const void *input, const void *table, const void *z, const void *l0,
                          const void *l_last, const void *l_active_row, const void *y, int rot, int n) {
    return zk_shuffle_eval_h_on(res, input, table, z, l0, l_last, l_active_row, y, rot, n, 0);
}

hipError_t zk_shuffle_eval_h_v2_on(void *res, const void *inputs, const void *tables, const void *betas, int group_len,
                             const void *z, const void *l0, const void *l_last, const void *l_active_row,
                             const void *y, int rot, int n, hipStream_t stream) {
    if (bad_n(n) || !res || !inputs || !tables || !betas || group_len <= 0 || !z || !l0 || !l_last || !l_active_row ||
        !y)
        return hipErrorInvalidValue;
    k_shuffle_v2<<<grid_for(n), kThreads, 0, stream>>>((Fr *)res, (const Fr *const *)inputs, (const Fr *const *)tables,
                                                  (const Fr *)betas, group_len, (const Fr *)z, (const Fr *)l0,
                                                  (const Fr *)l_last, (const Fr *)l_active_row, (const Fr *)y, rot,
                                                  (uint32_t)n);
    return hipGetLastError();
}

hipError_t shuffle_eval_h_v2(void *res, const void *inputs, const void *tables, const void *betas, int group_len,
                             const void *z, const void *l0, const void *l_last, const void *l_active_row,
                             const void *y, int rot, int n) {
    return zk_shuffle_eval_h_v2_on(res, inputs, tables, betas, group_len, z, l0, l_last, l_active_row, y, rot, n, 0);
}

// Extension (no reference entry; replaces the per-column field_op /
// permutation_eval_h_l / extended-NTT sequence of src/eval_h.rs:700-840):
// one permutation set's term folded into h in one pass.  v, sigma: device
// arrays of nc <= 16 coset columns; bd: nc Fr (beta * delta^column);
// X: the coset points; rot: the extended-domain shift of one row.
hipError_t zk_permutation_eval_h_set(void *h, const void *z, const void *v, const void *sigma, int nc,
                                     const void *beta, const void *gamma, const void *bd, const void *X,
                                     const void *l_active, const void *y, int rot, int n, hipStream_t stream) {
    if (bad_n(n) || !h || !z || !v || !sigma || nc <= 0 || nc > kMaxPermCols || !beta || !gamma || !bd || !X ||
        !l_active || !y)
        return hipErrorInvalidValue;
    k_perm_set_eval<<<grid_for((uint32_t)n), kThreads, 0, stream>>>(
        (Fr *)h, (const Fr *)z, (const Fr *const *)v, (const Fr *const *)sigma, nc, (const Fr *)beta,
        (const Fr *)gamma, (const Fr *)bd, (const Fr *)X, (const Fr *)l_active, (const Fr *)y, rot, (uint32_t)n);
    return hipGetLastError();
}

// cuda/bn254.cu:1217-1230 (declared at src/cuda/bn254_c.rs:71; the reference
// never calls it).  v, v_c: device arrays of v_n device pointers (v_c entries
// may be null), v_rot: device array of v_n rotations, omegas: w^i for i < n.
// Runs on the null stream, as the reference's does.
hipError_t field_sum(void *res, const void *v, const void *v_c, const void *v_rot, const void *omegas, int v_n,
                     int n) {
    if (bad_n(n) || v_n < 0 || v_n > kMaxSumTerms || !res || (v_n && (!v || !v_c || !v_rot || !omegas)))
        return hipErrorInvalidValue;
    k_field_sum<<<grid_for((uint32_t)n), kThreads, 0, 0>>>((Fr *)res, (const Fr *const *)v, (const Fr *const *)v_c,
                                                          (const int *)v_rot, (const Fr *)omegas, v_n, (uint32_t)n);
    return hipGetLastError();
}

// cuda/bn254.cu:1430-1456 (declared at src/cuda/bn254_c.rs:90; the reference
// never calls it)
hipError_t lookup_eval_h(void *res, const void *input, const void *table, const void *permuted_input,
                         const void *permuted_table, const void *z, const void *l0, const void *l_last,
                         const void *l_active_row, const void *y, const void *beta, const void *gamma, int rot, int n,
                         hipStream_t stream) {
    if (bad_n(n) || !res || !input || !table || !permuted_input || !permuted_table || !z || !l0 || !l_last ||
        !l_active_row || !y || !beta || !gamma)
        return hipErrorInvalidValue;
    k_lookup_eval_h<<<grid_for((uint32_t)n), kThreads, 0, stream>>>(
        (Fr *)res, (const Fr *)input, (const Fr *)table, (const Fr *)permuted_input, (const Fr *)permuted_table,
        (const Fr *)z, (const Fr *)l0, (const Fr *)l_last, (const Fr *)l_active_row, (const Fr *)y, (const Fr *)beta,
        (const Fr *)gamma, rot, (uint32_t)n);
    return hipGetLastError();
}

}  // extern "C"
