// CPU harness for the row arithmetic of the eval_h folds (csrc/evalh_rows.h)
// and its oracle, the same rows in full-width products reduced after every
// step (csrc/ff.h).  v: the row's values, c: the challenges; each fold names
// what it takes from them.
#include <stddef.h>

#include "evalh_rows.h"

using namespace zk;

namespace {

enum { PERM_P1, PERM_P2, LOGUP, LOGUP_EXTRA, SHUFFLE, PERM_SET, GATES };

Fr lazy(int which, const Fr *v, const Fr *c, int cols) {
    const F29 y = hi(c[0]);
    switch (which) {
        case PERM_P1: return perm_p1_row(v, v + 1, v + 2, v + 3, v + 4, 0, fe_one<FrParams>(), y);
        case PERM_P2: {
            F29 t = lo(v[0]);
            for (int j = 0; j < cols; j++) t = perm_p2_step(t, v[2 + 2 * j], v[3 + 2 * j], hi(v[1]), y);
            return f29_to_fr(t);
        }
        case LOGUP:  // z and its rotation are neighbours
            return logup_row(v, v + 6, v + 7, v + 4, v + 5, v + 1, v + 3, v + 8, v + 9, v + 10, 0, 1, y);
        case LOGUP_EXTRA: return logup_extra_row(v, v + 3, v + 4, v + 1, v + 5, 0, 1, y);
        case SHUFFLE: {
            F29 l = lo(v[6] + c[1]), r = lo(v[7] + c[1]);
            for (int j = 1; j < cols; j++) {
                l = shuffle_factor(l, v[6 + 2 * j], hi(c[1 + j]));
                r = shuffle_factor(r, v[7 + 2 * j], hi(c[1 + j]));
            }
            return shuffle_fold(v[0], l, r, v[1], v[2], v[3], v[4], v[5], y);
        }
        case PERM_SET: {
            F29 l = lo(v[1]), r = lo(v[2]);
            for (int j = 0; j < cols; j++) {
                const F29 vg = hi(v[5 + 2 * j] + c[2]);
                l = perm_set_factor(l, vg, hi(c[1]), hi(v[6 + 2 * j]));
                r = perm_set_factor(r, vg, hi(c[3 + j]), hi(v[3]));
            }
            return perm_set_fold(v[0], l, r, v[4], y);
        }
        default: {
            F29 acc = gate_first(hi(v[1]), v[2], v[3], v[4]);
            for (int j = 0; j < cols; j++) acc = gate_step(acc, hi(v[1]), v[5 + 2 * j], v[6 + 2 * j], y);
            return gate_last(acc, v[0]);
        }
    }
}

Fr full(int which, const Fr *v, const Fr *c, int cols) {
    const Fr y = c[0], one = fe_one<FrParams>();
    switch (which) {
        case PERM_P1: return (v[0] * y + (one - v[1]) * v[3]) * y + (v[2] * v[2] - v[2]) * v[4];
        case PERM_P2: {
            Fr t = v[0];
            for (int j = 0; j < cols; j++) t = t * y + (v[2 + 2 * j] - v[3 + 2 * j]) * v[1];
            return t;
        }
        case LOGUP:
            return ((v[0] * y + v[8] * v[1]) * y + v[9] * v[3]) * y +
                   (((v[2] - v[1]) * v[4] + v[5]) * v[6] - v[4] * v[7]) * v[10];
        case LOGUP_EXTRA: return v[0] * y + ((v[2] - v[1]) * v[3] - v[4]) * v[5];
        case SHUFFLE: {
            Fr l = v[6] + c[1], r = v[7] + c[1];
            for (int j = 1; j < cols; j++) {
                l = l * (v[6 + 2 * j] + c[1 + j]);
                r = r * (v[7 + 2 * j] + c[1 + j]);
            }
            return ((v[0] * y + v[3] * (one - v[1])) * y + v[4] * (v[1] * v[1] - v[1])) * y + (r * v[2] - l * v[1]) * v[5];
        }
        case PERM_SET: {
            Fr l = v[1], r = v[2];
            for (int j = 0; j < cols; j++) {
                const Fr vg = v[5 + 2 * j] + c[2];
                l = l * (vg + c[1] * v[6 + 2 * j]);
                r = r * (vg + c[3 + j] * v[3]);
            }
            return v[0] * y + v[4] * (l - r);
        }
        default: {
            Fr acc = v[1] * v[2] + v[3] - v[4];
            for (int j = 0; j < cols; j++) acc = acc * y + (v[5 + 2 * j] * v[1] - v[6 + 2 * j]);
            return v[0] * acc;
        }
    }
}

}  // namespace

extern "C" {
// rows of `width` values; out and exp receive one value per row
void folds_run(int which, const void *rows, int n, int width, const void *challenges, int cols, void *out, void *exp) {
    const Fr *v = (const Fr *)rows, *c = (const Fr *)challenges;
    for (int i = 0; i < n; i++) {
        ((Fr *)out)[i] = lazy(which, v + (size_t)i * width, c, cols);
        ((Fr *)exp)[i] = full(which, v + (size_t)i * width, c, cols);
    }
}
}
