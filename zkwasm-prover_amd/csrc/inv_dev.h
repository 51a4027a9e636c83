// One Fr inversion by a whole wave (device side of inv_wave.h).
#pragma once
#include "ff.h"
#include "inv_wave.h"

namespace zk {

// a^-1 in the Montgomery domain for a value that is the same in all 64 (active)
// lanes; 0 -> 0.  The result is checked by one product, as fe_inv's; should
// that fail, the one-bit-at-a-time extended Euclid gives it.
__device__ __forceinline__ Fr fr_inv_wave(const Fr &a) {
    uint32_t v[8];
    const bool ok = zkinv::bingcd_wave(v, a.v, FrParams::M, FrParams::INV);
    const Fr r = fe_from_raw<FrParams>(v) * fe_from_raw<FrParams>(FrParams::INVC);
    if (ok && fe_eq<FrParams>(a * r, fe_one<FrParams>())) return r;
    return fe_inv_raw<FrParams>(a) * fe_from_raw<FrParams>(FrParams::R3);
}

}  // namespace zk
