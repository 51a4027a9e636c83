// CPU harness for the wave-wide binary GCD (csrc/inv_wave.h), host branch.
#include "inv_wave.h"
namespace {
const uint32_t kR[8] = {0xf0000001u, 0x43e1f593u, 0x79b97091u, 0x2833e848u,
                        0x8181585du, 0xb85045b6u, 0xe131a029u, 0x30644e72u};
const uint32_t kP[8] = {0xd87cfd47u, 0x3c208c16u, 0x6871ca8du, 0x97816a91u,
                        0x8181585du, 0xb85045b6u, 0xe131a029u, 0x30644e72u};
}  // namespace
extern "C" {
int ib_inv(uint32_t *v, const uint32_t *y, int field) {
    return zkinv::bingcd_wave(v, y, field ? kP : kR, field ? 0xe4866389u : 0xefffffffu) ? 1 : 0;
}
int ib_bits() { return zkinv::kBits; }
int ib_steps() { return zkinv::kSteps; }
}
