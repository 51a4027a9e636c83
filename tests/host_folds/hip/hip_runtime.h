// What the arithmetic headers need of the HIP runtime header, for a host compiler.
#pragma once
#define __device__
#define __host__
#define __forceinline__ inline
#define __noinline__
struct uint4 {
    unsigned x, y, z, w;
};
inline uint4 make_uint4(unsigned x, unsigned y, unsigned z, unsigned w) { return uint4{x, y, z, w}; }
inline unsigned host_addc(unsigned a, unsigned b, unsigned c, unsigned *co) {
    const unsigned long long s = (unsigned long long)a + b + c;
    *co = (unsigned)(s >> 32);
    return (unsigned)s;
}
inline unsigned host_subc(unsigned a, unsigned b, unsigned c, unsigned *bo) {
    const unsigned long long s = (unsigned long long)a - b - c;
    *bo = (unsigned)(s >> 63);
    return (unsigned)s;
}
#define __builtin_addc host_addc
#define __builtin_subc host_subc
