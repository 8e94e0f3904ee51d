// sincos_unit.h -- sin and cos of pi x in FP32 for the facet rotors of the FP32 paths.
#pragma once
#include <stdint.h>

namespace bam {

// |x| <= 1: x = n/2 + r exactly, |r| <= 1/4, and polynomials in r^2, least-squares fits whose
// coefficients are rounded to FP32 one after the other, the rest refitted each time (the sine's
// constant term completes pi beyond its FP32 value, so the leading product carries it).
// Within 0.68 ulp (sine) and 0.88 ulp (cosine) of the true values for |x| <= 1/4; about 24
// instructions, where sincospif spends 45 on arguments that it has to reduce and classify first.
//
// A rotor multiplies every visibility, so an error of its amplitude that is the same for all phases
// scales the image and does not average out.  Over uniform phases (4 M, extended precision) the
// mean amplitude lies 0.6e-11 from 1, sincospif's 8.6e-11; the worst mean over a 128th of the
// circle is 0.9e-9 against 1.4e-9.  Coefficients fitted for the worst ulp alone left 2.1e-9
// (5.4e-9 at an eighth of a turn), the rounding of the cosine's first coefficient.
__device__ __forceinline__ void sincospi_unit(float x, float *sn, float *cs) {
    const float n = __builtin_rintf(2.0f * x);
    const float r = __builtin_fmaf(n, -0.5f, x);
    const float z = r * r;
    float u = __builtin_fmaf(z, 0x1.497906p-4f, -0x1.32bfc6p-1f);
    u = __builtin_fmaf(u, z, 0x1.466b98p+1f);
    u = __builtin_fmaf(u, z, -0x1.4abbcep+2f);
    u = __builtin_fmaf(u, z, -0x1.799212p-24f);
    const float s = __builtin_fmaf(0x1.921fb6p+1f, r, r * u);
    float v = __builtin_fmaf(z, 0x1.d60294p-3f, -0x1.55b6b2p+0f);
    v = __builtin_fmaf(v, z, 0x1.03c1b6p+2f);
    v = __builtin_fmaf(v, z, -0x1.3bd3ccp+2f);
    const float c = __builtin_fmaf(v, z, 1.0f);
    const uint32_t q = (uint32_t)(int)n;
    uint32_t sb, cb;
    __builtin_memcpy(&sb, &s, 4);
    __builtin_memcpy(&cb, &c, 4);
    const uint32_t a = ((q & 1u) ? cb : sb) ^ ((q & 2u) << 30);
    const uint32_t b = ((q & 1u) ? sb : cb) ^ (((q + 1u) & 2u) << 30);
    __builtin_memcpy(sn, &a, 4);
    __builtin_memcpy(cs, &b, 4);
}

}  // namespace bam
