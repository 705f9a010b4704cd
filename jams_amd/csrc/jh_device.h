// jh_device.h -- device-side building blocks of the gfx950 Heun-LLG engine:
// the Philox4x32-10 counter RNG, the thermostat's normal deviates, the LLG
// right-hand side and the spin renormalisation.
//
// Everything here is compiled with -ffp-contract=off: each +, -, *, / and
// sqrt is one correctly rounded IEEE-754 operation in the order written, so
// the FP64 path reproduces the reference CPU solver's arithmetic bit for bit
// (solvers/cpu_llg_heun.cc:84-144, containers/vec3.h:184-188, :276-283).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace jh {

// ---------------------------------------------------------------------------
// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11).  Multipliers 0xD2511F53,
// 0xCD9E8D57; Weyl key increments 0x9E3779B9, 0xBB67AE85; 10 rounds.
struct u32x4 { uint32_t x, y, z, w; };

// a ^ b ^ k as one v_bitop3_b32 (truth table 0x96, odd parity); the compiler
// issues two v_xor_b32 for the plain expression.
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t k) {
  return __builtin_amdgcn_bitop3_b32(a, b, k, 0x96);
}
// The whole 64-bit product of a round in one v_mad_u64_u32: the empty asm
// keeps the compiler from splitting it into v_mul_lo_u32 + v_mul_hi_u32 (each
// as slow as the v_mad).
__device__ __forceinline__ uint64_t mul_wide(uint32_t m, uint32_t x) {
  uint64_t p = (uint64_t)m * x;
  asm("" : "+v"(p));
  return p;
}
__device__ __forceinline__ uint32_t lo32(uint64_t v) { return (uint32_t)v; }
__device__ __forceinline__ uint32_t hi32(uint64_t v) { return (uint32_t)(v >> 32); }

// The two Philox blocks of a spin's draw: counter (spin, call, step lo, step
// hi), call = 0 and 1, key (k0, k1).  Their counters differ in one word only,
// and the step is the same in every lane, so the first three rounds are
// written out: the products that both calls share are formed once, and those
// of the step (with a wave-uniform key) on the scalar unit.  33 vector
// multiplies instead of 40.
__device__ __forceinline__ void philox4x32_10_pair(uint32_t spin, uint64_t step, uint32_t k0,
                                                   uint32_t k1, u32x4 (&c)[2]) {
  constexpr uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u, W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
  // round 1: (spin, call, step lo, step hi)
  const uint64_t a0 = mul_wide(M0, spin);
  const uint64_t a1 = (uint64_t)M1 * lo32(step);
  const uint32_t az = hi32(a0) ^ (hi32(step) ^ k1);  // word 2, either call
  // round 2: (hi(a1) ^ call ^ k0, lo(a1), az, lo(a0))
  const uint64_t b1 = mul_wide(M1, az);
  const uint32_t bx = hi32(b1) ^ (lo32(a1) ^ (k0 + W0));  // word 0, either call
  // round 3: (bx, lo(b1), word 2 of each call, lo of each call's M0 product)
  const uint64_t c0 = mul_wide(M0, bx);
#pragma unroll
  for (int call = 0; call < 2; ++call) {
    const uint64_t b0 = (uint64_t)M0 * (hi32(a1) ^ (uint32_t)call ^ k0);
    const uint64_t c1 = mul_wide(M1, lo32(a0) ^ (hi32(b0) ^ (k1 + W1)));
    c[call] = u32x4{xor3(hi32(c1), lo32(b1), k0 + 2 * W0), lo32(c1),
                    hi32(c0) ^ (lo32(b0) ^ (k1 + 2 * W1)), lo32(c0)};
  }
  k0 += 3 * W0;
  k1 += 3 * W1;
#pragma unroll
  for (int r = 3; r < 10; ++r) {
#pragma unroll
    for (int call = 0; call < 2; ++call) {
      const uint64_t p0 = mul_wide(M0, c[call].x), p1 = mul_wide(M1, c[call].z);
      c[call] = u32x4{xor3(hi32(p1), c[call].y, k0), lo32(p1), xor3(hi32(p0), c[call].w, k1),
                      lo32(p0)};
    }
    k0 += W0;
    k1 += W1;
  }
}

// ---------------------------------------------------------------------------
// Quotients and square roots of operands whose exponents are known to be
// moderate.  The compiler's FP64 division and square root scale their
// operands, fix up special values and unscale; the steps between (reciprocal
// or reciprocal square root estimate, Newton steps, one residual correction)
// are these, and with moderate operands the scaling is by 1, so the results
// are the same bit for bit.  Each caller says why its operands qualify.
__device__ __forceinline__ double rcp_mid(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
}
// n / d from r = rcp_mid(d)
__device__ __forceinline__ double quot_mid(double n, double d, double r) {
  const double q = n * r;
  return __builtin_fma(__builtin_fma(-d, q, n), r, q);
}
__device__ __forceinline__ double sqrt_mid(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}

// Coefficients of the draw's series: the odd atanh series of the log
// (1/21 .. 1/3), the sine's and the cosine's Taylor series.  They are read
// through the scalar unit into SGPRs, which an FP64 multiply-add takes as its
// addend; as literals each one costs two moves into vector registers per use
// (73 of the draw's 384 vector instructions).
static __constant__ double kNoiseCoef[28] = {
    1.0 / 21.0, 1.0 / 19.0, 1.0 / 17.0, 1.0 / 15.0, 1.0 / 13.0, 1.0 / 11.0, 1.0 / 9.0, 1.0 / 7.0,
    1.0 / 5.0, 1.0 / 3.0,
    -1.0 / 121645100408832000.0, 1.0 / 355687428096000.0, -1.0 / 1307674368000.0,
    1.0 / 6227020800.0, -1.0 / 39916800.0, 1.0 / 362880.0, -1.0 / 5040.0, 1.0 / 120.0, -1.0 / 6.0,
    1.0 / 6402373705728000.0, -1.0 / 20922789888000.0, 1.0 / 87178291200.0, -1.0 / 479001600.0,
    1.0 / 3628800.0, -1.0 / 40320.0, 1.0 / 720.0, -1.0 / 24.0, 0.5};
typedef const __attribute__((address_space(4))) double *NoiseCoef;

// One Horner series of `terms` coefficients from index `first`, at the
// arguments z[0] and z[1] of a draw's two blocks.  Both arguments share the
// coefficients; the asm statements have them read here (hoisted, the LINE
// kernels' scalar registers would spill) and kept in scalar registers past
// their last use (the compiler otherwise copies a coefficient into vector
// registers there and accumulates onto the copy).
template <int first, int terms>
__device__ __forceinline__ void noise_series(const double (&z)[2], double (&p)[2]) {
  NoiseCoef C = (NoiseCoef)kNoiseCoef + first;
  asm volatile("" : "+s"(C));
  p[0] = p[1] = C[0];
#pragma unroll
  for (int k = 1; k < terms; ++k) {
    const double c = C[k];
    p[0] = __builtin_fma(p[0], z[0], c);
    p[1] = __builtin_fma(p[1], z[1], c);
    asm volatile("" : : "s"(c));
  }
}

// The double with sign and exponent bits `top` and the top 52 bits of hi:lo
// as its significand.
__device__ __forceinline__ double with_bits52(uint32_t top, uint32_t hi, uint32_t lo) {
  return __hiloint2double((int)(top | (hi >> 12)), (int)__builtin_amdgcn_alignbit(hi, lo, 12));
}

// r = sqrt(-2 log u) for words x:y of both blocks: u = (2k + 1) 2^-53 in
// (0, 1) with k the top 52 bits of x:y, which is (1 + k 2^-52) - (1 - 2^-53)
// exactly.  log u: u = m 2^e, m in [sqrt(1/2), sqrt(2)), log m = 2 atanh(s)
// with s = (m-1)/(m+1) summed as the odd series to s^21 by fused multiply-add
// Horner steps.  Every operation is one correctly rounded IEEE-754 operation
// (fma included), so the CPU oracle reproduces the bits.  The quotient's
// divisor is in (1.7, 2.5) and its dividend is 0 or at least 2^-53 in
// magnitude; -2 log u is in (2^-53, 74).
__device__ __forceinline__ void noise_radius(const u32x4 (&w)[2], double (&r)[2]) {
  double s[2], z[2], p[2], e[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const double u = with_bits52(0x3FF00000u, w[b].x, w[b].y) - 0x1.fffffffffffffp-1;
    const uint32_t uh = (uint32_t)__double2hiint(u);
    int ex = (int)(uh >> 20) - 1023;
    double m = __hiloint2double((int)((uh & 0x000FFFFFu) | 0x3FF00000u), __double2loint(u));
    if (m > 1.4142135623730951) { m = m * 0.5; ex = ex + 1; }
    const double f = m - 1.0;
    const double d = 2.0 + f;
    s[b] = quot_mid(f, d, rcp_mid(d));
    z[b] = s[b] * s[b];
    e[b] = (double)ex;
  }
  noise_series<0, 10>(z, p);
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const double s2 = 2.0 * s[b];
    const double lm = __builtin_fma(s2, z[b] * p[b], s2);
    r[b] = sqrt_mid(-2.0 * __builtin_fma(e[b], 0.6931471805599453, lm));
  }
}

// cos(2 pi u) of both blocks and sin(2 pi u) of the first, u in (0, 1) as
// above from words z:w: 4u = (4 + 4k 2^-52) - (4 - 2^-51), exactly, whose
// nearest integer q is read off the top bits (4u is never half-way between
// integers); exact quadrant reduction, Taylor series on [-pi/4, pi/4] by fma
// Horner steps, exact quadrant rotation.
__device__ __forceinline__ void noise_sincos2pi(const u32x4 (&w)[2], double (&c)[2], double &s0) {
  double x[2], z[2], ps[2], pc[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const double v = with_bits52(0x40100000u, w[b].z, w[b].w) - 0x1.fffffffffffffp+1;
    x[b] = (v - rint(v)) * 1.5707963267948966;
    z[b] = x[b] * x[b];
  }
  noise_series<10, 9>(z, ps);
  noise_series<19, 9>(z, pc);
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const double sn = __builtin_fma(x[b], z[b] * ps[b], x[b]);
    const double cs = __builtin_fma(-z[b], pc[b], 1.0);
    // (c, s) = (cs, sn), (-sn, cs), (-cs, -sn), (sn, -cs) for q = 0 .. 3
    const uint32_t q = (w[b].z + 0x20000000u) >> 30;
    const double a = (q & 1u) ? sn : cs;
    c[b] = __hiloint2double(__double2hiint(a) ^ (int)(((q + 1u) & 2u) << 30), __double2loint(a));
    if (b == 0) {
      const double t = (q & 1u) ? cs : sn;
      s0 = __hiloint2double(__double2hiint(t) ^ (int)((q & 2u) << 30), __double2loint(t));
    }
  }
}

// Three standard normal deviates of the thermostat stream for (seed, step,
// spin): two Philox blocks with counter (spin, call, step lo, step hi) and
// key (seed lo, seed hi), Box-Muller on each block.  The stream's counter
// holds spin's high word beside the call; it is 0 here (a context holds at
// most 2^31 spins).  step is the same in every lane.
// 16.8 M draws written to memory: 203 -> 151 us against the form with literal
// coefficients, separate blocks, integer-to-double conversions and the
// compiler's division and square root, bit for bit.
__device__ __forceinline__ void normals3(uint64_t seed, uint64_t step, uint32_t spin, double &z0,
                                         double &z1, double &z2) {
  u32x4 w[2];
  philox4x32_10_pair(spin, step, lo32(seed), hi32(seed), w);
  double r[2], c[2], s0;
  noise_radius(w, r);
  noise_sincos2pi(w, c, s0);
  z0 = r[0] * c[0];
  z1 = r[0] * s0;
  z2 = r[1] * c[1];
}

// rhs = -gyro (s x h + alpha s x (s x h)) with the reference's grouping
// (solvers/cpu_llg_heun.cc:89; containers/vec3.h:184-188).
__device__ __forceinline__ void llg_rhs(double s0, double s1, double s2, double h0, double h1,
                                        double h2, double gyro, double alpha, double &r0,
                                        double &r1, double &r2) {
  const double c0 = s1 * h2 - s2 * h1;
  const double c1 = s2 * h0 - s0 * h2;
  const double c2 = s0 * h1 - s1 * h0;
  const double d0 = s1 * c2 - s2 * c1;
  const double d1 = s2 * c0 - s0 * c2;
  const double d2 = s0 * c1 - s1 * c0;
  const double g = -gyro;
  r0 = g * (c0 + alpha * d0);
  r1 = g * (c1 + alpha * d1);
  r2 = g * (c2 + alpha * d2);
}

// v / |v| as one reciprocal and three products (the FP32-field form, whose
// arithmetic need not reproduce the reference's operation for operation):
// within 1.5 ulp of unit_vector, two FP64 divisions fewer.
__device__ __forceinline__ void unit_vector_rcp(double &v0, double &v1, double &v2) {
  const double len = sqrt(v0 * v0 + v1 * v1 + v2 * v2);
  if (fabs(len) <= 2.220446049250313e-16) return;
  const double r = 1.0 / len;
  v0 = v0 * r;
  v1 = v1 * r;
  v2 = v2 * r;
}

// unit_vector (containers/vec3.h:276-283): v / |v| unless |v| <= DBL_EPSILON.
__device__ __forceinline__ void unit_vector(double &v0, double &v1, double &v2) {
  const double len = sqrt(v0 * v0 + v1 * v1 + v2 * v2);
  if (fabs(len) <= 2.220446049250313e-16) return;
  v0 = v0 / len;
  v1 = v1 / len;
  v2 = v2 / len;
}

// XCD-aware block order: hardware hands consecutive workgroups to the 8
// XCDs round robin; remap so each XCD walks one contiguous range of spins and
// neighbour gathers hit its own L2.
__device__ __forceinline__ int64_t xcd_block(int64_t bid, int64_t nb) {
  const int64_t q = nb >> 3, r = nb & 7;
  const int64_t x = bid & 7, k = bid >> 3;
  const int64_t start = x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q;
  return start + k;
}

}  // namespace jh
