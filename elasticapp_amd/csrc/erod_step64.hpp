// The FP64 step's director update and curvature, shared by the op-by-op
// kernels (erod_ops.hip) and the fused FP64 kernel (erod_fused64.hip), so that
// both round the same way.  Included by units built with -ffp-contract=off.
#pragma once

#include "erod_common.hpp"
#include "erod_math.hpp"

namespace erod {
  namespace step64 {

    // ---- division and square root without their special cases -------------------
    //
    // An FP64 division is 11 instructions: the divisor's reciprocal by Newton's
    // iteration from v_rcp_f64, the quotient by it, one correction from the
    // exact remainder (Markstein), and four more that scale extreme operands
    // and patch special results.  Where no operand is extreme the scaling is by
    // one, and the same steps without it give the same bits (a zero quotient
    // may lose its sign); several numerators over one divisor then share the
    // iteration, and a constant divisor's can be made once.  A square root is
    // 18 instructions of which 10 remain.  kPlain code below takes these forms
    // and notes in a Range whether every operand allowed them; a wave in which
    // one did not computes the terms again with the full forms.  The FP64 step is
    // bound by VALU issue: 1,190 -> 970 instructions of the fused one, 1,024 rods
    // of 64 elements 1.65 -> 1.50 ms per 500 steps, 2,048 ragged rods 8.4 -> 7.1 ms
    // per 300, op-by-op steps of 248,188 elements 14.4 -> 13.5 us each.

    // operands met so far: bad if a divisor or radicand lies outside 2^-100 ...
    // 2^100, a numerator other than zero below 2^-800, or one above 2^600
    struct Range {
      // smallest exponent e, 2^(e-1) <= |n| < 2^e, denormal numbers' true one
      // among them; a zero's, an infinity's and a NaN's is 0
      int least = 0;
      bool out = false;

      __device__ __forceinline__ static uint32_t high(double v) { return static_cast<uint32_t>(__double2hiint(v)); }
      __device__ __forceinline__ void divisor(double d) {
        out |= high(d) - ((1023u - 100u) << 20) >= (200u << 20);  // (a negative one, an infinity or a NaN too)
      }
      // a numerator known not to be large
      __device__ __forceinline__ void numerator(double n) { least = min(least, __builtin_amdgcn_frexp_exp(n)); }
      // the largest magnitude of numerators that may be
      __device__ __forceinline__ void largest(double a) { out |= !(a < 0x1p600); }
      __device__ __forceinline__ bool bad() const { return out || least < -799; }
    };

    // a divisor with its reciprocal
    struct Divisor {
      double d, r;
    };

    template <bool kPlain>
    __device__ __forceinline__ Divisor divisor(double d) {
      if constexpr (!kPlain) return {d, 0.0};
      double r = __builtin_amdgcn_rcp(d);
      r = __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
      r = __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
      return {d, r};
    }

    template <bool kPlain>
    __device__ __forceinline__ double over(double n, const Divisor& by) {
      if constexpr (!kPlain) return n / by.d;
      const double q = n * by.r;
      return __builtin_fma(__builtin_fma(-by.d, q, n), by.r, q);
    }

    template <bool kPlain>
    __device__ __forceinline__ double root(double x) {
      if constexpr (!kPlain) return sqrt(x);
      const double y = __builtin_amdgcn_rsq(x);
      double g = x * y, h = 0.5 * y;
      const double e = __builtin_fma(-h, g, 0.5);
      g = __builtin_fma(g, e, g);
      h = __builtin_fma(h, e, h);
      g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
      return __builtin_fma(__builtin_fma(-g, g, x), h, g);
    }

    // whether any lane of the wave has `b`
    __device__ __forceinline__ bool any(bool b) { return __ballot(b) != 0ull; }

    // the rotation exp(-[u]x), u = c w: its axis and the sine and cosine of
    // its angle
    struct Rotation {
      double u[3], beta, c_alpha;
    };

    __device__ __forceinline__ Rotation rotation(const double w[3], double c) {
      Rotation o;
      double u0 = c * w[0], u1 = c * w[1], u2 = c * w[2];
      const double theta = sqrt(u0 * u0 + u1 * u1 + u2 * u2);
      math::sincos(theta, &o.beta, &o.c_alpha);
      const double den = theta + 1e-14;
      // (|u| <= theta: no numerator is large when den is not)
      Range g;
      g.divisor(den);
      g.numerator(u0);
      g.numerator(u1);
      g.numerator(u2);
      if (any(g.bad())) {
        u0 /= den;
        u1 /= den;
        u2 /= den;
      } else {
        const Divisor by = divisor<true>(den);
        u0 = over<true>(u0, by);
        u1 = over<true>(u1, by);
        u2 = over<true>(u2, by);
      }
      o.u[0] = u0;
      o.u[1] = u1;
      o.u[2] = u2;
      return o;
    }

    // Q <- exp(-[u]x) Q
    __device__ __forceinline__ void rotate(double q[9], const Rotation& o) {
      const double u0 = o.u[0], u1 = o.u[1], u2 = o.u[2], beta = o.beta, c_alpha = o.c_alpha;
      const double alpha = 1.0 - c_alpha;
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const double a = q[j], b = q[3 + j], cc = q[6 + j];
        const double com = a * u0 + b * u1 + cc * u2;
        q[j] = c_alpha * a + alpha * u0 * com + beta * (b * u2 - cc * u1);
        q[3 + j] = c_alpha * b + alpha * u1 * com + beta * (cc * u0 - a * u2);
        q[6 + j] = c_alpha * cc + alpha * u2 * com + beta * (a * u1 - b * u0);
      }
    }

    // Q <- exp(-[u]x) Q with u = c w: SO3AddAssign<scalar>
    // (SO3PrimitiveAddAssign/Scalar.hpp:25-96)
    __device__ __forceinline__ void so3_update(double q[9], const double w[3], double c) {
      rotate(q, rotation(w, c));
    }

    // math::acos, for angles below 60 degrees with a root and a division that
    // need no range test: z = (1 - x) / 2 is zero (then y is no number, and the
    // result zero) or 2^-54 and more, the remainder z - h h a multiple of 2^-104.
    // With the quotient below: 1,024 rods of 64 elements, 500 steps 1.667 -> 1.614
    // ms, a pass with the state read back.
    __device__ __forceinline__ double acos(double x) {
      if (!(x > 0.5 && x <= 1.0)) return math::acos(x);
      const double z = (1.0 - x) * 0.5;
      const double y = root<true>(z);
      const double t = math::asin_tail(y, z);
      if (!(y > 0.0)) return 0.0;
      const double h = math::bits_head26(y);
      const double c = over<true>(z - h * h, divisor<true>(y + h));
      return 2.0 * (h + (c + t));
    }

    // curvature between neighbouring directors: InvRotateDivideOp<scalar>
    // (InvRotateDivide/Scalar.hpp:26-110)
    template <bool kPlain>
    __device__ __forceinline__ void curvature(const double qc[9], const double qn[9], const Divisor& D0, double kap[3]) {
      const double tr = qc[0] * qn[0] + qc[1] * qn[1] + qc[2] * qn[2] + qc[3] * qn[3] + qc[4] * qn[4] +
                        qc[5] * qn[5] + qc[6] * qn[6] + qc[7] * qn[7] + qc[8] * qn[8];
      const double theta = acos(0.5 * tr - (0.5 + 1e-10));
      // (theta is zero, NaN or 2^-27 to pi, the sine 2^-54 and more either way:
      // their quotient is zero, NaN or 1/2 to 2^54)
      const double st = over<kPlain>(over<true>(0.5 * theta, divisor<true>(math::sin(theta + 1e-14))), D0);
      kap[0] = st * (-qc[3] * qn[6] - qc[4] * qn[7] - qc[5] * qn[8] + qc[6] * qn[3] + qc[7] * qn[4] + qc[8] * qn[5]);
      kap[1] = st * (qc[0] * qn[6] + qc[1] * qn[7] + qc[2] * qn[8] - qc[6] * qn[0] - qc[7] * qn[1] - qc[8] * qn[2]);
      kap[2] = st * (-qc[0] * qn[3] - qc[1] * qn[4] - qc[2] * qn[5] + qc[3] * qn[0] + qc[4] * qn[1] + qc[5] * qn[2]);
    }

    // ramp of an end force (Rampup.hpp:95-150, 302-330)
    __device__ __forceinline__ double ramp_value(int kind, double t, double start, double interval) {
      if (kind == EROD_RAMP_NONE) return 1.0;
      if (t < start) return 0.0;
      if (t > start + interval) return 1.0;
      if (kind == EROD_RAMP_LINEAR) return (t - start) / interval;
      const double s = 2.0 * ((t - start) / interval) - 1.0;
      return 0.5 * (s + (1.0 + (math::sin(M_PI * s) / M_PI)));
    }

  }  // namespace step64
}  // namespace erod
