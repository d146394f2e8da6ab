// The FP64 step's director update and curvature, shared by the op-by-op
// kernels (erod_ops.hip) and the fused FP64 kernel (erod_fused64.hip), so that
// both round the same way.  Included by units built with -ffp-contract=off.
#pragma once

#include "erod_common.hpp"
#include "erod_math.hpp"

namespace erod {
  namespace step64 {

    // Q <- exp(-[u]x) Q with u = c w: SO3AddAssign<scalar>
    // (SO3PrimitiveAddAssign/Scalar.hpp:25-96)
    __device__ __forceinline__ void so3_update(double q[9], const double w[3], double c) {
      double u0 = c * w[0], u1 = c * w[1], u2 = c * w[2];
      const double theta = sqrt(u0 * u0 + u1 * u1 + u2 * u2);
      double beta, c_alpha;
      math::sincos(theta, &beta, &c_alpha);
      const double alpha = 1.0 - c_alpha;
      const double den = theta + 1e-14;
      u0 /= den;
      u1 /= den;
      u2 /= den;
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const double a = q[j], b = q[3 + j], cc = q[6 + j];
        const double com = a * u0 + b * u1 + cc * u2;
        q[j] = c_alpha * a + alpha * u0 * com + beta * (b * u2 - cc * u1);
        q[3 + j] = c_alpha * b + alpha * u1 * com + beta * (cc * u0 - a * u2);
        q[6 + j] = c_alpha * cc + alpha * u2 * com + beta * (a * u1 - b * u0);
      }
    }

    // curvature between neighbouring directors: InvRotateDivideOp<scalar>
    // (InvRotateDivide/Scalar.hpp:26-110)
    __device__ __forceinline__ void curvature(const double qc[9], const double qn[9], double D0, double kap[3]) {
      const double tr = qc[0] * qn[0] + qc[1] * qn[1] + qc[2] * qn[2] + qc[3] * qn[3] + qc[4] * qn[4] +
                        qc[5] * qn[5] + qc[6] * qn[6] + qc[7] * qn[7] + qc[8] * qn[8];
      const double theta = math::acos(0.5 * tr - (0.5 + 1e-10));
      const double st = 0.5 * theta / math::sin(theta + 1e-14) / D0;
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
