// The plain FP64 path: the reference's block timestep over every slot of the
// ghost-padded block (ghosts included), one kernel per call of its stepper,
// in the reference's evaluation order.  This file is built with
// -ffp-contract=off so that every product and sum is rounded on its own, as
// in the CPU restatement it is checked against.  acos, sin and cos are the
// library's own (erod_math.hpp), so that these kernels and a CPU build of the
// restatement with the same functions compute the same bits.
//
// Reference operators (paths under elastica/Systems/CosseratRods/):
//   spanwise geometry   Components/Geometry/detail/CosseratRodSpanwiseGeometry.hpp:578-664
//   radius              Components/Geometry/detail/CosseratRodCrossSectionInterface.hpp:445-456
//   internal loads      Components/Elasticity/WithDiagonalLinearHyperElasticModel.hpp:197-238
//   internal torques    Components/Elasticity/WithDiagonalLinearHyperElasticModel.hpp:246-391
//   damping             Components/Elasticity/detail/ExplicitDampingAdapterFacade.hpp:177-235
//   accelerations       Components/Kinematics/WithRodKinematics.hpp:683-714
//   operators           Traits/Operations/BlazeBackend/OpsTraits.hpp:88-346
//   director update     elastica/Systems/States/Expressions/backends/blaze/SO3PrimitiveAddAssign/Scalar.hpp:25-96
//
// The reference evaluates an operator at a time, each a pass over the block's
// arrays.  Here one thread takes slot k (node k, element k, Voronoi region k)
// through all of them: an operator needs only values of slots k - 1 ... k + 2,
// so its temporaries stay in registers.  Ghost slots take part like any other
// and get their ghost values where the reference refills them, so every field
// ends with the bits the pass-by-pass evaluation leaves in it, ghosts included.
#include "erod_common.hpp"
#include "erod_step64.hpp"

namespace erod {
  namespace {

#define GRID_STRIDE(i, n) \
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < (n); i += (uint64_t)gridDim.x * blockDim.x)

    __global__ void k_fill(double* __restrict__ p, double val, uint64_t n) {
      GRID_STRIDE(i, n) p[i] = val;
    }

    // fill_ghosts_for (Block.hpp:658-690): ghost node g, deficit d -> slots g, g-1, ..., g-d+1
    __global__ void k_fill_ghosts(double* __restrict__ p, const uint64_t* __restrict__ gn, uint64_t n_gn,
                                  int deficit, uint64_t slots, int ncomp, double ghost) {
      GRID_STRIDE(i, n_gn * (uint64_t)deficit) {
        const uint64_t g = gn[i / deficit];
        const uint64_t idx = g - (i % deficit);
        if (ghost < -1.0) {
          const double gd[9] = {0.8, 0.6, 0.0, 0.0, 0.0, 1.0, 0.6, -0.8, 0.0};
          for (int c = 0; c < 9; ++c) p[c * slots + idx] = gd[c];
        } else {
          for (int c = 0; c < ncomp; ++c) p[c * slots + idx] = ghost;
        }
      }
    }

    // ---- one slot of the block timestep ------------------------------------------

    // the fields of a block the kernels below read and write
    struct Lines {
      double *x, *v, *acc, *f_int, *f_ext;                                   // node, 3 lines
      const double *m, *im, *gf;                                             // node
      double *q;                                                             // element, 9 lines
      double *w, *alpha, *t, *sigma, *stress, *tau_int, *tau_ext, *d1, *d2;  // element, 3 lines
      const double *S, *J, *iJ, *sigma0;                                     // element, 3 lines
      double *l, *e, *r;                                                     // element
      const double *l0, *vol, *gt;                                           // element
      double *kappa, *couple, *dv;                                           // Voronoi, 3 lines
      const double *kappa0, *B;                                              // Voronoi, 3 lines
      double *D, *eps;                                                       // Voronoi
      const double* D0;                                                      // Voronoi
    };

    // the constants of slot k: node k, element k, Voronoi region k, and the
    // mass of node k + 1
    struct SlotConst {
      double m, mn, im, gf, l0, gt, S[3], sigma0[3], J[3], iJ[3], D0, kappa0[3], B[3];
      double il0, iD0;  // of step64::divisor
    };

    // bits of a slot's place: ghost node / element / Voronoi region, the
    // block's first and last node, element, and past-the-end flags
    enum : uint32_t {
      kGhostNode = 1u, kGhostElem = 2u, kGhostVor = 4u,
      kHasElem = 8u, kHasVor = 16u,      // slot k has an element, a Voronoi region
      kFirst = 32u,                      // k = 0
      kLastNode = 64u, kLastElem = 128u  // k = E (the last node), k = E - 1
    };

    // where slot k of a block of E elements lies: ghost node g makes element
    // slots g and g - 1 and Voronoi slots g, g - 1 and g - 2 ghosts
    // (fill_ghosts_for, Block.hpp:658-690)
    __device__ __forceinline__ uint32_t slot_place(uint64_t k, uint64_t E, const uint8_t* __restrict__ is_ghost) {
      const bool elem = k < E, vor = k + 1 < E;
      const bool g0 = is_ghost[k], g1 = elem && is_ghost[k + 1], g2 = vor && is_ghost[k + 2];
      return (g0 ? kGhostNode : 0u) | (g0 || g1 ? kGhostElem : 0u) | (g0 || g1 || g2 ? kGhostVor : 0u) |
             (elem ? kHasElem : 0u) | (vor ? kHasVor : 0u) | (k == 0 ? kFirst : 0u) | (k == E ? kLastNode : 0u) |
             (k + 1 == E ? kLastElem : 0u);
    }

    __device__ __forceinline__ void load_slot_const(const Lines& f, uint64_t k, uint64_t E, uint32_t place, SlotConst& K) {
      // (a missing element or Voronoi region reads slot 0: finite or not, its
      // terms are not used)
      const uint64_t ke = (place & kHasElem) ? k : 0, kv = (place & kHasVor) ? k : 0, V = E - 1;
      K.m = f.m[k];
      K.mn = f.m[ke + 1];
      K.im = f.im[k];
      K.gf = f.gf[k];
      K.l0 = f.l0[ke];
      K.gt = f.gt[ke];
      K.D0 = f.D0[kv];
      K.il0 = step64::divisor<true>(K.l0).r;
      K.iD0 = step64::divisor<true>(K.D0).r;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        K.S[c] = f.S[c * E + ke];
        K.sigma0[c] = f.sigma0[c * E + ke];
        K.J[c] = f.J[c * E + ke];
        K.iJ[c] = f.iJ[c * E + ke];
        K.kappa0[c] = f.kappa0[c * V + kv];
        K.B[c] = f.B[c * V + kv];
      }
    }

    __device__ __forceinline__ void cross(const double a[3], const double b[3], double o[3]) {
      o[0] = a[1] * b[2] - a[2] * b[1];
      o[1] = a[2] * b[0] - a[0] * b[2];
      o[2] = a[0] * b[1] - a[1] * b[0];
    }

    // element_length = batch_norm(difference_kernel(position))
    template <bool kPlain>
    __device__ __forceinline__ double length(const double d[3]) {
      return step64::root<kPlain>(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
    }

    // what slot k computes before it needs the terms of slot k - 1
    struct SlotTerms {
      double l, t[3], e;                          // element length (1 at a ghost), tangent, dilatation
      double qt[3], sigma[3], stress[3], c[3];    // Q t, strain, stress, Q^T n / e (0 at a ghost)
      double D, eps, kappa[3], couple[3], dv[3];  // Voronoi length, dilatation, curvature (0 at a ghost), couple, kappa x M
      double P[3], R[3];                          // M / eps^3, (kappa x M) D0 / eps^3
      double jw[3];                               // J w / e
    };

    // (kPlain: divisions and roots without their special cases; returns bit 0 if
    // an operand of the element's terms did not allow that, bit 1 if one of the
    // Voronoi region's did not)
    template <bool kPlain>
    __device__ __forceinline__ uint32_t slot_terms(const double x0[3], const double x1[3], const double x2[3],
                                               const double q[9], const double qn[9], const double w[3], uint32_t place,
                                               bool next_ghost_elem, const SlotConst& K, SlotTerms& o) {
      using step64::Divisor;
      using step64::divisor;
      using step64::over;
      // update_spanwise_variables
      const double d[3] = {x1[0] - x0[0], x1[1] - x0[1], x1[2] - x0[2]};
      const double dn[3] = {x2[0] - x1[0], x2[1] - x1[1], x2[2] - x1[2]};
      o.l = (place & kGhostElem) ? 1.0 : length<kPlain>(d);
      const double ln = next_ghost_elem ? 1.0 : length<kPlain>(dn);
      const Divisor byl = divisor<kPlain>(o.l), l0{K.l0, K.il0}, D0{K.D0, K.iD0};
#pragma unroll
      for (int c = 0; c < 3; ++c) o.t[c] = over<kPlain>(d[c], byl);
      o.e = over<kPlain>(o.l, l0);
      o.D = 0.5 * (o.l + ln);
      o.eps = over<kPlain>(o.D, D0);
      const Divisor bye = divisor<kPlain>(o.e);
      // update_shear_stretch_strain: sigma = (Q t) e - z; n = S % (sigma - sigma0)
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        o.qt[p] = q[3 * p] * o.t[0] + q[3 * p + 1] * o.t[1] + q[3 * p + 2] * o.t[2];
        o.sigma[p] = o.qt[p] * o.e;
      }
      o.sigma[2] -= 1.0;
#pragma unroll
      for (int p = 0; p < 3; ++p) o.stress[p] = K.S[p] * (o.sigma[p] - K.sigma0[p]);
      // Q^T n / e with zeroed ghosts, and J w / e
      double a[3], jw[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        a[j] = q[j] * o.stress[0] + q[3 + j] * o.stress[1] + q[6 + j] * o.stress[2];
        o.c[j] = (place & kGhostElem) ? 0.0 : over<kPlain>(a[j], bye);
        jw[j] = K.J[j] * w[j];
        o.jw[j] = over<kPlain>(jw[j], bye);
      }
      // curvature, couple, 1 / eps^3 and the terms of the torque sums
      step64::curvature<kPlain>(q, qn, D0, o.kappa);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        if (place & kGhostVor) o.kappa[c] = 0.0;
        o.couple[c] = K.B[c] * (o.kappa[c] - K.kappa0[c]);
      }
      cross(o.kappa, o.couple, o.dv);
      const double cube = o.eps * o.eps * o.eps;
      const double ic = over<kPlain>(1.0, divisor<kPlain>(cube)), icd = ic * K.D0;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        o.P[c] = o.couple[c] * ic;
        o.R[c] = o.dv[c] * icd;
      }
      if constexpr (!kPlain) return 0u;
      step64::Range elem, vor;
      elem.divisor(o.l);
      elem.divisor(o.e);
      elem.divisor(K.l0);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        elem.numerator(d[c]);
        elem.numerator(a[c]);
        elem.numerator(jw[c]);
      }
      elem.largest((((fabs(d[0]) + fabs(d[1])) + (fabs(d[2]) + fabs(a[0]))) + ((fabs(a[1]) + fabs(a[2])) + fabs(jw[0]))) +
                   (fabs(jw[1]) + fabs(jw[2])));
      vor.divisor(ln);
      vor.divisor(K.D0);
      vor.divisor(cube);
      return ((place & kHasElem) && elem.bad() ? 1u : 0u) | ((place & kHasVor) && vor.bad() ? 2u : 0u);
    }

    // two_point_difference_kernel (BlazeCalculus.hpp:29-45) at one output,
    // from this slot's and the previous slot's value
    __device__ __forceinline__ double two_point(double a, double am, bool first, bool last) {
      return first ? a : (last ? -am : a - am);
    }

    // internal force on node k
    __device__ __forceinline__ void slot_force(const double c[3], const double cm[3], const double v[3], uint32_t place,
                                               bool damped, const SlotConst& K, double f[3]) {
      const double mg = K.m * K.gf;
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        f[i] = two_point(c[i], cm[i], place & kFirst, place & kLastNode);
        if (damped) f[i] -= mg * v[i];
      }
    }

    // internal torque on element k: couple difference and quadrature, shear,
    // Lagrangian transport, unsteady dilatation, damping, added in this order
    __device__ __forceinline__ void slot_torque(const SlotTerms& s, const double Pm[3], const double Rm[3],
                                                const double v0[3], const double v1[3], const double w[3],
                                                uint32_t place, bool damped, const SlotConst& K, double dvel[3],
                                                double tau[3]) {
      double shear[3], lag[3];
      cross(s.qt, s.stress, shear);
      cross(s.jw, w, lag);
#pragma unroll
      for (int c = 0; c < 3; ++c) dvel[c] = v1[c] - v0[c];
      const double rate = (s.t[0] * dvel[0] + s.t[1] * dvel[1] + s.t[2] * dvel[2]) / (s.e * K.l0);
      const double eg = (0.5 * (K.m + K.mn)) * K.gt;
      const bool first = place & kFirst, last = place & kLastElem;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        double a = two_point(s.P[c], Pm[c], first, last);
        a += 0.5 * (first ? s.R[c] : (last ? Rm[c] : s.R[c] + Rm[c]));  // quadrature_kernel (BlazeCalculus.hpp:67-86)
        a += shear[c] * K.l0;
        a += lag[c];
        a += s.jw[c] * rate;
        if (damped) a -= eg * w[c];
        tau[c] = a;
      }
    }

    // ---- the stepper's calls ----------------------------------------------------

    // kinematic_states() += c * kinematic_rates(): x += c v on node k,
    // Q <- exp(-c [w]x) Q on element k.  Bound by memory, 240 B per slot: 5.6 us
    // at 67,584 slots (two kernels before)
    __global__ void __launch_bounds__(kThreads) k_kinematic(double* __restrict__ x, const double* __restrict__ v,
                                                            double* __restrict__ Q, const double* __restrict__ w,
                                                            double c, uint64_t E) {
      const uint64_t N = E + 1;
      GRID_STRIDE(k, N) {
#pragma unroll
        for (int d = 0; d < 3; ++d) x[d * N + k] += c * v[d * N + k];
        if (k < E) {
          double q[9], wk[3];
#pragma unroll
          for (int m = 0; m < 9; ++m) q[m] = Q[m * E + k];
#pragma unroll
          for (int d = 0; d < 3; ++d) wk[d] = w[d * E + k];
          step64::so3_update(q, wk, c);
#pragma unroll
          for (int m = 0; m < 9; ++m) Q[m * E + k] = q[m];
        }
      }
    }

    // ExternalLoads = ExternalTorques = 0, then every derived field
    // (compute_internal_dynamics), in one pass: bound by memory, 640 B per slot
    // and 14 us at 67,584 slots, where a pass per operator (37 of them) moved
    // 2.5 KB and took 86 us.  A workgroup of kThreads takes kThreads - 1
    // slots: its first thread computes the slot before them, whose Q^T n / e
    // and couple terms the first of them needs.
    __global__ void __launch_bounds__(kThreads) k_internal(Lines f, const uint8_t* __restrict__ is_ghost, bool damped,
                                                           uint64_t E) {
      const uint64_t N = E + 1, V = E - 1;
      const int tid = threadIdx.x;
      __shared__ double s[9][kThreads];
      const int64_t kk = int64_t(blockIdx.x) * (kThreads - 1) + tid - 1;
      const bool in = kk >= 0 && kk <= int64_t(E);
      const uint64_t k = in ? uint64_t(kk) : 0;
      const uint32_t place = slot_place(k, E, is_ghost);
      SlotConst K;
      SlotTerms o;
      double x[3][3], v0[3], v1[3], q[9], qn[9], w[3];
      load_slot_const(f, k, E, place, K);
      const uint64_t ke = (place & kHasElem) ? k : 0, kv = (place & kHasVor) ? k : 0;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        x[0][c] = f.x[c * N + k];
        x[1][c] = f.x[c * N + ke + 1];
        x[2][c] = f.x[c * N + kv + 2];
        v0[c] = f.v[c * N + k];
        v1[c] = f.v[c * N + ke + 1];
        w[c] = f.w[c * E + ke];
      }
#pragma unroll
      for (int m = 0; m < 9; ++m) {
        q[m] = f.q[m * E + ke];
        // (a ghost region's curvature is zero, and a missing one unused: its
        // wave need not run the large-angle form for it)
        qn[m] = f.q[m * E + ((place & kHasVor) && !(place & kGhostVor) ? k + 1 : ke)];
      }
      const double vol = f.vol[ke];
      const bool next_ghost = (place & kHasVor) && (is_ghost[k + 1] || is_ghost[k + 2]);
      slot_terms<false>(x[0], x[1], x[2], q, qn, w, place, next_ghost, K, o);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        s[c][tid] = o.c[c];
        s[3 + c][tid] = o.P[c];
        s[6 + c][tid] = o.R[c];
      }
      __syncthreads();
      if (tid == 0 || !in) return;
      double cm[3], Pm[3], Rm[3], fi[3], tau[3], dvel[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        cm[c] = s[c][tid - 1];
        Pm[c] = s[3 + c][tid - 1];
        Rm[c] = s[6 + c][tid - 1];
      }
      slot_force(o.c, cm, v0, place, damped, K, fi);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        f.f_int[c * N + k] = fi[c];
        f.f_ext[c * N + k] = 0.0;
      }
      if (place & kHasElem) {
        slot_torque(o, Pm, Rm, v0, v1, w, place, damped, K, dvel, tau);
        f.l[k] = o.e * K.l0;  // (the reference leaves e l0 here, and eps D0 below)
        f.e[k] = o.e;
        f.r[k] = sqrt(M_1_PI * vol / o.l);  // update_dimension
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          f.t[c * E + k] = o.t[c];
          f.sigma[c * E + k] = o.sigma[c];
          f.stress[c * E + k] = o.stress[c];
          f.tau_int[c * E + k] = tau[c];
          f.tau_ext[c * E + k] = 0.0;
          f.d1[c * E + k] = o.jw[c];
          f.d2[c * E + k] = dvel[c];
        }
      }
      if (place & kHasVor) {
        f.D[k] = o.eps * K.D0;
        f.eps[k] = o.eps;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          f.kappa[c * V + k] = o.kappa[c];
          f.couple[c * V + k] = o.couple[c];
          f.dv[c * V + k] = o.dv[c];
        }
      }
    }

    // accelerations from the loads and torques, then v += dt a, w += dt alpha
    __global__ void __launch_bounds__(kThreads) k_dynamic(Lines f, double dt, uint64_t E) {
      const uint64_t N = E + 1;
      GRID_STRIDE(k, N) {
        // (every load before the first store: the fields could alias for the compiler)
        const uint64_t ke = k < E ? k : 0;
        double fi[3], fe[3], v[3], iJ[3], ti[3], te[3], w[3];
        const double im = f.im[k], e = f.e[ke];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          fi[c] = f.f_int[c * N + k];
          fe[c] = f.f_ext[c * N + k];
          v[c] = f.v[c * N + k];
          iJ[c] = f.iJ[c * E + ke];
          ti[c] = f.tau_int[c * E + ke];
          te[c] = f.tau_ext[c * E + ke];
          w[c] = f.w[c * E + ke];
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const double a = (fi[c] + fe[c]) * im;
          f.acc[c * N + k] = a;
          f.v[c * N + k] = v[c] + dt * a;
        }
        if (k < E) {
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            const double al = (iJ[c] * (ti[c] + te[c])) * e;
            f.alpha[c * E + k] = al;
            f.w[c * E + k] = w[c] + dt * al;
          }
        }
      }
    }

    // ---- hooks ---------------------------------------------------------------

    // ConstrainPrimitives of a fixed clamp at index i: node i's position and
    // element min(i, n - 1)'s director are held
    __global__ void k_clamp_values(double* __restrict__ x, double* __restrict__ Q, const RodInfo* __restrict__ rods,
                                   uint64_t n_rods, uint64_t E) {
      const uint64_t N = E + 1;
      GRID_STRIDE(r, n_rods) {
        const RodInfo& ri = rods[r];
        for (int k = 0; k < 2; ++k) {
          const uint32_t i = ri.clamp_idx[k];
          if (!(ri.flags & clamp_bit(k)) || i > ri.n) continue;
          const uint64_t s = ri.start + i;
          const uint64_t se = ri.start + (i < ri.n ? i : ri.n - 1);
          for (int d = 0; d < 3; ++d) x[d * N + s] = ri.clamp[k].x[d];
          for (int m = 0; m < 9; ++m) Q[m * E + se] = ri.clamp[k].q[m];
        }
      }
    }

    // ConstrainRates of the same clamp: its node's velocity and its
    // element's angular velocity are zeroed
    __global__ void k_clamp_rates(double* __restrict__ v, double* __restrict__ w, const RodInfo* __restrict__ rods,
                                  uint64_t n_rods, uint64_t E) {
      const uint64_t N = E + 1;
      GRID_STRIDE(r, n_rods) {
        const RodInfo& ri = rods[r];
        for (int k = 0; k < 2; ++k) {
          const uint32_t i = ri.clamp_idx[k];
          if (!(ri.flags & clamp_bit(k)) || i > ri.n) continue;
          const uint64_t s = ri.start + i;
          const uint64_t se = ri.start + (i < ri.n ? i : ri.n - 1);
          for (int d = 0; d < 3; ++d) v[d * N + s] = 0.0;
          for (int d = 0; d < 3; ++d) w[d * E + se] = 0.0;
        }
      }
    }

    __global__ void k_end_force(double* __restrict__ fe, const RodInfo* __restrict__ rods, uint64_t n_rods, uint64_t E, double t) {
      const uint64_t N = E + 1;
      GRID_STRIDE(r, n_rods) {
        const RodInfo& ri = rods[r];
        if (!(ri.flags & 2u)) continue;
        const uint64_t node = ri.start + ri.n;
        const double rv = step64::ramp_value(ri.ramp, t, ri.ramp_start, ri.ramp_interval);
        for (int d = 0; d < 3; ++d) fe[d * N + node] = ri.force[d] * rv;
      }
    }

    // flags the ghost node between two rods
    __global__ void k_mark_ghost_nodes(uint8_t* __restrict__ flag, const uint64_t* __restrict__ ghost, uint64_t n) {
      GRID_STRIDE(i, n) flag[ghost[i]] = 1;
    }

    // gravity on every node (the block-wide update of GravityField.hpp:239-246);
    // plane contact on the rods' own nodes only
    __device__ __forceinline__ void add_environment(const Env& env, double m, const double x[3], const double v[3],
                                                    bool ghost, double fe[3]) {
      if (env.gravity)
        for (int c = 0; c < 3; ++c) fe[c] += env.g[c] * m;
      if (!env.contact) return;
      // the plane n . x = z0; the node's height above it, less the offset
      const double gap = ((env.n[0] * x[0] + env.n[1] * x[1]) + env.n[2] * x[2]) - env.z0 - env.offset;
      if (gap < 0.0 && !ghost) {
        const double delta = -gap;
        const double vnv = (env.n[0] * v[0] + env.n[1] * v[1]) + env.n[2] * v[2];
        const double vn = -vnv;  // approach speed along the normal
        const double fn = fmax(0.0, env.k * delta + env.c * vn);
        double vt[3];
        for (int c = 0; c < 3; ++c) vt[c] = v[c] - vnv * env.n[c];
        const double vtn = sqrt((vt[0] * vt[0] + vt[1] * vt[1]) + vt[2] * vt[2]);
        for (int c = 0; c < 3; ++c) fe[c] += fn * env.n[c];
        if (vtn > 0.0) {
          const double ft = fmin(env.ct * vtn, env.mu * fn);
          const double s = ft / vtn;  // f_T along the unit slip
          for (int c = 0; c < 3; ++c) fe[c] -= s * vt[c];
        }
      }
    }

    __global__ void k_environment(double* __restrict__ fe, const double* __restrict__ m, const double* __restrict__ x,
                                  const double* __restrict__ v, const uint8_t* __restrict__ is_ghost, uint64_t E,
                                  Env env) {
      const uint64_t N = E + 1;
      GRID_STRIDE(i, N) {
        double f[3], xi[3], vi[3];
        for (int c = 0; c < 3; ++c) {
          f[c] = fe[c * N + i];
          xi[c] = x[c * N + i];
          vi[c] = v[c * N + i];
        }
        add_environment(env, m[i], xi, vi, is_ghost[i], f);
        for (int c = 0; c < 3; ++c) fe[c * N + i] = f[c];
      }
    }

    // the rod of every slot; the ghost node between two rods goes with the first
    __global__ void k_slot_rods(uint32_t* __restrict__ rod_of, const RodInfo* __restrict__ rods, uint64_t n_rods) {
      for (uint64_t r = blockIdx.x; r < n_rods; r += gridDim.x) {
        const uint64_t s = rods[r].start, n = rods[r].n + (r + 1 < n_rods ? 2u : 1u);
        for (uint64_t i = threadIdx.x; i < n; i += blockDim.x) rod_of[s + i] = static_cast<uint32_t>(r);
      }
    }

    // ---- several whole steps in one launch -----------------------------------------

    // Steps per launch of k_steps: more of them amortise its loads and launch,
    // and cost 2 slots of a workgroup's 256 each.  Measured with 4 / 8 / 12 / 16 /
    // 20: 12.8 / 12.1 / 11.3 / 11.0 / 10.9 us a step at 248,188 elements, 46.5 /
    // 39.7 / 37.5 / 38.1 / 38.8 at 992,754.  One workgroup has nothing to recompute.
    constexpr uint64_t kStepsPerLaunch = 12, kStepsOneBlock = 100;

    // x, v, Q, w: the state a launch of k_steps reads or writes
    struct State {
      double *x, *v, *q, *w;
    };

    // hook bits of a slot: 0-1 the clamps that hold node k, 2-3 those that
    // hold element k, 4 the rod's end force acts on node k
    __device__ __forceinline__ uint32_t slot_hooks(const RodInfo& ri, uint64_t k) {
      uint32_t h = 0;
      for (int c = 0; c < 2; ++c) {
        const uint32_t i = ri.clamp_idx[c];
        if (!(ri.flags & clamp_bit(c)) || i > ri.n) continue;
        if (k == ri.start + i) h |= 1u << c;
        if (k == ri.start + (i < ri.n ? i : ri.n - 1)) h |= 4u << c;
      }
      if ((ri.flags & 2u) && k == ri.start + ri.n) h |= 16u;
      return h;
    }

    // `nsteps` steps of the op-by-op path on the state alone: what the
    // stepper's calls above do to x, v, Q, w, with the derived fields left in
    // registers.  One thread per slot, neighbours through LDS (two barriers a
    // step).  A workgroup recomputes slots beside its own: a step needs the
    // -1 slot's terms (from its own nodes and director) and, for the next
    // element's length, the +2 slot's node, but what is wrong past an edge
    // moves inward by one slot a step only: if nodes from a and directors
    // from b on are wrong, Q^T n / e is from min(a - 1, b) on, the couple from
    // min(a - 2, b - 1) on, hence a' = min(a - 1, b), b' = min(a - 2, b - 1):
    // from a = b = kThreads, b is kThreads - 1 - s after s steps.  So `left` =
    // nsteps slots before its own and nsteps + 1 after them are enough.  A
    // workgroup reads `in` and writes `out`, two copies of the state, so that
    // none writes what another reads.  A block of at most kThreads slots is
    // one workgroup (left = 0, own = its slots), in place, for any nsteps.
    // Bound by VALU issue like the fused FP64 kernel (208 VGPRs, two workgroups
    // per CU, 876 VALU instructions per wave and step); constants stay in
    // registers for the launch.  11.3 us a step at 248,188 elements against 209
    // with a pass per operator, 3.1 against 113 on one rod of 100 elements (46
    // launches a step before).
    __global__ void __launch_bounds__(kThreads) k_steps(State in, State out, Lines f, const uint8_t* __restrict__ is_ghost,
                                                        const uint32_t* __restrict__ rod_of,
                                                        const RodInfo* __restrict__ rods, Env env, bool damped, double dt,
                                                        double t, int nsteps, int left, int own, uint64_t E) {
      const uint64_t N = E + 1;
      const int tid = threadIdx.x;
      __shared__ double s1[15][kThreads], s3[9][kThreads];
      const int64_t first = int64_t(blockIdx.x) * own, kk = first + tid - left;
      const bool valid = kk >= 0 && kk <= int64_t(E);
      const uint64_t k = valid ? uint64_t(kk) : 0;
      const uint32_t place = slot_place(k, E, is_ghost);
      const bool next_ghost = (place & kHasVor) && (is_ghost[k + 1] || is_ghost[k + 2]);
      const uint64_t ke = (place & kHasElem) ? k : 0;
      double x[3], v[3], q[9], w[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        x[c] = in.x[c * N + k];
        v[c] = in.v[c * N + k];
        w[c] = in.w[c * E + ke];
      }
#pragma unroll
      for (int m = 0; m < 9; ++m) q[m] = in.q[m * E + ke];
      SlotConst K;
      load_slot_const(f, k, E, place, K);
      const uint32_t rod = rod_of ? rod_of[k] : 0u;
      const uint32_t hooks = rod_of ? slot_hooks(rods[rod], k) : 0u;
      const bool whooks = __ballot(hooks != 0u) != 0ull;
      const bool environment = env.gravity || env.contact;
      const int n1 = tid + 1 < kThreads ? tid + 1 : tid, n2 = tid + 2 < kThreads ? tid + 2 : n1, p1 = tid > 0 ? tid - 1 : 0;
      // Where a slot has no element, no Voronoi region, or no thread beside it
      // to take one from, its terms are never used, and the curvature of a ghost
      // region is zero: they get an unstrained element and their own director,
      // so that their waves don't run the large-angle forms or, over values that
      // are no numbers, the full ones.  Threads past the block's slots stand still.
      const bool no_elem = !valid || !(place & kHasElem) || tid + 1 >= kThreads;
      const bool no_vor = no_elem || !(place & kHasVor) || tid + 2 >= kThreads;
      const bool own_q = no_vor || (place & kGhostVor);
      const bool edge = step64::any(own_q);
      const double dtk = valid ? dt : 0.0, ch = 0.5 * dtk;
      // (the half step that closes a step turns by the rotation of the one that
      // opens the next)
      step64::Rotation turn = step64::rotation(w, ch);
      for (int step = 0; step < nsteps; ++step) {
#pragma unroll
        for (int c = 0; c < 3; ++c) x[c] += ch * v[c];
        step64::rotate(q, turn);
        t += 0.5 * dt;
        if (whooks && (hooks & 15u)) {
          const RodInfo& ri = rods[rod];
          for (int c = 0; c < 2; ++c) {
            if (hooks & (1u << c))
              for (int d = 0; d < 3; ++d) x[d] = ri.clamp[c].x[d];
            if (hooks & (4u << c))
              for (int m = 0; m < 9; ++m) q[m] = ri.clamp[c].q[m];
          }
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          s1[c][tid] = x[c];
          s1[3 + c][tid] = v[c];
        }
#pragma unroll
        for (int m = 0; m < 9; ++m) s1[6 + m][tid] = q[m];
        __syncthreads();
        double x1[3], x2[3], v1[3], qn[9];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          x1[c] = s1[c][n1];
          x2[c] = s1[c][n2];
          v1[c] = s1[3 + c][n1];
        }
#pragma unroll
        for (int m = 0; m < 9; ++m) qn[m] = s1[6 + m][n1];
        if (edge) {
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            if (no_elem) x1[c] = x[c] + K.l0 * q[6 + c];
            if (no_vor) x2[c] = x1[c] + (x1[c] - x[c]);
          }
#pragma unroll
          for (int m = 0; m < 9; ++m)
            if (own_q) qn[m] = q[m];
        }
        SlotTerms o;
        // (what lies past the last thread, and what a launch over several
        // workgroups has already got wrong beside it, has no say)
        const uint32_t bad = slot_terms<true>(x, x1, x2, q, qn, w, place, next_ghost, K, o);
        const int sound = kThreads - 1 - (left > 0 ? step : 0);
        if (step64::any(valid && (((bad & 1u) && tid < sound) || ((bad & 2u) && tid + 1 < sound))))
          slot_terms<false>(x, x1, x2, q, qn, w, place, next_ghost, K, o);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          s3[c][tid] = o.c[c];
          s3[3 + c][tid] = o.P[c];
          s3[6 + c][tid] = o.R[c];
        }
        __syncthreads();
        double cm[3], Pm[3], Rm[3], fi[3], tau[3], dvel[3], fe[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          cm[c] = s3[c][p1];
          Pm[c] = s3[3 + c][p1];
          Rm[c] = s3[6 + c][p1];
        }
        slot_force(o.c, cm, v, place, damped, K, fi);
        slot_torque(o, Pm, Rm, v, v1, w, place, damped, K, dvel, tau);
        // forcing first, then environments
        if (whooks && (hooks & 16u)) {
          const RodInfo& ri = rods[rod];
          const double rv = step64::ramp_value(ri.ramp, t, ri.ramp_start, ri.ramp_interval);
          for (int c = 0; c < 3; ++c) fe[c] = ri.force[c] * rv;
        }
        if (environment) add_environment(env, K.m, x, v, place & kGhostNode, fe);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          v[c] += dtk * ((fi[c] + fe[c]) * K.im);
          w[c] += dtk * ((K.iJ[c] * (tau[c] + 0.0)) * o.e);  // (the external torque is zero)
        }
        if (whooks) {
          if (hooks & 3u)
            for (int c = 0; c < 3; ++c) v[c] = 0.0;
          if (hooks & 12u)
            for (int c = 0; c < 3; ++c) w[c] = 0.0;
        }
        t += 0.5 * dt;
#pragma unroll
        for (int c = 0; c < 3; ++c) x[c] += ch * v[c];
        turn = step64::rotation(w, ch);
        step64::rotate(q, turn);
      }
      if (!valid || tid < left || tid >= left + own) return;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        out.x[c * N + k] = x[c];
        out.v[c * N + k] = v[c];
      }
      if (!(place & kHasElem)) return;
#pragma unroll
      for (int c = 0; c < 3; ++c) out.w[c * E + k] = w[c];
#pragma unroll
      for (int m = 0; m < 9; ++m) out.q[m * E + k] = q[m];
    }

  }  // namespace

#define L(kernel, n, ...) hipLaunchKernelGGL(kernel, dim3(grid_for(n)), dim3(kThreads), 0, b->stream, __VA_ARGS__)
#define F(id) (b->d_field[id])

  int ops_set_rod_clocks(erod_batch* b, double t) {
    L(k_fill, b->n_rods, b->d_time, t, b->n_rods);
    return hip_check(hipGetLastError(), "set rod clocks");
  }

  int ops_mark_ghost_nodes(erod_batch* b) {
    EROD_HIP(hipMemsetAsync(b->d_node_is_ghost, 0, b->E + 1, b->stream));
    if (!b->ghost_nodes.empty()) L(k_mark_ghost_nodes, b->ghost_nodes.size(), b->d_node_is_ghost, b->d_ghost_nodes,
                                   static_cast<uint64_t>(b->ghost_nodes.size()));
    return hip_check(hipGetLastError(), "mark ghost nodes");
  }

  int ops_fill_ghosts(erod_batch* b, int field) {
    if (b->ghost_nodes.empty()) return EROD_OK;
    const FieldInfo& fi = field_info(field);
    const int deficit = fi.stagger == EROD_NODE ? 1 : (fi.stagger == EROD_ELEMENT ? 2 : 3);
    const uint64_t n = b->ghost_nodes.size();
    L(k_fill_ghosts, n * deficit, F(field), b->d_ghost_nodes, n, deficit, b->field_slots(field), fi.ncomp, fi.ghost);
    return hip_check(hipGetLastError(), "fill_ghosts");
  }

  // the fields of the block for the kernels that take all of them
  static Lines lines_of(erod_batch* b) {
    Lines f;
    f.x = F(EROD_POSITION);
    f.v = F(EROD_VELOCITY);
    f.acc = F(EROD_ACCELERATION);
    f.f_int = F(EROD_INTERNAL_LOADS);
    f.f_ext = F(EROD_EXTERNAL_LOADS);
    f.m = F(EROD_MASS);
    f.im = F(EROD_INV_MASS);
    f.gf = F(EROD_FORCE_DAMPING_RATE);
    f.q = F(EROD_DIRECTOR);
    f.w = F(EROD_ANGULAR_VELOCITY);
    f.alpha = F(EROD_ANGULAR_ACCELERATION);
    f.t = F(EROD_TANGENT);
    f.sigma = F(EROD_SHEAR_STRETCH_STRAIN);
    f.stress = F(EROD_INTERNAL_STRESS);
    f.tau_int = F(EROD_INTERNAL_TORQUES);
    f.tau_ext = F(EROD_EXTERNAL_TORQUES);
    f.d1 = F(EROD_DUMMY_ELEMENT_VECTOR);
    f.d2 = F(EROD_DUMMY_ELEMENT_VECTOR2);
    f.S = F(EROD_SHEAR_STRETCH_RIGIDITY);
    f.J = F(EROD_MASS_SECOND_MOMENT_OF_INERTIA);
    f.iJ = F(EROD_INV_MASS_SECOND_MOMENT_OF_INERTIA);
    f.sigma0 = F(EROD_REFERENCE_SHEAR_STRETCH_STRAIN);
    f.l = F(EROD_ELEMENT_LENGTH);
    f.e = F(EROD_ELEMENT_DILATATION);
    f.r = F(EROD_ELEMENT_DIMENSION);
    f.l0 = F(EROD_REFERENCE_ELEMENT_LENGTH);
    f.vol = F(EROD_ELEMENT_VOLUME);
    f.gt = F(EROD_TORQUE_DAMPING_RATE);
    f.kappa = F(EROD_CURVATURE);
    f.couple = F(EROD_INTERNAL_COUPLE);
    f.dv = F(EROD_DUMMY_VORONOI_VECTOR);
    f.kappa0 = F(EROD_REFERENCE_CURVATURE);
    f.B = F(EROD_BENDING_TWIST_RIGIDITY);
    f.D = F(EROD_VORONOI_LENGTH);
    f.eps = F(EROD_VORONOI_DILATATION);
    f.D0 = F(EROD_REFERENCE_VORONOI_LENGTH);
    return f;
  }

  // kinematic_states() += c * kinematic_rates(): x += c v, Q <- exp(-c [w]x) Q
  int ops_kinematic_update_by(erod_batch* b, double c) {
    L(k_kinematic, b->E + 1, F(EROD_POSITION), F(EROD_VELOCITY), F(EROD_DIRECTOR), F(EROD_ANGULAR_VELOCITY), c, b->E);
    return hip_check(hipGetLastError(), "kinematic_update");
  }

  // PositionVerlet's kinematic substep: the coefficient (1/2) dt
  int ops_kinematic_update(erod_batch* b, double dt) { return ops_kinematic_update_by(b, 0.5 * dt); }

  // every slot of a field (ghosts included) set to one value: the block-wide
  // assignment of a scalar to a variable
  int ops_fill_field(erod_batch* b, int field, double v) {
    const uint64_t n = uint64_t(field_info(field).ncomp) * b->field_slots(field);
    L(k_fill, n, b->d_field[field], v, n);
    return hip_check(hipGetLastError(), "fill_field");
  }

  int ops_compute_internal_dynamics(erod_batch* b) {
    const uint64_t blocks = (b->E + 1 + kThreads - 2) / (kThreads - 1);
    hipLaunchKernelGGL(k_internal, dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0, b->stream, lines_of(b),
                       b->d_node_is_ghost, b->damped, b->E);
    return hip_check(hipGetLastError(), "compute_internal_dynamics");
  }

  int ops_dynamic_update(erod_batch* b, double dt) {
    L(k_dynamic, b->E + 1, lines_of(b), dt, b->E);
    return hip_check(hipGetLastError(), "dynamic_update");
  }

  int ops_apply_post_kinematic(erod_batch* b) {
    if (!b->has_clamps) return EROD_OK;
    L(k_clamp_values, b->n_rods, F(EROD_POSITION), F(EROD_DIRECTOR), b->d_rods, b->n_rods, b->E);
    return hip_check(hipGetLastError(), "post_kinematic");
  }

  // Forcing first, then environments (the module order of the oracle).
  int ops_apply_pre_dynamic(erod_batch* b, double time) {
    const uint64_t N = b->E + 1;
    if (b->has_forces) L(k_end_force, b->n_rods, F(EROD_EXTERNAL_LOADS), b->d_rods, b->n_rods, b->E, time);
    if (b->env.gravity || b->env.contact)
      L(k_environment, N, F(EROD_EXTERNAL_LOADS), F(EROD_MASS), F(EROD_POSITION), F(EROD_VELOCITY), b->d_node_is_ghost,
        b->E, b->env);
    return hip_check(hipGetLastError(), "pre_dynamic");
  }

  int ops_apply_post_dynamic(erod_batch* b) {
    if (!b->has_clamps) return EROD_OK;
    L(k_clamp_rates, b->n_rods, F(EROD_VELOCITY), F(EROD_ANGULAR_VELOCITY), b->d_rods, b->n_rods, b->E);
    return hip_check(hipGetLastError(), "post_dynamic");
  }

  // the second copy of the state and the slots' rods, for k_steps; false when
  // the device has no room for them
  static bool steps_buffers(erod_batch* b) {
    const OnDevice here(b->device);
    static const int fields[4] = {EROD_POSITION, EROD_VELOCITY, EROD_DIRECTOR, EROD_ANGULAR_VELOCITY};
    const bool two = b->E + 1 > kThreads;
    bool ok = !two || shadow_fits(b);
    if (two && ok)
      for (int i = 0; i < 4 && ok; ++i)
        if (!b->d_shadow[i])
          ok = hipMalloc(&b->d_shadow[i], sizeof(double) * field_info(fields[i]).ncomp * b->field_slots(fields[i])) == hipSuccess;
    if (two && !ok)  // (no part of a copy that is of no use)
      for (double*& p : b->d_shadow) {
        (void)hipFree(p);
        p = nullptr;
      }
    if (ok && !b->d_slot_rods && (b->has_clamps || b->has_forces)) {
      ok = hipMalloc(&b->d_slot_rods, sizeof(uint32_t) * (b->E + 1)) == hipSuccess;
      if (ok)
        hipLaunchKernelGGL(k_slot_rods, dim3(static_cast<unsigned>(b->n_rods < 65535 ? b->n_rods : 65535)), dim3(kThreads), 0,
                           b->stream, b->d_slot_rods, b->d_rods, b->n_rods);
    }
    if (!ok) (void)hipGetLastError();
    return ok;
  }

  // The first n - 1 steps of a call change the state only (the last one
  // rewrites every derived field), so they go through k_steps, at most
  // kStepsPerLaunch a launch; without memory for its second copy of the
  // state, every step goes call by call.
  static int steps_before_last(erod_batch* b, double* t, double dt, uint64_t n, uint64_t* done) {
    *done = 0;
    const uint64_t N = b->E + 1;
    const bool one = N <= kThreads;
    // two copies: an even number of launches ends in the fields
    if (n < (one ? 1u : 2u) || !steps_buffers(b)) return EROD_OK;
    const State fields{F(EROD_POSITION), F(EROD_VELOCITY), F(EROD_DIRECTOR), F(EROD_ANGULAR_VELOCITY)};
    const State shadow{b->d_shadow[0], b->d_shadow[1], b->d_shadow[2], b->d_shadow[3]};
    const uint64_t most = one ? kStepsOneBlock : kStepsPerLaunch;
    uint64_t launches = (n + most - 1) / most;
    if (!one) launches += launches & 1;
    for (uint64_t i = 0; i < launches; ++i) {
      const int s = static_cast<int>(n / launches + (i < n % launches ? 1 : 0));
      const int left = one ? 0 : s, own = one ? static_cast<int>(N) : kThreads - 1 - 2 * s;
      const bool odd = !one && (i & 1);
      hipLaunchKernelGGL(k_steps, dim3(static_cast<unsigned>((N + own - 1) / own)), dim3(kThreads), 0, b->stream,
                         odd ? shadow : fields, one || odd ? fields : shadow, lines_of(b), b->d_node_is_ghost,
                         b->has_clamps || b->has_forces ? b->d_slot_rods : nullptr, b->d_rods, b->env, b->damped, dt, *t, s,
                         left, own, b->E);
      if (int rc = hip_check(hipGetLastError(), "k_steps")) return rc;
      for (int j = 0; j < 2 * s; ++j) *t += 0.5 * dt;
    }
    *done = n;
    return EROD_OK;
  }

  int ops_step(erod_batch* b, double* time, double dt, uint64_t n) {
    double t = *time;
    uint64_t done = 0;
    int rc = n > 1 ? steps_before_last(b, &t, dt, n - 1, &done) : EROD_OK;
    if (rc) return rc;
    for (; done < n; ++done) {
      if ((rc = ops_kinematic_update(b, dt))) return rc;
      t += 0.5 * dt;
      if ((rc = ops_apply_post_kinematic(b))) return rc;
      if ((rc = ops_compute_internal_dynamics(b))) return rc;
      if ((rc = ops_apply_pre_dynamic(b, t))) return rc;
      if ((rc = ops_dynamic_update(b, dt))) return rc;
      if ((rc = ops_apply_post_dynamic(b))) return rc;
      t += 0.5 * dt;
      if ((rc = ops_kinematic_update(b, dt))) return rc;
    }
    *time = t;
    // every rod clock follows the caller's clock, so checkpoints carry it
    return ops_set_rod_clocks(b, t);
  }

#undef L
#undef F

}  // namespace erod
