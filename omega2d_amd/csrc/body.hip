// body.hip - the small vector work of a body in a device step: the right-hand side of its
// boundary-element system (src/RHS.h:54-115, src/BEMHelper.h:116-137), the solution taken apart, and
// the panel strengths with the solved rotation's added (src/Surfaces.h:556-620). Every operation is
// rounded by itself, in the order of the formulas.
//
// Bound by launches: a stage made about 35 elementwise operations on a few hundred to a few thousand
// panels, 2 to 3 us each, for kilobytes of data. One launch for each of the three takes a step of 2,000
// particles around 100 panels from 615 to 397 us.
#include "nbody.h"
#include "o2d_runtime.h"

namespace o2d {

namespace {

constexpr int kBlock = 256;

inline unsigned blocks(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

// rhs[nunk p] = -(u . t), rhs[nunk p + 1] = -(u . n) (two unknowns) with u = fs + factor (pu, pv), and
// the last row reabsorbed + vol2 omega_error
__global__ __launch_bounds__(kBlock) void body_rhs_kernel(
    int64_t np, int nunk, double fsx, double fsy, double factor, const double* __restrict__ pu,
    const double* __restrict__ pv, const double* __restrict__ tx, const double* __restrict__ ty,
    const double* __restrict__ nx, const double* __restrict__ ny,
    const double* __restrict__ reabsorbed, double vol2, const double* __restrict__ omega_error,
    double* __restrict__ rhs) {
#pragma clang fp contract(off)
  const int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (p == 0) rhs[nunk * np] = (0.0 + *reabsorbed) + vol2 * *omega_error;
  if (p >= np) return;
  const double u = fsx + pu[p] * factor, v = fsy + pv[p] * factor;
  rhs[nunk * p] = -(u * tx[p] + v * ty[p]);
  if (nunk == 2) rhs[2 * p + 1] = -(u * nx[p] + v * ny[p]);
}

__global__ __launch_bounds__(kBlock) void body_unpack_kernel(int64_t np, int nunk,
                                                             const double* __restrict__ sol,
                                                             double* __restrict__ vs,
                                                             double* __restrict__ ss,
                                                             double* __restrict__ omega,
                                                             double* __restrict__ omega_error) {
  const int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (p == 0) *omega = *omega_error = sol[nunk * np];
  if (p >= np) return;
  vs[p] = sol[nunk * p];
  ss[p] = nunk == 2 ? sol[2 * p + 1] : 0.0;
}

// ovs = vs - (ui tx + vi ty), oss = ss - (ui ty - vi tx) with (ui, vi) = omega (-ddy, ddx)
__global__ __launch_bounds__(kBlock) void body_strengths_kernel(
    int64_t np, const double* __restrict__ vs, const double* __restrict__ ss,
    const double* __restrict__ omega, const double* __restrict__ tx, const double* __restrict__ ty,
    const double* __restrict__ ddx, const double* __restrict__ ddy, double* __restrict__ ovs,
    double* __restrict__ oss) {
#pragma clang fp contract(off)
  const int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (p >= np) return;
  const double w = *omega;
  const double ui = -w * ddy[p], vi = w * ddx[p];
  ovs[p] = vs[p] + -1.0 * (ui * tx[p] + vi * ty[p]);
  oss[p] = ss[p] + -1.0 * (ui * ty[p] - vi * tx[p]);
}

int check_body(const o2d_env* env, int64_t np, int32_t nunk, bool given) {
  if (!env) return fail(O2D_ERR_ARG, "env is NULL");
  if (np < 0) return fail(O2D_ERR_SIZE, "negative count");
  if (nunk != 1 && nunk != 2) return fail(O2D_ERR_SIZE, "nunk must be 1 or 2");
  if (!given) return fail(O2D_ERR_ARG, "NULL array");
  return 0;
}

}  // namespace

}  // namespace o2d

using namespace o2d;

extern "C" {

int o2d_hip_body_rhs_dev_d(const o2d_env* env, int64_t np, int32_t nunk, double fsx, double fsy,
                           double factor, const double* pu, const double* pv, const double* tx,
                           const double* ty, const double* nx, const double* ny,
                           const double* reabsorbed, double vol2, const double* omega_error,
                           double* rhs) {
  clear_error();
  const bool given = reabsorbed && omega_error && rhs &&
                     (np == 0 || (pu && pv && tx && ty && (nunk == 1 || (nx && ny))));
  O2D_TRY(check_body(env, np, nunk, given));
  Device* d;
  O2D_TRY(device(env->device, &d));
  body_rhs_kernel<<<blocks(np + 1), kBlock, 0, dev_stream(env)>>>(
      np, nunk, fsx, fsy, factor, pu, pv, tx, ty, nx, ny, reabsorbed, vol2, omega_error, rhs);
  O2D_LAUNCH_CHECK();
  return 0;
}

int o2d_hip_body_unpack_dev_d(const o2d_env* env, int64_t np, int32_t nunk, const double* sol,
                              double* vs, double* ss, double* omega, double* omega_error) {
  clear_error();
  O2D_TRY(check_body(env, np, nunk, sol && omega && omega_error && (np == 0 || (vs && ss))));
  Device* d;
  O2D_TRY(device(env->device, &d));
  body_unpack_kernel<<<blocks(np + 1), kBlock, 0, dev_stream(env)>>>(np, nunk, sol, vs, ss, omega,
                                                                     omega_error);
  O2D_LAUNCH_CHECK();
  return 0;
}

int o2d_hip_body_strengths_dev_d(const o2d_env* env, int64_t np, const double* vs, const double* ss,
                                 const double* omega, const double* tx, const double* ty,
                                 const double* ddx, const double* ddy, double* ovs, double* oss) {
  clear_error();
  O2D_TRY(check_body(env, np, 1,
                     omega && (np == 0 || (vs && ss && tx && ty && ddx && ddy && ovs && oss))));
  Device* d;
  O2D_TRY(device(env->device, &d));
  if (np == 0) return 0;
  body_strengths_kernel<<<blocks(np), kBlock, 0, dev_stream(env)>>>(np, vs, ss, omega, tx, ty, ddx,
                                                                    ddy, ovs, oss);
  O2D_LAUNCH_CHECK();
  return 0;
}

}  // extern "C"
