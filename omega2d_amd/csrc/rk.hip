// rk.hip - fp64 Runge-Kutta position update, ElementBase::move (src/ElementBase.h:276-359).
//
// Stage weights combine in the reference's order: one stage x += (dt*w0)*u0; two or three
// stages u = w0*u0 + w1*u1 (+ w2*u2), x += dt*u. Every operation is an explicitly rounded IEEE
// double operation (no fused multiply-add), so the update is bit-identical to a plain C loop.
//
// A step's vector work is bound by launches, not by memory, at the sizes where it matters (10,000
// particles are 80 kB an array, 0.02 us, against 2 to 3 us a launch), so one launch finalizes both
// velocity components, and one makes the update out of place or together with the combined velocity
// that a step returns: 22 launches a Ralston RK2 step became 6 (209 -> 165 us at 10,000 particles).
#include "nbody.h"
#include "o2d_runtime.h"

namespace o2d {

namespace {

constexpr int kBlock = 256;

struct Stages {
  const double* u[3];
  const double* v[3];
  double w[3];
};

// x = x0 + ..., y = y0 + ... (x0, y0 may be x, y); uc, vc (or null): the combined stage velocity
__global__ __launch_bounds__(kBlock) void rk_kernel(int64_t n, double dt, int nstage, Stages st,
                                                    const double* x0, const double* y0, double* x,
                                                    double* y, double* __restrict__ uc,
                                                    double* __restrict__ vc) {
#pragma clang fp contract(off)
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  // plain operators on purpose: the pragma keeps exactly these from being fused
  if (nstage == 1) {
    const double f = dt * st.w[0];
    x[i] = x0[i] + f * st.u[0][i];
    y[i] = y0[i] + f * st.v[0][i];
    if (uc) {
      uc[i] = st.w[0] * st.u[0][i];
      vc[i] = st.w[0] * st.v[0][i];
    }
    return;
  }
  double u = st.w[0] * st.u[0][i] + st.w[1] * st.u[1][i];
  double v = st.w[0] * st.v[0][i] + st.w[1] * st.v[1][i];
  if (nstage == 3) {
    u = u + st.w[2] * st.u[2][i];
    v = v + st.w[2] * st.v[2][i];
  }
  x[i] = x0[i] + dt * u;
  y[i] = y0[i] + dt * v;
  if (uc) {
    uc[i] = u;
    vc[i] = v;
  }
}

// u = fsx + u * factor, v = fsy + v * factor
__global__ __launch_bounds__(kBlock) void finalize_kernel(int64_t n, double fsx, double fsy,
                                                          double factor, double* __restrict__ u,
                                                          double* __restrict__ v) {
#pragma clang fp contract(off)
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  u[i] = fsx + u[i] * factor;
  v[i] = fsy + v[i] * factor;
}

}  // namespace

int rk_move_dev(hipStream_t s, int64_t n, double dt, int nstage, const double* w,
                const double* const* u, const double* const* v, const double* x0,
                const double* y0, double* x, double* y, double* uc, double* vc) {
  if (n == 0) return 0;
  Stages st = {};
  for (int k = 0; k < nstage; ++k) {
    st.u[k] = u[k];
    st.v[k] = v[k];
    st.w[k] = w[k];
  }
  rk_kernel<<<(unsigned)((n + kBlock - 1) / kBlock), kBlock, 0, s>>>(n, dt, nstage, st, x0, y0,
                                                                     x, y, uc, vc);
  O2D_LAUNCH_CHECK();
  return 0;
}

static int check_rk(const o2d_env* env, int64_t n, int32_t nstage, const double* w,
                    const double* const* u, const double* const* v, double* x, double* y) {
  if (!env) return fail(O2D_ERR_ARG, "env is NULL");
  if (nstage < 1 || nstage > 3) return fail(O2D_ERR_RESULTS, "nstage must be 1, 2 or 3");
  if (n < 0) return fail(O2D_ERR_SIZE, "negative count");
  if (!w || !u || !v) return fail(O2D_ERR_ARG, "NULL weights or stage arrays");
  if (n > 0) {
    if (!x || !y) return fail(O2D_ERR_ARG, "NULL positions");
    for (int k = 0; k < nstage; ++k)
      if (!u[k] || !v[k]) return fail(O2D_ERR_ARG, "NULL stage velocity %d", k);
  }
  return 0;
}

}  // namespace o2d

using namespace o2d;

extern "C" {

// u and v are host arrays of nstage device pointers
int o2d_hip_rk_move_dev_d(const o2d_env* env, int64_t n, double dt, int32_t nstage,
                          const double* w, const double* const* u, const double* const* v,
                          double* x, double* y) {
  clear_error();
  O2D_TRY(check_rk(env, n, nstage, w, u, v, x, y));
  Device* d;
  O2D_TRY(device(env->device, &d));
  return rk_move_dev(dev_stream(env), n, dt, nstage, w, u, v, x, y, x, y, nullptr, nullptr);
}

int o2d_hip_rk_advance_dev_d(const o2d_env* env, int64_t n, double dt, int32_t nstage,
                             const double* w, const double* const* u, const double* const* v,
                             const double* x0, const double* y0, double* x, double* y, double* uc,
                             double* vc) {
  clear_error();
  O2D_TRY(check_rk(env, n, nstage, w, u, v, x, y));
  if (n > 0 && (!x0 || !y0)) return fail(O2D_ERR_ARG, "NULL initial positions");
  if (!uc != !vc) return fail(O2D_ERR_ARG, "uc and vc go together");
  Device* d;
  O2D_TRY(device(env->device, &d));
  return rk_move_dev(dev_stream(env), n, dt, nstage, w, u, v, x0, y0, x, y, uc, vc);
}

int o2d_hip_finalize_dev_d(const o2d_env* env, int64_t n, double fsx, double fsy, double factor,
                           double* u, double* v) {
  clear_error();
  if (!env) return fail(O2D_ERR_ARG, "env is NULL");
  if (n < 0) return fail(O2D_ERR_SIZE, "negative count");
  if (n > 0 && (!u || !v)) return fail(O2D_ERR_ARG, "NULL velocities");
  Device* d;
  O2D_TRY(device(env->device, &d));
  if (n == 0) return 0;
  finalize_kernel<<<(unsigned)((n + kBlock - 1) / kBlock), kBlock, 0, dev_stream(env)>>>(
      n, fsx, fsy, factor, u, v);
  O2D_LAUNCH_CHECK();
  return 0;
}

int o2d_hip_rk_move_d(const o2d_env* env, int64_t n, double dt, int32_t nstage, const double* w,
                      const double* const* u, const double* const* v, double* x, double* y) {
  clear_error();
  O2D_TRY(check_rk(env, n, nstage, w, u, v, x, y));
  if (n == 0) return 0;
  Device* d;
  O2D_TRY(device(env->device, &d));
  hipStream_t s = stream_of(env, d);
  static const Slot us[3] = {kStageF0, kStageF1, kStageF2};
  static const Slot vs[3] = {kStageF3, kStageF4, kStageF5};
  const double* du[3];
  const double* dv[3];
  for (int k = 0; k < nstage; ++k) {
    double *a, *b;
    O2D_TRY(upload<double>(d, us[k], u[k], n, s, &a));
    O2D_TRY(upload<double>(d, vs[k], v[k], n, s, &b));
    du[k] = a;
    dv[k] = b;
  }
  double *dx, *dy;
  O2D_TRY(upload<double>(d, kTrgX, x, n, s, &dx));
  O2D_TRY(upload<double>(d, kTrgY, y, n, s, &dy));
  O2D_TRY(rk_move_dev(s, n, dt, nstage, w, du, dv, dx, dy, dx, dy, nullptr, nullptr));
  O2D_TRY(download<double>(x, dx, n, s));
  O2D_TRY(download<double>(y, dy, n, s));
  O2D_HIP(hipStreamSynchronize(s));
  return 0;
}

}  // extern "C"
