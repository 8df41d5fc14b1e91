// capi_nbody.hip - C ABI for particles on points (host and device pointer forms) and the
// float/double staging shared by the synchronous entry points.
#include <cstring>

#include "nbody.h"
#include "o2d_runtime.h"

namespace o2d {

namespace {

__global__ void f2d_kernel(int64_t n, const float* __restrict__ a, double* __restrict__ b) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = (double)a[i];
}

__global__ void d2f_kernel(int64_t n, const double* __restrict__ a, float* __restrict__ b) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = (float)a[i];
}

// A call on host arrays whose packed size is at most kPackBytes copies all of its inputs, and all of
// its outputs, at once through page-locked memory: an array by itself costs a copy of 3 us on the
// device and about as much on the host, and in float a conversion launch. 1,531 float particles on
// themselves: 160 us with nine uploads and two downloads, 77 packed; in double 119 and 68; 60,000
// (1.9 and 3.8 MB) 1,052 and 935, 1,037 and 997; 500,000 on 100 points (15 MB in double) 1,271 and 749.
// Outputs pass through that memory three times, and from kPackOut bytes of them array by array is the
// faster: 100 on 150,000, 200,000 and 240,000 points in double 492, 554 and 601 us, packed 425, 552 and
// 640; on 400,000 and 500,000 in float 649 and 716, packed 602 and 753.
constexpr size_t kPackBytes = size_t(16) << 20, kPackOut = size_t(3) << 20;
constexpr int64_t kPackAlign = 32;  // elements: each array starts on 128 bytes or more

template <class T>
struct Packed {
  T* host = nullptr;      // the packed arrays in page-locked memory
  double* dev = nullptr;  // and on the device, in double
  int64_t n = 0;          // elements so far
  int64_t add(int64_t count) {
    const int64_t at = n;
    n += (count + kPackAlign - 1) / kPackAlign * kPackAlign;
    return at;
  }
};

// Waits for the stream where a call that copies from or to the page-locked memory ends early: the next
// call fills that memory again.
struct Drain {
  hipStream_t s;
  bool pending = true;
  ~Drain() {
    if (pending) (void)hipStreamSynchronize(s);
  }
};

// particles on points, packed: the inputs, then the outputs (which are inputs too: sums add to them)
template <class T>
int points_packed(Device* d, hipStream_t s, const o2d_env* env, int64_t ns, const T* sx, const T* sy,
                  const T* ss, const T* sr, int64_t nt, const T* tx, const T* ty, const T* tr, T* tu,
                  T* tv, T* aux, bool* done) {
  // a collection acting on itself (the usual particle case) passes the same host arrays as
  // sources and targets: their device copies serve both
  const bool self = nt == ns;
  const T* in[7] = {sx, sy, ss, sr, self && tx == sx ? nullptr : tx, self && ty == sy ? nullptr : ty,
                    self && tr == sr ? nullptr : tr};
  T* out[3] = {tu, tv, aux};
  *done = false;
  if (ns > (int64_t)(kPackBytes / sizeof(T)) || nt > (int64_t)(kPackBytes / sizeof(T))) return 0;
  Packed<T> p;
  int64_t at[7], ot[3];
  for (int k = 0; k < 7; ++k) at[k] = in[k] ? p.add(k < 4 ? ns : nt) : -1;
  const int64_t first = p.n;  // of the outputs
  for (int k = 0; k < 3; ++k) ot[k] = out[k] ? p.add(nt) : -1;
  if (sizeof(T) * (size_t)p.n > kPackBytes || sizeof(T) * (size_t)(p.n - first) > kPackOut) return 0;
  *done = true;
  void *h, *v;
  O2D_TRY(pinned(d, sizeof(T) * p.n, &h));
  p.host = static_cast<T*>(h);
  O2D_TRY(slot(d, kSrcX, sizeof(double) * p.n, s, &v));
  p.dev = static_cast<double*>(v);
  for (int k = 0; k < 7; ++k)
    if (in[k]) std::memcpy(p.host + at[k], in[k], sizeof(T) * (k < 4 ? ns : nt));
  for (int k = 0; k < 3; ++k)
    if (out[k]) std::memcpy(p.host + ot[k], out[k], sizeof(T) * nt);
  float* f = nullptr;
  Drain drain{s};
  if constexpr (sizeof(T) == sizeof(float)) {
    O2D_TRY(slot(d, kStageF0, sizeof(float) * p.n, s, &v));
    f = static_cast<float*>(v);
    O2D_HIP(hipMemcpyAsync(f, p.host, sizeof(float) * p.n, hipMemcpyHostToDevice, s));
    f2d_kernel<<<(unsigned)((p.n + 255) / 256), 256, 0, s>>>(p.n, f, p.dev);
    O2D_LAUNCH_CHECK();
  } else {
    O2D_HIP(hipMemcpyAsync(p.dev, p.host, sizeof(double) * p.n, hipMemcpyHostToDevice, s));
  }
  const auto dev = [&](int64_t a) { return a < 0 ? nullptr : p.dev + a; };
  O2D_TRY(nbody_dev(d, s, env->core, env->precision, env->results, ns, dev(at[0]), dev(at[1]),
                    dev(at[2]), dev(at[3]), nt, in[4] ? dev(at[4]) : dev(at[0]),
                    in[5] ? dev(at[5]) : dev(at[1]),
                    in[6] ? dev(at[6]) : (tr ? dev(at[3]) : nullptr), dev(ot[0]), dev(ot[1]),
                    dev(ot[2])));
  const int64_t nout = p.n - first;
  if constexpr (sizeof(T) == sizeof(float)) {
    d2f_kernel<<<(unsigned)((nout + 255) / 256), 256, 0, s>>>(nout, p.dev + first, f + first);
    O2D_LAUNCH_CHECK();
    O2D_HIP(hipMemcpyAsync(p.host + first, f + first, sizeof(float) * nout, hipMemcpyDeviceToHost, s));
  } else {
    O2D_HIP(hipMemcpyAsync(p.host + first, p.dev + first, sizeof(double) * nout,
                           hipMemcpyDeviceToHost, s));
  }
  O2D_HIP(hipStreamSynchronize(s));
  drain.pending = false;
  for (int k = 0; k < 3; ++k)
    if (out[k]) std::memcpy(out[k], p.host + ot[k], sizeof(T) * nt);
  return 0;
}

}  // namespace

int upload_f2d(Device* d, Slot stage, Slot dst, const float* h, int64_t n, hipStream_t s,
               double** out) {
  float* f;
  O2D_TRY(upload<float>(d, stage, h, n, s, &f));
  void* p;
  O2D_TRY(slot(d, dst, sizeof(double) * (n > 0 ? n : 1), s, &p));
  if (n > 0) {
    f2d_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(n, f, static_cast<double*>(p));
    O2D_LAUNCH_CHECK();
  }
  *out = static_cast<double*>(p);
  return 0;
}

int download_d2f(Device* d, Slot stage, float* h, const double* dptr, int64_t n, hipStream_t s) {
  if (n <= 0) return 0;
  void* p;
  O2D_TRY(slot(d, stage, sizeof(float) * n, s, &p));
  d2f_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(n, dptr, static_cast<float*>(p));
  O2D_LAUNCH_CHECK();
  return download<float>(h, static_cast<const float*>(p), n, s);
}

int check_pp(const o2d_env* env, int64_t ns, const void* sx, const void* sy,
                    const void* ss, const void* sr, int64_t nt, const void* tx, const void* ty,
                    const void* tu, const void* tv, const void* tw, const void* te) {
  O2D_TRY(check_env(env));
  if (ns < 0 || nt < 0) return fail(O2D_ERR_SIZE, "negative count (ns=%lld, nt=%lld)",
                                    (long long)ns, (long long)nt);
  if (nt > 0x7fffffffLL) return fail(O2D_ERR_SIZE, "nt=%lld exceeds 2^31-1", (long long)nt);
  if (ns > 0 && (!sx || !sy || !ss || !sr)) return fail(O2D_ERR_ARG, "NULL source array");
  if (nt > 0 && (!tx || !ty || !tu || !tv)) return fail(O2D_ERR_ARG, "NULL target array");
  if (nt > 0 && env->results == O2D_VELANDVORT && !tw)
    return fail(O2D_ERR_ARG, "results=VELANDVORT needs tw");
  if (nt > 0 && env->results == O2D_VELANDSHEAR && !te)
    return fail(O2D_ERR_ARG, "results=VELANDSHEAR needs te");
  return 0;
}

}  // namespace o2d

using namespace o2d;

extern "C" {

int o2d_hip_points_on_points_dev_d(const o2d_env* env, int64_t ns, const double* sx,
                                   const double* sy, const double* sstr, const double* srad,
                                   int64_t nt, const double* tx, const double* ty,
                                   const double* trad, double* tu, double* tv, double* tw,
                                   double* te) {
  clear_error();
  O2D_TRY(check_pp(env, ns, sx, sy, sstr, srad, nt, tx, ty, tu, tv, tw, te));
  Device* d;
  O2D_TRY(device(env->device, &d));
  double* aux = env->results == O2D_VELANDVORT ? tw : (env->results == O2D_VELANDSHEAR ? te : nullptr);
  return nbody_dev(d, dev_stream(env), env->core, env->precision, env->results, ns, sx, sy, sstr,
                   srad, nt, tx, ty, trad, tu, tv, aux);
}

int o2d_hip_points_on_points_d(const o2d_env* env, int64_t ns, const double* sx, const double* sy,
                               const double* sstr, const double* srad, int64_t nt,
                               const double* tx, const double* ty, const double* trad,
                               double* tu, double* tv, double* tw, double* te) {
  clear_error();
  O2D_TRY(check_pp(env, ns, sx, sy, sstr, srad, nt, tx, ty, tu, tv, tw, te));
  if (ns == 0 || nt == 0) return 0;
  Device* d;
  O2D_TRY(device(env->device, &d));
  hipStream_t s = stream_of(env, d);
  double* haux = env->results == O2D_VELANDVORT ? tw : (env->results == O2D_VELANDSHEAR ? te : nullptr);
  bool done;
  O2D_TRY(points_packed<double>(d, s, env, ns, sx, sy, sstr, srad, nt, tx, ty, trad, tu, tv, haux,
                                &done));
  if (done) return 0;
  double *dsx, *dsy, *dss, *dsr, *dtx, *dty, *dtr = nullptr, *du, *dv, *dw = nullptr;
  O2D_TRY(upload<double>(d, kSrcX, sx, ns, s, &dsx));
  O2D_TRY(upload<double>(d, kSrcY, sy, ns, s, &dsy));
  O2D_TRY(upload<double>(d, kSrcS, sstr, ns, s, &dss));
  O2D_TRY(upload<double>(d, kSrcR, srad, ns, s, &dsr));
  // a collection acting on itself (the usual particle case) passes the same host arrays as
  // sources and targets: their device copies serve both
  const bool self = nt == ns;
  if (self && tx == sx) dtx = dsx;
  else O2D_TRY(upload<double>(d, kTrgX, tx, nt, s, &dtx));
  if (self && ty == sy) dty = dsy;
  else O2D_TRY(upload<double>(d, kTrgY, ty, nt, s, &dty));
  if (trad && self && trad == srad) dtr = dsr;
  else if (trad) O2D_TRY(upload<double>(d, kTrgR, trad, nt, s, &dtr));
  O2D_TRY(upload<double>(d, kOutU, tu, nt, s, &du));
  O2D_TRY(upload<double>(d, kOutV, tv, nt, s, &dv));
  if (haux) O2D_TRY(upload<double>(d, kOutW, haux, nt, s, &dw));
  O2D_TRY(nbody_dev(d, s, env->core, env->precision, env->results, ns, dsx, dsy, dss, dsr, nt, dtx,
                    dty, dtr, du, dv, dw));
  O2D_TRY(download<double>(tu, du, nt, s));
  O2D_TRY(download<double>(tv, dv, nt, s));
  if (haux) O2D_TRY(download<double>(haux, dw, nt, s));
  O2D_HIP(hipStreamSynchronize(s));
  return 0;
}

int o2d_hip_points_on_points_f(const o2d_env* env, int64_t ns, const float* sx, const float* sy,
                               const float* sstr, const float* srad, int64_t nt, const float* tx,
                               const float* ty, const float* trad, float* tu, float* tv,
                               float* tw, float* te) {
  clear_error();
  O2D_TRY(check_pp(env, ns, sx, sy, sstr, srad, nt, tx, ty, tu, tv, tw, te));
  if (ns == 0 || nt == 0) return 0;
  Device* d;
  O2D_TRY(device(env->device, &d));
  hipStream_t s = stream_of(env, d);
  float* haux = env->results == O2D_VELANDVORT ? tw : (env->results == O2D_VELANDSHEAR ? te : nullptr);
  bool done;
  O2D_TRY(points_packed<float>(d, s, env, ns, sx, sy, sstr, srad, nt, tx, ty, trad, tu, tv, haux,
                               &done));
  if (done) return 0;
  double *dsx, *dsy, *dss, *dsr, *dtx, *dty, *dtr = nullptr, *du, *dv, *dw = nullptr;
  O2D_TRY(upload_f2d(d, kStageF0, kSrcX, sx, ns, s, &dsx));
  O2D_TRY(upload_f2d(d, kStageF1, kSrcY, sy, ns, s, &dsy));
  O2D_TRY(upload_f2d(d, kStageF2, kSrcS, sstr, ns, s, &dss));
  O2D_TRY(upload_f2d(d, kStageF3, kSrcR, srad, ns, s, &dsr));
  const bool self = nt == ns;
  if (self && tx == sx) dtx = dsx;
  else O2D_TRY(upload_f2d(d, kStageF4, kTrgX, tx, nt, s, &dtx));
  if (self && ty == sy) dty = dsy;
  else O2D_TRY(upload_f2d(d, kStageF5, kTrgY, ty, nt, s, &dty));
  if (trad && self && trad == srad) dtr = dsr;
  else if (trad) O2D_TRY(upload_f2d(d, kStageF6, kTrgR, trad, nt, s, &dtr));
  O2D_TRY(upload_f2d(d, kStageF7, kOutU, tu, nt, s, &du));
  O2D_TRY(upload_f2d(d, kStageF8, kOutV, tv, nt, s, &dv));
  if (haux) O2D_TRY(upload_f2d(d, kStageF9, kOutW, haux, nt, s, &dw));
  O2D_TRY(nbody_dev(d, s, env->core, env->precision, env->results, ns, dsx, dsy, dss, dsr, nt, dtx,
                    dty, dtr, du, dv, dw));
  O2D_TRY(download_d2f(d, kStageF7, tu, du, nt, s));
  O2D_TRY(download_d2f(d, kStageF8, tv, dv, nt, s));
  if (haux) O2D_TRY(download_d2f(d, kStageF9, haux, dw, nt, s));
  O2D_HIP(hipStreamSynchronize(s));
  return 0;
}

int o2d_hip_morton_order_dev_d(const o2d_env* env, int64_t n, const double* x, const double* y,
                               double x0, double y0, double inv_extent, uint32_t* keys,
                               uint32_t* order) {
  clear_error();
  if (!env) return fail(O2D_ERR_ARG, "env is NULL");
  if (n < 0 || n > 0x7fffffffLL) return fail(O2D_ERR_SIZE, "bad count %lld", (long long)n);
  if (n > 0 && (!x || !y || !keys || !order)) return fail(O2D_ERR_ARG, "NULL array");
  Device* d;
  O2D_TRY(device(env->device, &d));
  return morton_order(d, dev_stream(env), n, x, y, false, x0, y0, inv_extent, keys, order,
                      nullptr, true);
}

}  // extern "C"
