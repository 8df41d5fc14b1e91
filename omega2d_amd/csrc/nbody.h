// nbody.h - internal interfaces between the kernel modules and the C ABI layer.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "o2d_runtime.h"

namespace o2d {

// particles on points, device pointers, enqueued on s (tw is the vorticity or shear output);
// temporaries come from the device's buffer pool, or from *ws when it is given
int nbody_dev(Device* d, hipStream_t s, int core, int prec, int res, int64_t ns, const double* sx,
              const double* sy, const double* ss, const double* sr, int64_t nt, const double* tx,
              const double* ty, const double* tr, double* tu, double* tv, double* tw,
              Workspace* ws = nullptr);

// argument checks of the particles-on-points entry points (counts, NULL arrays, outputs the
// result type needs)
int check_pp(const o2d_env* env, int64_t ns, const void* sx, const void* sy, const void* ss,
             const void* sr, int64_t nt, const void* tx, const void* ty, const void* tu,
             const void* tv, const void* tw, const void* te);

// 32-bit Morton keys and stable order (bbox: derive the box on device from x, y); keys_out
// holds the sorted keys when want_keys, else scratch. sort.hip
int morton_order(Device* d, hipStream_t s, int64_t n, const double* x, const double* y,
                 bool bbox, double x0, double y0, double inv, uint32_t* keys_out,
                 uint32_t* order_out, Workspace* ws, bool want_keys);

int panels_on_points_dev(Device* d, hipStream_t s, int64_t nnodes, const double* nx,
                         const double* ny, int64_t np, const uint32_t* idx, const double* vs,
                         const double* ss, int64_t nt, const double* tx, const double* ty,
                         double* tu, double* tv);

int points_on_panels_dev(Device* d, hipStream_t s, int64_t ns, const double* sx, const double* sy,
                         const double* ss, int64_t nnodes, const double* nx, const double* ny,
                         int64_t np, const uint32_t* idx, double* pu, double* pv);

int bem_assemble_dev(Device* d, hipStream_t s, int64_t nnodes, const double* nx, const double* ny,
                     int64_t np, const uint32_t* idx, int nunk, int augmented,
                     const double* urot_u, const double* urot_v, double vol, double* A,
                     int64_t lda);

int bem_factor_dev(Device* d, hipStream_t s, int64_t n, const double* A, int64_t lda);

// blocked LU with partial pivoting (lu.hip), n <= lu_max_order(); ipiv 1-based, info device int
int64_t lu_max_order();
int lu_factor_dev(Device* d, hipStream_t s, int n, double* A, int lda, int* ipiv, int* perm,
                  int* info);
// solves with those factors (lusolve.hip): lu_prepare_solve once per factorisation
int lu_prepare_solve(Device* d, hipStream_t s, int n, const double* lu);
int lu_solve_dev(Device* d, hipStream_t s, int n, const double* lu, const int* perm,
                 const double* b, double* x);
// bytes of the kSolveTmp slot that lu_solve_dev and matvec_dev take for order n
size_t solve_scratch(int64_t n);
// x = A b, A n x n column-major
int matvec_dev(Device* d, hipStream_t s, int n, const double* a, const double* b, double* x);
int bem_solve_dev(Device* d, hipStream_t s, int64_t n, const double* b, double* x);

// o_f[order[i]] += sum over chunks c of part[(f nchunk + c) nt + i], for the nf (2 to 4) components f
// (order null: the identity). gate: a device flag (or null); unless it is set to `open`, nothing is done.
// nbody.hip
int reduce_chunks(hipStream_t s, int64_t nchunk, int64_t nt, const uint32_t* order, int nf,
                  const double* part, double* o0, double* o1, double* o2, double* o3,
                  const int* gate = nullptr, int open = 1);

int rk_move_dev(hipStream_t s, int64_t n, double dt, int nstage, const double* w,
                const double* const* u, const double* const* v, const double* x0,
                const double* y0, double* x, double* y, double* uc, double* vc);

int adjoint_dev(Device* d, hipStream_t s, int core, int64_t ns, const double* sx,
                const double* sy, const double* ss, const double* sr, int64_t nt,
                const double* tx, const double* ty, const double* gu, const double* gv,
                double* gx, double* gy, double* gs, double* gr);

// the fp64 Gaussian velocity sum and its adjoint with the sources beyond the compact cutoff taken
// by clusters, to rounding (treecode.hip), and the sizes from which they are faster than the pair by
// pair sums. Where the cores hold so much of the set that they are not, which only the device knows, the
// same calls sum pair by pair.
int64_t sum64_targets(const Device* d, int64_t ns, int64_t nt);  // targets in a workgroup of the pairs
constexpr int kAdjointTileS = 512, kAdjointTileT = 256;          // particles and probes in a tile of theirs
bool gauss_clusters(const Device* d, int64_t ns, int64_t nt);
int gauss_tree_dev(Device* d, hipStream_t s, int64_t ns, const double* sx, const double* sy,
                   const double* ss, const double* sr, int64_t nt, const double* tx,
                   const double* ty, const double* tr, double* tu, double* tv);
bool gauss_adjoint_clusters(int64_t ns, int64_t nt);
int gauss_adjoint_tree_dev(Device* d, hipStream_t s, int64_t ns, const double* sx,
                           const double* sy, const double* ss, const double* sr, int64_t nt,
                           const double* tx, const double* ty, const double* gu,
                           const double* gv, double* gx, double* gy, double* gs, double* gr);

// The pair by pair forms of the two, launched behind a gate: they do nothing unless *gate (on the
// device) is set when they run. src, trg: records (x, y, strength, radius term) in order, those of the
// targets mapped to the outputs by torder (nbody.hip, adjoint.hip).
int gauss_pairs_gated(Device* d, hipStream_t s, int64_t ns, const void* src, int64_t nt,
                      const void* trg, bool radii, const uint32_t* torder, double* tu, double* tv,
                      const int* gate);
int adjoint_pairs_dev(Device* d, hipStream_t s, int core, int64_t ns, const double* sx,
                      const double* sy, const double* ss, const double* sr, int64_t nt,
                      const double* tx, const double* ty, const double* gu, const double* gv,
                      double* gx, double* gy, double* gs, double* gr, const int* gate);

// Gaussian vorticity of particles at targets (fp64, +=), device pointers
int vorticity_dev(Device* d, hipStream_t s, int64_t ns, const double* sx, const double* sy,
                  const double* ss, const double* sr, int64_t nt, const double* tx,
                  const double* ty, double* tw);

// particle/panel proximity (mode 0 nearest distances, 1 reflect, 2 clear), device pointers
int near_dev(Device* d, hipStream_t s, int mode, int method, double cutoff_mult, double ips,
             int64_t nnodes, const double* nx, const double* ny, int64_t np,
             const uint32_t* idx, const double* pnx, const double* pny, int64_t nt, double* tx,
             double* ty, double* ts, const double* tr, double* dist, double* value,
             int64_t* counts);

// host <-> device staging for the synchronous entry points
template <class T>
int upload(Device* d, Slot sl, const T* h, int64_t n, hipStream_t s, T** out) {
  void* p;
  O2D_TRY(slot(d, sl, sizeof(T) * (n > 0 ? n : 1), s, &p));
  if (n > 0) O2D_HIP(hipMemcpyAsync(p, h, sizeof(T) * n, hipMemcpyHostToDevice, s));
  *out = static_cast<T*>(p);
  return 0;
}

template <class T>
int download(T* h, const T* dptr, int64_t n, hipStream_t s) {
  if (n > 0) O2D_HIP(hipMemcpyAsync(h, dptr, sizeof(T) * n, hipMemcpyDeviceToHost, s));
  return 0;
}

// float host array -> double device array (through a float staging slot)
int upload_f2d(Device* d, Slot stage, Slot dst, const float* h, int64_t n, hipStream_t s,
               double** out);
// double device array -> float host array (through a float staging slot)
int download_d2f(Device* d, Slot stage, float* h, const double* dptr, int64_t n, hipStream_t s);

}  // namespace o2d
