// vb_ops.hpp -- per-transform-length launch table.  Each supported length N
// is compiled in its own translation unit (vb_n<N>.hip) so the build runs in
// parallel; the host pipeline picks the table of nx (x and y kernels) and the
// table of nz (z kernels) at solver creation.
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "vb_device.hpp"

namespace vb {

// Launch recording for batched launches.  While a Recorder is installed on
// the calling thread, the pipeline launchers append each launch (its kernel,
// its argument struct and its grid) instead of issuing it; the batched form
// then issues one launch per recorded position for all solves of a size
// group, with the solves' argument structs in a device table.
enum PipeOp {
  OP_XA_RS, OP_XA_F, OP_XA_S, OP_XA_SUMS, OP_Y_FWD, OP_Y_INV, OP_Y_FWD_GM, OP_ZLAP, OP_ZPREP,
  OP_ZS41, OP_ZS42, OP_ZS43, OP_ZS44, OP_ZS21, OP_ZS22, OP_FIN, OP_KEEP, OP_ZS44P, OP_RELAYOUT,
  OP_PL_ETD, OP_PL_SUMS, OP_PL_ROWSUMS
};
// x-kernel outputs: the partial sums of v, (v^2-1)^2 and f^2 only (k_xrow
// without its forward transform: the integrals of a field), tmp1 and f
// (Euler), tmp1 and s (spectral N), the partial sums of v and (v^2-1)^2 only
// (from P alone: k_xsums)
enum XaMode { XA_ROWSUMS = 0, XA_WITHF = 1, XA_WITHS = 2, XA_SUMS = 3 };
// modes of the plane kernel (k_plane)
enum PlaneMode { PL_ETD = 0, PL_SUMS = 1, PL_ROWSUMS = 2, PL_EULER = 3 };
struct RecLaunch {
  // issues the table form of the recorded kernel over `lanes` solves
  void (*launch_tab)(int op, const void* tab, dim3 grid, dim3 block, int lanes, hipStream_t s);
  int op;
  std::vector<unsigned char> args;
  dim3 grid, block;
};
struct Recorder {
  std::vector<RecLaunch> seq;
};
extern thread_local Recorder* g_recorder;

template <class A>
inline void record_launch(void (*tabfn)(int, const void*, dim3, dim3, int, hipStream_t), int op, const A& a,
                          dim3 grid, dim3 block) {
  RecLaunch r;
  r.launch_tab = tabfn;
  r.op = op;
  r.args.assign(reinterpret_cast<const unsigned char*>(&a), reinterpret_cast<const unsigned char*>(&a) + sizeof(A));
  r.grid = grid;
  r.block = block;
  g_recorder->seq.push_back(std::move(r));
}

template <typename T>
struct PlaneArgs {
  const cpx<T>* P;   // z-inverse of v^
  const cpx<T>* Q;   // z-inverse of -|k|^2 v^ (PL_SUMS: unused)
  cpx<T>* U;         // PL_ETD out: x,y-forward of tmp1 and eps^3 s (k_xrow's units),
  cpx<T>* U2;        // in the z kernels' group-major layout, column tile ztb
  double* part;      // [workgroup][3]
  double* dcpart;    // FP32 PL_ETD: [workgroup][2], or nullptr
  const cpx<T>* tw;
  Geo g;
  int ztb, pad;
  double eps, kappa, D;
  T* v;              // PL_EULER out: the real fields v and f, and the x,y-forward
  T* f;              // of f times inv_n in the row layout
  cpx<T>* W;
  double inv_n;
};

template <typename T> struct XaArgs;
template <typename T> struct XeArgs;
template <typename T> struct ZsArgs;

template <typename T>
struct SizeOps {
  int N;
  int sched;       // kernel schedule (z tile, x plan) this table launches
  int xr_passes;   // passes of the ETD x kernel's plan
  int xr_radix;    // radix of its first pass
  int xlanes;      // row pairs per x workgroup
  int ytile;       // columns per workgroup of the z stage kernels
  int ctile;       // columns per workgroup of the y passes and the z Laplacian
  int ythreads;    // threads per y / z workgroup
  void (*xr2c_d)(const double* in, cpx<T>* out, long long npairs, const cpx<T>* tw, double scl, const Geo& g,
                 hipStream_t s);
  void (*xr2c)(const T* in, cpx<T>* out, long long npairs, const cpx<T>* tw, double scl, const Geo& g, hipStream_t s);
  void (*xc2r_d)(const cpx<T>* in, double* out, long long npairs, const cpx<T>* tw, const Geo& g, hipStream_t s);
  void (*xc2r)(const cpx<T>* in, T* out, long long npairs, const cpx<T>* tw, const Geo& g, hipStream_t s);
  void (*xa)(const XaArgs<T>& a, int mode, hipStream_t s);   // mode: XaMode
  void (*xe)(const XeArgs<T>& a, hipStream_t s);
  // fin (or nullptr): integrals evaluated by extra workgroups of the launch
  void (*ypass)(cpx<T>* b0, cpx<T>* b1, int narr, int sign, const Geo& g, const cpx<T>* tw, const FinArgs* fin,
                hipStream_t s);
  // forward y pass of two arrays into the z kernels' group-major layout of a
  // grid of nzt planes (g: the planes of b0, b1, which start at plane 0 of o0, o1)
  void (*ypass_gm)(const cpx<T>* b0, const cpx<T>* b1, cpx<T>* o0, cpx<T>* o1, int ztb, int nzt, const Geo& g,
                   const cpx<T>* tw, const FinArgs* fin, hipStream_t s);
  void (*zpass)(cpx<T>* b, int sign, const Geo& g, const cpx<T>* tw, hipStream_t s);
  // fin (or nullptr): integrals evaluated by one extra workgroup of the launch
  void (*zlap)(cpx<T>* b, const Geo& g, const cpx<T>* tw, const FinArgs* fin, hipStream_t s);
  void (*zprep)(const cpx<double>* vh, cpx<T>* P, cpx<T>* Q, double* part, double* dc, const Geo& g, const cpx<T>* tw,
                hipStream_t s);
  // stg 1..sch; 5: the probe form of ETDRK4 stage 4 (V and A of the result
  // only: no state store, P alone)
  void (*zstage)(const ZsArgs<T>& a, int sch, int stg, hipStream_t s);
  // the prefix with a whole xy plane in LDS (vb_plane.hpp), mode: PlaneMode;
  // nullptr where a plane does not fit.  Its partials are one set per
  // workgroup: nz of them (PL_SUMS: nz / sums_planes).
  int sums_planes;
  bool plane_euler;   // it has the mode PL_EULER
  int plane_min_nz;   // the planes from which it is used
  void (*plane)(const PlaneArgs<T>& a, int mode, hipStream_t s);
  // The Forward-Euler update with x and y of a plane in one kernel (nullptr
  // where a plane does not fit; nz partials of rhs^2), used from xe_min_nz planes
  // on, and the z pass that
  // follows it: the new state from W, and the prepared field's P, Q
  int xe_min_nz;
  void (*xe_plane)(const XeArgs<T>& a, const Geo& g, hipStream_t s);
  void (*zeuler)(const cpx<T>* W, cpx<double>* uh, cpx<T>* P, cpx<T>* Q, double* part, double* dc, const Geo& g,
                 const cpx<T>* tw, hipStream_t s);
  // out of place z pass of a layout gi into a layout go, the input times op
  // (ZmOp; sign < 0: ZM_ONE only)
  void (*zmul)(const cpx<T>* in, cpx<T>* out, int sign, int op, const Geo& gi, const Geo& go, const cpx<T>* tw,
               hipStream_t s);
  // x and y transforms of whole planes in LDS (k_pair), real rows to half
  // spectra times scl and back; nullptr where a plane does not fit.  Used from
  // pair_r2c_nz and pair_c2r_nz planes on.
  int pair_r2c_nz, pair_c2r_nz;
  void (*pair_r2c)(const T* u, cpx<T>* so, double scl, const Geo& g, const cpx<T>* tw, hipStream_t s);
  void (*pair_c2r)(const cpx<T>* si, T* uo, const Geo& g, const cpx<T>* tw, hipStream_t s);
};

// launch table of kernel schedule sc of length N (nullptr if not compiled),
// and the number of schedules compiled for it
template <typename T, int N> const SizeOps<T>* ops_for(int sc);
template <typename T, int N> int sched_count();

#define VB_SIZE_LIST(X) X(16) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384) X(512)

#define VB_DECL(n)                                              \
  template <> const SizeOps<double>* ops_for<double, n>(int);   \
  template <> const SizeOps<float>* ops_for<float, n>(int);     \
  template <> int sched_count<double, n>();                     \
  template <> int sched_count<float, n>();
VB_SIZE_LIST(VB_DECL)
#undef VB_DECL

template <typename T>
inline int sched_count_of(int N) {
  switch (N) {
#define VB_CASE(n) case n: return sched_count<T, n>();
    VB_SIZE_LIST(VB_CASE)
#undef VB_CASE
    default: return 0;
  }
}

// The schedule in use for (precision, N): the autotuner's or the caller's
// choice (vb_schedule_set), else 0; a thread's override (>= 0) wins while
// set (the autotuner builds its candidate solvers under one).
int sched_selected(bool fp32, int N);
extern thread_local int g_sched_override;

template <typename T>
inline const SizeOps<T>* get_ops(int N, int sc) {
  switch (N) {
#define VB_CASE(n) case n: return ops_for<T, n>(sc);
    VB_SIZE_LIST(VB_CASE)
#undef VB_CASE
    default: return nullptr;
  }
}
template <typename T>
inline const SizeOps<T>* get_ops(int N) {
  int sc = g_sched_override >= 0 ? g_sched_override : sched_selected(sizeof(T) == 4, N);
  if (sc >= sched_count_of<T>(N)) sc = 0;
  return get_ops<T>(N, sc);
}

// The z kernels' table of a grid: under a large plane the short lengths take the
// wide tile on the default plan (kWideZ, tbw_wide) in place of one wave's columns.
// There the combines stream from memory, and 64-byte pieces of P and Q cost more
// than the barriers and the longer threads.  us per step, the narrow tile / this:
//   FP32 192 x 64 480 / 466, 256 x 64 661 / 645, 512 x 64 2485 / 2300, batches of 8
//   of 192 x 64 2490 / 2375, 4 of 256 x 64 2225 / 2100; 256 x 32 447 / 436;
//   128 x 32 215 / 255
//   FP64 192 x 64 710 / 704, 512 x 64 4290 / 4010; 256 x 128 1797 / 1801, 384 x 128
//   4590 / 4395, two of 256 x 128 3890 / 3750, but 192 x 128 1209 / 1222; 512 x 32
//   2155 / 2120, but 256 x 32 562 / 592
// mixed: the FP64 integrals of a mixed solver, whose tile should be the FP32 one's
// (a pass regroups the state where it is not).
constexpr int kWideZ = 8;   // a schedule number past those that can be selected
template <typename T>
inline const SizeOps<T>* get_zops(int nx, int nz, bool mixed) {
  const SizeOps<T>* const o = get_ops<T>(nz);
  const int from = sizeof(T) == 4 || mixed || nz == 64 ? 192 : nz == 128 ? 256 : 384;
  if (nx < from || o != get_ops<T>(nz, 0)) return o;   // (a schedule that was chosen stays)
  const SizeOps<T>* const w = get_ops<T>(nz, kWideZ);
  return w ? w : o;
}

inline bool size_supported(int N) {
  switch (N) {
#define VB_CASE(n) case n: return true;
    VB_SIZE_LIST(VB_CASE)
#undef VB_CASE
    default: return false;
  }
}

}  // namespace vb
