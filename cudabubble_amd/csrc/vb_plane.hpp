// vb_plane.hpp -- the ETD prefix of one field with a whole xy plane in LDS.
//
// For grids whose plane of v and lap v (as half spectra: N x (N + 2) complex
// values) fits the 160 KB of LDS, the y-inverse, the x kernel (k_xrow) and the
// y-forward run as one kernel, one workgroup per z: P and Q are read once and
// the spectra of tmp1 and s written once, instead of three kernels that each
// read and write both arrays.
//
// What bounds it: the chain of its phases (one workgroup per CU at most at the
// larger lengths).  So the transforms stay inside a wave (no workgroup barrier
// but between the phases), the twiddles are read from LDS, the Nyquist columns
// have a wave of their own, and the sums go through DPP moves.  Measured: 32^3
// FP64 6.2 us against 13.1 for the three kernels, 128^3 FP32 (k_plane2) 19
// against 33; a penalty-drift step of 32^3 FP64, 64^3 FP32, 128^3 FP32 173 -> 104,
// 195 -> 138, 489 -> 388 us (with the combines evaluating the integrals and their
// wave tiles), batches of 16 x 32^3, 16 x 64^3, 12 x 128^3 302 -> 186, 712 ->
// 576, 3465 -> 2800 us.
#pragma once
#include "vb_kernels.hpp"

namespace vb {

template <typename T, int N>
struct PlaneCfg {
  // plans with every transform inside one wave: the two-pass plan at 128, 12 x
  // 4 (x 2) at 48 and 96, else the default
  static constexpr int V = N == 128 ? 1 : (N == 48 || N == 96) ? 3 : 0;
  static constexpr int E = N <= 128 ? Plan<N, V>::E : 8;
  static constexpr int TF = N / E;
  static constexpr int NT = N * TF;                 // TF lanes per row, and per column of P and Q but Nyquist
  // the two Nyquist columns are a wave's of their own, so that no wave runs
  // two column transforms one after the other, where there is room for one
  static constexpr int XW = NT + 64 <= 1024 ? 1 : 0;
  static constexpr int NA = NT + 64 * XW;           // threads of the workgroup
  static constexpr int PS = (N == 96 || N == 128) ? 4 : 3;
  // a row holds the N points of its transform, or its N + 2 half-spectrum
  // modes: P[0, N/2), Q[0, N/2), then the two Nyquist modes
  static constexpr int LL = N + 2 + ((N + 1) >> PS);
  static constexpr int bytes = N * LL * int(sizeof(cpx<T>));
  static constexpr bool ok = N <= 128 && NT <= 1024 && bytes + N * int(sizeof(cpx<T>)) + 1024 <= 160 * 1024;
};

// Element (ky, kx) of a plane of half-spectrum rows (see Geo).
__device__ __forceinline__ int plane_pos(const Geo& g, int ky, int kx) {
  return (g.nq >= 0 && kx == g.nx / 2) ? int(g.nq) + ky : ky * g.pitch + kx;
}

// PL_ETD: the prefix of a stage (k_ypass, k_xrow and the group-major k_ypass
// in one; the same terms and units as k_xrow).  PL_EULER: the Euler paths'
// (k_ypass, k_xa and the y-forward of f): v and f stored, pointwise terms in
// FP64 as in k_xa.  PL_ROWSUMS: the partial sums
// of v, (v^2-1)^2 and f^2 only.  PL_SUMS: the partial sums of v and (v^2-1)^2
// from P alone, two planes per workgroup, the second in Q's place.
template <typename T, int N, int MODE, bool TAB = false>
__global__ void __launch_bounds__((PlaneCfg<T, N>::NA)) k_plane(PlaneArgs<T> a0, const PlaneArgs<T>* tab) {
  using C = PlaneCfg<T, N>;
  constexpr int E = C::E, TF = C::TF, LL = C::LL, PS = C::PS, V = C::V, NT = C::NT, NA = C::NA, CW = 64 / TF,
                H = N / 2;
  static_assert(64 % TF == 0 && N % CW == 0, "whole lane groups per wave");
  const PlaneArgs<T> a = TAB ? tab[blockIdx.z] : a0;
  const Geo& g = a.g;
  __shared__ cpx<T> sm[N * LL];
  __shared__ cpx<T> tw[N];
  __shared__ double red[5 * (NA / 64)];
  const int z = MODE == PL_SUMS ? 2 * int(blockIdx.x) : pair_item(int(blockIdx.x), int(gridDim.x));
  const cpx<T>* const pA = a.P + (long long)z * g.pp;
  const cpx<T>* const pB = MODE == PL_SUMS ? pA + g.pp : a.Q + (long long)z * g.pp;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  // columns: CW consecutive ones per wave; column c of [0, N) is P's kx = c,
  // then Q's; the two Nyquist columns are the extra wave's, or (XW = 0) the
  // first wave's second ones
  const int cj = lane / CW, cc = wave * CW + lane % CW;
  auto slot = [](int c) { return c + (c >> PS); };
  // which array a column is of: by wave where no wave has both
  auto second = [&](int c) { return H % CW == 0 && c < N ? wave * CW >= H : c < N ? c >= H : c > N; };
  auto load = [&](cpx<T>* x, int c) {
    const cpx<T>* const p = second(c) ? pB : pA;
    const int kx = c < N ? c % H : H;
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = p[unsigned(plane_pos(g, cj + TF * e, kx))];
  };
  auto inv = [&](cpx<T>* x, int c) {
    PlaneCol<T, LL> col{sm + slot(c)};
    fft<T, N, +1, V>(x, cj, tw, col);
#pragma unroll
    for (int e = 0; e < E; ++e) col(cj + TF * e) = x[e];
  };
  const bool main = wave < NT / 64, act = main || lane % CW < 2;
  {
    cpx<T> x[E];
    if (act) load(x, cc);
    // the twiddles from LDS: a pass's loads of them would be a round trip to L2
    if (threadIdx.x < N) tw[threadIdx.x] = a.tw[threadIdx.x];
    __syncthreads();
    if (act) inv(x, cc);
    if (!C::XW && wave == 0 && lane % CW < 2) {
      load(x, N + lane % CW);
      inv(x, N + lane % CW);
    }
  }
  __syncthreads();
  constexpr int K = (MODE == PL_ETD && sizeof(T) == 4) ? 5 : 3;
  double acc[K] = {};
  if (main) {
    const int r = threadIdx.x / TF, j = threadIdx.x % TF;
    PlaneRow<T, PS> row{sm + r * LL};
    cpx<T> x[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      // pack2 over the row's slots
      const int p = j + TF * e;
      const bool mir = p > H;
      const int k = mir ? N - p : p;
      cpx<T> u = row(k == H ? N : k), w = row(k == H ? N + 1 : H + k);
      if (k == 0 || k == H) { u.y = T(0); w.y = T(0); }
      if (mir) { u.y = -u.y; w.y = -w.y; }
      x[e] = mk<T>(u.x - w.y, u.y + w.x);
    }
    row.sync();
    fft<T, N, +1, V>(x, j, tw, row);
    const double eps = a.eps, kappa = a.kappa, ieps = 1.0 / eps, D = a.D;
    T ts[5] = {T(0), T(0), T(0), T(0), T(0)};
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if constexpr (MODE == PL_SUMS) {
        const T v0 = x[e].x, v1 = x[e].y;
        const double w0 = double(v0 * v0 - T(1)), w1 = double(v1 * v1 - T(1));
        acc[0] += double(v0) + double(v1);
        acc[1] += w0 * w0 + w1 * w1;
      } else if constexpr (MODE == PL_EULER) {
        const double v = double(x[e].x), lv = double(x[e].y), w = v * v - 1.0, f = -lv * eps + w * v * ieps;
        acc[0] += v; acc[1] += w * w; acc[2] += f * f;
        const long long i = ((long long)z * N + r) * N + j + TF * e;
        a.v[i] = T(v);
        a.f[i] = T(f);
        x[e] = mk<T>(T(f), T(0));
      } else {
        const T v = x[e].x, lv = x[e].y;
        const T w = v * v - T(1);
        const T f = -lv * T(eps) + w * v * T(ieps);                               // f_kernel, Calc.cu:160
        const T t1 = v * (w - T(kappa));                                          // nld_kernel1, Calc.cu:270
        const T sv = T(D) * t1 + (T(3 * eps) * v * v - T(eps * (D + 1))) * f;     // Calc.cu:282, times eps^3
        if constexpr (sizeof(T) == 4) {
          ts[0] += v; ts[1] += w * w; ts[2] += f * f; ts[3] += t1; ts[4] += sv;
        } else {
          acc[0] += double(v); acc[1] += double(w) * double(w); acc[2] += double(f) * double(f);
        }
        x[e] = mk<T>(t1, sv);
      }
    }
    if constexpr ((MODE == PL_ETD || MODE == PL_ROWSUMS) && sizeof(T) == 4) {
#pragma unroll
      for (int q = 0; q < K; ++q) acc[q] = double(ts[q]);
    }
    if constexpr (MODE == PL_ETD || MODE == PL_EULER) {
      constexpr int NH = H + 1, U = (NH + TF - 1) / TF;
      fft<T, N, -1, V>(x, j, tw, row);
#pragma unroll
      for (int e = 0; e < E; ++e) row(j + TF * e) = x[e];
      row.sync();
      // unpack_store without SCALE, over the row's own slots
      cpx<T> ua[U], ub[U];
#pragma unroll
      for (int i = 0; i < U; ++i) {
        const int k = j + TF * i;
        if (k < NH) {
          const cpx<T> zk = row(k), zm = row(k == 0 ? 0 : N - k);
          ua[i] = mk<T>(zk.x + zm.x, zk.y - zm.y);
          ub[i] = mk<T>(zk.y + zm.y, zm.x - zk.x);
          if constexpr (MODE == PL_EULER) ua[i] = scale(ua[i], T(0.5) * T(a.inv_n));
        }
      }
      row.sync();
#pragma unroll
      for (int i = 0; i < U; ++i) {
        const int k = j + TF * i;
        if (k < NH) {
          row(k == H ? N : k) = ua[i];
          if constexpr (MODE == PL_ETD) row(k == H ? N + 1 : H + k) = ub[i];
        }
      }
    }
  }
  wave_part<K, NA>(acc, red);
  __syncthreads();
  if (threadIdx.x < K) {
    const double s = wave_total<NA>(red, threadIdx.x);
    if (threadIdx.x < 3) a.part[3 * (long long)blockIdx.x + threadIdx.x] = s;
    else if (a.dcpart) a.dcpart[2 * (long long)blockIdx.x + threadIdx.x - 3] = s;
  }
  if constexpr (MODE == PL_EULER) {
    auto fwd = [&](int c) {   // f's columns: kx = c, or Nyquist
      PlaneCol<T, LL> col{sm + slot(c)};
      cpx<T> x[E];
#pragma unroll
      for (int e = 0; e < E; ++e) x[e] = col(cj + TF * e);
      col.sync();
      fft<T, N, -1, V>(x, cj, tw, col);
      cpx<T>* const o = a.W + (long long)z * g.pp;
#pragma unroll
      for (int e = 0; e < E; ++e) o[unsigned(plane_pos(g, cj + TF * e, c < H ? c : H))] = x[e];
    };
    if (act && (cc < H || cc == N)) fwd(cc);
    if (!C::XW && wave == 0 && lane % CW == 0) fwd(N);
  }
  if constexpr (MODE == PL_ETD) {
    auto fwd = [&](int c) {
      PlaneCol<T, LL> col{sm + slot(c)};
      cpx<T> x[E];
#pragma unroll
      for (int e = 0; e < E; ++e) x[e] = col(cj + TF * e);
      col.sync();
      fft<T, N, -1, V>(x, cj, tw, col);
      const int kx = c < N ? c % H : H;
      cpx<T>* const out = second(c) ? a.U2 : a.U;
      if (g.aligned && c < N) {
        // ky = cj + TF e: one ky step is one row of column groups of all z
        const unsigned o = unsigned(gm_index(g, a.ztb, z, cj, kx)),
                       st = unsigned(((H >> __builtin_ctz((unsigned)a.ztb)) * TF) * g.nz * a.ztb);
#pragma unroll
        for (int e = 0; e < E; ++e) out[o + e * st] = x[e];
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e) out[unsigned(gm_index(g, a.ztb, z, cj + TF * e, kx))] = x[e];
      }
    };
    if (act) fwd(cc);
    if (!C::XW && wave == 0 && lane % CW < 2) fwd(N + lane % CW);
  }
}

// ---------------------------------------------------------------------------
// The x and y transforms of one real plane in LDS (the Calc level's r2c and
// c2r): two real rows travel as one complex transform, and a row pair's storage
// holds its N points or its two half spectra.  A 3-D transform is then this
// kernel and a z pass, two sweeps of the data instead of three: 32^3 FP64
// forward and back 45 -> 35 us with the copy of c2r's input gone as well, an
// FP64 c2r at 128^3 about 31 -> 25 us.
// ---------------------------------------------------------------------------
template <typename T, int N>
struct PairCfg {
  static constexpr int V = (N == 128 || N == 192) ? 1 : (N == 48 || N == 96) ? 3 : 0;
  static constexpr bool fits = N <= 128 || (N == 192 && sizeof(T) == 4);
  static constexpr int E = fits ? Plan<N, V>::E : 8;
  static constexpr int TF = N / E;
  static constexpr int CW = fits ? 64 / TF : 1;                // columns, and row pairs, per wave
  static constexpr int NA = 64 * ((N / 2 + CW) / CW);           // lanes for N / 2 + 1 columns
  static constexpr int PS = N >= 96 ? 4 : 3;
  static constexpr int LL = N + 2 + ((N + 1) >> PS);
  static constexpr int bytes = N / 2 * LL * int(sizeof(cpx<T>)) + N * int(sizeof(cpx<T>));
  static constexpr bool ok = fits && NA <= 1024 && bytes + 512 <= 160 * 1024;
};

// column kx of a plane of row pairs: position y is row y % 2 of pair y / 2
template <typename T, int LL>
struct PairCol {
  cpx<T>* base;
  int odd;   // offset of the odd row's slot
  __device__ __forceinline__ cpx<T>& operator()(int pos) const { return base[(pos >> 1) * LL + (pos & 1) * odd]; }
  __device__ __forceinline__ void sync() const { wave_sync(); }
};

template <typename T>
struct PairArgs {
  const T* u;          // real rows [nz][ny][nx] (r2c: in)
  T* uo;               // (c2r: out)
  const cpx<T>* si;    // half spectra, x and y transformed (c2r: in)
  cpx<T>* so;          // (r2c: out, times scl)
  const cpx<T>* tw;
  Geo g;
  double scl;
};

template <typename T, int N, int S>
__global__ void __launch_bounds__((PairCfg<T, N>::NA)) k_pair(PairArgs<T> a) {
  using C = PairCfg<T, N>;
  constexpr int E = C::E, TF = C::TF, LL = C::LL, PS = C::PS, V = C::V, CW = C::CW, H = N / 2;
  static_assert(64 % TF == 0, "transforms inside a wave");
  const Geo& g = a.g;
  __shared__ cpx<T> sm[H * LL];
  __shared__ cpx<T> tw[N];
  const int z = int(blockIdx.x);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int cj = lane / CW, kx = wave * CW + lane % CW;    // column
  const int r = threadIdx.x / TF, j = threadIdx.x % TF;    // row pair
  PlaneRow<T, PS> row{sm + (r < H ? r : 0) * LL};
  auto slot = [](int c) { return c + (c >> PS); };
  const PairCol<T, LL> col{sm + slot(kx < H ? kx : N), kx < H ? slot(H + kx) - slot(kx) : slot(N + 1) - slot(N)};
  const bool isrow = r < H, iscol = kx <= H;
  cpx<T> x[E];
  if constexpr (S < 0) {
    if (isrow) {
      const T* const u = a.u + ((long long)z * N + 2 * r) * N;
#pragma unroll
      for (int e = 0; e < E; ++e) x[e] = mk<T>(u[j + TF * e], u[N + j + TF * e]);
    }
    for (int i = threadIdx.x; i < N; i += C::NA) tw[i] = a.tw[i];
    __syncthreads();
    if (isrow) {
      fft<T, N, -1, V>(x, j, tw, row);
      constexpr int NH = H + 1, U = (NH + TF - 1) / TF;
#pragma unroll
      for (int e = 0; e < E; ++e) row(j + TF * e) = x[e];
      row.sync();
      cpx<T> ua[U], ub[U];
      const T h = T(0.5) * T(a.scl);
#pragma unroll
      for (int i = 0; i < U; ++i) {
        const int k = j + TF * i;
        if (k < NH) {
          const cpx<T> zk = row(k), zm = row(k == 0 ? 0 : N - k);
          ua[i] = mk<T>((zk.x + zm.x) * h, (zk.y - zm.y) * h);
          ub[i] = mk<T>((zk.y + zm.y) * h, (zm.x - zk.x) * h);
        }
      }
      row.sync();
#pragma unroll
      for (int i = 0; i < U; ++i) {
        const int k = j + TF * i;
        if (k < NH) {
          row(k == H ? N : k) = ua[i];
          row(k == H ? N + 1 : H + k) = ub[i];
        }
      }
    }
    __syncthreads();
    if (iscol) {
#pragma unroll
      for (int e = 0; e < E; ++e) x[e] = col(cj + TF * e);
      col.sync();
      fft<T, N, -1, V>(x, cj, tw, col);
      cpx<T>* const o = a.so + (long long)z * g.pp;
#pragma unroll
      for (int e = 0; e < E; ++e) o[unsigned(plane_pos(g, cj + TF * e, kx))] = x[e];
    }
  } else {
    if (iscol) {
      const cpx<T>* const i0 = a.si + (long long)z * g.pp;
#pragma unroll
      for (int e = 0; e < E; ++e) x[e] = i0[unsigned(plane_pos(g, cj + TF * e, kx))];
    }
    for (int i = threadIdx.x; i < N; i += C::NA) tw[i] = a.tw[i];
    __syncthreads();
    if (iscol) {
      fft<T, N, +1, V>(x, cj, tw, col);
#pragma unroll
      for (int e = 0; e < E; ++e) col(cj + TF * e) = x[e];
    }
    __syncthreads();
    if (isrow) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int p = j + TF * e;
        const bool mir = p > H;
        const int k = mir ? N - p : p;
        cpx<T> u = row(k == H ? N : k), w = row(k == H ? N + 1 : H + k);
        if (k == 0 || k == H) { u.y = T(0); w.y = T(0); }
        if (mir) { u.y = -u.y; w.y = -w.y; }
        x[e] = mk<T>(u.x - w.y, u.y + w.x);
      }
      row.sync();
      fft<T, N, +1, V>(x, j, tw, row);
      T* const u = a.uo + ((long long)z * N + 2 * r) * N;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        u[j + TF * e] = x[e].x;
        u[N + j + TF * e] = x[e].y;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The prefix with two rows travelling as one transform (k_pair's storage): half
// the rows and columns per array, so a workgroup has half the waves of k_plane's
// and each has twice the phases.  Where both planes fit LDS (two) they go through
// a phase together; else (FP64 at 128) the plane of P goes through y and x first,
// its v kept in registers, then Q's, then the spectra of tmp1 and of s one after
// the other.  The same arguments and units as k_plane.
//
// A workgroup does not get faster with fewer of them, so a launch whose last
// round of planes fills at most half of the 256 CUs gives these planes two
// workgroups each (nsplit): both invert P and Q and take the pointwise terms, one
// transforms tmp1 and writes the sums, the other s; the second read of P and Q
// comes from the XCD's L2.  What remains is arithmetic, latency and LDS: in a
// batch of 12 x 128^3 FP32 the SIMDs issue VALU work in 48 % of the cycles and the
// waves wait in 35 % of theirs (one solve: 37 and 29).  FP64 at 128 spills 25
// registers: nine waves, the Nyquist column's being the ninth, leave 168 each.
// Measured, us per step:
//   128^3 FP64 drift: three kernels 627, one workgroup per plane 606, two 556;
//     batches of 3 and 4 (the rest of 384 split; 512) 1375 -> 1303, 1594
//   128^3 FP32 drift: k_plane 418, here 388; batches of 2, 3, 12: 572, 863,
//     2832 -> 572, 832, 2800
//   96^3 FP64: k_plane 414, here 380; batches of 2, 6: 605, 1445 -> 589, 1401
//   64^3 FP32: 138 both; batches of 6, 16: 307, 617 -> 287, 577
// k_plane stays at the others, k_plane / here: 96^3 FP32 288 / 287, batches of 2
// and 6 363, 822 / 385, 880; 64^3 FP64 172 / 171, a batch of 4 284 / 299; 48^3 FP64
// 171 / 181, FP32 156 / 167, 4 of FP64 242 / 269; 32^3 FP64 98 / 104, FP32 97 / 103,
// 16 of FP64 232 / 247.  (FP32 at 192 fits as well but spills 78 registers: 76 us a
// launch against 75.)  PL_SUMS takes one plane per workgroup here; it and
// PL_ROWSUMS run here only where k_plane does not fit.
// ---------------------------------------------------------------------------
template <typename T, int N>
struct Plane2Cfg {
  static constexpr bool ok = N == 128 || N == (sizeof(T) == 4 ? 64 : 96);
  static constexpr bool two = sizeof(T) == 4 || N <= 96;   // both planes do fit
};

// Planes from which the plane kernels are the faster ones: a workgroup's time
// does not shrink with fewer of them.  128 x 128 x nz drift steps, plane kernels
// against three kernels, us: FP32 nz = 16 213 / 160, 32 246 / 215, 48 297 / 285,
// 64 (one workgroup per plane) 343 / 345, 128 388 / 459; FP64 nz = 32 351 / 262,
// 64 399 / 361, 96 558 / 562, 128 556 / 627, 192 878 / 1023.  At the shorter
// lengths they won at every depth measured (16 and up).
template <typename T, int N> constexpr int plane_min_nz() { return N < 128 ? 0 : sizeof(T) == 8 ? 128 : 64; }

template <typename T, int N, int MODE, bool TAB = false>
__global__ void __launch_bounds__((PairCfg<T, N>::NA)) k_plane2(PlaneArgs<T> a0, const PlaneArgs<T>* tab,
                                                                    int nsplit) {
  using C = PairCfg<T, N>;
  constexpr int E = C::E, TF = C::TF, LL = C::LL, PS = C::PS, V = C::V, CW = C::CW, NA = C::NA, H = N / 2;
  // the last nsplit solves have two workgroups per plane: the first writes
  // tmp1's spectra and the sums, the second, at the end of the grid, s's
  const int lanes = int(gridDim.z) - nsplit, second = int(blockIdx.z) >= lanes;
  const int lane_z = second ? int(blockIdx.z) - nsplit : int(blockIdx.z);
  const bool split = lane_z >= lanes - nsplit;
  const PlaneArgs<T> a = TAB ? tab[lane_z] : a0;
  const Geo& g = a.g;
  // FP32: a plane each for P and Q, tmp1 and s; FP64: one, in turn
  constexpr bool TWO = Plane2Cfg<T, N>::two;
  __shared__ cpx<T> sm[(TWO ? 2 : 1) * H * LL];
  __shared__ cpx<T> tw[N];
  constexpr int K = (MODE == PL_ETD && sizeof(T) == 4) ? 5 : 3;
  __shared__ double red[K * (NA / 64)];
  const int z = pair_item(int(blockIdx.x), int(gridDim.x));
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int cj = lane / CW, kx = wave * CW + lane % CW;    // column
  const int r = threadIdx.x / TF, j = threadIdx.x % TF;    // row pair
  constexpr int B2 = TWO ? H * LL : 0;
  const PlaneRow<T, PS> row1{sm + (r < H ? r : 0) * LL}, row2{row1.base + B2};
  auto slot = [](int c) { return c + (c >> PS); };
  const PairCol<T, LL> col1{sm + slot(kx < H ? kx : N), kx < H ? slot(H + kx) - slot(kx) : slot(N + 1) - slot(N)},
      col2{col1.base + B2, col1.odd};
  const bool isrow = r < H, iscol = kx <= H;
  const long long pz = (long long)z * g.pp;

  auto col_load = [&](cpx<T>* x, const cpx<T>* src) {
    if (iscol) {
#pragma unroll
      for (int e = 0; e < E; ++e) x[e] = src[unsigned(plane_pos(g, cj + TF * e, kx))];
    }
  };
  auto col_inv = [&](cpx<T>* x, const PairCol<T, LL>& col) {
    if (iscol) {
      fft<T, N, +1, V>(x, cj, tw, col);
#pragma unroll
      for (int e = 0; e < E; ++e) col(cj + TF * e) = x[e];
    }
  };
  auto row_inv = [&](cpx<T>* x, const PlaneRow<T, PS>& row) {   // two real rows, as re and im
    if (isrow) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int p = j + TF * e;
        const bool mir = p > H;
        const int k = mir ? N - p : p;
        cpx<T> u = row(k == H ? N : k), w = row(k == H ? N + 1 : H + k);
        if (k == 0 || k == H) { u.y = T(0); w.y = T(0); }
        if (mir) { u.y = -u.y; w.y = -w.y; }
        x[e] = mk<T>(u.x - w.y, u.y + w.x);
      }
      row.sync();
      fft<T, N, +1, V>(x, j, tw, row);
    }
  };
  auto row_fwd = [&](cpx<T>* x, const PlaneRow<T, PS>& row) {
    if (isrow) {
      constexpr int NH = H + 1, U = (NH + TF - 1) / TF;
      fft<T, N, -1, V>(x, j, tw, row);
#pragma unroll
      for (int e = 0; e < E; ++e) row(j + TF * e) = x[e];
      row.sync();
      cpx<T> ua[U], ub[U];
#pragma unroll
      for (int i = 0; i < U; ++i) {
        const int k = j + TF * i;
        if (k < NH) {
          const cpx<T> zk = row(k), zm = row(k == 0 ? 0 : N - k);
          ua[i] = mk<T>(zk.x + zm.x, zk.y - zm.y);
          ub[i] = mk<T>(zk.y + zm.y, zm.x - zk.x);
        }
      }
      row.sync();
#pragma unroll
      for (int i = 0; i < U; ++i) {
        const int k = j + TF * i;
        if (k < NH) {
          row(k == H ? N : k) = ua[i];
          row(k == H ? N + 1 : H + k) = ub[i];
        }
      }
    }
  };
  auto col_fwd = [&](const PairCol<T, LL>& col, cpx<T>* out) {
    if (iscol) {
      cpx<T> y[E];
#pragma unroll
      for (int e = 0; e < E; ++e) y[e] = col(cj + TF * e);
      col.sync();
      fft<T, N, -1, V>(y, cj, tw, col);
      if (g.aligned && kx < H) {
        const unsigned o = unsigned(gm_index(g, a.ztb, z, cj, kx)),
                       st = unsigned(((H >> __builtin_ctz((unsigned)a.ztb)) * TF) * g.nz * a.ztb);
#pragma unroll
        for (int e = 0; e < E; ++e) out[o + e * st] = y[e];
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e) out[unsigned(gm_index(g, a.ztb, z, cj + TF * e, kx))] = y[e];
      }
    }
  };

  cpx<T> v[E], x[E];
  col_load(x, a.P + pz);
  if constexpr (TWO && MODE != PL_SUMS) col_load(v, a.Q + pz);
  for (int i = threadIdx.x; i < N; i += NA) tw[i] = a.tw[i];
  __syncthreads();
  col_inv(x, col1);
  if constexpr (MODE == PL_SUMS) {
    __syncthreads();
    row_inv(x, row1);
  } else if constexpr (TWO) {
    col_inv(v, col2);
    __syncthreads();
    row_inv(v, row1);
    row_inv(x, row2);    // lap v
  } else {
    __syncthreads();
    row_inv(v, row1);
    col_load(x, a.Q + pz);
    __syncthreads();     // the rows of P are read
    col_inv(x, col1);
    __syncthreads();
    row_inv(x, row1);
  }
  double acc[K] = {};
  if (isrow) {
    const double eps = a.eps, kappa = a.kappa, ieps = 1.0 / eps, D = a.D;
    // as in k_xrow, a thread's E values of a row are added in T, the rows in FP64
    T ts[2][5] = {};
#pragma unroll
    for (int e = 0; e < E; ++e) {
      T t1[2], sv[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if constexpr (MODE == PL_SUMS) {
          const T q = h ? x[e].y : x[e].x;
          const double w = double(q * q - T(1));
          acc[0] += double(q);
          acc[1] += w * w;
        } else {
          const T q = h ? v[e].y : v[e].x, lq = h ? x[e].y : x[e].x;
          const T w = q * q - T(1);
          const T f = -lq * T(eps) + w * q * T(ieps);                               // f_kernel, Calc.cu:160
          t1[h] = q * (w - T(kappa));                                               // nld_kernel1, Calc.cu:270
          sv[h] = T(D) * t1[h] + (T(3 * eps) * q * q - T(eps * (D + 1))) * f;       // Calc.cu:282, times eps^3
          if constexpr (sizeof(T) == 4) {
            ts[h][0] += q; ts[h][1] += w * w; ts[h][2] += f * f; ts[h][3] += t1[h]; ts[h][4] += sv[h];
          } else {
            acc[0] += double(q); acc[1] += double(w) * double(w); acc[2] += double(f) * double(f);
          }
        }
      }
      if constexpr (MODE == PL_ETD) {
        v[e] = mk<T>(sv[0], sv[1]);
        x[e] = mk<T>(t1[0], t1[1]);
      }
    }
    if constexpr (MODE != PL_SUMS && sizeof(T) == 4) {
#pragma unroll
      for (int q = 0; q < K; ++q) acc[q] = double(ts[0][q]) + double(ts[1][q]);
    }
  }
  wave_part<K, NA>(acc, red);
  if constexpr (MODE == PL_ETD) {
    // the barriers order the sums' partials too
    if constexpr (TWO) {
      if (!second) row_fwd(x, row1);
      if (second || !split) row_fwd(v, row2);
      __syncthreads();
      if (!second) col_fwd(col1, a.U);
      if (second || !split) col_fwd(col2, a.U2);
    } else {
      if (!second) {
        row_fwd(x, row1);
        __syncthreads();
        col_fwd(col1, a.U);
      }
      if (!split) __syncthreads();
      if (second || !split) {
        row_fwd(v, row1);
        __syncthreads();
        col_fwd(col1, a.U2);
      }
    }
  } else {
    __syncthreads();
  }
  if (threadIdx.x < K && !second) {
    const double s = wave_total<NA>(red, threadIdx.x);
    if (threadIdx.x < 3) a.part[3 * (long long)blockIdx.x + threadIdx.x] = s;
    else if (a.dcpart) a.dcpart[2 * (long long)blockIdx.x + threadIdx.x - 3] = s;
  }
}

// ---------------------------------------------------------------------------
// The Forward-Euler update of a plane in LDS: the y and x inverse of W (x and y
// spectra of lap f), k_xe's update, the x and y forward of the new field over W.
// With PL_EULER and k_zeuler a fixed-dt Euler step is four kernels instead of
// ten: 64^3 FP64 53 -> 33 us, 32^3 FP32 38 -> 19, 128^3 FP32 98 -> 68.  Used where
// it is the faster form (kXePlane, xe_min_nz).
// ---------------------------------------------------------------------------
template <typename T, int N>
__global__ void __launch_bounds__((PairCfg<T, N>::NA)) k_xe_plane(XeArgs<T> a, Geo g) {
  using C = PairCfg<T, N>;
  constexpr int E = C::E, TF = C::TF, LL = C::LL, PS = C::PS, V = C::V, CW = C::CW, NA = C::NA, H = N / 2;
  __shared__ cpx<T> sm[H * LL];
  __shared__ cpx<T> tw[N];
  __shared__ double red[NA / 64];
  const int z = int(blockIdx.x);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int cj = lane / CW, kx = wave * CW + lane % CW;    // column
  const int r = threadIdx.x / TF, j = threadIdx.x % TF;    // row pair
  PlaneRow<T, PS> row{sm + (r < H ? r : 0) * LL};
  auto slot = [](int c) { return c + (c >> PS); };
  const PairCol<T, LL> col{sm + slot(kx < H ? kx : N), kx < H ? slot(H + kx) - slot(kx) : slot(N + 1) - slot(N)};
  const bool isrow = r < H, iscol = kx <= H;
  const long long r0 = ((long long)z * N + 2 * r) * N;
  cpx<T> x[E];
  T v[2][E], f[2][E];
  if (iscol) {
    const cpx<T>* const i0 = a.W + (long long)z * g.pp;
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = i0[unsigned(plane_pos(g, cj + TF * e, kx))];
  }
  if (isrow) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        v[h][e] = a.v[r0 + h * N + j + TF * e];
        f[h][e] = a.f[r0 + h * N + j + TF * e];
      }
    }
  }
  const double l1 = a.sc->l1, l2 = a.sc->l2, eta = a.eta, eps = a.eps, t = a.tp ? *a.tp : a.t, ie2 = 1.0 / (eps * eps);
  for (int i = threadIdx.x; i < N; i += NA) tw[i] = a.tw[i];
  __syncthreads();
  if (iscol) {
    fft<T, N, +1, V>(x, cj, tw, col);
#pragma unroll
    for (int e = 0; e < E; ++e) col(cj + TF * e) = x[e];
  }
  __syncthreads();
  double acc[1] = {0.0};
  if (isrow) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int p = j + TF * e;
      const bool mir = p > H;
      const int k = mir ? N - p : p;
      cpx<T> u = row(k == H ? N : k), w = row(k == H ? N + 1 : H + k);
      if (k == 0 || k == H) { u.y = T(0); w.y = T(0); }
      if (mir) { u.y = -u.y; w.y = -w.y; }
      x[e] = mk<T>(u.x - w.y, u.y + w.x);
    }
    row.sync();
    fft<T, N, +1, V>(x, j, tw, row);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      double nv[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const double lf = double(h ? x[e].y : x[e].x), vv = double(v[h][e]), ff = double(f[h][e]);
        const double g0 = -lf + (3.0 * vv * vv - 1.0) * ff * ie2;           // Calc.cu:178
        const double rhs = a.shape ? g0 : l1 * 0.5 + l2 * ff + g0 * eta;    // Calc.cu:417
        nv[h] = vv + t * rhs;                                               // Calc.cu:400
        acc[0] += rhs * rhs;
      }
      x[e] = mk<T>(T(nv[0]), T(nv[1]));
    }
  }
  if (a.part) {   // uniform over the grid: the residual sum only
    block_sum_store<1, NA>(acc, red, a.part + blockIdx.x);
    return;
  }
  if (isrow) {
    fft<T, N, -1, V>(x, j, tw, row);
    constexpr int NH = H + 1, U = (NH + TF - 1) / TF;
#pragma unroll
    for (int e = 0; e < E; ++e) row(j + TF * e) = x[e];
    row.sync();
    cpx<T> ua[U], ub[U];
    const T h = T(0.5) * T(a.inv_n);
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int k = j + TF * i;
      if (k < NH) {
        const cpx<T> zk = row(k), zm = row(k == 0 ? 0 : N - k);
        ua[i] = mk<T>((zk.x + zm.x) * h, (zk.y - zm.y) * h);
        ub[i] = mk<T>((zk.y + zm.y) * h, (zm.x - zk.x) * h);
      }
    }
    row.sync();
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int k = j + TF * i;
      if (k < NH) {
        row(k == H ? N : k) = ua[i];
        row(k == H ? N + 1 : H + k) = ub[i];
      }
    }
  }
  __syncthreads();
  if (iscol) {
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = col(cj + TF * e);
    col.sync();
    fft<T, N, -1, V>(x, cj, tw, col);
    cpx<T>* const o = a.out + (long long)z * g.pp;
#pragma unroll
    for (int e = 0; e < E; ++e) o[unsigned(plane_pos(g, cj + TF * e, kx))] = x[e];
  }
}

}  // namespace vb
