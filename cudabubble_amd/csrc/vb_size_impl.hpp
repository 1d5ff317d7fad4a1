// vb_size_impl.hpp -- launch wrappers for one transform length.  Included by
// exactly one translation unit per length with VB_N defined.
#pragma once
#include <algorithm>

#include "vb_kernels.hpp"
#include "vb_ops.hpp"
#include "vb_plane.hpp"

namespace vb {

// Kernel schedules of one length: bit 0 selects the other z tile (tbw_alt),
// bit 1 the other plan of the ETD x kernel (xrplan_alt).  Only FP32 has
// alternatives; a schedule is compiled where its choice differs from the
// default (see schedules()).
template <typename T, int N>
constexpr int schedules() {
  return sizeof(T) == 8 ? 1 : (xrplan_alt<T, N>() != xrplan<T, N>() ? 4 : 2);
}

template <typename T, int N, int SC = 0>
struct Launch {
  static constexpr int TF = TFof<N>();
  static constexpr int G = xlanes<T, N>();
  static constexpr int TB = (SC & kWideZ) ? tbw_wide<T, N>() : (SC & 1) ? tbw_alt<T, N>() : tbw<T, N>();
  static constexpr int ZV = (SC & kWideZ) ? 0 : zsplan<T, N>();   // plan of the z kernels
  static constexpr int XR = (SC & 2) ? xrplan_alt<T, N>() : xrplan<T, N>();
  static constexpr int YT = TB * TFof<N, ZV>();
  // tile, plan and threads of the plain z passes (k_zpass, k_zmul)
  static constexpr int PB = zpassw<T, N, TB>();
  static constexpr int PV = PB == TB ? ZV : 0;
  static constexpr int PT = PB * TFof<N, PV>();
  static constexpr int CV = colplan<T, N>();          // plan of the y passes and the z Laplacian
  static constexpr int CB = colw<T, N>();             // their columns per workgroup
  static constexpr int CT = CB * TFof<N, CV>();       // and threads per workgroup
  // workgroups of the integrals in a launch that evaluates them (nullptr: none)
  static int fin_groups(const FinArgs* fin) {
    return fin ? std::min(kFinShares, std::max(1, (fin->nxb + 1023) / 1024)) : 0;
  }

  static unsigned xgrid(long long npairs) { return unsigned((npairs + G - 1) / G); }

  static Rows rows(const Geo& g) { return Rows{g.ny, g.pitch, g.pp, g.nq}; }
  // The real input past the caches where it and the spectra together come near the
  // 256 MB of the memory-side cache, so that the next kernel finds the spectra there.
  // An r2c with cached input / past the caches, us: 192^3 FP64 (108 MB) 74.5 / 77.7,
  // 256^3 FP32 (128) 112 / 116, 384 x 192 FP32 (216) 141 / 134, 384 x 96 FP64 (216) 140
  // / 135, 256^3 FP64 (256) 166 / 150, 384^3 FP32 (432) 281 / 268; and 384^3 FP64
  // (864), past any help, 657 / 675.
  template <typename TI>
  static void xr2c_any(const TI* in, cpx<T>* out, long long np, const cpx<T>* tw, double scl, const Geo& g, hipStream_t s) {
    const double mb = double(np) * N * (2 * sizeof(TI) + sizeof(cpx<T>)) / (1 << 20);
    if (mb >= 192 && mb < 768)
      hipLaunchKernelGGL((k_xr2c<TI, T, N, true>), dim3(xgrid(np)), dim3(XWG), 0, s, in, out, np, tw, scl, rows(g));
    else
      hipLaunchKernelGGL((k_xr2c<TI, T, N, false>), dim3(xgrid(np)), dim3(XWG), 0, s, in, out, np, tw, scl, rows(g));
  }
  static void xr2c_d(const double* in, cpx<T>* out, long long np, const cpx<T>* tw, double scl, const Geo& g,
                     hipStream_t s) {
    xr2c_any(in, out, np, tw, scl, g, s);
  }
  static void xr2c(const T* in, cpx<T>* out, long long np, const cpx<T>* tw, double scl, const Geo& g,
                   hipStream_t s) {
    xr2c_any(in, out, np, tw, scl, g, s);
  }
  static void xc2r_d(const cpx<T>* in, double* out, long long np, const cpx<T>* tw, const Geo& g, hipStream_t s) {
    hipLaunchKernelGGL((k_xc2r<T, double, N>), dim3(xgrid(np)), dim3(XWG), 0, s, in, out, np, tw, rows(g));
  }
  static void xc2r(const cpx<T>* in, T* out, long long np, const cpx<T>* tw, const Geo& g, hipStream_t s) {
    hipLaunchKernelGGL((k_xc2r<T, T, N>), dim3(xgrid(np)), dim3(XWG), 0, s, in, out, np, tw, rows(g));
  }
  static void xa(const XaArgs<T>& a, int mode, hipStream_t s) {
    // k_xrow: one row per lane, over the same rows per workgroup; k_xsums:
    // kXsLoop row groups per workgroup
    const dim3 gr(mode == XA_SUMS ? (xgrid(a.npairs) + kXsLoop - 1) / kXsLoop : xgrid(a.npairs)),
        bl(mode == XA_WITHS || mode == XA_ROWSUMS ? xrthreads<T, N, XR>() : XWG);
    if (g_recorder) {
      const int op = mode == XA_WITHF ? OP_XA_F : mode == XA_WITHS ? OP_XA_S : mode == XA_SUMS ? OP_XA_SUMS : OP_XA_RS;
      return record_launch(&launch_tab, op, a, gr, bl);
    }
    if (mode == XA_WITHF)
      hipLaunchKernelGGL((k_xa<T, N>), gr, bl, 0, s, a, nullptr);
    else if (mode == XA_WITHS)
      hipLaunchKernelGGL((k_xrow<T, N, false, XR>), gr, bl, 0, s, a, nullptr);
    else if (mode == XA_SUMS)
      hipLaunchKernelGGL((k_xsums<T, N>), gr, bl, 0, s, a, nullptr);
    else
      hipLaunchKernelGGL((k_xrow<T, N, false, XR, true>), gr, bl, 0, s, a, nullptr);
  }
  static void xe(const XeArgs<T>& a, hipStream_t s) {
    hipLaunchKernelGGL((k_xe<T, N>), dim3(xgrid(a.npairs)), dim3(XWG), 0, s, a);
  }
  static int ypad(const Geo& g, int nf) {
    return g.aligned ? (kXcds - (nf + (g.nz + CB - 1) / CB) % kXcds) % kXcds : 0;
  }
  static void ypass(cpx<T>* b0, cpx<T>* b1, int narr, int sign, const Geo& g, const cpx<T>* tw, const FinArgs* fin,
                    hipStream_t s) {
    const int nf = fin_groups(fin);
    const int pad = ypad(g, nf);
    const dim3 grid(unsigned(ygroups(g, CB)) + unsigned(nf + pad), unsigned(narr)), bl(CT);
    YArgs<T> a{b0, b1, tw, g, fin ? *fin : FinArgs{}, nf, pad, nullptr, nullptr, 0, g.nz, 0};
    if (g_recorder) return record_launch(&launch_tab, sign < 0 ? OP_Y_FWD : OP_Y_INV, a, grid, bl);
    if (sign < 0)
      hipLaunchKernelGGL((k_ypass<T, N, -1, CB, false, CV>), grid, bl, 0, s, a, nullptr);
    else
      hipLaunchKernelGGL((k_ypass<T, N, +1, CB, false, CV>), grid, bl, 0, s, a, nullptr);
  }
  // forward y pass of two arrays, written out of place in the z kernels'
  // group-major layout (column tile ztb)
  static void ypass_gm(const cpx<T>* b0, const cpx<T>* b1, cpx<T>* o0, cpx<T>* o1, int ztb, int nzt, const Geo& g,
                       const cpx<T>* tw, const FinArgs* fin, hipStream_t s) {
    const int nf = fin_groups(fin);
    const int pad = ypad(g, nf);
    const dim3 grid(unsigned(ygroups(g, CB)) + unsigned(nf + pad), 2u), bl(CT);
    YArgs<T> a{const_cast<cpx<T>*>(b0), const_cast<cpx<T>*>(b1), tw, g, fin ? *fin : FinArgs{}, nf, pad, o0, o1, ztb, nzt, 0};
    if (g_recorder) return record_launch(&launch_tab, OP_Y_FWD_GM, a, grid, bl);
    hipLaunchKernelGGL((k_ypass<T, N, -1, CB, false, CV, true>), grid, bl, 0, s, a, nullptr);
  }
  static unsigned zgrid(const Geo& g) { return unsigned(zgroups(g, TB)); }
  static void zpass(cpx<T>* b, int sign, const Geo& g, const cpx<T>* tw, hipStream_t s) {
    if (sign < 0)
      hipLaunchKernelGGL((k_zpass<T, N, -1, PB, PV>), dim3(unsigned(zgroups(g, PB))), dim3(PT), 0, s, b, g, tw);
    else
      hipLaunchKernelGGL((k_zpass<T, N, +1, PB, PV>), dim3(unsigned(zgroups(g, PB))), dim3(PT), 0, s, b, g, tw);
  }
  // FP32 at 192 would spill its 24 elements' v and f (a step 199 -> 209 us); FP64 at
  // 128 spilled 60 registers: nz = 16, 64, 128, 256 62, 84, 110, 169 us a step against
  // 46, 76, 106, 158 with separate kernels.  FP32 at 128 spills 18 and is faster.
  static constexpr bool kXePlane = PairCfg<T, N>::ok && (N <= 96 || (N == 128 && sizeof(T) == 4));
  static void xe_plane(const XeArgs<T>& a, const Geo& g, hipStream_t s) {
    if constexpr (kXePlane)
      hipLaunchKernelGGL((k_xe_plane<T, N>), dim3(unsigned(g.nz)), dim3(PairCfg<T, N>::NA), 0, s, a, g);
  }
  static void zeuler(const cpx<T>* W, cpx<double>* uh, cpx<T>* P, cpx<T>* Q, double* part, double* dc, const Geo& g,
                     const cpx<T>* tw, hipStream_t s) {
    hipLaunchKernelGGL((k_zeuler<T, N, TB, ZV>), dim3(zgrid(g)), dim3(YT), 0, s, W, uh,
                       (ZprArgs<T>{nullptr, P, Q, part, dc, tw, g}));
  }
  static void zmul(const cpx<T>* in, cpx<T>* out, int sign, int op, const Geo& gi, const Geo& go, const cpx<T>* tw,
                   hipStream_t s) {
    const ZmArgs<T> a{in, out, tw, gi, go};
    const dim3 gr(unsigned(zgroups(go.aligned ? go : gi, PB))), bl(PT);
    if (sign < 0) {
      hipLaunchKernelGGL((k_zmul<T, N, -1, PB, ZM_ONE, PV>), gr, bl, 0, s, a);
      return;
    }
    switch (op) {
      case ZM_LAP: hipLaunchKernelGGL((k_zmul<T, N, +1, PB, ZM_LAP, PV>), gr, bl, 0, s, a); break;
      case ZM_DX: hipLaunchKernelGGL((k_zmul<T, N, +1, PB, ZM_DX, PV>), gr, bl, 0, s, a); break;
      case ZM_DY: hipLaunchKernelGGL((k_zmul<T, N, +1, PB, ZM_DY, PV>), gr, bl, 0, s, a); break;
      case ZM_DZ: hipLaunchKernelGGL((k_zmul<T, N, +1, PB, ZM_DZ, PV>), gr, bl, 0, s, a); break;
      default: hipLaunchKernelGGL((k_zmul<T, N, +1, PB, ZM_ONE, PV>), gr, bl, 0, s, a); break;
    }
  }
  static void pair_r2c(const T* u, cpx<T>* so, double scl, const Geo& g, const cpx<T>* tw, hipStream_t s) {
    if constexpr (PairCfg<T, N>::ok)
      hipLaunchKernelGGL((k_pair<T, N, -1>), dim3(unsigned(g.nz)), dim3(PairCfg<T, N>::NA), 0, s,
                         (PairArgs<T>{u, nullptr, nullptr, so, tw, g, scl}));
  }
  static void pair_c2r(const cpx<T>* si, T* uo, const Geo& g, const cpx<T>* tw, hipStream_t s) {
    if constexpr (PairCfg<T, N>::ok)
      hipLaunchKernelGGL((k_pair<T, N, +1>), dim3(unsigned(g.nz)), dim3(PairCfg<T, N>::NA), 0, s,
                         (PairArgs<T>{nullptr, uo, si, nullptr, tw, g, 1.0}));
  }
  static void zlap(cpx<T>* b, const Geo& g, const cpx<T>* tw, const FinArgs* fin, hipStream_t s) {
    const int nf = fin_groups(fin);
    const dim3 gr(unsigned(zgroups(g, CB)) + unsigned(nf)), bl(CT);
    ZlArgs<T> a{b, tw, g, fin ? *fin : FinArgs{}, nf};
    if (g_recorder) return record_launch(&launch_tab, OP_ZLAP, a, gr, bl);
    hipLaunchKernelGGL((k_zlap<T, N, CB, false, CV>), gr, bl, 0, s, a, nullptr);
  }
  static void zprep(const cpx<double>* vh, cpx<T>* P, cpx<T>* Q, double* part, double* dc, const Geo& g,
                    const cpx<T>* tw, hipStream_t s) {
    const dim3 gr(zgrid(g)), bl(YT);
    ZprArgs<T> a{vh, P, Q, part, dc, tw, g};
    if (g_recorder) return record_launch(&launch_tab, OP_ZPREP, a, gr, bl);
    hipLaunchKernelGGL((k_zprep<T, N, TB, false, ZV>), gr, bl, 0, s, a, nullptr);
  }
  template <int SCH, int STG, bool TAB, bool PROBE = false>
  static void zs_launch(dim3 gr, const ZsArgs<T>& a, const ZsArgs<T>* tab, hipStream_t s) {
    hipLaunchKernelGGL((k_zstage<T, N, SCH, STG, TB, TAB, ZV, PROBE>), gr, dim3(YT), 0, s, a, tab);
  }
  template <bool TAB>
  static void zs_dispatch(int sch, int stg, dim3 gr, const ZsArgs<T>& a, const ZsArgs<T>* tab, hipStream_t s) {
    if (sch == 4) {
      switch (stg) {
        case 1: zs_launch<4, 1, TAB>(gr, a, tab, s); break;
        case 2: zs_launch<4, 2, TAB>(gr, a, tab, s); break;
        case 3: zs_launch<4, 3, TAB>(gr, a, tab, s); break;
        case 4: zs_launch<4, 4, TAB>(gr, a, tab, s); break;
        default: zs_launch<4, 4, TAB, true>(gr, a, tab, s); break;   // 5: the probe form of stage 4
      }
    } else if (stg == 1) {
      zs_launch<2, 1, TAB>(gr, a, tab, s);
    } else {
      zs_launch<2, 2, TAB>(gr, a, tab, s);
    }
  }
  static void zstage(const ZsArgs<T>& a, int sch, int stg, hipStream_t s) {
    const dim3 gr(zgrid(a.g));
    if (g_recorder)
      return record_launch(&launch_tab, stg == 5 ? OP_ZS44P : (sch == 4 ? OP_ZS41 : OP_ZS21) + (stg - 1), a, gr,
                           dim3(YT));
    zs_dispatch<false>(sch, stg, gr, a, nullptr, s);
  }

  // solves, of `lanes` with nz planes each, whose planes get two workgroups of
  // k_plane2 each: those of a last round of planes that fills at most half of
  // the compute units (measured at k_plane2)
  static int plane2_split(int nz, int lanes) {
    const int rest = nz * lanes % kCus;
    return 2 * rest <= kCus ? rest / nz : 0;
  }
  template <bool TAB>
  static void pl_launch(int mode, dim3 gr, const PlaneArgs<T>& a, const PlaneArgs<T>* tab, hipStream_t s) {
    if constexpr (Plane2Cfg<T, N>::ok) {
      if (mode == PL_ETD) {
        const int k = plane2_split(int(gr.x), int(gr.z));
        gr.z += unsigned(k);
        hipLaunchKernelGGL((k_plane2<T, N, PL_ETD, TAB>), gr, dim3(PairCfg<T, N>::NA), 0, s, a, tab, k);
        return;
      }
    }
    const dim3 bl(kPlaneThreads);
    if constexpr (PlaneCfg<T, N>::ok) {
      if (!TAB && mode == PL_EULER)
        hipLaunchKernelGGL((k_plane<T, N, PL_EULER>), gr, bl, 0, s, a, nullptr);
      else if (mode == PL_SUMS)
        hipLaunchKernelGGL((k_plane<T, N, PL_SUMS, TAB>), gr, bl, 0, s, a, tab);
      else if (mode == PL_ROWSUMS)
        hipLaunchKernelGGL((k_plane<T, N, PL_ROWSUMS, TAB>), gr, bl, 0, s, a, tab);
      else if constexpr (!Plane2Cfg<T, N>::ok)
        hipLaunchKernelGGL((k_plane<T, N, PL_ETD, TAB>), gr, bl, 0, s, a, tab);
    } else if constexpr (Plane2Cfg<T, N>::ok) {
      if (mode == PL_SUMS)
        hipLaunchKernelGGL((k_plane2<T, N, PL_SUMS, TAB>), gr, bl, 0, s, a, tab, 0);
      else
        hipLaunchKernelGGL((k_plane2<T, N, PL_ROWSUMS, TAB>), gr, bl, 0, s, a, tab, 0);
    }
  }
  static constexpr int kPlaneThreads = PlaneCfg<T, N>::ok ? PlaneCfg<T, N>::NA : PairCfg<T, N>::NA;
  static constexpr int kSumsPlanes = PlaneCfg<T, N>::ok ? 2 : 1;
  static void plane(const PlaneArgs<T>& a, int mode, hipStream_t s) {
    const dim3 gr(unsigned(mode == PL_SUMS ? a.g.nz / kSumsPlanes : a.g.nz));
    if (g_recorder) return record_launch(&launch_tab, OP_PL_ETD + mode, a, gr, dim3(kPlaneThreads));
    pl_launch<false>(mode, gr, a, nullptr, s);
  }

  // the table form of a recorded launch, over `lanes` solves (blockIdx.z)
  static void launch_tab(int op, const void* tab, dim3 gr, dim3 bl, int lanes, hipStream_t s) {
    gr.z = unsigned(lanes);
    // the workgroups' order (see kXcds): by the bytes of the batch's P and Q
    auto past = [&](double modes, int mb) { return int(2.0 * sizeof(cpx<T>) * modes * lanes > double(mb << 20)); };
    XaArgs<T> xa{};
    YArgs<T> ya{};
    xa.in_order = past(double(gr.x) * 2 * G * (N / 2), 32);
    ya.in_order = past(double(gr.x) * CB * N, 256);
    switch (op) {
      case OP_XA_RS:
        hipLaunchKernelGGL((k_xrow<T, N, true, XR, true>), gr, bl, 0, s, xa, (const XaArgs<T>*)tab);
        break;
      case OP_XA_F: hipLaunchKernelGGL((k_xa<T, N, true>), gr, bl, 0, s, XaArgs<T>{}, (const XaArgs<T>*)tab); break;
      case OP_XA_S:
        hipLaunchKernelGGL((k_xrow<T, N, true, XR>), gr, bl, 0, s, xa, (const XaArgs<T>*)tab);
        break;
      case OP_XA_SUMS:
        hipLaunchKernelGGL((k_xsums<T, N, true>), gr, bl, 0, s, XaArgs<T>{}, (const XaArgs<T>*)tab);
        break;
      case OP_Y_FWD:
        hipLaunchKernelGGL((k_ypass<T, N, -1, CB, true, CV>), gr, bl, 0, s, ya, (const YArgs<T>*)tab);
        break;
      case OP_Y_INV:
        hipLaunchKernelGGL((k_ypass<T, N, +1, CB, true, CV>), gr, bl, 0, s, ya, (const YArgs<T>*)tab);
        break;
      case OP_Y_FWD_GM:
        hipLaunchKernelGGL((k_ypass<T, N, -1, CB, true, CV, true>), gr, bl, 0, s, ya, (const YArgs<T>*)tab);
        break;
      case OP_ZLAP:
        hipLaunchKernelGGL((k_zlap<T, N, CB, true, CV>), gr, bl, 0, s, ZlArgs<T>{}, (const ZlArgs<T>*)tab);
        break;
      case OP_ZPREP:
        hipLaunchKernelGGL((k_zprep<T, N, TB, true, ZV>), gr, bl, 0, s, ZprArgs<T>{}, (const ZprArgs<T>*)tab);
        break;
      case OP_ZS41: case OP_ZS42: case OP_ZS43: case OP_ZS44:
        zs_dispatch<true>(4, op - OP_ZS41 + 1, gr, ZsArgs<T>{}, (const ZsArgs<T>*)tab, s);
        break;
      case OP_PL_ETD: case OP_PL_SUMS: case OP_PL_ROWSUMS:
        pl_launch<true>(op - OP_PL_ETD, gr, PlaneArgs<T>{}, (const PlaneArgs<T>*)tab, s);
        break;
      case OP_ZS44P: zs_dispatch<true>(4, 5, gr, ZsArgs<T>{}, (const ZsArgs<T>*)tab, s); break;
      case OP_ZS21: case OP_ZS22:
        zs_dispatch<true>(2, op - OP_ZS21 + 1, gr, ZsArgs<T>{}, (const ZsArgs<T>*)tab, s);
        break;
      default: break;
    }
  }

  static SizeOps<T> table() {
    SizeOps<T> o;
    o.N = N;
    o.sched = SC;
    o.xr_passes = Plan<N, XR>::NP;
    o.xr_radix = Plan<N, XR>::R[0];
    o.xlanes = G;
    o.ytile = TB;
    o.ctile = CB;
    o.ythreads = YT;
    o.xr2c_d = &xr2c_d;
    o.xr2c = &xr2c;
    o.xc2r_d = &xc2r_d;
    o.xc2r = &xc2r;
    o.xa = &xa;
    o.xe = &xe;
    o.ypass = &ypass;
    o.ypass_gm = &ypass_gm;
    o.zpass = &zpass;
    o.zlap = &zlap;
    o.zprep = &zprep;
    o.zstage = &zstage;
    o.plane = PlaneCfg<T, N>::ok || Plane2Cfg<T, N>::ok ? &plane : nullptr;
    o.sums_planes = kSumsPlanes;
    o.plane_min_nz = plane_min_nz<T, N>();
    o.plane_euler = PlaneCfg<T, N>::ok;
    o.xe_plane = kXePlane ? &xe_plane : nullptr;
    // few planes leave the chip idle.  us per step (and with a residual after it),
    // one kernel / separate ones: FP32 128 nz = 16 43.8 (101.5) / 39.1 (87.9), 48 59.0
    // (117) / 54.4 (103), 64 61.9 (121) / 62.1 (112), 96 67.6 / 70.0, 128 69.8 / 75.2;
    // FP64 96 nz = 16 50.9 (106) / 50.2 (99), 32 56.3 / 57.6; FP32 96 nz = 16 35.3 / 37.6
    o.xe_min_nz = N == 128 ? 96 : N == 96 && sizeof(T) == 8 ? 32 : 0;
    o.zeuler = &zeuler;
    o.zmul = &zmul;
    // few planes leave the chip idle.  A call, separate kernels / by plane, us: r2c FP64
    // 128 nz = 16 23.1 / 27.0, 32 27.0 / 28.5, 48 31.4 / 30.5; FP32 128 nz = 16 21.6 /
    // 22.2, 32 23.4 / 23.9, 48 26.2 / 24.1; FP32 192 nz = 16 25.2 / 29.5, 32 30.3 / 33.3,
    // 48 36.1 / 33.6; c2r FP32 192 nz = 16 28.9 / 29.4, 32 35.0 / 31.0 (96 and shorter:
    // by plane at 16 too)
    o.pair_r2c_nz = N < 128 ? 0 : 48;
    o.pair_c2r_nz = N < 128 ? 0 : 32;
    o.pair_r2c = PairCfg<T, N>::ok ? &pair_r2c : nullptr;
    o.pair_c2r = PairCfg<T, N>::ok ? &pair_c2r : nullptr;
    return o;
  }
};

}  // namespace vb

namespace vb {
// the launch table of schedule sc of length N (nullptr: not compiled)
template <typename T, int N>
const SizeOps<T>* ops_table(int sc) {
  if (sc == kWideZ) {
    if constexpr (tbw_wide<T, N>() != 0) {
      static const SizeOps<T> w = Launch<T, N, kWideZ>::table();
      return &w;
    }
    return nullptr;
  }
  if (sc < 0 || sc >= schedules<T, N>()) return nullptr;
  static const SizeOps<T> t[4] = {
      Launch<T, N, 0>::table(), Launch<T, N, (schedules<T, N>() > 1 ? 1 : 0)>::table(),
      Launch<T, N, (schedules<T, N>() > 2 ? 2 : 0)>::table(), Launch<T, N, (schedules<T, N>() > 2 ? 3 : 0)>::table()};
  return &t[sc];
}
}  // namespace vb

#define VB_DEFINE_SIZE(n)                                                                     \
  namespace vb {                                                                              \
  template <> const SizeOps<double>* ops_for<double, n>(int sc) { return ops_table<double, n>(sc); } \
  template <> const SizeOps<float>* ops_for<float, n>(int sc) { return ops_table<float, n>(sc); }    \
  template <> int sched_count<double, n>() { return schedules<double, n>(); }                 \
  template <> int sched_count<float, n>() { return schedules<float, n>(); }                   \
  }
