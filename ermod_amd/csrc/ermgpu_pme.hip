// ermgpu_pme.hip -- the register-FFT kernels of one precision and grid
// length: z columns, in FP32 the y columns and the x slab with the gather, and
// the adjoint's solvent-potential transforms.  Compiled once per (ERM_T,
// ERM_K), or per list ERM_ZLENS of FP32 lengths of k_pme_zcol_dit, so that the
// instantiations build in parallel; ermgpu.hip dispatches on the grid length at
// run time.
#include <algorithm>

#include "ermgpu_ctx.h"
#include "ermgpu_fft2.h"
#include "ermgpu_grad.h"

#ifndef ERM_T
#error "ERM_T (float or double) and ERM_K (grid length), or ERM_ZLENS, select the instantiations"
#endif

namespace ermh {

template <typename T, int K, int XT>
int launch_zcol_reg_t(erm_ctx *c, const Params &k, int n, int nblk) {
  using V = typename C2<T>::type;
  const size_t lds = zcol_reg_lds<T>(k.H, k.K2, K, XT);
  TRY(set_lds(c, (const void *)k_pme_zcol_reg<T, K, XT>, lds, "k_pme_zcol_reg"));
  hipLaunchKernelGGL((k_pme_zcol_reg<T, K, XT>), dim3(nblk, n), dim3(XT), lds, c->st, k, dp<T>(c->d_engfac),
                     dp<T>(c->d_sqv), dp<V>(c->d_w1h), dp<V>(c->d_w2h), dp<V>(c->d_w3h), dp<V>(c->d_tw3),
                     dp<V>(c->d_Hk), dp<double>(c->d_selfp));
  return ERM_OK;
}
// z columns with the tuned workgroup size (256 or 512)
template <typename T, int K> int launch_zcol_reg(erm_ctx *c, const Params &k, int n, int nblk) {
  if (c->zcol_T == 512) return launch_zcol_reg_t<T, K, 512>(c, k, n, nblk);
  return launch_zcol_reg_t<T, K, NTHR>(c, k, n, nblk);
}
template <typename T, int K, int PP, int XT>
int launch_zcol_fft_t(erm_ctx *c, const Params &k, int n, int nblk, size_t site0, size_t cfg0) {
  using V = typename C2<T>::type;
  const size_t lds = zcol_fft_lds<T>(k.H, k.K2, XT, zfft_lanes(sizeof(T), K));
  const size_t hk = cfg0 * k.K3 * (size_t)k.K2 * k.H;
  TRY(set_lds(c, (const void *)k_pme_zcol_fft<T, K, PP, XT>, lds, "k_pme_zcol_fft"));
  hipLaunchKernelGGL((k_pme_zcol_fft<T, K, PP, XT>), dim3(nblk, n), dim3(XT), lds, c->st, k, dp<T>(c->d_engfac),
                     dp<T>(c->d_sqv) + site0, dp<V>(c->d_w1h) + site0 * k.H, dp<V>(c->d_w2h) + site0 * k.K2,
                     dp<int>(c->d_sg3) + site0, dp<T>(c->d_sw3) + site0 * k.p, dp<V>(c->d_Hk) + hk,
                     dp<double>(c->d_selfp) + cfg0 * nblk);
  return ERM_OK;
}
// z columns spread and transformed along z (spline orders 4 and 6; not FP64
// columns of 64, which z_kernel gives to the two-step kernel)
template <typename T, int K>
int launch_zcol_fft(erm_ctx *c, const Params &k, int n, int nblk, size_t site0, size_t cfg0) {
  if constexpr (sizeof(T) == 4 || K < 64) {
    if (k.p == 4) {
      if (c->zcol_T == 512) return launch_zcol_fft_t<T, K, 4, 512>(c, k, n, nblk, site0, cfg0);
      return launch_zcol_fft_t<T, K, 4, NTHR>(c, k, n, nblk, site0, cfg0);
    }
    if (c->zcol_T == 512) return launch_zcol_fft_t<T, K, 6, 512>(c, k, n, nblk, site0, cfg0);
    return launch_zcol_fft_t<T, K, 6, NTHR>(c, k, n, nblk, site0, cfg0);
  }
  return fail(c, ERM_E_ENG_BUG, "register z columns of 64 in FP64");
}
// z columns of a heterogeneous batch (run table in device memory): a
// persistent grid (as many workgroups as fit the device at once) pulling
// items through the counter
template <typename T, int K, int PP, int XT>
int launch_zcol_runs_t(erm_ctx *c, const Params &k, int nblk, const GRun *runs, int nrun, int nitem, int *counter) {
  using V = typename C2<T>::type;
  const size_t lds = zcol_fft_lds<T>(k.H, k.K2, XT, zfft_lanes(sizeof(T), K));
  const void *f = (const void *)k_pme_zcol_fft_runs<T, K, PP, XT>;
  TRY(set_lds(c, f, lds, "k_pme_zcol_fft_runs"));
  int occ = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, f, XT, lds) != hipSuccess || occ < 1) {
    (void)hipGetLastError();
    occ = 1;
  }
  const int grid = std::min(nitem, std::max(1, occ * c->ncu));
  hipLaunchKernelGGL((k_pme_zcol_fft_runs<T, K, PP, XT>), dim3(grid), dim3(XT), lds, c->st, k, dp<T>(c->d_engfac),
                     dp<T>(c->d_sqv), dp<V>(c->d_w1h), dp<V>(c->d_w2h), dp<int>(c->d_sg3), dp<T>(c->d_sw3),
                     dp<V>(c->d_Hk), dp<double>(c->d_selfp), runs, nrun, nblk, nitem, counter);
  return ERM_OK;
}
template <typename T, int K>
int launch_zcol_fft_runs(erm_ctx *c, const Params &k, int nblk, const GRun *runs, int nrun, int nitem, int *counter) {
  if constexpr (sizeof(T) == 4 || K < 64) {
    if (k.p == 4) {
      if (c->zcol_T == 512) return launch_zcol_runs_t<T, K, 4, 512>(c, k, nblk, runs, nrun, nitem, counter);
      return launch_zcol_runs_t<T, K, 4, NTHR>(c, k, nblk, runs, nrun, nitem, counter);
    }
    if (c->zcol_T == 512) return launch_zcol_runs_t<T, K, 6, 512>(c, k, nblk, runs, nrun, nitem, counter);
    return launch_zcol_runs_t<T, K, 6, NTHR>(c, k, nblk, runs, nrun, nitem, counter);
  }
  return fail(c, ERM_E_ENG_BUG, "register z columns of 64 in FP64");
}
// inverse y columns, one lane per column
template <typename T, int K> int launch_ycol_reg(erm_ctx *c, const Params &k, int n) {
  if constexpr (sizeof(T) == 4) {
    using V = typename C2<T>::type;
    int nblk = (k.K3 * k.H + NTHR - 1) / NTHR;
    hipLaunchKernelGGL((k_pme_ycol_reg<T, K>), dim3(nblk, n), dim3(NTHR), 0, c->st, k, dp<V>(c->d_tw2),
                       dp<V>(c->d_Hk));
    return launch_check(c, "k_pme_ycol_reg");
  }
  return fail(c, ERM_E_ENG_BUG, "y columns in FP64");
}
template <typename T, int K, int R, int XT = NTHR, bool YF = false>
int launch_xslab_r(erm_ctx *c, const Params &k, int n, const XsShape &s) {
  using V = typename C2<T>::type;
  const size_t lds = sizeof(V) * (size_t)s.Q * k.H * k.K2;
  TRY(set_lds(c, (const void *)k_pme_xslab<T, K, R, XT, YF>, lds, "k_pme_xslab"));
  const int nslab = (k.K3 + s.S - 1) / s.S;
  hipLaunchKernelGGL((k_pme_xslab<T, K, R, XT, YF>), dim3(nslab, n), dim3(XT), lds, c->st, k, s.S, s.Q, c->nsites,
                     dp<V>(c->d_Hk), dp<V>(c->d_tw1), dp<int>(c->d_zstart), dp<int>(c->d_zg), dp<T>(c->d_zq),
                     dp<T>(c->d_zw), dp<int>(c->d_zsite), dp<double>(c->d_esite));
  return launch_check(c, "k_pme_xslab");
}
// a 512-thread workgroup owns the same sites as one of 256 with half as many
// per thread
template <typename T, int K> int launch_xslab(erm_ctx *c, const Params &k, int n, const XsShape &s) {
  if constexpr (sizeof(T) == 4) {
    if (s.fold) {
      if (s.R == 8) return launch_xslab_r<T, K, 4, 512, true>(c, k, n, s);
      if (s.R == 16) return launch_xslab_r<T, K, 8, 512, true>(c, k, n, s);
      return launch_xslab_r<T, K, 16, 512, true>(c, k, n, s);
    }
    if (s.T == 512) {
      if (s.R == 8) return launch_xslab_r<T, K, 4, 512>(c, k, n, s);
      if (s.R == 16) return launch_xslab_r<T, K, 8, 512>(c, k, n, s);
      return launch_xslab_r<T, K, 16, 512>(c, k, n, s);
    }
    if (s.R == 8) return launch_xslab_r<T, K, 8>(c, k, n, s);
    if (s.R == 16) return launch_xslab_r<T, K, 16>(c, k, n, s);
    return launch_xslab_r<T, K, 32>(c, k, n, s);
  }
  return fail(c, ERM_E_ENG_BUG, "x slab in FP64");
}
template <typename T, int K> void launch_xr2c(erm_ctx *c, const Params &k) {
  using V = typename C2<T>::type;
  const int nt = k.K3 * ((k.K2 + 1) / 2);
  hipLaunchKernelGGL((k_xrow_r2c<T, K>), dim3((nt + NTHR - 1) / NTHR), dim3(NTHR), 0, c->st, k,
                     dp<T>(c->d_ggrid), dp<V>(c->d_tw1), dp<V>(c->d_gHk));
}
template <typename T, int K> void launch_xc2r(erm_ctx *c, const Params &k) {
  using V = typename C2<T>::type;
  const int nt = k.K3 * ((k.K2 + 1) / 2);
  hipLaunchKernelGGL((k_xrow_c2r<T, K>), dim3((nt + NTHR - 1) / NTHR), dim3(NTHR), 0, c->st, k,
                     dp<V>(c->d_gHk), dp<V>(c->d_tw1), dp<T>(c->d_ggrid));
}
template <typename T, int K, int SIGN> void launch_ydense(erm_ctx *c, const Params &k) {
  using V = typename C2<T>::type;
  const int nt = k.K3 * k.H;
  hipLaunchKernelGGL((k_pme_ycol_reg<T, K, SIGN>), dim3((nt + NTHR - 1) / NTHR, 1), dim3(NTHR), 0, c->st, k,
                     dp<V>(c->d_tw2), dp<V>(c->d_gHk));
}
template <typename T, int K> void launch_zgreen(erm_ctx *c, const Params &k) {
  using V = typename C2<T>::type;
  const int nt = k.H * k.K2;
  hipLaunchKernelGGL((k_zcol_green<T, K>), dim3((nt + NTHR - 1) / NTHR), dim3(NTHR), 0, c->st, k,
                     dp<T>(c->d_engfac), dp<V>(c->d_tw3), dp<V>(c->d_gHk));
}

#ifdef ERM_ZLENS
template <int K, int PP> int launch_zcol_dit_t(erm_ctx *c, const Params &k, int n, int nblk) {
  const size_t lds = zdit_lds(k.H, k.K2, K, PP);
  TRY(set_lds(c, (const void *)k_pme_zcol_dit<K, PP>, lds, "k_pme_zcol_dit"));
  hipLaunchKernelGGL((k_pme_zcol_dit<K, PP>), dim3(nblk, n), dim3(NTHR), lds, c->st, k, dp<float>(c->d_engfac),
                     dp<int>(c->d_sg3), dp<float>(c->d_sw3), dp<float>(c->d_sqv), dp<float2>(c->d_w1h),
                     dp<float2>(c->d_w2h), dp<float2>(c->d_tw3), dp<float2>(c->d_Hk), dp<double>(c->d_selfp));
  return launch_check(c, "k_pme_zcol_dit");
}
template <int K> int launch_zcol_dit(erm_ctx *c, const Params &k, int n, int nblk) {
  return k.p == 4 ? launch_zcol_dit_t<K, 4>(c, k, n, nblk) : launch_zcol_dit_t<K, 6>(c, k, n, nblk);
}
#define ERM_Z(K) template int launch_zcol_dit<K>(erm_ctx *, const Params &, int, int);
ERM_ZLENS
#else
template int launch_zcol_reg<ERM_T, ERM_K>(erm_ctx *, const Params &, int, int);
template int launch_zcol_fft<ERM_T, ERM_K>(erm_ctx *, const Params &, int, int, size_t, size_t);
template int launch_zcol_fft_runs<ERM_T, ERM_K>(erm_ctx *, const Params &, int, const GRun *, int, int, int *);
template int launch_ycol_reg<ERM_T, ERM_K>(erm_ctx *, const Params &, int);
template int launch_xslab<ERM_T, ERM_K>(erm_ctx *, const Params &, int, const XsShape &);
template void launch_xr2c<ERM_T, ERM_K>(erm_ctx *, const Params &);
template void launch_xc2r<ERM_T, ERM_K>(erm_ctx *, const Params &);
template void launch_ydense<ERM_T, ERM_K, -1>(erm_ctx *, const Params &);
template void launch_ydense<ERM_T, ERM_K, +1>(erm_ctx *, const Params &);
template void launch_zgreen<ERM_T, ERM_K>(erm_ctx *, const Params &);
#endif

}  // namespace ermh
