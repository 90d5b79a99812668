// ermgpu_grad.h -- adjoint kernels: gradient of the solute-solvent energy
// u = sum_{k>=1} uvengy(k) with respect to the solute's per-site charge q_i,
// LJ epsilon_i and sigma_i.
//
//  real space   per (configuration, solute site): sums over the candidate
//               solvent sites of the pair kernel
//                 dU/dq_i      += q_v erfc(alpha r) / r
//                 U_LJ,i       += rep - att          (dU/deps_i = U_LJ,i / 2 eps_i)
//                 dU/dsigma_i  += (6 rep - 3 att) f_iv
//               where every LJ variant of realcal.F90:708-776 is rep - att
//               with rep proportional to sigma^12 and att to sigma^6, and
//               f_iv = d(sigma_iv^2)/d(sigma_i) / sigma_iv^2.
//  reciprocal   the PME energy is the symmetric bilinear form
//               q_slt^T W^T Phi W q_slv (recpcal.F90:342-502), so dU/dq_i is
//               the solvent's PME potential at site i: once per frame the
//               solvent charges are spread, transformed (register FFTs),
//               multiplied by the Green's function and transformed back; per
//               configuration each solute site interpolates that grid.
//  residual     residual_ene (engproc.F90:859-869): -pi Q_slt Q_solv / (alpha^2 V).
#pragma once

#include "ermgpu_kern.h"

namespace erm {

// rep and att of one LJ pair (U = rep - att) for the four switches of
// realcal.F90:708-776; rep scales with sigma^12, att with sigma^6
template <typename T>
__device__ __forceinline__ void lj_parts_t(const Params &P, T eps, T sig2, T dist, T &rep, T &att) {
  T invr2 = sig2 / dist;
  T invr6 = invr2 * invr2 * invr2;
  T sg6 = sig2 * sig2 * sig2;
  const bool low = dist <= (T)P.lw2;
  if (P.ljswitch <= 1) {
    T sw = (T)1;
    if (!low) {
      if (P.ljswitch == 0) {
        T up2 = (T)P.up2, lw2 = (T)P.lw2;
        T d = dist - up2, w = up2 - lw2;
        sw = ((T)2 * dist + up2 - (T)3 * lw2) * (d * d) / (w * w * w);
      } else {
        T x = (sqrt(dist) - (T)P.lwljcut) / (T)(P.upljcut - P.lwljcut);
        T x3 = x * x * x;
        sw = (T)1 - (T)10 * x3 + (T)15 * (x3 * x) - (T)6 * (x3 * x * x);
      }
    }
    rep = (T)4 * eps * invr6 * invr6 * sw;
    att = (T)4 * eps * invr6 * sw;
    return;
  }
  if (P.ljswitch == 2) {
    if (low) {
      rep = (T)4 * eps * (invr6 * invr6 - sg6 * sg6 / (T)(P.lw6 * P.up6));
      att = (T)4 * eps * (invr6 - sg6 / (T)(P.lw3 * P.up3));
    } else {
      T invr3 = sqrt(invr6), sg3 = sqrt(sg6);
      T a = invr6 - sg6 / (T)P.up6, c = invr3 - sg3 / (T)P.up3;
      rep = (T)4 * eps * (T)(P.up6 / (P.up6 - P.lw6)) * (a * a);
      att = (T)4 * eps * (T)(P.up3 / (P.up3 - P.lw3)) * (c * c);
    }
    return;
  }
  T a = (T)P.repC, b = (T)P.attC;
  if (!low) {
    T sw = sqrt(dist) - (T)P.lwljcut;
    T sw3 = sw * sw * sw, sw4 = sw3 * sw;
    a = (T)P.repA * sw3 + (T)P.repB * sw4 + (T)P.repC;
    b = (T)P.attA * sw3 + (T)P.attB * sw4 + (T)P.attC;
  }
  rep = (T)4 * eps * (invr6 * invr6 - sg6 * sg6 * a);
  att = (T)4 * eps * (invr6 - sg6 * b);
}

template <typename T> __device__ __forceinline__ T erfc_over_r(T r, T alpha);
template <> __device__ __forceinline__ float erfc_over_r<float>(float r, float alpha) { return erfcf(alpha * r) / r; }
template <> __device__ __forceinline__ double erfc_over_r<double>(double r, double alpha) {
  return (1.0 - erf(alpha * r)) / r;
}

// Real-space adjoint.  Grid (n, nsplit); every workgroup of configuration b
// builds the pair kernel's candidate segments and takes every nsplit-th
// solvent site of them.  The sites are staged in LDS in chunks, relative to
// the solute's centre; a thread holds one solute site and every nsl-th site of
// the chunk.  It first tests up to 64 distances into a bit mask and then
// evaluates the marked pairs, so that the lanes of a wave meet in the
// expensive part (erfc and Lennard-Jones) rather than each waiting for the
// others' hits: a third of the tested pairs is within the cutoff.  A chunk
// takes its sites from all over the candidates, which evens the lanes' counts.
// Per-site sums are added in slice order and written as
// part[(b * nsplit + y)][4][ns] = {u, dU/dq, U_LJ, dU/dsigma}: deterministic.
// Bound by FP64 (erf, square root and division).  Walking the candidate
// molecules once per solute site, displacement and cutoff branch inside, took
// 246 us for 256 configurations of 30 sites in 4000 waters, this 115.
// LDS: ns T (x, y, z, charge; in FP32 also the coordinates' low parts) + 3 ns
// nvt T (eps_iv, sigma_iv^2, f_iv) + segments + the larger of a chunk and the
// slices' sums.
template <typename T> constexpr int grad_site_bytes() { return (sizeof(T) == 4 ? 7 : 4) * sizeof(T) + sizeof(int); }
template <typename T> inline size_t grad_lds(int ns, int nvt, int nsl, int chunk) {
  const size_t red = nsl > 1 ? sizeof(double) * 4 * (size_t)nsl * ns : 0;
  const size_t stage = (size_t)chunk * grad_site_bytes<T>();
  return (std::max(red, stage) + 15) / 16 * 16 + sizeof(T) * ((size_t)(sizeof(T) == 4 ? 7 : 4) * ns + (size_t)3 * ns * nvt) +
         sizeof(int) * (2 * MAXSEG + 2);
}

template <typename T>
__global__ __launch_bounds__(NTHR) void k_pair_grad(Params P, int nsl, int chunk, const double *__restrict__ spos,
                                                    const double *__restrict__ sref, const T *__restrict__ gq,
                                                    const T *__restrict__ gtab, const int *__restrict__ cell_start,
                                                    const int *__restrict__ mol_first, const double *__restrict__ sx,
                                                    const double *__restrict__ sy, const double *__restrict__ sz,
                                                    const T *__restrict__ sq, const int *__restrict__ sct,
                                                    const int *__restrict__ slt_j,
                                                    const double *__restrict__ rm_ord_p, double *part) {
  constexpr bool LOW = sizeof(T) == 4;  // FP32 offsets carry low parts
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const int ns = P.ns, nvt = P.nvt;
  const size_t nred = nsl > 1 ? sizeof(double) * 4 * (size_t)nsl * ns : 0;
  const size_t nst = (size_t)chunk * grad_site_bytes<T>();
  double *red = reinterpret_cast<double *>(lds_raw);  // [nsl][4][ns], after the last chunk
  T *vx = reinterpret_cast<T *>(lds_raw);             // the chunk
  T *vy = vx + chunk;
  T *vz = vy + chunk;
  T *vq = vz + chunk;
  T *vlo = vq + chunk;  // FP32: [3][chunk]
  int *vt = reinterpret_cast<int *>(vlo + (LOW ? 3 * chunk : 0));
  T *ux = reinterpret_cast<T *>(lds_raw + ((nred > nst ? nred : nst) + 15) / 16 * 16);
  T *uy = ux + ns;
  T *uz = uy + ns;
  T *uq = uz + ns;
  T *ulo = uq + ns;                          // FP32: [3][ns]
  T *tab = ulo + (LOW ? 3 * ns : 0);         // [ns][nvt][3]
  int *seg_beg = reinterpret_cast<int *>(tab + 3 * ns * nvt);
  int *seg_pre = seg_beg + MAXSEG;
  const int b = blockIdx.x;
  const double C0 = sref[4 * b], C1 = sref[4 * b + 1], C2v = sref[4 * b + 2];
  const double Rs = sref[4 * b + 3];
  const double *xs = spos + (size_t)b * ns * 3;
  for (int s = threadIdx.x; s < ns; s += blockDim.x) {
    const double d0 = xs[3 * s] - C0, d1 = xs[3 * s + 1] - C1, d2 = xs[3 * s + 2] - C2v;
    ux[s] = (T)d0;
    uy[s] = (T)d1;
    uz[s] = (T)d2;
    uq[s] = gq[s];
    if constexpr (LOW) {
      ulo[s] = (T)(d0 - (double)ux[s]);
      ulo[ns + s] = (T)(d1 - (double)uy[s]);
      ulo[2 * ns + s] = (T)(d2 - (double)uz[s]);
    }
  }
  for (int t = threadIdx.x; t < 3 * ns * nvt; t += blockDim.x) tab[t] = gtab[t];
  const double Rm = ord_to_dbl(*(const unsigned long long *)rm_ord_p);
  const double R = P.rcmax + Rs + Rm + 1e-6 * (1.0 + P.rcmax);
  const double Cw[3] = {wrap1(C0, P.L[0]), wrap1(C1, P.L[1]), wrap1(C2v, P.L[2])};
  const int nsg = pillar_segments(P, Cw, R, cell_start, seg_beg, seg_pre);
  // segments of molecules -> segments of their sites, which lie in the same
  // order; from the last block down, since a block reads its lower
  // neighbour's last prefix sum
  for (int t0 = (nsg - 1) / (int)blockDim.x * (int)blockDim.x; t0 >= 0; t0 -= blockDim.x) {
    const int t = t0 + threadIdx.x;
    int s0 = 0, len = 0;
    if (t < nsg) {
      const int m0 = seg_beg[t], nm = seg_pre[t + 1] - seg_pre[t];
      s0 = mol_first[m0];
      len = mol_first[m0 + nm] - s0;
    }
    __syncthreads();
    if (t < nsg) {
      seg_beg[t] = s0;
      seg_pre[t + 1] = len;
    }
  }
  __syncthreads();
  block_inclusive_scan(seg_pre + 1, nsg);
  const int total = seg_pre[nsg];
  const int sj = slt_j[b];
  const int e0 = sj >= 0 ? mol_first[sj] : -1, e1 = sj >= 0 ? mol_first[sj + 1] : -1;  // the solute's own sites
  const T L0 = (T)P.L[0], L1 = (T)P.L[1], L2 = (T)P.L[2];
  const T h0 = (T)P.halfL[0], h1 = (T)P.halfL[1], h2 = (T)P.halfL[2];
  const T up2 = (T)P.up2, el2 = (T)P.el2, cut2 = (T)P.cut2, alpha = (T)P.screen;
  const int nsplit = gridDim.y, y = blockIdx.y;
  const int mine = total > y ? (total - y + nsplit - 1) / nsplit : 0;
  const int nch = (mine + chunk - 1) / chunk;
  double *out = part + ((size_t)b * nsplit + y) * 4 * ns;
  for (int r0 = 0; r0 < ns; r0 += NTHR) {  // more than one round only with one slice
    const int sl = nsl > 1 ? (int)threadIdx.x / ns : 0;
    const int s = r0 + (int)threadIdx.x - sl * ns;
    const bool on = nsl > 1 ? sl < nsl : s < ns;
    T usx = 0, usy = 0, usz = 0, qs = 0, lsx = 0, lsy = 0, lsz = 0;
    if (on) {
      usx = ux[s], usy = uy[s], usz = uz[s], qs = uq[s];
      if constexpr (LOW) lsx = ulo[s], lsy = ulo[ns + s], lsz = ulo[2 * ns + s];
    }
    double a_u = 0.0, a_q = 0.0, a_lj = 0.0, a_sg = 0.0;
    for (int ch = 0; ch < nch; ++ch) {
      const int cnt = (mine - ch + nch - 1) / nch;  // sites y + nsplit (ch + nch i), i < cnt <= chunk
      __syncthreads();
      for (int i = threadIdx.x; i < cnt; i += blockDim.x) {
        const int idx = y + nsplit * (ch + nch * i);
        int lo_s = 0, hi_s = nsg;
        while (hi_s - lo_s > 1) {
          int mid = (lo_s + hi_s) >> 1;
          if (seg_pre[mid] <= idx)
            lo_s = mid;
          else
            hi_s = mid;
        }
        const int t = seg_beg[lo_s] + (idx - seg_pre[lo_s]);
        double dx = sx[t] - C0, dy = sy[t] - C1, dz = sz[t] - C2v;
        dx -= P.L[0] * rint(dx / P.L[0]);
        dy -= P.L[1] * rint(dy / P.L[1]);
        dz -= P.L[2] * rint(dz / P.L[2]);
        vx[i] = (T)dx;
        vy[i] = (T)dy;
        vz[i] = (T)dz;
        if constexpr (LOW) {
          vlo[i] = (T)(dx - (double)vx[i]);
          vlo[chunk + i] = (T)(dy - (double)vy[i]);
          vlo[2 * chunk + i] = (T)(dz - (double)vz[i]);
        }
        vq[i] = sq[t];
        vt[i] = (t >= e0 && t < e1) ? -1 : sct[t];
      }
      __syncthreads();
      if (!on) continue;
      auto dist2 = [&](int i) {
        T dx = vx[i] - usx, dy = vy[i] - usy, dz = vz[i] - usz;
        if constexpr (LOW) {
          dx = (dx + vlo[i]) - lsx;
          dy = (dy + vlo[chunk + i]) - lsy;
          dz = (dz + vlo[2 * chunk + i]) - lsz;
        }
        T ax = fabs(dx), ay = fabs(dy), az = fabs(dz);
        ax = (ax > h0) ? L0 - ax : ax;
        ay = (ay > h1) ? L1 - ay : ay;
        az = (az > h2) ? L2 - az : az;
        return ax * ax + ay * ay + az * az;
      };
      for (int i0 = sl; i0 < cnt; i0 += 64 * nsl) {
        unsigned long long m = 0;
        const int ne = min(64, (cnt - i0 + nsl - 1) / nsl);
        for (int e = 0; e < ne; ++e) {
          const int i = i0 + e * nsl;
          if (dist2(i) <= cut2 && vt[i] >= 0) m |= 1ull << e;
        }
        while (m) {
          const int i = i0 + (__ffsll((long long)m) - 1) * nsl;
          m &= m - 1;
          const T r2 = dist2(i);
          const T *tb = tab + (s * nvt + vt[i]) * 3;
          if (tb[0] > (T)0 && r2 <= up2) {
            T rep, att;
            lj_parts_t<T>(P, tb[0], tb[1], r2, rep, att);
            const double lj = (double)(rep - att);
            a_u += lj;
            a_lj += lj;
            a_sg += (double)(((T)6 * rep - (T)3 * att) * tb[2]);
          }
          if (r2 <= el2) {
            const T c = vq[i] * erfc_over_r<T>(sqrt(r2), alpha);
            a_u += (double)(qs * c);
            a_q += (double)c;
          }
        }
      }
    }
    if (nsl == 1) {
      if (on) {
        out[s] = a_u;
        out[ns + s] = a_q;
        out[2 * ns + s] = a_lj;
        out[3 * ns + s] = a_sg;
      }
      continue;
    }
    __syncthreads();
    if (on) {
      red[(sl * 4 + 0) * ns + s] = a_u;
      red[(sl * 4 + 1) * ns + s] = a_q;
      red[(sl * 4 + 2) * ns + s] = a_lj;
      red[(sl * 4 + 3) * ns + s] = a_sg;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < 4 * ns; t += blockDim.x) {
      double v = 0.0;
      for (int k = 0; k < nsl; ++k) v += red[k * 4 * ns + t];
      out[t] = v;
    }
  }
}

// ---- per-frame solvent potential grid -----------------------------------
template <typename T> __global__ void k_fill(T *p, size_t n, T v) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// spreads the sites of every sorted physical molecule except `excl` onto the
// real grid grid[z][y][x] (recpcal.F90:357-373 with the solvent's charges).  A
// workgroup per z plane sums the sites of the p planes that reach it (the
// z-sorted sites; zsite is their index in cell order) in LDS, thread per (site,
// y, x), and writes the plane.  Bound by the LDS adds.  Global adds of a
// thread per molecule, on a cleared grid, took 131 us for 12000 sites of order 4 on
// 48^3 in FP64, this 21.
constexpr int SPREAD_THR = 1024;
template <typename T>
__global__ __launch_bounds__(SPREAD_THR) void k_spread_slv(Params P, int excl, const int *__restrict__ mol_first,
                                                           const int *__restrict__ zst,
                                                           const int *__restrict__ zsite, const int *__restrict__ zg,
                                                           const T *__restrict__ zw, const T *__restrict__ zq,
                                                           T *__restrict__ grid) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  T *pl = reinterpret_cast<T *>(lds_raw);
  const int p = P.p, pp = p * p, K1 = P.K1, K2 = P.K2, K3 = P.K3, z = blockIdx.x;
  const int e0 = excl >= 0 ? mol_first[excl] : -1, e1 = excl >= 0 ? mol_first[excl + 1] : -1;
  for (int i = threadIdx.x; i < K1 * K2; i += SPREAD_THR) pl[i] = (T)0;
  __syncthreads();
  for (int c3 = 0; c3 < p; ++c3) {
    int g3 = z + c3;
    g3 -= (g3 >= K3) ? K3 : 0;
    const int t0 = zst[g3], n = (zst[g3 + 1] - t0) * pp;
    for (int i = threadIdx.x; i < n; i += SPREAD_THR) {
      const int ts = i / pp, r = i - ts * pp, c2 = r / p, c1 = r - c2 * p, t = t0 + ts;
      const int s = zsite[t];
      if (s >= e0 && s < e1) continue;
      const int gp = zg[t];
      int x = (gp & 1023) - c1, y = ((gp >> 10) & 1023) - c2;
      x += (x < 0) ? K1 : 0;
      y += (y < 0) ? K2 : 0;
      const T *w = zw + (size_t)t * 3 * p;
      const T f3 = zq[t] * w[2 * p + c3];
      const T f2 = f3 * w[p + c2];
      atomicAdd(pl + y * K1 + x, f2 * w[c1]);
    }
  }
  __syncthreads();
  T *d = grid + (size_t)z * K1 * K2;
  for (int i = threadIdx.x; i < K1 * K2; i += SPREAD_THR) d[i] = pl[i];
}

// forward x transform of real rows, two rows per complex FFT: thread per
// (z, row pair); Hk[z][y][m1], m1 < K1/2 + 1
template <typename T, int K1>
__global__ __launch_bounds__(NTHR) void k_xrow_r2c(Params P, const T *__restrict__ grid,
                                                   const typename C2<T>::type *__restrict__ tw1,
                                                   typename C2<T>::type *Hk) {
  using V = typename C2<T>::type;
  constexpr int H = K1 / 2 + 1;
  const int K2 = P.K2, K3 = P.K3, npair = (K2 + 1) / 2;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= K3 * npair) return;
  const int z = t / npair, y0 = 2 * (t - z * npair), y1 = y0 + 1;
  const bool has1 = y1 < K2;
  const T *r0 = grid + ((size_t)z * K2 + y0) * K1;
  V Z[K1];
#pragma unroll
  for (int x = 0; x < K1; ++x) {
    Z[x].x = r0[x];
    Z[x].y = has1 ? r0[K1 + x] : (T)0;
  }
  reg_fft<K1, -1>(Z, tw1);
  V *o0 = Hk + ((size_t)z * K2 + y0) * H;
#pragma unroll
  for (int m = 0; m < H; ++m) {
    const V a = Z[m], w = Z[(K1 - m) % K1];
    V A, Cc;
    A.x = (T)0.5 * (a.x + w.x);
    A.y = (T)0.5 * (a.y - w.y);
    Cc.x = (T)0.5 * (a.y + w.y);
    Cc.y = (T)-0.5 * (a.x - w.x);
    o0[m] = A;
    if (has1) o0[H + m] = Cc;
  }
}

// z columns of the half spectrum: forward FFT, Green's function, inverse FFT
template <typename T, int K3>
__global__ __launch_bounds__(NTHR) void k_zcol_green(Params P, const T *__restrict__ engfac,
                                                     const typename C2<T>::type *__restrict__ tw3,
                                                     typename C2<T>::type *Hk) {
  using V = typename C2<T>::type;
  const int ncol = P.H * P.K2;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncol) return;
  V X[K3];
#pragma unroll
  for (int z = 0; z < K3; ++z) X[z] = Hk[(size_t)z * ncol + c];
  reg_fft<K3, -1>(X, tw3);
#pragma unroll
  for (int z = 0; z < K3; ++z) {
    const T g = engfac[(size_t)z * ncol + c];
    X[z].x *= g;
    X[z].y *= g;
  }
  reg_fft<K3, +1>(X, tw3);
#pragma unroll
  for (int z = 0; z < K3; ++z) Hk[(size_t)z * ncol + c] = X[z];
}

// inverse x transform of Hermitian row pairs into real rows grid[z][y][x]
template <typename T, int K1>
__global__ __launch_bounds__(NTHR) void k_xrow_c2r(Params P, const typename C2<T>::type *__restrict__ Hk,
                                                   const typename C2<T>::type *__restrict__ tw1, T *grid) {
  using V = typename C2<T>::type;
  constexpr int H = K1 / 2 + 1;
  const int K2 = P.K2, K3 = P.K3, npair = (K2 + 1) / 2;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= K3 * npair) return;
  const int z = t / npair, y0 = 2 * (t - z * npair), y1 = y0 + 1;
  const bool has1 = y1 < K2;
  const V *r0 = Hk + ((size_t)z * K2 + y0) * H;
  V Z[K1];
#pragma unroll
  for (int x = 0; x < H; ++x) {
    V a = r0[x];
    V cc = has1 ? r0[H + x] : V{0, 0};
    if (x == 0 || x == K1 / 2) {
      a.y = 0;
      cc.y = 0;
    }
    Z[x].x = a.x - cc.y;
    Z[x].y = a.y + cc.x;
    if (x > 0 && x < K1 - x) {
      Z[K1 - x].x = a.x + cc.y;
      Z[K1 - x].y = -a.y + cc.x;
    }
  }
  reg_fft<K1, +1>(Z, tw1);
  T *d0 = grid + ((size_t)z * K2 + y0) * K1;
#pragma unroll
  for (int x = 0; x < K1; ++x) d0[x] = Z[x].x;
  if (has1) {
#pragma unroll
    for (int x = 0; x < K1; ++x) d0[K1 + x] = Z[x].y;
  }
}

// solvent potential at every solute site of every configuration
// (calc_spline_molecule, recpcal.F90:408-442, then the gather of
// recpcal.F90:451-502 against the solvent grid); RECIP_LANES lanes per (b, s), one
// per plane of the site's support.  Bound by the latency of the p^2 loads of a
// lane and of the spline recursion (7680 sites: 33 us with a lane per site, 17 so).
constexpr int RECIP_LANES = 16;  // a power of two >= MAXP
template <typename T>
__global__ __launch_bounds__(NTHR) void k_grad_recip(Params P, int n, const double *__restrict__ spos,
                                                     const T *__restrict__ grid, double *phi) {
#pragma clang fp contract(off)
  const int i = (blockIdx.x * blockDim.x + threadIdx.x) / RECIP_LANES, c3 = threadIdx.x % RECIP_LANES;
  const int p = P.p;
  double acc = 0.0;
  if (i < n * P.ns && c3 < p) {
    const double *x = spos + (size_t)i * 3;
    const int Ks[3] = {P.K1, P.K2, P.K3};
    double w[2][MAXP], w3 = 0.0;
    int g[3];
    for (int d = 0; d < 3; ++d) {
      double f = P.invcl[d] * x[0] + P.invcl[3 + d] * x[1] + P.invcl[6 + d] * x[2];
      f = f - floor(f);
      double factor = f * (double)Ks[d];
      int rci = (factor >= 0.0 && factor <= (double)Ks[d]) ? (int)factor : 0;
      if (d == 2) w3 = spline_value_dev(P.coeff, p, factor - (double)(rci - c3));
      else
        for (int k = 0; k < MAXP; ++k)
          w[d][k] = (k < p) ? spline_value_dev(P.coeff, p, factor - (double)(rci - k)) : 0.0;
      g[d] = rci % Ks[d];
    }
    int z = g[2] - c3;
    z += (z < 0) ? P.K3 : 0;
    for (int c2 = 0; c2 < p; ++c2) {
      int y = g[1] - c2;
      y += (y < 0) ? P.K2 : 0;
      const T *row = grid + ((size_t)z * P.K2 + y) * P.K1;
      double rs = 0.0;
      for (int c1 = 0; c1 < p; ++c1) {
        int xx = g[0] - c1;
        xx += (xx < 0) ? P.K1 : 0;
        rs += w[0][c1] * (double)row[xx];
      }
      acc += w3 * w[1][c2] * rs;
    }
  }
  for (int o = RECIP_LANES / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, RECIP_LANES);
  if (c3 == 0 && i < n * P.ns) phi[i] = acc;
}

// sum of v over a workgroup of GRAD_THR threads, in a fixed order; thread 0
// returns it
constexpr int GRAD_THR = 256;
__device__ __forceinline__ double block_sum(double v) {
  __shared__ double red[GRAD_THR / 64];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = red[0];
  for (int w = 1; w < GRAD_THR / 64; ++w) t += red[w];
  return t;
}

// per configuration (one wave each; a thread each: 21 us for 256 of 30 sites,
// this 5): u_b = sum_s (u_real + q_s phi_s) + Q_slt * rf
static __global__ __launch_bounds__(GRAD_THR) void k_grad_ub(Params P, int n, int nsplit,
                          const double *__restrict__ part, const double *__restrict__ phi,
                          const double *__restrict__ qd, double rf, double qslt, double *ub) {
  const int b = blockIdx.x * (GRAD_THR / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (b >= n) return;
  const int ns = P.ns;
  double u = 0.0;
  for (int s = lane; s < ns; s += 64) {
    u += qd[s] * phi[(size_t)b * ns + s];
    for (int y = 0; y < nsplit; ++y) u += part[((size_t)b * nsplit + y) * 4 * ns + s];
  }
  for (int o = 32; o > 0; o >>= 1) u += __shfl_xor(u, o, 64);
  if (lane == 0) ub[b] = u + qslt * rf;
}

// weighted batch sums: out = [sum w, sum w u, sum w du/dq (ns),
// sum w du/deps (ns), sum w du/dsigma (ns)]; a workgroup per output, its
// threads over the configurations (a thread per output walked n nsplit
// dependent loads: 256 configurations of 30 sites 282 us, this 7)
static __global__ __launch_bounds__(GRAD_THR) void k_grad_reduce(Params P, int n, int nsplit,
                              const double *__restrict__ part, const double *__restrict__ phi,
                              const double *__restrict__ ub, const double *__restrict__ w,
                              const double *__restrict__ epsd, double rf, double *out) {
  const int o = blockIdx.x;
  const int ns = P.ns;
  double acc = 0.0;
  if (o == 0) {
    for (int b = threadIdx.x; b < n; b += GRAD_THR) acc += w[b];
  } else if (o == 1) {
    for (int b = threadIdx.x; b < n; b += GRAD_THR) acc += w[b] * ub[b];
  } else {
    const int c = (o - 2) / ns, s = (o - 2) - c * ns;  // 0 q, 1 eps, 2 sigma
    const int comp = (c == 0) ? 1 : (c == 1) ? 2 : 3;
    for (int b = threadIdx.x; b < n; b += GRAD_THR) {
      double v = 0.0;
      for (int y = 0; y < nsplit; ++y) v += part[(((size_t)b * nsplit + y) * 4 + comp) * ns + s];
      if (c == 0) v += phi[(size_t)b * ns + s] + rf;
      if (c == 1) v = (epsd[s] > 0.0) ? v / (2.0 * epsd[s]) : 0.0;
      acc += w[b] * v;
    }
  }
  acc = block_sum(acc);
  if (threadIdx.x == 0) out[o] = acc;
}

}  // namespace erm
