// ermgpu_fft2.h -- PME kernels for grid lengths K = A B transformed in two
// steps: an A-point DFT of x[n1 + B n2] over n2, the twiddle w_K^(n1 k2), a
// B-point DFT over n1.  Both steps run in registers (A, B <= 20 values) with
// one exchange through LDS between them, so a length needs no kernel of its
// own: the radices are launch arguments.  fft2_split() lists the lengths.
#pragma once

#include "ermgpu_kern.h"

namespace erm {

struct Fft2 {
  int A, B;
};

// K = A B with cases in the radix switches below.  FP64: A <= B <= 12, where a
// step's values still fit 128 registers beside their addresses.  FP32: A is a
// product of the first radices of K in the order 4, 2, 3, 5 and B of the
// others, so that the two steps are the radix steps of lds_fft (dit_steps).
template <typename T> inline bool fft2_split(int K, Fft2 &f) {
  static const int t64[][3] = {{16, 4, 4},   {18, 3, 6},  {20, 4, 5},  {24, 4, 6},  {25, 5, 5},  {27, 3, 9},
                               {30, 5, 6},   {32, 4, 8},  {36, 6, 6},  {40, 5, 8},  {45, 5, 9},  {48, 6, 8},
                               {50, 5, 10},  {54, 6, 9},  {60, 6, 10}, {64, 8, 8},  {72, 8, 9},  {80, 8, 10},
                               {81, 9, 9},   {90, 9, 10}, {96, 8, 12}, {100, 10, 10}, {108, 9, 12}, {120, 10, 12}};
  static const int t32[][3] = {{16, 4, 4},   {18, 6, 3},  {20, 4, 5},  {24, 4, 6},  {25, 5, 5},  {27, 9, 3},
                               {30, 6, 5},   {32, 4, 8},  {36, 4, 9},  {40, 8, 5},  {45, 9, 5},  {48, 4, 12},
                               {50, 10, 5},  {54, 6, 9},  {60, 12, 5}, {64, 16, 4}, {72, 8, 9},  {75, 15, 5},
                               {80, 16, 5},  {81, 9, 9},  {90, 6, 15}, {96, 16, 6}, {100, 20, 5}, {108, 12, 9},
                               {120, 8, 15}, {128, 16, 8}};
  auto find = [&](const auto &tab) {
    for (const auto &t : tab)
      if (t[0] == K) {
        f.A = t[1];
        f.B = t[2];
        return true;
      }
    return false;
  };
  return sizeof(T) == 4 ? find(t32) : find(t64);
}

#define ERM_RADIX(R, CALL) \
  case R: { constexpr int RR = R; CALL; } break;
// FP64
#define ERM_RADIX_A(A, CALL)                                                                                \
  switch (A) {                                                                                              \
    ERM_RADIX(3, CALL) ERM_RADIX(4, CALL) ERM_RADIX(5, CALL) ERM_RADIX(6, CALL) ERM_RADIX(8, CALL)          \
    ERM_RADIX(9, CALL) ERM_RADIX(10, CALL)                                                                  \
    default: break;                                                                                         \
  }
#define ERM_RADIX_B(B, CALL)                                                                                \
  switch (B) {                                                                                              \
    ERM_RADIX(4, CALL) ERM_RADIX(5, CALL) ERM_RADIX(6, CALL) ERM_RADIX(8, CALL) ERM_RADIX(9, CALL)          \
    ERM_RADIX(10, CALL)                                                                                     \
    case 12: if constexpr (BMAX >= 12) { constexpr int RR = 12; CALL; } break;                              \
    default: break;                                                                                         \
  }
// FP32
#define ERM_RADIX_A32(A, CALL)                                                                              \
  switch (A) {                                                                                              \
    ERM_RADIX(4, CALL) ERM_RADIX(5, CALL) ERM_RADIX(6, CALL) ERM_RADIX(8, CALL) ERM_RADIX(9, CALL)          \
    ERM_RADIX(10, CALL) ERM_RADIX(12, CALL) ERM_RADIX(15, CALL) ERM_RADIX(16, CALL) ERM_RADIX(20, CALL)     \
    default: break;                                                                                         \
  }
#define ERM_RADIX_B32(B, CALL)                                                                              \
  switch (B) {                                                                                              \
    ERM_RADIX(3, CALL) ERM_RADIX(4, CALL) ERM_RADIX(5, CALL) ERM_RADIX(6, CALL) ERM_RADIX(8, CALL)          \
    ERM_RADIX(9, CALL) ERM_RADIX(12, CALL) ERM_RADIX(15, CALL)                                              \
    default: break;                                                                                         \
  }

// --------------------------------------------------------------------------
// The FP32 steps.  They give bit for bit what lds_fft gives with one radix
// step per trip through LDS, since the bins' counts of an FP32 run move with
// the transforms' rounding (launch_yx): the same radices in the same order,
// each input times its table twiddle before the butterfly, products and sums
// fused where that code's are, which is written out here (explicit fmaf,
// nothing else contracted).
// --------------------------------------------------------------------------
// a times w of a table e^{-2 pi i j / K} (SIGN < 0), or its conjugate.  Of the
// imaginary part's products lds_fft rounds a.x w.y for a step's twiddles and
// a.y w.x for a root within a butterfly (ROOT); the same with the conjugate.
template <int SIGN, bool ROOT = false> __device__ __forceinline__ float2 tmul(float2 a, float2 w) {
#pragma clang fp contract(off)
  float2 r;
  if constexpr (SIGN < 0) {
    r.x = fmaf(a.x, w.x, -(a.y * w.y));
    r.y = ROOT ? fmaf(a.x, w.y, a.y * w.x) : fmaf(a.y, w.x, a.x * w.y);
  } else {
    r.x = fmaf(a.x, w.x, a.y * w.y);
    r.y = fmaf(a.y, w.x, -(a.x * w.y));
  }
  return r;
}
// an axis' table at places that are the same in every lane: through the
// constant address space it comes by scalar loads, also behind barriers
struct UTab {
  const __attribute__((address_space(4))) float *t;
  __device__ __forceinline__ explicit UTab(const float2 *tw)
      : t((const __attribute__((address_space(4))) float *)(uintptr_t)tw) {}
  __device__ __forceinline__ float2 operator[](int i) const { return make_float2(t[2 * i], t[2 * i + 1]); }
};
// R-point DFT; tw, str: w_R^j = tw[str j]
template <int R, int SIGN>
__device__ __forceinline__ void dit_dft(float2 (&x)[R], UTab tw, int str) {
#pragma clang fp contract(off)
  if constexpr (R == 4) {
    const float2 s0 = cadd(x[0], x[2]), d0 = csub(x[0], x[2]), s1 = cadd(x[1], x[3]), d1 = csub(x[1], x[3]);
    const float2 j = make_float2(-SIGN * d1.y, SIGN * d1.x);
    x[0] = cadd(s0, s1);
    x[1] = cadd(d0, j);
    x[2] = csub(s0, s1);
    x[3] = csub(d0, j);
  } else if constexpr (R == 2) {
    const float2 a = x[0];
    x[0] = cadd(a, x[1]);
    x[1] = csub(a, x[1]);
  } else {
    float2 y[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      y[q] = x[0];
#pragma unroll
      for (int s = 1; s < R; ++s)
        y[q] = cadd(y[q], (s * q) % R ? tmul<SIGN, true>(x[s], tw[(s * q) % R * str]) : x[s]);
    }
#pragma unroll
    for (int q = 0; q < R; ++q) x[q] = y[q];
  }
}
// The radix steps of an N-point block of a K-point transform, those before it
// (with product A) giving its place k: x[n1] in, frequency k + A kk out at
// x[kk].  tw is the table in memory (read at uniform places), lt the same in
// LDS (read at the lane's own); A = 1 for the first block (FIRST), N = K where
// that is the whole transform.
template <int N, int PP, int SIGN, bool FIRST, bool WHOLE = false>
__device__ __forceinline__ void dit_steps(float2 (&x)[N], int K, int A, int k, UTab tw, const float2 *lt) {
  constexpr int R = first_radix(N / PP), M = N / (PP * R);
  if constexpr (WHOLE)
    K = N;
  else
    asm volatile("" : "+s"(K));  // the table's values stay out of the registers of other steps
  float2 y[N];
#pragma unroll
  for (int r = 0; r < M; ++r)
#pragma unroll
    for (int kk = 0; kk < PP; ++kk) {
      float2 v[R];
#pragma unroll
      for (int q = 0; q < R; ++q) {
        v[q] = x[kk + PP * (r + q * M)];
        if constexpr (FIRST) {
          if (q && kk) v[q] = tmul<SIGN>(v[q], tw[q * kk * (K / (PP * R))]);
        } else {
          if (q) v[q] = tmul<SIGN>(v[q], lt[q * (k + A * kk) * M]);
        }
      }
      dit_dft<R, SIGN>(v, tw, K / R);
#pragma unroll
      for (int q = 0; q < R; ++q) {
        // a whole transform's butterflies stay in this order and in this place:
        // mixed or moved to where their results are used they take twice the registers
        if constexpr (WHOLE) asm volatile("" : "+v"(v[q].x), "+v"(v[q].y));
        y[kk + PP * (q + R * r)] = v[q];
      }
    }
#pragma unroll
  for (int i = 0; i < N; ++i) x[i] = y[i];
  if constexpr (PP * R < N) dit_steps<N, PP * R, SIGN, FIRST, WHOLE>(x, K, A, k, tw, lt);
}

// a times the conjugate of w (the twiddle tables hold e^{-2 pi i j / K})
template <typename V> __device__ __forceinline__ V cmulc(V a, V w) {
  V r;
  r.x = a.x * w.x + a.y * w.y;
  r.y = a.y * w.x - a.x * w.y;
  return r;
}

// --------------------------------------------------------------------------
// z columns.  A workgroup takes C consecutive columns (m1, m2) of one
// configuration: the solute's sites, in chunks of Z2_SCH in plane order, are
// added to the columns (each plane over the sites whose p planes hold it),
// transformed forward, multiplied by the Green's function (self energy on the
// way, recpcal.F90:385-394), transformed back and written to Hk.  The spread
// leaves the values in the registers of the first forward step, and the
// Green's function meets those of the second, which run the first inverse
// step as well: a column makes four trips through LDS and none through memory
// but its write.
// Bound by the latency of its four phases and the spread; a workgroup's threads
// take one first step each.  500 FP64 configurations of 40 x 40 x 80 with 20
// solute sites: 0.25 ms (2.2 TB/s of spectrum written), where the stages of 2
// to 5 points through LDS (k_pme_zcol) took 2.38 ms and 32 columns spread in
// LDS 0.35; one of 96^3 with 300 sites, order 6: 0.26 -> 0.053 ms.
// --------------------------------------------------------------------------
constexpr int Z2_SCH = 64;   // solute sites per chunk
constexpr int Z2_COLS = 16;  // columns per workgroup: 128 or 256 contiguous bytes of a plane
// threads: one per column and value of n1 (whole waves), so every thread
// takes one first step and those with k2 < A one second step
inline int z2_threads(int B) { return (Z2_COLS * B + 63) & ~63; }
constexpr int Z2_MAXT = 256;

// (the columns take the place of the last chunk's amplitudes)
template <typename T> __host__ __device__ inline size_t z2_lds(int K3, int p) {
  const size_t buf = 2 * sizeof(T) * (size_t)K3 * Z2_COLS;
  const size_t chunk = 2 * sizeof(T) * (size_t)Z2_SCH * Z2_COLS + sizeof(T) * (size_t)Z2_SCH * p +
                       sizeof(int) * (Z2_SCH + (size_t)K3 + 1);
  return (((buf > chunk ? buf : chunk) + 15) & ~(size_t)15) + 2 * sizeof(T) * K3 + sizeof(double) * (Z2_MAXT / 64);
}

struct Z2Args {
  int ns, p, K2, K3, H, m1, m2, cl, sub, nsub;
  bool on;
};

// Spread and first forward step of (n1 = sub, column): the thread's A planes
// n1 + B i are summed over the sites whose p planes hold them, chunk by
// chunk, in registers, transformed and written to the column.
template <typename T, int A>
__device__ __forceinline__ void z2_front(const Z2Args &q, int B, unsigned char *lds,
                                         const typename C2<T>::type *tw, const int *__restrict__ sg3,
                                         const T *__restrict__ sw3, const T *__restrict__ sqv,
                                         const typename C2<T>::type *__restrict__ w1h,
                                         const typename C2<T>::type *__restrict__ w2h) {
  using V = typename C2<T>::type;
  constexpr int C = Z2_COLS;
  const int p = q.p, K3 = q.K3;
  V *amp = reinterpret_cast<V *>(lds);                       // [Z2_SCH][C] q what1 what2 of the chunk's sites
  T *wz = reinterpret_cast<T *>(amp + (size_t)Z2_SCH * C);   // [Z2_SCH][p] z weights
  int *gz = reinterpret_cast<int *>(wz + (size_t)Z2_SCH * p);  // [Z2_SCH] planes g3, ascending
  int *first = gz + Z2_SCH;                                  // [K3 + 1] first site of the chunk with g3 >= z
  V x[A];
#pragma unroll
  for (int i = 0; i < A; ++i) {
    x[i].x = 0;
    x[i].y = 0;
  }
  for (int s0 = 0; s0 < q.ns; s0 += Z2_SCH) {
    const int nc = min(Z2_SCH, q.ns - s0);
    if (s0) __syncthreads();  // the previous chunk's sites are used up
    // site j opens the planes (g3 of j - 1, g3 of j], the last site also
    // those above it
    if (threadIdx.x < (unsigned)nc) {
      const int j = threadIdx.x, g = sg3[s0 + j], g0 = j ? sg3[s0 + j - 1] : -1;
      gz[j] = g;
      for (int z = g0 + 1; z <= g; ++z) first[z] = j;
      if (j == nc - 1)
        for (int z = g + 1; z <= K3; ++z) first[z] = nc;
    }
    for (int t = threadIdx.x; t < nc * p; t += blockDim.x) wz[t] = sw3[(size_t)s0 * p + t];
    for (int j = q.sub; j < nc; j += q.nsub) {
      const size_t s = (size_t)s0 + j;
      V a = cmul(w1h[s * q.H + q.m1], w2h[s * q.K2 + q.m2]);
      const T c = q.on ? sqv[s] : (T)0;
      a.x *= c;
      a.y *= c;
      amp[j * C + q.cl] = a;
    }
    __syncthreads();
    if (q.sub < B) {
#pragma unroll
      for (int i = 0; i < A; ++i) {
        // plane z holds the sites with g3 - z in [0, p) (mod K3)
        int z = q.sub + B * i;
        asm volatile("" : "+v"(z));  // the planes' addresses are formed one plane at a time
        const int zt = z + p;
        for (int j = first[z]; j < first[min(zt, K3)]; ++j) {
          const V a = amp[j * C + q.cl];
          const T w = wz[j * p + gz[j] - z];
          x[i].x += a.x * w;
          x[i].y += a.y * w;
        }
        if (zt > K3)  // planes wrapped past the top
          for (int j = 0; j < first[zt - K3]; ++j) {
            const V a = amp[j * C + q.cl];
            const T w = wz[j * p + gz[j] + K3 - z];
            x[i].x += a.x * w;
            x[i].y += a.y * w;
          }
      }
    }
  }
  __syncthreads();
  if (q.sub < B) {
    V *col = reinterpret_cast<V *>(lds) + q.cl;
    reg_fft<A, -1>(x);
    col[q.sub * C] = x[0];
#pragma unroll
    for (int k = 1; k < A; ++k) col[(q.sub + B * k) * C] = cmul(x[k], tw[q.sub * k]);
  }
}

// second forward step of (k2, column), Green's function, first inverse step:
// in place; returns the column's share of the self energy (weight 1)
template <typename T, int B>
__device__ __forceinline__ double z2_mid(typename C2<T>::type *col, int A, int k2, const T *__restrict__ g,
                                         size_t gstr, const typename C2<T>::type *tw) {
  using V = typename C2<T>::type;
  constexpr int C = Z2_COLS;
  T gv[B];
#pragma unroll
  for (int k = 0; k < B; ++k) gv[k] = g[(size_t)(k2 + A * k) * gstr];
  V x[B];
#pragma unroll
  for (int n = 0; n < B; ++n) x[n] = col[(B * k2 + n) * C];
  reg_fft<B, -1>(x);
  double self = 0.0;
#pragma unroll
  for (int k = 0; k < B; ++k) {
    self += (double)gv[k] * ((double)x[k].x * (double)x[k].x + (double)x[k].y * (double)x[k].y);
    x[k].x *= gv[k];
    x[k].y *= gv[k];
  }
  reg_fft<B, +1>(x);
  col[(B * k2) * C] = x[0];
#pragma unroll
  for (int n = 1; n < B; ++n) col[(B * k2 + n) * C] = cmulc(x[n], tw[k2 * n]);
  return self;
}

// last inverse step of (n1, column), into Hk
template <typename T, int A>
__device__ __forceinline__ void z2_last(const typename C2<T>::type *col, int B, int n1, typename C2<T>::type *out,
                                        size_t ostr) {
  using V = typename C2<T>::type;
  constexpr int C = Z2_COLS;
  V x[A];
#pragma unroll
  for (int k = 0; k < A; ++k) x[k] = col[(n1 + B * k) * C];
  reg_fft<A, +1>(x);
#pragma unroll
  for (int i = 0; i < A; ++i) out[(size_t)(n1 + B * i) * ostr] = x[i];
}

// (FP64; BMAX bounds the registers)
template <typename T, int BMAX>
__global__ __launch_bounds__(Z2_MAXT) void k_pme_zcol2(Params P, int A, int B, const T *__restrict__ engfac,
                                                       const int *__restrict__ sg3, const T *__restrict__ sw3,
                                                       const T *__restrict__ sqv,
                                                       const typename C2<T>::type *__restrict__ w1h,
                                                       const typename C2<T>::type *__restrict__ w2h,
                                                       const typename C2<T>::type *__restrict__ tw3,
                                                       typename C2<T>::type *Hk, double *selfp) {
  using V = typename C2<T>::type;
  constexpr int C = Z2_COLS;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const int b = blockIdx.y, K3 = P.K3;
  V *buf = reinterpret_cast<V *>(lds_raw);       // [K3][C], after the last chunk
  double *red = reinterpret_cast<double *>(lds_raw + z2_lds<T>(K3, P.p) - sizeof(double) * (Z2_MAXT / 64));
  V *tw = reinterpret_cast<V *>(red) - K3;       // [K3]
  Z2Args q;
  q.ns = P.ns;
  q.p = P.p;
  q.K2 = P.K2;
  q.K3 = K3;
  q.H = P.H;
  q.cl = threadIdx.x % C;
  q.sub = threadIdx.x / C;
  q.nsub = blockDim.x / C;
  const int ncol = P.H * P.K2, c = blockIdx.x * C + q.cl;
  q.on = c < ncol;
  q.m2 = q.on ? c / P.H : 0;
  q.m1 = q.on ? c - q.m2 * P.H : 0;
  for (int t = threadIdx.x; t < K3; t += blockDim.x) tw[t] = tw3[t];
  const size_t bs = (size_t)b * q.ns;
  ERM_RADIX_A(A, (z2_front<T, RR>(q, B, lds_raw, tw, sg3 + bs, sw3 + bs * q.p, sqv + bs, w1h + bs * q.H,
                                  w2h + bs * q.K2)))
  __syncthreads();
  double self = 0.0;
  if (q.sub < A) {
    const T *g = engfac + (size_t)q.m2 * q.H + q.m1;
    ERM_RADIX_B(B, (self = z2_mid<T, RR>(buf + q.cl, A, q.sub, g, (size_t)ncol, tw)))
  }
  self = q.on ? ((q.m1 == 0 || 2 * q.m1 == P.K1) ? 0.5 : 1.0) * self : 0.0;
  for (int o = 32; o > 0; o >>= 1) self += __shfl_xor(self, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = self;
  __syncthreads();
  if (threadIdx.x == 0) {
    double sum = red[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) sum += red[w];
    selfp[(size_t)b * gridDim.x + blockIdx.x] = sum;
  }
  if (q.on && q.sub < B) {
    V *out = Hk + (size_t)b * K3 * ncol + c;
    ERM_RADIX_A(A, (z2_last<T, RR>(buf + q.cl, B, q.sub, out, (size_t)ncol)))
  }
}

// The FP32 z columns: the same division of work, with the sums and steps in
// lds_fft's order.  The chunk's sites are added to a plane in the solute's own
// order (a bit mask per plane holds the sites that reach it), and the inverse
// transform starts with an A-point step as the forward one does, so a column
// makes one trip through LDS more.  701 configurations of 45 x 60 x 75 with 33
// solute sites: 0.66 ms (k_pme_zcol 6.08); 500 of 60^3, order 6: 0.43 (3.37).
constexpr int Z2_MAXT32 = 320;  // 16 columns x 20 values of n1 or k2
inline int z2_threads32(int A, int B) { return (Z2_COLS * (A > B ? A : B) + 63) & ~63; }
__host__ __device__ inline size_t z2_lds32(int K3, int p) {
  const size_t buf = sizeof(float2) * (size_t)K3 * Z2_COLS;
  const size_t chunk = sizeof(float2) * (size_t)Z2_SCH * Z2_COLS + sizeof(unsigned long long) * K3 +
                       (sizeof(float) * p + sizeof(int)) * (size_t)Z2_SCH;
  return (((buf > chunk ? buf : chunk) + 15) & ~(size_t)15) + sizeof(float2) * K3 + sizeof(double) * (Z2_MAXT32 / 64);
}
template <typename T> __host__ __device__ inline size_t z2_lds_of(int K3, int p) {
  return sizeof(T) == 4 ? z2_lds32(K3, p) : z2_lds<T>(K3, p);
}

// spread and first forward step of (n1 = sub, column)
template <int A>
__device__ __forceinline__ void z2_front32(const Z2Args &q, int B, unsigned char *lds, const float2 *__restrict__ tw,
                                           const int *__restrict__ sg3, const float *__restrict__ sw3,
                                           const float *__restrict__ sqv, const float2 *__restrict__ w1h,
                                           const float2 *__restrict__ w2h) {
  constexpr int C = Z2_COLS;
  const int p = q.p, K3 = q.K3;
  float2 *amp = reinterpret_cast<float2 *>(lds);  // [Z2_SCH][C] q what1 what2 of the chunk's sites
  unsigned long long *mask = reinterpret_cast<unsigned long long *>(amp + (size_t)Z2_SCH * C);  // [K3]
  float *wz = reinterpret_cast<float *>(mask + K3);            // [Z2_SCH][p] z weights
  int *gz = reinterpret_cast<int *>(wz + (size_t)Z2_SCH * p);  // [Z2_SCH] planes g3
  static_assert(Z2_SCH <= 64, "a bit per site");
  float2 x[A];
#pragma unroll
  for (int i = 0; i < A; ++i) x[i] = make_float2(0.0f, 0.0f);
  for (int s0 = 0; s0 < q.ns; s0 += Z2_SCH) {
    const int nc = min(Z2_SCH, q.ns - s0);
    if (s0) __syncthreads();  // the previous chunk's sites are used up
    for (int z = threadIdx.x; z < K3; z += blockDim.x) mask[z] = 0ull;
    for (int t = threadIdx.x; t < nc * p; t += blockDim.x) wz[t] = sw3[(size_t)s0 * p + t];
    for (int j = q.sub; j < nc; j += q.nsub) {
      const size_t s = (size_t)s0 + j;
      float2 a = tmul<-1>(w1h[s * q.H + q.m1], w2h[s * q.K2 + q.m2]);
      const float c = q.on ? sqv[s] : 0.0f;
      a.x *= c;
      a.y *= c;
      amp[j * C + q.cl] = a;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < nc * p; t += blockDim.x) {
      const int j = t / p, k = t - j * p, g = sg3[s0 + j], z = g - k + (g < k ? K3 : 0);
      if (k == 0) gz[j] = g;
      atomicOr(mask + z, 1ull << j);
    }
    __syncthreads();
    if (q.sub < B) {
#pragma unroll
      for (int i = 0; i < A; ++i) {
        int z = q.sub + B * i;
        asm volatile("" : "+v"(z));  // the planes' addresses are formed one plane at a time
        for (unsigned long long m = mask[z]; m; m &= m - 1) {
          const int j = __ffsll((long long)m) - 1;
          const int d = gz[j] - z;
          const float2 a = amp[j * C + q.cl];
          const float w = wz[j * p + d + (d < 0 ? K3 : 0)];
          x[i].x = fmaf(a.x, w, x[i].x);
          x[i].y = fmaf(a.y, w, x[i].y);
        }
      }
    }
  }
  __syncthreads();
  if (q.sub < B) {
    float2 *col = reinterpret_cast<float2 *>(lds) + q.cl;
    dit_steps<A, 1, -1, true>(x, K3, 1, 0, UTab(tw), tw);
#pragma unroll
    for (int k = 0; k < A; ++k) col[(q.sub + B * k) * C] = x[k];
  }
}

// a product that no sum after it is fused with
__device__ __forceinline__ float2 zscale(float2 a, float g) {
#pragma clang fp contract(off)
  return make_float2(a.x * g, a.y * g);
}

// second forward step of (k2 < A, column) and the Green's function, the
// spectrum in the place of the first step's values; returns the column's share
// of the self energy (weight 1).  Every thread calls it.
template <int B>
__device__ __forceinline__ double z2_mid32(float2 *col, int K3, int A, int k2, const float *__restrict__ g,
                                           size_t gstr, const float2 *__restrict__ tw, const float2 *lt) {
#pragma clang fp contract(off)
  float2 x[B];
  double self = 0.0;
  if (k2 < A) {
    float gv[B];
#pragma unroll
    for (int k = 0; k < B; ++k) gv[k] = g[(size_t)(k2 + A * k) * gstr];
#pragma unroll
    for (int n = 0; n < B; ++n) x[n] = col[(B * k2 + n) * Z2_COLS];
    dit_steps<B, 1, -1, false>(x, K3, A, k2, UTab(tw), lt);
#pragma unroll
    for (int k = 0; k < B; ++k) {
      self += (double)gv[k] * ((double)x[k].x * (double)x[k].x + (double)x[k].y * (double)x[k].y);
      x[k].x *= gv[k];
      x[k].y *= gv[k];
    }
  }
  __syncthreads();
  if (k2 < A) {
#pragma unroll
    for (int k = 0; k < B; ++k) col[(k2 + A * k) * Z2_COLS] = x[k];
  }
  return self;
}

// first inverse step of (n1, column), in place
template <int A>
__device__ __forceinline__ void z2_back32(float2 *col, int K3, int B, int n1, const float2 *__restrict__ tw) {
  float2 x[A];
#pragma unroll
  for (int i = 0; i < A; ++i) x[i] = col[(n1 + B * i) * Z2_COLS];
  dit_steps<A, 1, +1, true>(x, K3, 1, 0, UTab(tw), tw);
#pragma unroll
  for (int k = 0; k < A; ++k) col[(n1 + B * k) * Z2_COLS] = x[k];
}

// last inverse step of (k2, column), into Hk
template <int B>
__device__ __forceinline__ void z2_last32(const float2 *col, int K3, int A, int k2, const float2 *__restrict__ tw,
                                          const float2 *lt, float2 *out, size_t ostr) {
  float2 x[B];
#pragma unroll
  for (int n = 0; n < B; ++n) x[n] = col[(B * k2 + n) * Z2_COLS];
  dit_steps<B, 1, +1, false>(x, K3, A, k2, UTab(tw), lt);
#pragma unroll
  for (int k = 0; k < B; ++k) out[(size_t)(k2 + A * k) * ostr] = x[k];
}

static __global__ __launch_bounds__(Z2_MAXT32) void k_pme_zcol2_f32(
    Params P, int A, int B, const float *__restrict__ engfac, const int *__restrict__ sg3,
    const float *__restrict__ sw3, const float *__restrict__ sqv, const float2 *__restrict__ w1h,
    const float2 *__restrict__ w2h, const float2 *__restrict__ tw3, float2 *Hk, double *selfp) {
  constexpr int C = Z2_COLS;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const int b = blockIdx.y, K3 = P.K3;
  float2 *buf = reinterpret_cast<float2 *>(lds_raw);  // [K3][C], after the last chunk
  double *red = reinterpret_cast<double *>(lds_raw + z2_lds32(K3, P.p) - sizeof(double) * (Z2_MAXT32 / 64));
  float2 *lt = reinterpret_cast<float2 *>(red) - K3;  // [K3] twiddles
  Z2Args q;
  q.ns = P.ns;
  q.p = P.p;
  q.K2 = P.K2;
  q.K3 = K3;
  q.H = P.H;
  q.cl = threadIdx.x % C;
  q.sub = threadIdx.x / C;
  q.nsub = blockDim.x / C;
  const int ncol = P.H * P.K2, c = blockIdx.x * C + q.cl;
  q.on = c < ncol;
  q.m2 = q.on ? c / P.H : 0;
  q.m1 = q.on ? c - q.m2 * P.H : 0;
  for (int t = threadIdx.x; t < K3; t += blockDim.x) lt[t] = tw3[t];
  const size_t bs = (size_t)b * q.ns;
  ERM_RADIX_A32(A, (z2_front32<RR>(q, B, lds_raw, tw3, sg3 + bs, sw3 + bs * q.p, sqv + bs, w1h + bs * q.H,
                                   w2h + bs * q.K2)))
  __syncthreads();
  float2 *col = buf + q.cl;
  double self = 0.0;
  const float *g = engfac + (size_t)q.m2 * q.H + q.m1;
  ERM_RADIX_B32(B, (self = z2_mid32<RR>(col, K3, A, q.sub, g, (size_t)ncol, tw3, lt)))
  self = q.on ? ((q.m1 == 0 || 2 * q.m1 == P.K1) ? 0.5 : 1.0) * self : 0.0;
  for (int o = 32; o > 0; o >>= 1) self += __shfl_xor(self, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = self;
  __syncthreads();
  if (threadIdx.x == 0) {
    double sum = red[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) sum += red[w];
    selfp[(size_t)b * gridDim.x + blockIdx.x] = sum;
  }
  if (q.sub < B) ERM_RADIX_A32(A, (z2_back32<RR>(col, K3, B, q.sub, tw3)))
  __syncthreads();
  if (q.on && q.sub < A) {
    float2 *out = Hk + (size_t)b * K3 * ncol + c;
    ERM_RADIX_B32(B, (z2_last32<RR>(col, K3, A, q.sub, tw3, lt, out, (size_t)ncol)))
  }
}

// FP32 z columns of up to 100 points and spline orders 4 and 6 with one lane per
// column (m1, m2), the whole column in its registers: spread plane by plane
// from a list of each plane's sites in the solute's order, transformed by all
// radix steps at once.  The same values as k_pme_zcol2_f32 without its trips
// through LDS: 701 configurations of 45 x 60 x 75 with 33 solute sites 0.66 ->
// 0.42 ms, 500 of 60^3, order 6, 0.43 -> 0.27, 40 of 90^3 with 300 sites 0.33 ->
// 0.29.  Bound by issue in the transforms (two waves per SIMD) and by latency in
// the spread, whose reads run one entry ahead.
constexpr int ZD_SCH = 64;  // solute sites per chunk, a bit each
constexpr int ZD_KMAX = 127;
__host__ __device__ inline size_t zdit_lds(int H, int K2, int K3, int p) {
  return sizeof(int4) * ((size_t)ZD_SCH * p + 2) + sizeof(unsigned long long) * K3 + sizeof(double) * (NTHR / 64) +
         sizeof(float2) * (size_t)ZD_SCH * (H + zcol_fft_rows(H, K2, NTHR, 1)) + sizeof(float) * ZD_SCH +
         sizeof(int) * (K3 + 1);
}
template <int K3, int PP>
__global__ __launch_bounds__(NTHR) __attribute__((amdgpu_waves_per_eu(2))) void k_pme_zcol_dit(
    Params P, const float *__restrict__ engfac, const int *__restrict__ sg3, const float *__restrict__ sw3,
    const float *__restrict__ sqv, const float2 *__restrict__ w1h, const float2 *__restrict__ w2h,
    const float2 *__restrict__ tw3, float2 *Hk, double *selfp) {
  static_assert(K3 <= ZD_KMAX, "two planes per lane of the scan");
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const int b = blockIdx.y, ns = P.ns, H = P.H, K2 = P.K2, ncol = H * K2;
  const int c = blockIdx.x * NTHR + (int)threadIdx.x;
  const bool on = c < ncol;
  const int m2 = on ? c / H : 0, m1 = on ? c - m2 * H : 0;
  const int m2lo = blockIdx.x * NTHR / H, nm2 = min((int)(blockIdx.x + 1) * NTHR - 1, ncol - 1) / H - m2lo + 1;
  // [ZD_SCH PP + 2] the planes' sites in order: places in l1 and l2, z weight, charge
  int4 *ent = reinterpret_cast<int4 *>(lds_raw);
  unsigned long long *mask = reinterpret_cast<unsigned long long *>(ent + ZD_SCH * PP + 2);  // [K3] sites of a plane
  double *red = reinterpret_cast<double *>(mask + K3);
  float2 *l1 = reinterpret_cast<float2 *>(red + NTHR / 64);  // [ZD_SCH][H] spectra along x
  float2 *l2 = l1 + ZD_SCH * H;                              // [ZD_SCH][nm2] the block's rows of those along y
  float *lq = reinterpret_cast<float *>(l2 + ZD_SCH * zcol_fft_rows(H, K2, NTHR, 1));  // [ZD_SCH] charges
  int *st = reinterpret_cast<int *>(lq + ZD_SCH);            // [K3 + 1] first entry of a plane
  float2 x[K3];
#pragma unroll
  for (int z = 0; z < K3; ++z) x[z] = make_float2(0.0f, 0.0f);
  const size_t bs = (size_t)b * ns;
  const int row = on ? m2 - m2lo : 0;
  for (int s0 = 0; s0 < ns; s0 += ZD_SCH) {
    const int nc = min(ZD_SCH, ns - s0);
    const size_t o = bs + s0;
    __syncthreads();  // the previous chunk is used up
    for (int z = threadIdx.x; z < K3; z += NTHR) mask[z] = 0ull;
    for (int t = threadIdx.x; t < nc * H; t += NTHR) l1[t] = w1h[o * H + t];
    for (int t = threadIdx.x; t < nc * nm2; t += NTHR) {
      const int j = t / nm2;
      l2[t] = w2h[(o + j) * K2 + m2lo + (t - j * nm2)];
    }
    for (int t = threadIdx.x; t < nc; t += NTHR) lq[t] = sqv[o + t];
    __syncthreads();
    auto plane = [&](int t, int &j) {
      j = t / PP;
      const int k = t - j * PP, g = sg3[o + j];
      return g - k + (g < k ? K3 : 0);
    };
    for (int t = threadIdx.x; t < nc * PP; t += NTHR) {
      int j;
      const int z = plane(t, j);
      atomicOr(mask + z, 1ull << j);
    }
    __syncthreads();
    if (threadIdx.x < 64) {  // first entries: a scan over the planes, two per lane
      const int z = 2 * threadIdx.x;
      const int n0 = z < K3 ? __popcll(mask[z]) : 0, n1 = z + 1 < K3 ? __popcll(mask[z + 1]) : 0;
      int inc = n0 + n1;
      for (int d = 1; d < 64; d <<= 1) {
        const int u = __shfl_up(inc, d, 64);
        if ((int)threadIdx.x >= d) inc += u;
      }
      if (z <= K3) st[z] = inc - n0 - n1;
      if (z + 1 <= K3) st[z + 1] = inc - n1;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < nc * PP; t += NTHR) {
      int j;
      const int z = plane(t, j), e = st[z] + __popcll(mask[z] & ((1ull << j) - 1));
      ent[e] = make_int4(j * H, j * nm2, __float_as_int(sw3[o * PP + t]), __float_as_int(lq[j]));
    }
    if (threadIdx.x < 2) ent[nc * PP + threadIdx.x] = make_int4(0, 0, 0, 0);  // read ahead, not used
    __syncthreads();
    // one entry after another, its spectra loaded one entry ahead and its place two
    int e = 0;
    int4 h = ent[0], h1 = ent[1];
    float2 u = l1[h.x + m1], v = l2[h.y + row];
#pragma unroll
    for (int z = 0; z < K3; ++z) {
      const int e1 = __builtin_amdgcn_readfirstlane(st[z + 1]);
      while (e < e1) {
        const int4 h2 = ent[e + 2];
        const float2 u1 = l1[h1.x + m1], v1 = l2[h1.y + row];
        float2 a = tmul<-1>(u, v);
        const float w = __int_as_float(h.z), q = __int_as_float(h.w);
        a.x *= q;
        a.y *= q;
        x[z].x = fmaf(a.x, w, x[z].x);
        x[z].y = fmaf(a.y, w, x[z].y);
        h = h1;
        h1 = h2;
        u = u1;
        v = v1;
        ++e;
      }
    }
  }
  dit_steps<K3, 1, -1, true, true>(x, K3, 1, 0, UTab(tw3), tw3);
  // the Green's function in groups of 8 values, loaded a group ahead
  constexpr int GL = 8, NG = (K3 + GL - 1) / GL;
  int gi = on ? c : 0;
  float gv[2][GL];
  auto load = [&](float (&v)[GL], int m0) {
    asm volatile("" : "+v"(gi));  // not before the transform, nor all at once
#pragma unroll
    for (int i = 0; i < GL; ++i)
      if (m0 + i < K3) v[i] = engfac[gi + (size_t)i * ncol];
    gi += GL * ncol;
  };
  load(gv[0], 0);
  double self = 0.0;
#pragma unroll
  for (int q = 0; q < NG; ++q) {
    if (q + 1 < NG) load(gv[(q + 1) & 1], (q + 1) * GL);
#pragma unroll
    for (int i = 0; i < GL; ++i)
      if (q * GL + i < K3) {
        float2 &v = x[q * GL + i];
        const float g = gv[q & 1][i];
        self += (double)g * ((double)v.x * (double)v.x + (double)v.y * (double)v.y);
        v = zscale(v, g);
      }
    asm volatile("" : "+v"(self));  // here, not after the inverse transform
  }
  dit_steps<K3, 1, +1, true, true>(x, K3, 1, 0, UTab(tw3), tw3);
  if (on) {
    float2 *out = Hk + (size_t)b * K3 * ncol + c;
#pragma unroll
    for (int z = 0; z < K3; ++z) out[(size_t)z * ncol] = x[z];
  }
  self = on ? ((m1 == 0 || 2 * m1 == P.K1) ? 0.5 : 1.0) * self : 0.0;
  for (int d = 32; d > 0; d >>= 1) self += __shfl_xor(self, d, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = self;
  __syncthreads();
  if (threadIdx.x == 0) {
    double sum = red[0];
    for (int w = 1; w < NTHR / 64; ++w) sum += red[w];
    selfp[(size_t)b * gridDim.x + blockIdx.x] = sum;
  }
}

// --------------------------------------------------------------------------
// y and x transforms of a slab of z planes, and the gather (the owned planes
// [zb, zb + S) and their p - 1 halo planes, Q planes in LDS at a time; the
// sites of the slab summed in the z order).  A wave owns whole
// columns (y) and whole row pairs (x), several at once over its lanes: both
// steps of a transform and their exchange stay within the wave (LDS
// operations of a wave complete in order), so a group of planes passes
// three barriers.  The y transform's first step reads Hk straight into
// registers; the x transform takes two Hermitian rows as one complex row of
// length K1 (even or odd), and its real rows end in natural order behind
// a copy of their last p - 1 values for the gather.  Bound in FP64 by LDS (65%
// busy at 48^3), in FP32 by VALU issue and LDS in turn, a group's phases
// overlapping with the other workgroup of the CU; the gather is 40 to 60% of the
// time, and half its LDS cycles are bank conflicts between sites of a plane's
// largest class.  Measured: 500 FP64
// configurations of 40 x 40 x 80, 12000 sites, 0.29 ms (k_pme_slab 2.71); 701
// FP32 ones of 45 x 60 x 75, 18000 sites, 0.61 ms (3.61).  Against a register
// FFT per row with the planes staged in LDS and y columns transformed in HBM
// (FP64's register lengths until then): 1000 configurations of 48^3, 12000
// sites, 1.24 -> 0.49 ms; 500 of 64^3, order 6, 21000 sites, 2.23 -> 0.86.
// --------------------------------------------------------------------------
// (off lanes, on = false, read where they may and write nothing)
template <typename T, int A>
__device__ __forceinline__ void xy2_yfirst(bool on, const typename C2<T>::type *__restrict__ src, unsigned off,
                                           unsigned sstr, typename C2<T>::type *dst, int dstr, int n1, int K,
                                           const typename C2<T>::type *__restrict__ gtw,
                                           const typename C2<T>::type *tw) {
  using V = typename C2<T>::type;
  V x[A];
#pragma unroll
  for (int i = 0; i < A; ++i) x[i] = src[off + i * sstr];
  if constexpr (sizeof(T) == 4)
    dit_steps<A, 1, +1, true>(x, K, 1, 0, UTab(gtw), gtw);
  else
    reg_fft<A, +1>(x);
  if (!on) return;
  dst[0] = x[0];
#pragma unroll
  for (int k = 1; k < A; ++k) dst[k * dstr] = sizeof(T) == 4 ? x[k] : cmulc(x[k], tw[n1 * k]);
}
template <typename T, int B>
__device__ __forceinline__ void xy2_ysecond(bool on, typename C2<T>::type *col, int rs, int A, int k2, int K,
                                            const typename C2<T>::type *__restrict__ gtw,
                                            const typename C2<T>::type *tw) {
  using V = typename C2<T>::type;
  V x[B];
#pragma unroll
  for (int n = 0; n < B; ++n) x[n] = col[(k2 * B + n) * rs];
  wave_lds_sync();
  if constexpr (sizeof(T) == 4)
    dit_steps<B, 1, +1, false>(x, K, A, k2, UTab(gtw), tw);
  else
    reg_fft<B, +1>(x);
  if (!on) return;
#pragma unroll
  for (int k = 0; k < B; ++k) col[(k2 + A * k) * rs] = x[k];
}
// LDS banks.  The second x step reads blocks of B values, a lane a block: with
// B a multiple of 4 the blocks' starts fall on few banks (6 blocks of 8 in FP64
// all on one), so the values that a pair's two rows of rs hold beyond K1 are
// dealt out between the blocks (pad: 256ths of a value per block).  1000
// configurations on 48^3 in FP64 525 -> 508 us, on 40x40x80 316 -> 307; FP32
// the same within 1 %.
__device__ __forceinline__ int xy2_blk(int k, int B, int pad) { return B * k + ((k * pad) >> 8); }
// o2: offset of the pair's second row, 0 for a last row without a partner
// (its values then end in the imaginary parts too).  n = n1 + B i lies in the
// upper half, X[n] = conj X[K1 - n], for every i > A / 2 and for i = A / 2
// beyond K1 / 2; X[0] and X[K1 / 2] are real and their imaginary parts are
// not read, i = 0 and i = A / 2 again.
template <typename T, int A>
__device__ __forceinline__ void xy2_xfirst(bool on, int o2, typename C2<T>::type *pr, int K1, int B, int pad, int n1,
                                           const typename C2<T>::type *__restrict__ gtw,
                                           const typename C2<T>::type *tw) {
#pragma clang fp contract(off)
  using V = typename C2<T>::type;
  V x[A];
#pragma unroll
  for (int i = 0; i < A; ++i) {
    const int n = n1 + B * i;
    V a, c;
    if (i < A / 2) {
      a = pr[n];
      c = pr[o2 + n];
      if (i == 0) {
        a.y = (n1 == 0) ? (T)0 : a.y;
        c.y = (n1 == 0) ? (T)0 : c.y;
      }
    } else if (i > A / 2) {
      a = pr[K1 - n];
      c = pr[o2 + K1 - n];
      a.y = -a.y;
      c.y = -c.y;
    } else {
      const int t = 2 * n - K1, k = (t > 0) ? K1 - n : n;
      a = pr[k];
      c = pr[o2 + k];
      const T sg = (T)((t < 0) - (t > 0));
      a.y = sg * a.y;
      c.y = sg * c.y;
    }
    if constexpr (sizeof(T) == 4) {  // no partner: a row of zeros, which rounds as itself
      c.x = o2 ? c.x : (T)0;
      c.y = o2 ? c.y : (T)0;
    }
    x[i].x = a.x - c.y;
    x[i].y = a.y + c.x;
  }
  wave_lds_sync();
  if constexpr (sizeof(T) == 4)
    dit_steps<A, 1, +1, true>(x, K1, 1, 0, UTab(gtw), gtw);
  else
    reg_fft<A, +1>(x);
  if (!on) return;
  pr[n1] = x[0];
#pragma unroll
  for (int k = 1; k < A; ++k) pr[xy2_blk(k, B, pad) + n1] = sizeof(T) == 4 ? x[k] : cmulc(x[k], tw[n1 * k]);
}
// the real rows, x[n] at n + h, with x[K1 - h + i] again at i < h (the
// gather's wrap, h = p - 1)
template <typename T, int B>
__device__ __forceinline__ void xy2_xsecond(bool on, bool two, typename C2<T>::type *pr, int rs, int K1, int A, int h,
                                            int pad, int k2, const typename C2<T>::type *__restrict__ gtw,
                                            const typename C2<T>::type *tw) {
  using V = typename C2<T>::type;
  V x[B];
#pragma unroll
  for (int n = 0; n < B; ++n) x[n] = pr[xy2_blk(k2, B, pad) + n];
  wave_lds_sync();
  if constexpr (sizeof(T) == 4)
    dit_steps<B, 1, +1, false>(x, K1, A, k2, UTab(gtw), tw);
  else
    reg_fft<B, +1>(x);
  if (!on) return;
  T *r0 = reinterpret_cast<T *>(pr) + h + k2, *r1 = r0 + 2 * rs;
#pragma unroll
  for (int k = 0; k < B; ++k) r0[A * k] = x[k].x;
  if (two) {
#pragma unroll
    for (int k = 0; k < B; ++k) r1[A * k] = x[k].y;
  }
#pragma unroll
  for (int k = B - 1; k >= 0; --k) {
    if (A * (k + 1) <= K1 - h) break;  // uniform: no lane's value lies in the wrap
    if (k2 + A * k >= K1 - h) {
      r0[A * k - K1] = x[k].x;
      if (two) r1[A * k - K1] = x[k].y;
    }
  }
}
// v / d for 0 <= v < 2^20 from f = 1 / d: (v + 1/2) f lies at least 1 / 2d
// from an integer, far above the rounding of the product
__device__ __forceinline__ int div_by(int v, float f) { return (int)(((float)v + 0.5f) * f); }

// complex values of a row in LDS: the half spectrum, then the real row with
// its p - 1 repeated values
__host__ __device__ inline int xy2_row(int K1, int p) {
  const int H = K1 / 2 + 1, r = (K1 + p) / 2;
  return r > H ? r : H;
}
// complex values of a plane: its rows, an even number of them, padded to
// whole turns of the 32 LDS banks (the site sort's bank classes then hold for
// every plane)
__host__ __device__ inline int xy2_plane(int K2, int rs) { return ((K2 + (K2 & 1)) * rs + 15) & ~15; }
template <typename T> __host__ __device__ inline size_t xy2_lds(int Q, int K1, int K2, int p) {
  return 2 * sizeof(T) * ((size_t)Q * xy2_plane(K2, xy2_row(K1, p)) + K1 + K2);
}

constexpr int XY2_THR = 512;
// Gather of a group of nq real planes in LDS (first plane zz0) into the
// per-site sums: the sites whose p planes meet the group are one run
// [lo, hi) of the z order, dealt over the threads.  A site's first group
// (first: g3 - p + 1 >= zz0) stores its sum, a later one adds to it; the
// barrier between groups orders the two.  The planes are added in ascending
// order, so a sum does not depend on where the groups or slabs end (one
// configuration in any batch gives the same bits).
// A site's x values g1 - p + 1 .. g1 lie at g1 .. g1 + p - 1 of a row.
template <typename T, int PP>
__device__ __forceinline__ void xy2_gather(const Params &P, const T *real, const int rstr, const int pstr, int zz0,
                                           int nq, int lo, int hi, const int *__restrict__ zg,
                                           const T *__restrict__ zq, const T *__restrict__ zw, double *es) {
  const int K2 = P.K2, p = PP ? PP : P.p;
  for (int idx = lo + (int)threadIdx.x; idx < hi; idx += XY2_THR) {
    const int gp = zg[idx];
    const T qv = zq[idx];
    const T *wz = zw + (size_t)idx * 3 * p;  // [3][p]
    const int g1 = gp & 1023, g2 = (gp >> 10) & 1023, g3 = (gp >> 20) & 1023;
    const int clo = max(0, g3 - (zz0 + nq - 1)), chi = min(p - 1, g3 - zz0);
    const bool add = g3 - p + 1 < zz0;
    double acc = add ? es[idx] : 0.0;
    // rstr, pstr < 2^24
    const T *ph0 = real + __mul24(g3 - zz0, pstr) + g1;  // plane c3 = 0
    if constexpr (PP > 0) {
      T w[3 * PP];
      if constexpr (PP == 4) wz = static_cast<const T *>(__builtin_assume_aligned(wz, 16));
#pragma unroll
      for (int k = 0; k < 3 * PP; ++k) w[k] = wz[k];
      int ro[PP];
#pragma unroll
      for (int k = 0; k < PP; ++k) {
        const int y = g2 - k;
        ro[k] = __mul24(y + ((y < 0) ? K2 : 0), rstr);
      }
#pragma unroll
      for (int c3 = PP - 1; c3 >= 0; --c3) {
        if (c3 < clo || c3 > chi) continue;
        const T *ph = ph0 - c3 * pstr;
        T sum = 0;
#pragma unroll
        for (int c2 = 0; c2 < PP; ++c2) {
          const T *row = ph + ro[c2];
          T rs = 0;
#pragma unroll
          for (int c1 = 0; c1 < PP; ++c1) rs += w[c1] * row[PP - 1 - c1];
          sum += w[PP + c2] * rs;
        }
        acc += (double)(qv * w[2 * PP + c3] * sum);
      }
    } else {
      for (int c3 = chi; c3 >= clo; --c3) {
        const T *ph = ph0 - c3 * pstr;
        T sum = 0;
        for (int c2 = 0; c2 < p; ++c2) {
          int y = g2 - c2;
          y += (y < 0) ? K2 : 0;
          const T *row = ph + y * rstr;
          T rs = 0;
          for (int c1 = 0; c1 < p; ++c1) rs += wz[c1] * row[p - 1 - c1];
          sum += wz[p + c2] * rs;
        }
        acc += (double)(qv * wz[2 * p + c3] * sum);
      }
    }
    es[idx] = acc;
  }
}

#define ERM_XY_A(A, CALL)                                                                    \
  if constexpr (sizeof(T) == 4) { ERM_RADIX_A32(A, CALL) } else { ERM_RADIX_A(A, CALL) }
#define ERM_XY_B(B, CALL)                                                                    \
  if constexpr (sizeof(T) == 4) { ERM_RADIX_B32(B, CALL) } else { ERM_RADIX_B(B, CALL) }
template <typename T>
__global__ __launch_bounds__(XY2_THR) __attribute__((amdgpu_waves_per_eu(4))) void k_pme_xyslab(Params P, int S, int Q, Fft2 fy, Fft2 fx, int nsites,
                                                        const typename C2<T>::type *__restrict__ Hk,
                                                        const typename C2<T>::type *__restrict__ tw1,
                                                        const typename C2<T>::type *__restrict__ tw2,
                                                        const int *__restrict__ z_start, const int *__restrict__ zg,
                                                        const T *__restrict__ zq, const T *__restrict__ zw,
                                                        double *e_site) {
  using V = typename C2<T>::type;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const int K1 = P.K1, K2 = P.K2, K3 = P.K3, H = P.H, p = P.p;
  const int rs = xy2_row(K1, p), plane = xy2_plane(K2, rs);
  [[maybe_unused]] constexpr int BMAX = 12;
  V *stage = reinterpret_cast<V *>(lds_raw);   // [Q][plane]
  V *twy = stage + (size_t)Q * plane;          // [K2]
  V *twx = twy + K2;                           // [K1]
  for (int t = threadIdx.x; t < K2; t += XY2_THR) twy[t] = tw2[t];
  for (int t = threadIdx.x; t < K1; t += XY2_THR) twx[t] = tw1[t];
  // XCD-aware order: workgroups go to the 8 XCDs round-robin by linear index,
  // so XCD x takes the x-th contiguous share of the (configuration, slab)
  // items and finds the halo planes of consecutive slabs in its L2
  const int nwg = gridDim.x * gridDim.y;
  int L = blockIdx.y * gridDim.x + blockIdx.x;
  if (nwg % 8 == 0) L = (L % 8) * (nwg / 8) + L / 8;
  const int b = L / gridDim.x;
  const int zb = (L - b * gridDim.x) * S, ze = min(zb + S, K3);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  constexpr int NW = XY2_THR / 64;
  // A wave's round: Cy columns, dealt over its lanes by n1 (lane = n1 Gya +
  // column) in the first step and by k2 in the second, and Cx row pairs (lane =
  // pair B + n1, then pair A + k2).  FP64 has A <= B < 2 A and takes a round's
  // columns in one part each; the FP32 radices are as unlike as 4 and 12, so
  // there the step with fewer lanes per column sets the round and the
  // other takes it in parts.
  constexpr bool F32 = sizeof(T) == 4;
  const int Gya = 64 / fy.B, Gyb = F32 ? 64 / fy.A : Gya;
  const int Gxa = 64 / fx.B, Gxb = F32 ? 64 / fx.A : Gxa;
  auto round = [](int a, int b) { return min(a, b) * (max(a, b) / min(a, b)); };
  const int Cy = round(Gya, Gyb), Cx = round(Gxa, Gxb);
  const int lya = lane / Gya, lga = lane - lya * Gya, lyb = lane / Gyb, lgb = lane - lyb * Gyb;
  const int xg1 = lane / fx.B, xn0 = lane - xg1 * fx.B, xg2 = lane / fx.A, xk0 = lane - xg2 * fx.A;
  const int npair = (K2 + 1) / 2;
  const int pad = (fx.B & 3) ? 0 : min((2 * rs - K1) * 256 / (fx.A - 1), 256);
  const float fH = 1.0f / (float)H, fpair = 1.0f / (float)npair;
  double *es = e_site + (size_t)b * nsites;
  const V *src = Hk + (size_t)b * K3 * K2 * H;  // K1 K2 K3 < 2^29 values
  __syncthreads();
  for (int zz0 = zb - p + 1; zz0 < ze; zz0 += Q) {
    const int nq = min(Q, ze - zz0), ncol = nq * H;
    for (int c0 = wv * Cy; c0 < ncol; c0 += NW * Cy) {
      const int c1 = min(c0 + Cy, ncol);
      for (int g = c0; g < c1; g += Gya) {
        int ly = lya;
        asm volatile("" : "+v"(ly));  // no radix's addresses are hoisted out of the loop
        const bool in = lga < Gya && g + lga < c1;  // lanes past B Gya have ly >= B
        const int cid = in ? g + lga : c0, q = div_by(cid, fH), m1 = cid - q * H;
        const int z = zz0 + q + ((zz0 + q < 0) ? K3 : 0);
        V *col = stage + q * plane + m1;
        const int l1 = min(ly, fy.B - 1);
        ERM_XY_A(fy.A, (xy2_yfirst<T, RR>(in && ly < fy.B, src, (unsigned)((z * K2 + l1) * H + m1),
                                          (unsigned)(fy.B * H), col + l1 * rs, fy.B * rs, l1, K2, tw2, twy)))
      }
      wave_lds_sync();
      for (int g = c0; g < c1; g += Gyb) {
        int ly = lyb;
        asm volatile("" : "+v"(ly));
        const bool in = lgb < Gyb && g + lgb < c1;
        const int cid = in ? g + lgb : c0, q = div_by(cid, fH), m1 = cid - q * H;
        V *col = stage + q * plane + m1;
        ERM_XY_B(fy.B, (xy2_ysecond<T, RR>(in && ly < fy.A, col, rs, fy.A, min(ly, fy.A - 1), K2, tw2, twy)))
      }
    }
    __syncthreads();
    const int nrow = nq * npair;
    for (int p0 = wv * Cx; p0 < nrow; p0 += NW * Cx) {
      const int p1 = min(p0 + Cx, nrow);
      for (int g = p0; g < p1; g += Gxa) {
        int xn1 = xn0;
        asm volatile("" : "+v"(xn1));
        const bool in = xg1 < Gxa && g + xg1 < p1;
        const int pid = in ? g + xg1 : p0, q = div_by(pid, fpair), pr = pid - q * npair;
        V *row = stage + q * plane + 2 * pr * rs;
        ERM_XY_A(fx.A, (xy2_xfirst<T, RR>(in, (2 * pr + 1 < K2) ? rs : 0, row, K1, fx.B, pad, xn1, tw1, twx)))
      }
      wave_lds_sync();
      for (int g = p0; g < p1; g += Gxb) {
        int xk2 = xk0;
        asm volatile("" : "+v"(xk2));
        const bool in = xg2 < Gxb && g + xg2 < p1;
        const int pid = in ? g + xg2 : p0, q = div_by(pid, fpair), pr = pid - q * npair;
        V *row = stage + q * plane + 2 * pr * rs;
        ERM_XY_B(fx.B, (xy2_xsecond<T, RR>(in, 2 * pr + 1 < K2, row, rs, K1, fx.A, p - 1, pad, xk2, tw1, twx)))
      }
      wave_lds_sync();
    }
    __syncthreads();
    const T *real = reinterpret_cast<const T *>(stage);
    const int lo = z_start[max(zb, zz0)], hi = z_start[min(ze, zz0 + nq + p - 1)];
    if (p == 4)
      xy2_gather<T, 4>(P, real, 2 * rs, 2 * plane, zz0, nq, lo, hi, zg, zq, zw, es);
    else if (p == 6)
      xy2_gather<T, 6>(P, real, 2 * rs, 2 * plane, zz0, nq, lo, hi, zg, zq, zw, es);
    else
      xy2_gather<T, 0>(P, real, 2 * rs, 2 * plane, zz0, nq, lo, hi, zg, zq, zw, es);
    __syncthreads();
  }
}

}  // namespace erm
