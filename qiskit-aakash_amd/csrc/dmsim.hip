// dmsim.hip -- CDNA4 (gfx950) kernels and the C ABI of the Pauli-basis
// density-matrix engine.  See include/dmsim.h for the contract.
//
// Layout: a flat vector of N = 4^n coefficients; the 2-bit digit at
// "position" p = n-1-q of the flat index is the Pauli component of qubit q
// (stride 4^p).  All kernels update the vector in place; every element is
// read and written by exactly one thread (or one workgroup for tiles), so
// in-place updates are race free.

#include <hip/hip_runtime.h>

#include <math.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <type_traits>
#include <vector>

#include "dmsim.h"
#include "reg_plan.h"

namespace {

constexpr int kBlock = 256;
constexpr int kMaxQubits = 20;
constexpr int kFamilies = 10;  // profiling slots, see dm_profile_read

thread_local char g_err[512] = "";

int fail(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

#define HIP_TRY(expr)                                                            \
  do {                                                                           \
    hipError_t e_ = (expr);                                                      \
    if (e_ != hipSuccess)                                                        \
      return fail(DM_ERR_HIP, "%s failed: %s", #expr, hipGetErrorString(e_));    \
  } while (0)

// ---------------------------------------------------------------------------
// Small vector helpers
// ---------------------------------------------------------------------------

template <typename T, int W>
struct alignas(W * sizeof(T)) Pack {
  T v[W];
};

template <typename P, typename T>
__device__ __forceinline__ P ldp(const T *p) {
  return *reinterpret_cast<const P *>(p);
}
template <typename P, typename T>
__device__ __forceinline__ void stp(T *p, const P &x) {
  *reinterpret_cast<P *>(p) = x;
}

// 16-byte loads / stores, with the nontemporal hint when NT (streamed data
// not re-read before eviction; measured faster on gfx950 for strides of
// >= 16 coefficients, slower for stride 4).
template <typename T, bool NT>
__device__ __forceinline__ Pack<T, 16 / sizeof(T)> ld16(const T *p) {
  using P = Pack<T, 16 / sizeof(T)>;
  if (!NT) return ldp<P>(p);
  using V = T __attribute__((ext_vector_type(16 / sizeof(T))));
  const V v = __builtin_nontemporal_load(reinterpret_cast<const V *>(p));
  P r;
#pragma unroll
  for (int e = 0; e < (int)(16 / sizeof(T)); ++e) r.v[e] = v[e];
  return r;
}
template <typename T, bool NT>
__device__ __forceinline__ void st16(T *p, const Pack<T, 16 / sizeof(T)> &x) {
  if (!NT) {
    stp(p, x);
    return;
  }
  using V = T __attribute__((ext_vector_type(16 / sizeof(T))));
  V v;
#pragma unroll
  for (int e = 0; e < (int)(16 / sizeof(T)); ++e) v[e] = x.v[e];
  __builtin_nontemporal_store(v, reinterpret_cast<V *>(p));
}
// Insert a zero 2-bit digit at each of the ascending positions pos[0..m-1].
__device__ __forceinline__ uint64_t insert_digits(uint64_t r, const int *pos, int m) {
  for (int j = 0; j < m; ++j) {
    const int s = 2 * pos[j];
    const uint64_t low = r & ((1ull << s) - 1ull);
    r = ((r >> s) << (s + 2)) | low;
  }
  return r;
}

__host__ __device__ __forceinline__ uint64_t pow4(int p) { return 1ull << (2 * p); }

// ---------------------------------------------------------------------------
// K1: single-qubit PTM (rows X,Y,Z), any stride.
// ---------------------------------------------------------------------------

template <typename T>
struct Rows3 {
  T r[3][4];
};

template <typename T>
Rows3<T> make_rows3(const double *R) {
  Rows3<T> m;
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 4; ++j) m.r[i][j] = (T)R[4 * i + j];
  return m;
}

// Stride S = 4^p >= W: each unit covers W consecutive low indices of one
// (hi) slab; the four components are four coalesced W-vectors.
template <typename T, bool USE_I, bool NT>
__global__ __launch_bounds__(kBlock) void k_1q_wide(T *__restrict__ a, uint64_t units, int sh,
                                                    uint64_t S, Rows3<T> m) {
  constexpr int W = 16 / sizeof(T);
  using P = Pack<T, W>;
  const uint64_t mask = (1ull << sh) - 1ull;
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  for (uint64_t u = (uint64_t)blockIdx.x * kBlock + threadIdx.x; u < units; u += step) {
    T *b = a + ((u >> sh) * 4ull) * S + (u & mask) * W;
    P x0;
    if (USE_I) x0 = ld16<T, NT>(b);
    const P x1 = ld16<T, NT>(b + S), x2 = ld16<T, NT>(b + 2 * S), x3 = ld16<T, NT>(b + 3 * S);
    P y1, y2, y3;
#pragma unroll
    for (int e = 0; e < W; ++e) {
      T s1 = m.r[0][1] * x1.v[e] + m.r[0][2] * x2.v[e] + m.r[0][3] * x3.v[e];
      T s2 = m.r[1][1] * x1.v[e] + m.r[1][2] * x2.v[e] + m.r[1][3] * x3.v[e];
      T s3 = m.r[2][1] * x1.v[e] + m.r[2][2] * x2.v[e] + m.r[2][3] * x3.v[e];
      if (USE_I) {
        s1 += m.r[0][0] * x0.v[e];
        s2 += m.r[1][0] * x0.v[e];
        s3 += m.r[2][0] * x0.v[e];
      }
      y1.v[e] = s1;
      y2.v[e] = s2;
      y3.v[e] = s3;
    }
    st16<T, NT>(b + S, y1);
    st16<T, NT>(b + 2 * S, y2);
    st16<T, NT>(b + 3 * S, y3);
  }
}

// Stride 1 (the last qubit): the four components of a group are adjacent.
template <typename T, bool USE_I>
__global__ __launch_bounds__(kBlock) void k_1q_p0(T *__restrict__ a, uint64_t groups, Rows3<T> m) {
  using P = Pack<T, 4>;
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  for (uint64_t g = (uint64_t)blockIdx.x * kBlock + threadIdx.x; g < groups; g += step) {
    P x = ldp<P>(a + 4 * g);
    P y;
    y.v[0] = x.v[0];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      T s = m.r[r][1] * x.v[1] + m.r[r][2] * x.v[2] + m.r[r][3] * x.v[3];
      if (USE_I) s += m.r[r][0] * x.v[0];
      y.v[r + 1] = s;
    }
    stp(a + 4 * g, y);
  }
}

// ---------------------------------------------------------------------------
// K2: CX as a signed permutation of the 16 (control, target) pairs, with an
// optional per-pair scale.  Pairs are addressed in position order (hi, lo);
// CTRL_HI says whether the control qubit sits at the higher position.
// ---------------------------------------------------------------------------

template <typename T>
struct Scale16 {
  T s[16];
};

// Output pair (c,t) <- sign * input pair src(c,t), for the 12 moving pairs.
// (0,2)<-(3,2) (3,2)<-(0,2) (0,3)<-(3,3) (3,3)<-(0,3) (1,0)<-(1,1) (1,1)<-(1,0)
// (1,2)<-(2,3) (1,3)<--(2,2) (2,0)<-(2,1) (2,1)<-(2,0) (2,2)<--(1,3) (2,3)<-(1,2)
template <typename V, typename T, bool CTRL_HI, bool SCALED>
__device__ __forceinline__ void cx_map(V (&x)[4][4], const Scale16<T> &sc) {
  auto X = [&](int c, int t) -> V & { return CTRL_HI ? x[c][t] : x[t][c]; };
  auto S = [&](int c, int t) -> T { return SCALED ? sc.s[4 * c + t] : T(1); };
  V t02 = X(0, 2), t32 = X(3, 2), t03 = X(0, 3), t33 = X(3, 3);
  V t10 = X(1, 0), t11 = X(1, 1), t12 = X(1, 2), t13 = X(1, 3);
  V t20 = X(2, 0), t21 = X(2, 1), t22 = X(2, 2), t23 = X(2, 3);
  X(0, 2) = t32 * S(0, 2);
  X(3, 2) = t02 * S(3, 2);
  X(0, 3) = t33 * S(0, 3);
  X(3, 3) = t03 * S(3, 3);
  X(1, 0) = t11 * S(1, 0);
  X(1, 1) = t10 * S(1, 1);
  X(1, 2) = t23 * S(1, 2);
  X(1, 3) = -t22 * S(1, 3);
  X(2, 0) = t21 * S(2, 0);
  X(2, 1) = t20 * S(2, 1);
  X(2, 2) = -t13 * S(2, 2);
  X(2, 3) = t12 * S(2, 3);
  if (SCALED) {
    X(0, 1) = X(0, 1) * S(0, 1);
    X(3, 0) = X(3, 0) * S(3, 0);
    X(3, 1) = X(3, 1) * S(3, 1);
  }
}

// Whether pair (i_hi, i_lo) in position order is written by the CX map.
__host__ __device__ constexpr bool cx_writes(bool ctrl_hi, bool scaled, int ih, int il) {
  return (ih == 0 && il == 0) ? false
         : scaled             ? true
         : ctrl_hi            ? !((ih == 0 && il == 1) || (ih == 3 && il == 0) || (ih == 3 && il == 1))
                              : !((il == 0 && ih == 1) || (il == 3 && ih == 0) || (il == 3 && ih == 1));
}

// Low position >= 1 (stride >= W): units of W consecutive low indices.
template <typename T, bool CTRL_HI, bool SCALED, bool NT>
__global__ __launch_bounds__(kBlock) void k_cx_wide(T *__restrict__ a, uint64_t units, int sh_lo,
                                                    int sh_mid, uint64_t Sh, uint64_t Sl,
                                                    Scale16<T> sc) {
  constexpr int W = 16 / sizeof(T);
  using P = Pack<T, W>;
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  for (uint64_t u = (uint64_t)blockIdx.x * kBlock + threadIdx.x; u < units; u += step) {
    const uint64_t lo = u & ((1ull << sh_lo) - 1ull);
    const uint64_t rest = u >> sh_lo;
    const uint64_t mid = rest & ((1ull << sh_mid) - 1ull);
    const uint64_t hi = rest >> sh_mid;
    T *b = a + hi * 4ull * Sh + mid * 4ull * Sl + lo * W;
    P x[4][4];
#pragma unroll
    for (int ih = 0; ih < 4; ++ih)
#pragma unroll
      for (int il = 0; il < 4; ++il)
        if (cx_writes(CTRL_HI, SCALED, ih, il)) x[ih][il] = ld16<T, NT>(b + ih * Sh + il * Sl);
    // per-lane permutation
    P y[4][4];
#pragma unroll
    for (int e = 0; e < W; ++e) {
      T v[4][4];
#pragma unroll
      for (int ih = 0; ih < 4; ++ih)
#pragma unroll
        for (int il = 0; il < 4; ++il) v[ih][il] = cx_writes(CTRL_HI, SCALED, ih, il) ? x[ih][il].v[e] : T(0);
      cx_map<T, T, CTRL_HI, SCALED>(v, sc);
#pragma unroll
      for (int ih = 0; ih < 4; ++ih)
#pragma unroll
        for (int il = 0; il < 4; ++il) y[ih][il].v[e] = v[ih][il];
    }
#pragma unroll
    for (int ih = 0; ih < 4; ++ih)
#pragma unroll
      for (int il = 0; il < 4; ++il)
        if (cx_writes(CTRL_HI, SCALED, ih, il)) st16<T, NT>(b + ih * Sh + il * Sl, y[ih][il]);
  }
}

// Low position 0: each of the four high components is a contiguous quad.
template <typename T, bool CTRL_HI, bool SCALED>
__global__ __launch_bounds__(kBlock) void k_cx_p0(T *__restrict__ a, uint64_t groups, int sh_mid,
                                                  uint64_t Sh, Scale16<T> sc) {
  using P = Pack<T, 4>;
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  for (uint64_t g = (uint64_t)blockIdx.x * kBlock + threadIdx.x; g < groups; g += step) {
    const uint64_t mid = g & ((1ull << sh_mid) - 1ull);
    const uint64_t hi = g >> sh_mid;
    T *b = a + hi * 4ull * Sh + mid * 4ull;
    T v[4][4];
#pragma unroll
    for (int ih = 0; ih < 4; ++ih) {
      P q = ldp<P>(b + ih * Sh);
#pragma unroll
      for (int il = 0; il < 4; ++il) v[ih][il] = q.v[il];
    }
    cx_map<T, T, CTRL_HI, SCALED>(v, sc);
#pragma unroll
    for (int ih = 0; ih < 4; ++ih) {
      bool any = false;
#pragma unroll
      for (int il = 0; il < 4; ++il) any = any || cx_writes(CTRL_HI, SCALED, ih, il);
      if (any) {
        P q;
#pragma unroll
        for (int il = 0; il < 4; ++il) q.v[il] = v[ih][il];
        stp(b + ih * Sh, q);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// K2': dense two-qubit PTM (16x16), pairs in position order (hi, lo).
// ---------------------------------------------------------------------------

template <typename T>
struct Mat16 {
  T m[16][16];
};

template <typename T>
__global__ __launch_bounds__(kBlock) void k_2q_dense(T *__restrict__ a, uint64_t groups, int sh_lo,
                                                     int sh_mid, uint64_t Sh, uint64_t Sl,
                                                     Mat16<T> R, uint32_t rowmask) {
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  for (uint64_t u = (uint64_t)blockIdx.x * kBlock + threadIdx.x; u < groups; u += step) {
    const uint64_t lo = u & ((1ull << sh_lo) - 1ull);
    const uint64_t rest = u >> sh_lo;
    const uint64_t mid = rest & ((1ull << sh_mid) - 1ull);
    const uint64_t hi = rest >> sh_mid;
    T *b = a + hi * 4ull * Sh + mid * 4ull * Sl + lo;
    T x[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) x[j] = b[(j >> 2) * Sh + (j & 3) * Sl];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      if (rowmask & (1u << r)) {
        T s = T(0);
#pragma unroll
        for (int c = 0; c < 16; ++c) s += R.m[r][c] * x[c];
        b[(r >> 2) * Sh + (r & 3) * Sl] = s;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// K3: register tile of M qubits (positions pos[0..M-1], ascending): each
// thread owns the 4^M coefficients that differ only on those qubits and
// applies one 4x4 map per tile qubit.  Used for memory noise with a thermal
// feed (x,y <- h x,h y; z <- g z + d a_I) where the update is not diagonal.
// ---------------------------------------------------------------------------

template <typename T, int M>
struct TileMaps {
  int pos[M];
  T A[M][4][4];
};

template <typename T, int M>
__global__ __launch_bounds__(kBlock) void k_tile_maps(T *__restrict__ a, uint64_t units,
                                                      TileMaps<T, M> tm) {
  constexpr int E = 1 << (2 * M);
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  uint64_t S[M];
#pragma unroll
  for (int j = 0; j < M; ++j) S[j] = pow4(tm.pos[j]);
  for (uint64_t u = (uint64_t)blockIdx.x * kBlock + threadIdx.x; u < units; u += step) {
    const uint64_t base = insert_digits(u, tm.pos, M);
    T x[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      uint64_t off = 0;
#pragma unroll
      for (int j = 0; j < M; ++j) off += (uint64_t)((e >> (2 * j)) & 3) * S[j];
      x[e] = a[base + off];
    }
#pragma unroll
    for (int j = 0; j < M; ++j) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        if (((e >> (2 * j)) & 3) != 0) continue;
        const int st = 1 << (2 * j);
        T v0 = x[e], v1 = x[e + st], v2 = x[e + 2 * st], v3 = x[e + 3 * st];
        x[e + st] = tm.A[j][1][0] * v0 + tm.A[j][1][1] * v1 + tm.A[j][1][2] * v2 + tm.A[j][1][3] * v3;
        x[e + 2 * st] = tm.A[j][2][0] * v0 + tm.A[j][2][1] * v1 + tm.A[j][2][2] * v2 + tm.A[j][2][3] * v3;
        x[e + 3 * st] = tm.A[j][3][0] * v0 + tm.A[j][3][1] * v1 + tm.A[j][3][2] * v2 + tm.A[j][3][3] * v3;
      }
    }
#pragma unroll
    for (int e = 1; e < E; ++e) {
      uint64_t off = 0;
#pragma unroll
      for (int j = 0; j < M; ++j) off += (uint64_t)((e >> (2 * j)) & 3) * S[j];
      a[base + off] = x[e];
    }
  }
}

// ---------------------------------------------------------------------------
// K4: diagonal scalings.
//   k_diag_tab:  a_i *= prod_p tab[p][digit_p(i)]       (per-qubit tables)
//   k_diag_pow:  a_i *= hpow[#X/Y digits] * gpow[#Z digits] (same map on all)
//   k_product:   a_i  = scale * prod_p vec[p][digit_p(i)]  (product states)
// ---------------------------------------------------------------------------

struct Tab4 {
  double t[kMaxQubits * 4];
};

// The factor of a coefficient is the product of one table entry per digit:
// a workgroup keeps the products over the lowest kTabDigits digits in LDS
// (built from the products over their two halves) and multiplies them with
// the product over the others, which is the same for the 4^kTabDigits
// consecutive coefficients of a chunk.  Bound by HBM writes.  |0..0>, FP32:
// 16 qubits 8.4 ms with n multiplications a coefficient, 4.2 ms with chunks
// of 4^5, 3.2 ms (5.4 TB/s) with 4^6; 13 qubits 148, 74 and 49 us.
// Up to 10 qubits chunks are of 4^5, as building a larger table takes longer
// than the few coefficients of a workgroup (8 qubits FP64, 4^6 7.4 us, 4^5 6.1).
// NT: nontemporal accesses (states above the last-level cache).
constexpr int kTabDigits = 6;

template <typename T, bool WRITE_ONLY, bool NT>
__global__ __launch_bounds__(kBlock) void k_diag_tab(T *__restrict__ a, uint64_t chunks, int low, int n, Tab4 tab,
                                                     double scale) {
  constexpr int W = 16 / sizeof(T);
  using P = Pack<T, W>;
  __shared__ double s_low[1 << (2 * kTabDigits)], s_half[2][1 << kTabDigits];
  const int len = 1 << (2 * low), l0 = low / 2;
  for (int i = threadIdx.x; i < 2 << kTabDigits; i += kBlock) {
    const int half = i >> kTabDigits, k = i & ((1 << kTabDigits) - 1);
    const int p0 = half ? l0 : 0, p1 = half ? low : l0;
    double f = 1.0;
    for (int p = p0; p < p1; ++p) f *= tab.t[4 * p + ((k >> (2 * (p - p0))) & 3)];
    s_half[half][k] = f;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < len; i += kBlock) s_low[i] = s_half[0][i & ((1 << (2 * l0)) - 1)] * s_half[1][i >> (2 * l0)];
  __syncthreads();
  for (uint64_t c = blockIdx.x; c < chunks; c += gridDim.x) {
    double hi = scale;
    for (int p = low; p < n; ++p) hi *= tab.t[4 * p + ((c >> (2 * (p - low))) & 3)];
    T *b = a + c * len;
    for (int u = threadIdx.x; u < len / W; u += kBlock) {
      P x;
      if (!WRITE_ONLY) x = ld16<T, NT>(b + u * W);
#pragma unroll
      for (int e = 0; e < W; ++e) {
        const double f = hi * s_low[u * W + e];
        x.v[e] = WRITE_ONLY ? (T)f : (T)(x.v[e] * f);
      }
      st16<T, NT>(b + u * W, x);
    }
  }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_diag_pow(T *__restrict__ a, uint64_t units, int n,
                                                     double h, double g) {
  constexpr int W = 16 / sizeof(T);
  using P = Pack<T, W>;
  __shared__ T s_h[kMaxQubits + 1], s_g[kMaxQubits + 1];
  if (threadIdx.x == 0) {
    double ph = 1.0, pg = 1.0;
    for (int k = 0; k <= n; ++k) {
      s_h[k] = (T)ph;
      s_g[k] = (T)pg;
      ph *= h;
      pg *= g;
    }
  }
  __syncthreads();
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  const uint64_t m55 = 0x5555555555555555ull;
  for (uint64_t u = (uint64_t)blockIdx.x * kBlock + threadIdx.x; u < units; u += step) {
    P x = ldp<P>(a + u * W);
#pragma unroll
    for (int e = 0; e < W; ++e) {
      const uint64_t i = u * W + e;
      const uint64_t lo = i & m55, hi = (i >> 1) & m55;
      const int nz = __popcll(lo & hi);
      const int nxy = __popcll(lo ^ hi);
      x.v[e] = x.v[e] * (s_h[nxy] * s_g[nz]);
    }
    stp(a + u * W, x);
  }
}

// FP64 in place from 12 qubits on: a thread multiplies the n factors of its
// two coefficients.  Bound by HBM, and the workgroups pass over the state in
// the order of addresses, which streams better than chunks do (12 / 14 qubits
// 43 / 702 us against 46 / 730).
__global__ __launch_bounds__(kBlock) void k_diag_units(double *__restrict__ a, uint64_t units, int n, Tab4 tab,
                                                       double scale) {
  using P = Pack<double, 2>;
  __shared__ double s_tab[kMaxQubits * 4];
  for (int i = threadIdx.x; i < 4 * n; i += kBlock) s_tab[i] = tab.t[i];
  __syncthreads();
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  for (uint64_t u = (uint64_t)blockIdx.x * kBlock + threadIdx.x; u < units; u += step) {
    P x = ldp<P>(a + u * 2);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const uint64_t i = u * 2 + e;
      double f = scale;
      for (int p = 0; p < n; ++p) f *= s_tab[4 * p + ((i >> (2 * p)) & 3)];
      x.v[e] = x.v[e] * f;
    }
    stp(a + u * 2, x);
  }
}

// ---------------------------------------------------------------------------
// K5: fused k-qubit block on the matrix cores.
//
// The block's 4^K components (rows) times W contiguous "column" indices form
// a tile; C = S * B with S the 4^K x 4^K block PTM.  The tile rows are the
// digits at positions P[0..K-1]; the columns are the lowest L positions not
// in P (4^L = W); the remaining positions enumerate tiles.  B is staged in
// LDS; for K = 3 S^T is staged in LDS too, for K = 4 (256x256) it is read
// through the L2.  v_mfma_*_16x16x4 operand layout (per lane l of a wave):
//   A[16x4]: A[l%16][l/16]   B[4x16]: B[l/16][l%16]
//   D[16x16] in 4 registers: D[MfmaT<T>::row(l/16, i)][l%16]
// ---------------------------------------------------------------------------

typedef double dx4 __attribute__((ext_vector_type(4)));
typedef float fx4 __attribute__((ext_vector_type(4)));

template <typename T>
struct MfmaT;
// Accumulator row of register v in lane group lk = lane/16 (column lane%16),
// as measured on gfx950: f32 holds rows 4*lk+v, f64 holds rows lk+4*v.
template <>
struct MfmaT<double> {
  typedef dx4 acc;
  static __device__ __forceinline__ acc mma(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lk, int v) { return lk + 4 * v; }
};
template <>
struct MfmaT<float> {
  typedef fx4 acc;
  static __device__ __forceinline__ acc mma(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lk, int v) { return 4 * lk + v; }
};

struct BlockGeom {
  int n;
  int pos[4];       // block positions, ascending (digit j of the row index)
  int lpos[4];      // column positions, ascending
  int rpos[kMaxQubits];  // tile-enumerating positions, ascending
  int nr;
  uint64_t tiles;
};

template <typename T, int K, int L>
__global__ __launch_bounds__(kBlock) void k_block_mfma(T *__restrict__ a, const T *__restrict__ ST,
                                                       BlockGeom geo) {
  constexpr int ROWS = 1 << (2 * K);
  constexpr int W = 1 << (2 * L);
  constexpr int PAD = (sizeof(T) == 4 && (W % 32) == 0) ? 16 : 0;
  constexpr int LDW = W + PAD;
  constexpr bool ST_IN_LDS = (K <= 3);
  constexpr int LDR = ROWS + ((sizeof(T) == 4 && (ROWS % 32) == 0) ? 16 : 0);
  using MT = MfmaT<T>;
  using Acc = typename MT::acc;

  __shared__ T s_b[ROWS * LDW];
  __shared__ T s_st[ST_IN_LDS ? ROWS * LDR : 1];
  __shared__ uint64_t s_offr[ROWS];
  __shared__ uint64_t s_offc[W];

  const int tid = threadIdx.x;
  for (int r = tid; r < ROWS; r += kBlock) {
    uint64_t o = 0;
    for (int j = 0; j < K; ++j) o += (uint64_t)((r >> (2 * j)) & 3) << (2 * geo.pos[j]);
    s_offr[r] = o;
  }
  for (int c = tid; c < W; c += kBlock) {
    uint64_t o = 0;
    for (int j = 0; j < L; ++j) o += (uint64_t)((c >> (2 * j)) & 3) << (2 * geo.lpos[j]);
    s_offc[c] = o;
  }
  if (ST_IN_LDS) {
    for (int i = tid; i < ROWS * ROWS; i += kBlock) s_st[(i / ROWS) * LDR + (i % ROWS)] = ST[i];
  }
  __syncthreads();

  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int lr = lane & 15;   // row (A) / column (B, D) within a 16-block
  const int lk = lane >> 4;   // k index (A, B) / row quad (D)

  // Work split per wave: K=3 -> 16 row-blocks? no: 4 row-blocks x (W/16) col-blocks.
  constexpr int RB = ROWS / 16;          // row blocks
  constexpr int CB = W / 16;             // column blocks
  constexpr int NB = RB * CB;            // 16x16 output blocks per tile
  constexpr int PER_WAVE = NB / 4;       // blocks per wave (4 waves)
  static_assert(NB % 4 == 0, "tile must split over 4 waves");

  for (uint64_t t = blockIdx.x; t < geo.tiles; t += gridDim.x) {
    // tile base: deposit t's digits on the enumerating positions
    uint64_t base = 0;
    {
      uint64_t r = t;
      for (int j = 0; j < geo.nr; ++j) {
        base += (r & 3ull) << (2 * geo.rpos[j]);
        r >>= 2;
      }
    }
    // stage B
    for (int e = tid; e < ROWS * W; e += kBlock) {
      const int r = e / W, c = e % W;
      s_b[r * LDW + c] = a[base + s_offr[r] + s_offc[c]];
    }
    __syncthreads();

    Acc acc[PER_WAVE];
#pragma unroll
    for (int i = 0; i < PER_WAVE; ++i) acc[i] = Acc{0, 0, 0, 0};

    // output block index ob = wave * PER_WAVE + i -> (rb, cb) row-major over CB
#pragma unroll 4
    for (int k0 = 0; k0 < ROWS; k0 += 4) {
      const int kk = k0 + lk;
#pragma unroll
      for (int i = 0; i < PER_WAVE; ++i) {
        const int ob = wave * PER_WAVE + i;
        const int rb = ob / CB, cb = ob % CB;
        const T av = ST_IN_LDS ? s_st[kk * LDR + rb * 16 + lr] : ST[(uint64_t)kk * ROWS + rb * 16 + lr];
        const T bv = s_b[kk * LDW + cb * 16 + lr];
        acc[i] = MT::mma(av, bv, acc[i]);
      }
    }
    // write D straight to HBM
#pragma unroll
    for (int i = 0; i < PER_WAVE; ++i) {
      const int ob = wave * PER_WAVE + i;
      const int rb = ob / CB, cb = ob % CB;
      const uint64_t oc = s_offc[cb * 16 + lr];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int row = rb * 16 + MT::row(lk, j);
        a[base + s_offr[row] + oc] = acc[i][j];
      }
    }
    __syncthreads();  // s_b is restaged by the next tile
  }
}

// ---------------------------------------------------------------------------
// K5': tile program.  One workgroup stages a tile of 4^M coefficients -- the
// digits at positions tpos[0..M-1] (ascending; tpos[j] == j for j < w, so
// runs of 4^w coefficients are contiguous in HBM) with the other positions
// fixed -- in LDS, applies a short list of operations to it and writes it
// back: one HBM round trip for a whole group of gates.  Operations address
// tile digits:
//   TOP_1Q     digit d0, 12 values (rows X,Y,Z of a 4x4 PTM)
//   TOP_CX     control digit d0, target digit d1, k=1: 16 per-pair scales
//   TOP_2Q     digits d0, d1, 256 values (16x16 PTM, pair index 4 i_d0 + i_d1)
//   TOP_DENSE  k = 3 or 4 digits d0..d{k-1}: 4^k x 4^k PTM on the matrix
//              cores, values stored transposed (ST[col][row]); the other
//              tile digits index the 4^(M-k) columns.
//   TOP_STAGE  digits d0 < d1 and k members, the k records that follow it
//              (TOP_1Q on d0 or d1, TOP_CX or TOP_2Q on {d0, d1} in either
//              order), applied in order to each group of 16 coefficients in
//              registers: one LDS round trip for all of them.
// The kernels run TOP_STAGE and TOP_DENSE records; the host turns every
// other operation of a pass into a stage member (group_stages), marks the
// single-qubit members whose PTM is unital (first column (0, 0, 0): no term
// in the identity component) as TOP_1QU, and gives every CX member its 16
// scales (ones for a plain CX).  TileOp and the kinds: reg_plan.h.
// ---------------------------------------------------------------------------

struct TileGeom {
  int m;                  // tile digits (== template M)
  int w;                  // leading digits with tpos[j] == j
  int tpos[8];            // HBM position of each tile digit (ascending)
  int nr;
  int rpos[kMaxQubits];
  uint64_t tiles;
  // ident: tile index i sits at LDS index i.  Otherwise the LDS index is
  // lds_swz(i), and the operations enumerate their elements in the order of
  // TileOp::lanes.
  int ident;
};

// Swizzled LDS index.  The 64 banks of 4 bytes are LDS index bits 0-5 (tile
// digits 0-2); bits 2-3 and 4-5 take the XOR of tile digits 3 and 4, so the
// bank fields are [d0, d1 ^ d3, d2 ^ d4].  An operation on digit 1 or 2
// still has a free digit (3 or 4) that sweeps the field it occupies, and
// the quads of tile digit 0 stay contiguous.  A bijection on [0, 4^M) for
// M >= 5 that only permutes bits 2-5.
template <bool SWZ>
__device__ __forceinline__ int lds_swz(int i) {
  return SWZ ? (i ^ (((i >> 6) & 15) << 2)) : i;
}

// Tile index with the base-4 digits of g placed at the tile digits listed in
// ord (3 bits each), the operation's own digits left zero.
__device__ __forceinline__ int lane_deposit(int g, int ord, int nf) {
  int b = 0;
  for (int k = 0; k < nf; ++k) b |= ((g >> (2 * k)) & 3) << (2 * ((ord >> (3 * k)) & 7));
  return b;
}

// A quad (4 consecutive coefficients: 16 bytes in FP32, 32 in FP64) from or
// to HBM, with the nontemporal hint when NT.
template <typename T, bool NT>
__device__ __forceinline__ Pack<T, 4> ldq(const T *p) {
  constexpr int H = 16 / sizeof(T);
  Pack<T, 4> q;
#pragma unroll
  for (int h = 0; h < 4 / H; ++h) {
    const Pack<T, H> v = ld16<T, NT>(p + h * H);
#pragma unroll
    for (int e = 0; e < H; ++e) q.v[h * H + e] = v.v[e];
  }
  return q;
}
template <typename T, bool NT>
__device__ __forceinline__ void stq(T *p, const Pack<T, 4> &q) {
  constexpr int H = 16 / sizeof(T);
#pragma unroll
  for (int h = 0; h < 4 / H; ++h) {
    Pack<T, H> v;
#pragma unroll
    for (int e = 0; e < H; ++e) v.v[e] = q.v[h * H + e];
    st16<T, NT>(p + h * H, v);
  }
}

template <typename T>
__device__ __forceinline__ void lds_put_quad(T *s, int lb, const Pack<T, 4> &q) {
  *reinterpret_cast<Pack<T, 4> *>(&s[lb]) = q;
}
template <typename T>
__device__ __forceinline__ Pack<T, 4> lds_get_quad(const T *s, int lb) {
  return *reinterpret_cast<const Pack<T, 4> *>(&s[lb]);
}

// LDS accesses at a byte offset.  A stage addresses a coefficient as the
// XOR of a per-thread offset and a uniform one (scalar registers); in bytes
// that is one vector instruction per access instead of two.
template <typename V, typename T>
__device__ __forceinline__ V lds_ld(const T *s, uint32_t off) {
  return *reinterpret_cast<const V *>(reinterpret_cast<const char *>(s) + off);
}
template <typename V, typename T>
__device__ __forceinline__ void lds_st(T *s, uint32_t off, const V &x) {
  *reinterpret_cast<V *>(reinterpret_cast<char *>(s) + off) = x;
}

__device__ __forceinline__ int ins_zero(int g, int j) {
  const int lo = g & ((1 << (2 * j)) - 1);
  return ((g >> (2 * j)) << (2 * j + 2)) | lo;
}

template <typename T, int M>
__device__ __forceinline__ void tile_dense(T *s, const TileOp &op, const T *__restrict__ ST) {
  // rows: digits op.d[0..k-1] (row digit j -> tile digit d[j]); cols: the
  // remaining tile digits in ascending order.
  using MT = MfmaT<T>;
  using Acc = typename MT::acc;
  const int k = op.k;
  const int rows = 1 << (2 * k);
  const int cols = 1 << (2 * (M - k));
  int cdig[8];
  {
    int c = 0;
    for (int j = 0; j < M; ++j) {
      bool inrow = false;
      for (int r = 0; r < k; ++r) inrow = inrow || (op.d[r] == j);
      if (!inrow) cdig[c++] = j;
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  const int CB = cols / 16;
  const int NB = (rows / 16) * CB;
  const int per_wave = NB / 4;  // 4 for (M,k) = (6,3), (6,4)
  Acc acc[4];
  int rb_[4], cb_[4], coff[4];
  for (int i = 0; i < 4; ++i) {
    acc[i] = Acc{0, 0, 0, 0};
    const int ob = wave * per_wave + i;
    rb_[i] = ob / CB;
    cb_[i] = ob % CB;
    const int col = cb_[i] * 16 + lr;
    int o = 0;
    for (int j = 0; j < M - k; ++j) o |= ((col >> (2 * j)) & 3) << (2 * cdig[j]);
    coff[i] = o;
  }
  for (int k0 = 0; k0 < rows; k0 += 4) {
    const int kk = k0 + lk;
    int roff = 0;
    for (int j = 0; j < k; ++j) roff |= ((kk >> (2 * j)) & 3) << (2 * op.d[j]);
    for (int i = 0; i < per_wave; ++i) {
      const T av = ST[(size_t)kk * rows + rb_[i] * 16 + lr];
      const T bv = s[roff + coff[i]];
      acc[i] = MT::mma(av, bv, acc[i]);
    }
  }
  __syncthreads();  // every wave has read its B fragments
  for (int i = 0; i < per_wave; ++i) {
    for (int v = 0; v < 4; ++v) {
      const int row = rb_[i] * 16 + MT::row(lk, v);
      int roff = 0;
      for (int j = 0; j < k; ++j) roff |= ((row >> (2 * j)) & 3) << (2 * op.d[j]);
      s[roff + coff[i]] = acc[i][v];
    }
  }
}

template <typename T, int M>
__device__ __forceinline__ uint64_t tile_offset(int t, int w, int lomask, const TileGeom &geo) {
  uint64_t off = (uint64_t)(t & lomask);
  for (int j = w; j < M; ++j) off |= (uint64_t)((t >> (2 * j)) & 3) << (2 * geo.tpos[j]);
  return off;
}

// a * b + c with one rounding (v_fma_f32 / v_fma_f64).  The library is
// compiled without floating-point contraction (its host planner must match
// the Python planner bit for bit), so the register stages ask for it.
template <typename T>
__device__ __forceinline__ T fmad(T a, T b, T c) {
  if constexpr (sizeof(T) == 4) return __builtin_fmaf(a, b, c);
  else return __builtin_fma(a, b, c);
}

// Single-qubit member on stage digit a (LO) or b: rows X, Y, Z of the PTM;
// AFF adds the identity-component column (non-unital maps).
template <typename T, int NG, bool LO, bool AFF>
__device__ __forceinline__ void member_1q(T (&v)[NG][4][4], const T *__restrict__ pv) {
  T r[3][4];
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y) r[x][y] = pv[4 * x + y];
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      const T x0 = LO ? v[g][0][y] : v[g][y][0], x1 = LO ? v[g][1][y] : v[g][y][1];
      const T x2 = LO ? v[g][2][y] : v[g][y][2], x3 = LO ? v[g][3][y] : v[g][y][3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const T o = fmad(r[c][3], x3, fmad(r[c][2], x2, AFF ? fmad(r[c][1], x1, r[c][0] * x0) : r[c][1] * x1));
        if (LO) v[g][c + 1][y] = o;
        else v[g][y][c + 1] = o;
      }
    }
}

// CX member, control digit a (LO: pair (c, t) is v[c][t]) or b (v[t][c]),
// with its 16 per-pair scales.
template <typename T, int NG, bool LO>
__device__ __forceinline__ void member_cx(T (&v)[NG][4][4], const T *__restrict__ pv) {
  Scale16<T> sv;
#pragma unroll
  for (int u = 0; u < 16; ++u) sv.s[u] = pv[u];
#pragma unroll
  for (int g = 0; g < NG; ++g) cx_map<T, T, LO, true>(v[g], sv);
}

// 16x16 PTM member, pair index 4 i_d0 + i_d1 (first row the identity's),
// digit d0 a (lo) or b.
template <typename T, int NG>
__device__ __forceinline__ void member_2q(T (&v)[NG][4][4], const T *__restrict__ pv, bool lo) {
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    T w[16];
#pragma unroll
    for (int r = 1; r < 16; ++r) {
      T acc = T(0);
#pragma unroll
      for (int c = 0; c < 16; ++c) acc = fmad(pv[16 * r + c], lo ? v[g][c >> 2][c & 3] : v[g][c & 3][c >> 2], acc);
      w[r] = acc;
    }
#pragma unroll
    for (int r = 1; r < 16; ++r) {
      if (lo) v[g][r >> 2][r & 3] = w[r];
      else v[g][r & 3][r >> 2] = w[r];
    }
  }
}

// The member operations of a stage on NG groups of 16 coefficients in
// registers: v[g][x][y], x the component index along stage digit a (the
// lower one), y along the other digit.
template <typename T, bool GEN2Q, int NG>
__device__ __forceinline__ void stage_apply(T (&v)[NG][4][4], int a, const TileOp *__restrict__ mem, int nm,
                                            const T *__restrict__ prm) {
  for (int q = 0; q < nm; ++q) {
    const TileOp m = mem[q];
    const T *pv = prm + m.param;
    const bool lo = m.d[0] == a;
    if (m.kind == TOP_1QU) {
      if (lo) member_1q<T, NG, true, false>(v, pv);
      else member_1q<T, NG, false, false>(v, pv);
    } else if (m.kind == TOP_1Q) {
      if (lo) member_1q<T, NG, true, true>(v, pv);
      else member_1q<T, NG, false, true>(v, pv);
    } else if (!GEN2Q || m.kind == TOP_CX) {
      if (lo) member_cx<T, NG, true>(v, pv);
      else member_cx<T, NG, false>(v, pv);
    } else if (NG > 1) {
      // (7-digit FP32 tiles; with one group the selects are faster than a
      // second copy of the code and its scalar registers)
      if (lo) member_2q<T, NG>(v, pv, true);
      else member_2q<T, NG>(v, pv, false);
    } else {
      member_2q<T, NG>(v, pv, lo);
    }
  }
}

// The operations of a tile program on the LDS tile s (all threads of the
// workgroup take part; a barrier follows each operation).  Every operation
// is a stage (TOP_STAGE, digits ja < jb) or, in DENSE variants, a matrix-core
// PTM.  A stage reads each group of 16 coefficients (the 4 x 4 components
// along ja and jb) once, applies its members in registers and writes the 15
// that can change (the (I, I) component never does).  Access forms:
//  - ja = 0: one quad (16 bytes along digit 0) per component of jb;
//  - VEC, FP32, ja >= 1, at least 32 coefficients per thread (7-digit tiles
//    of 512 threads): the two groups that differ in the low bit of digit 0,
//    one 8-byte access per component pair;
//  - otherwise one 4- or 8-byte access per coefficient.
// SWZ: the tile is stored at lds_swz of each tile index, and a stage
// enumerates its groups in the digit order of TileOp::lanes (quad and
// element forms) or TileOp::qlanes (8-byte form), so that the lanes of a
// wave fall on distinct banks.  VEC is off in the 64-register one-tile
// kernel of 6-digit tiles (measured on MI355X: the 8-byte form's registers
// spill there).
template <typename T, int M, bool DENSE, bool GEN2Q, int NT, bool SWZ, bool VEC = true>
__device__ __forceinline__ void tile_ops(T *s, const TileOp *__restrict__ ops, int nops, const T *__restrict__ prm) {
  constexpr int E = 1 << (2 * M);
  constexpr int GPT = (E / 16 + NT - 1) / NT;  // groups of 16 per thread
  using Q = Pack<T, 4>;
  const int tid = threadIdx.x;
  for (int i = 0; i < nops; ++i) {
    const TileOp op = ops[i];
    if (DENSE && op.kind == TOP_DENSE) {
      if (M == 6) tile_dense<T, M>(s, op, prm + op.param);
      __syncthreads();
      continue;
    }
    // TOP_STAGE: the members follow the header in the list
    const int ja = op.d[0], jb = op.d[1];
    const TileOp *mem = ops + i + 1;
    const int nm = op.k;
    i += nm;
    uint32_t ka[4], kb[4];  // byte offsets of the components along ja, jb
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      ka[u] = lds_swz<SWZ>(u << (2 * ja)) * (uint32_t)sizeof(T);
      kb[u] = lds_swz<SWZ>(u << (2 * jb)) * (uint32_t)sizeof(T);
    }
    if (ja == 0) {
      // VEC kernels with 32+ FP32 coefficients per thread (7-digit tiles of
      // 512 threads: 2 groups) load all of a thread's groups before the
      // first operation; the others take one group at a time (their
      // register budget)
      constexpr int GB = (VEC && sizeof(T) == 4 && E / NT >= 32) ? GPT : 1;
      for (int g0 = tid; g0 < E / 16; g0 += GB * NT) {
        uint32_t bq[GB];
        T v[GB][4][4];
#pragma unroll
        for (int q = 0; q < GB; ++q) {
          const int g = g0 + q * NT;
          bq[q] = (SWZ ? lds_swz<true>(lane_deposit(g, op.lanes, M - 2)) : ins_zero(ins_zero(g, 0), jb)) * (uint32_t)sizeof(T);
          if (g < E / 16) {
#pragma unroll
            for (int y = 0; y < 4; ++y) {
              const Q qd = lds_ld<Q>(s, bq[q] ^ kb[y]);
#pragma unroll
              for (int x = 0; x < 4; ++x) v[q][x][y] = qd.v[x];
            }
          }
        }
        stage_apply<T, GEN2Q, GB>(v, 0, mem, nm, prm);
#pragma unroll
        for (int q = 0; q < GB; ++q) {
          if (g0 + q * NT >= E / 16) continue;
          // the (I, I) coefficient never changes; left visible, the compiler
          // drops it from the first quad's store and splits that store into
          // 4-byte writes that hit each bank 4 times
          asm volatile("" : "+v"(v[q][0][0]));
#pragma unroll
          for (int y = 0; y < 4; ++y) {
            Q qd;
#pragma unroll
            for (int x = 0; x < 4; ++x) qd.v[x] = v[q][x][y];
            lds_st(s, bq[q] ^ kb[y], qd);
          }
        }
      }
    } else if (VEC && sizeof(T) == 4 && E / NT >= 32) {
      // (with fewer than 32 coefficients per thread the 8-byte form would
      // leave threads idle)
      using P2 = Pack<T, 2>;
      constexpr int UN = E / 32;
      for (int un = tid; un < UN; un += NT) {
        const uint32_t b = lds_swz<SWZ>(((un & 1) << 1) | lane_deposit(un >> 1, op.qlanes, M - 3)) * (uint32_t)sizeof(T);
        T v[2][4][4];
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
          for (int y = 0; y < 4; ++y) {
            const P2 p = lds_ld<P2>(s, b ^ ka[x] ^ kb[y]);
            v[0][x][y] = p.v[0];
            v[1][x][y] = p.v[1];
          }
        stage_apply<T, GEN2Q, 2>(v, ja, mem, nm, prm);
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
          for (int y = 0; y < 4; ++y)
            if (x | y) {
              P2 p;
              p.v[0] = v[0][x][y];
              p.v[1] = v[1][x][y];
              lds_st(s, b ^ ka[x] ^ kb[y], p);
            }
      }
    } else {
      for (int g = tid; g < E / 16; g += NT) {
        const uint32_t b = (SWZ ? lds_swz<true>(lane_deposit(g, op.lanes, M - 2)) : ins_zero(ins_zero(g, ja), jb)) * (uint32_t)sizeof(T);
        T v[1][4][4];
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
          for (int y = 0; y < 4; ++y) v[0][x][y] = lds_ld<T>(s, b ^ ka[x] ^ kb[y]);
        stage_apply<T, GEN2Q, 1>(v, ja, mem, nm, prm);
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
          for (int y = 0; y < 4; ++y)
            if (x | y) lds_st(s, b ^ ka[x] ^ kb[y], v[0][x][y]);
      }
    }
    __syncthreads();
  }
}

// A fused pass: each workgroup loads a tile (the M tile digits of geo) into
// LDS, applies the pass's operations and writes it back, looping over tiles
// with stride gridDim.x and prefetching its next tile into registers.  The
// host launches grid = tiles or a persistent grid; mode bit 0 (persistent
// grids) keeps consecutive tiles on one XCD, bit 1 (FP32 runs of >= 4^3)
// makes the tile loads and stores nontemporal.  SWZ: the tile sits in LDS
// at lds_swz of each index.
template <typename T, int M, bool DENSE, bool GEN2Q, int NT, bool SWZ>
__global__ __launch_bounds__(NT) void k_tile_prog(T *__restrict__ a, TileGeom geo, const TileOp *__restrict__ ops,
                                                      int nops, const T *__restrict__ prm, int mode) {
  constexpr int E = 1 << (2 * M);
  constexpr int QPT = (E / 4 + NT - 1) / NT;  // quads per thread (4 for M=6, 1 for M=5)
  using Q = Pack<T, 4>;
  __shared__ __align__(32) T s[E];
  const int tid = threadIdx.x;
  const int w = geo.w;
  const int lomask = (1 << (2 * w)) - 1;
  // Workgroups are dispatched round-robin over the 8 XCDs (each with its own
  // L2).  With remap set (persistent grids over short runs, where
  // neighbouring tiles share HBM lines) consecutive tiles go to workgroups of
  // the same XCD: logical id = (b % 8) * (grid / 8) + b / 8.
  const uint64_t g8 = gridDim.x / 8;
  const bool remap = mode & 1;
  const uint64_t lid = (remap && gridDim.x % 8 == 0) ? (blockIdx.x % 8) * g8 + blockIdx.x / 8 : blockIdx.x;
  auto tile_base = [&](uint64_t tile) {
    uint64_t base = 0, r = tile;
    for (int j = 0; j < geo.nr; ++j) {
      base |= (r & 3ull) << (2 * geo.rpos[j]);
      r >>= 2;
    }
    return base;
  };
  // quad c = tid + i * NT is tile indices 4c..4c+3, 4 consecutive
  // coefficients in HBM and (swizzled or not) in LDS
  // nontemporal loads and stores (FP32 runs of >= 4^3 coefficients); runs
  // of 4^2 share HBM lines between neighbouring tiles through L2
  const bool nt = mode & 2;
  Q buf[QPT];
  auto load_tile = [&](uint64_t b) {
    if (nt) {
#pragma unroll
      for (int i = 0; i < QPT; ++i) {
        const int c = tid + i * NT;
        if (c < E / 4) buf[i] = ldq<T, true>(a + b + tile_offset<T, M>(4 * c, w, lomask, geo));
      }
    } else {
#pragma unroll
      for (int i = 0; i < QPT; ++i) {
        const int c = tid + i * NT;
        if (c < E / 4) buf[i] = ldq<T, false>(a + b + tile_offset<T, M>(4 * c, w, lomask, geo));
      }
    }
  };
  uint64_t tile = lid;
  if (tile < geo.tiles) load_tile(tile_base(tile));
  for (; tile < geo.tiles; tile += gridDim.x) {
    const uint64_t base = tile_base(tile);
#pragma unroll
    for (int i = 0; i < QPT; ++i) {
      const int c = tid + i * NT;
      if (c < E / 4) lds_put_quad(s, lds_swz<SWZ>(4 * c), buf[i]);
    }
    // prefetch the next tile while this one is computed
    const uint64_t next = tile + gridDim.x;
    if (next < geo.tiles) load_tile(tile_base(next));
    __syncthreads();
    tile_ops<T, M, DENSE, GEN2Q, NT, SWZ>(s, ops, nops, prm);
    if (nt) {
#pragma unroll
      for (int i = 0; i < QPT; ++i) {
        const int c = tid + i * NT;
        if (c < E / 4) stq<T, true>(a + base + tile_offset<T, M>(4 * c, w, lomask, geo), lds_get_quad(s, lds_swz<SWZ>(4 * c)));
      }
    } else {
#pragma unroll
      for (int i = 0; i < QPT; ++i) {
        const int c = tid + i * NT;
        if (c < E / 4) stq<T, false>(a + base + tile_offset<T, M>(4 * c, w, lomask, geo), lds_get_quad(s, lds_swz<SWZ>(4 * c)));
      }
    }
    __syncthreads();
  }
}

// The first or last stage of a one-tile pass, fused with the HBM copy: DIR
// 0 reads the stage's groups of 16 coefficients from HBM and writes its
// result to the LDS tile, DIR 1 reads the groups from LDS and writes the
// result to HBM, DIR 2 (a pass of one stage) goes from HBM to HBM without
// LDS.  Saves one LDS round trip on either side.  Only for stages whose
// group order is contiguous in HBM and conflict-free in LDS (stage_io_ok):
// digit 0 with a digit >= 3 (one quad per component; lanes over digits 1, 2
// first), or two digits >= 3 (lanes over digits 0-2 first; FP32 7-digit
// tiles pair the groups that differ in the low bit of digit 0 into 8-byte
// accesses).  A thread loads all its groups before the first operation.
// NTM: nontemporal HBM accesses (one-tile passes over whole states; the
// batch's small states keep them cached).
__host__ __device__ __forceinline__ bool stage_io_ok(const TileOp &op) {
  return (op.d[0] == 0 && op.d[1] >= 3) || op.d[0] >= 3;
}

template <typename T, int M, bool GEN2Q, int NT, bool SWZ, bool VEC, int DIR, bool NTM = true>
__device__ __forceinline__ void stage_io(T *__restrict__ a, uint64_t base, int w, int lomask, const TileGeom &geo,
                                         T *s, const TileOp *__restrict__ ops, int at, const T *__restrict__ prm) {
  constexpr int E = 1 << (2 * M);
  constexpr int GPT = (E / 16 + NT - 1) / NT;  // groups per thread
  using Q = Pack<T, 4>;
  const TileOp op = ops[at];
  const int ja = op.d[0], jb = op.d[1];
  const TileOp *mem = ops + at + 1;
  const int nm = op.k;
  const int tid = threadIdx.x;
  uint32_t ka[4], kb[4];  // LDS byte offsets of the components along ja, jb
  uint64_t ha[4], hb[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    ka[u] = lds_swz<SWZ>(u << (2 * ja)) * (uint32_t)sizeof(T);
    kb[u] = lds_swz<SWZ>(u << (2 * jb)) * (uint32_t)sizeof(T);
    ha[u] = (uint64_t)u << (2 * geo.tpos[ja]);
    hb[u] = (uint64_t)u << (2 * geo.tpos[jb]);
  }
  if (VEC && sizeof(T) == 4 && ja != 0) {
    // one unit per thread: the two groups that differ in the low bit of
    // digit 0, one 8-byte access per component pair
    using P2 = Pack<T, 2>;
    const int un = tid;
    if (un < E / 32) {
      const int bt = ((un & 1) << 1) | lane_deposit(un >> 1, op.qlanes, M - 3);
      const uint32_t lb = lds_swz<SWZ>(bt) * (uint32_t)sizeof(T);
      T *hp = a + base + tile_offset<T, M>(bt, w, lomask, geo);
      T v[2][4][4];
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) {
          P2 p;
          if (DIR == 1) {
            p = lds_ld<P2>(s, lb ^ ka[x] ^ kb[y]);
          } else {
            using V2 = T __attribute__((ext_vector_type(2)));
            const V2 *qp = reinterpret_cast<const V2 *>(hp + ha[x] + hb[y]);
            const V2 q = NTM ? __builtin_nontemporal_load(qp) : *qp;
            p.v[0] = q[0];
            p.v[1] = q[1];
          }
          v[0][x][y] = p.v[0];
          v[1][x][y] = p.v[1];
        }
      stage_apply<T, GEN2Q, 2>(v, ja, mem, nm, prm);
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) {
          if (DIR == 0) {
            P2 p;
            p.v[0] = v[0][x][y];
            p.v[1] = v[1][x][y];
            lds_st(s, lb ^ ka[x] ^ kb[y], p);
          } else {
            using V2 = T __attribute__((ext_vector_type(2)));
            V2 q;
            q[0] = v[0][x][y];
            q[1] = v[1][x][y];
            if (NTM) __builtin_nontemporal_store(q, reinterpret_cast<V2 *>(hp + ha[x] + hb[y]));
            else *reinterpret_cast<V2 *>(hp + ha[x] + hb[y]) = q;
          }
        }
    }
    return;
  }
  uint32_t lb[GPT];
  T *hp[GPT];
  T v[GPT][4][4];
#pragma unroll
  for (int q = 0; q < GPT; ++q) {
    const int g = tid + q * NT;
    const int bt = SWZ ? lane_deposit(g, op.lanes, M - 2) : ins_zero(ins_zero(g, ja), jb);
    lb[q] = lds_swz<SWZ>(bt) * (uint32_t)sizeof(T);
    hp[q] = a + base + tile_offset<T, M>(bt, w, lomask, geo);
    if (ja == 0) {
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        const Q qd = DIR == 1 ? lds_ld<Q>(s, lb[q] ^ kb[y]) : ldq<T, NTM>(hp[q] + hb[y]);
#pragma unroll
        for (int x = 0; x < 4; ++x) v[q][x][y] = qd.v[x];
      }
    } else {
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y)
          v[q][x][y] = DIR == 1 ? lds_ld<T>(s, lb[q] ^ ka[x] ^ kb[y])
                                : NTM ? __builtin_nontemporal_load(hp[q] + ha[x] + hb[y]) : hp[q][ha[x] + hb[y]];
    }
  }
  stage_apply<T, GEN2Q, GPT>(v, ja, mem, nm, prm);
#pragma unroll
  for (int q = 0; q < GPT; ++q) {
    if (ja == 0) {
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        Q qd;
#pragma unroll
        for (int x = 0; x < 4; ++x) qd.v[x] = v[q][x][y];
        if (DIR == 0) lds_st(s, lb[q] ^ kb[y], qd);
        else stq<T, NTM>(hp[q] + hb[y], qd);
      }
    } else {
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) {
          if (DIR == 0) lds_st(s, lb[q] ^ ka[x] ^ kb[y], v[q][x][y]);
          else if (NTM) __builtin_nontemporal_store(v[q][x][y], hp[q] + ha[x] + hb[y]);
          else hp[q][ha[x] + hb[y]] = v[q][x][y];
        }
    }
  }
}

// One tile per workgroup (grid = tiles, tile = block index): no prefetch of
// a next tile, so fewer registers during the operations and more resident
// workgroups per CU, which overlap each other's HBM and LDS phases.  Runs
// are >= 4^3 coefficients: nontemporal loads and stores (NTM; measured
// faster on MI355X for FP32 runs, 6 % on 7-digit tiles; FP64 keeps plain
// accesses).  FP32: 8 waves per SIMD (64
// VGPRs), 7 for swizzled tiles (72 VGPRs: their XOR addresses cannot use
// instruction offsets; 64 spilled); 7-digit tiles 4 waves (128 VGPRs), the
// two 512-thread workgroups their 64 KB of LDS allow per CU.
template <typename T, int M, bool GEN2Q, int NT, bool SWZ, bool NTM = true>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? ((1 << (2 * M)) / NT >= 32 ? 4 : SWZ && NT <= 256 ? 7 : 8) : 1))) void k_tile_stream(T *__restrict__ a, TileGeom geo, const TileOp *__restrict__ ops,
                                                        int nops, const T *__restrict__ prm, int io, int last_at) {
  constexpr int E = 1 << (2 * M);
  constexpr int QPT = (E / 4 + NT - 1) / NT;
  using Q = Pack<T, 4>;
  __shared__ __align__(32) T s[E];
  const uint64_t tile = blockIdx.x;
  if (tile >= geo.tiles) return;  // uniform over the workgroup
  const int tid = threadIdx.x;
  const int w = geo.w;
  const int lomask = (1 << (2 * w)) - 1;
  uint64_t base = 0, r = tile;
  for (int j = 0; j < geo.nr; ++j) {
    base |= (r & 3ull) << (2 * geo.rpos[j]);
    r >>= 2;
  }
  // io bit 0: the first operation is a stage that reads HBM itself, bit 1:
  // the stage with header last_at (the last operation) writes HBM itself
  constexpr bool VEC = E / NT >= 32;
  if ((io & 3) == 3 && last_at == 0) {
    stage_io<T, M, GEN2Q, NT, SWZ, VEC, 2, NTM>(a, base, w, lomask, geo, s, ops, 0, prm);
    return;
  }
  int i0 = 0;
  if (io & 1) {
    stage_io<T, M, GEN2Q, NT, SWZ, VEC, 0, NTM>(a, base, w, lomask, geo, s, ops, 0, prm);
    i0 = 1 + ops[0].k;
  } else if constexpr (VEC) {
    // 2 workgroups per CU: every load of the tile is issued before the first
    // LDS write (and every LDS read before the first store), so a thread
    // waits for HBM once.  6-digit tiles (8 workgroups per CU, 64 VGPRs)
    // keep one quad in flight per thread, which needs no buffer registers.
    Q buf[QPT];
#pragma unroll
    for (int i = 0; i < QPT; ++i) {
      const int c = tid + i * NT;
      if (c < E / 4) buf[i] = ldq<T, NTM>(a + base + tile_offset<T, M>(4 * c, w, lomask, geo));
    }
#pragma unroll
    for (int i = 0; i < QPT; ++i) {
      const int c = tid + i * NT;
      if (c < E / 4) lds_put_quad(s, lds_swz<SWZ>(4 * c), buf[i]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < QPT; ++i) {
      const int c = tid + i * NT;
      if (c < E / 4) lds_put_quad(s, lds_swz<SWZ>(4 * c), ldq<T, NTM>(a + base + tile_offset<T, M>(4 * c, w, lomask, geo)));
    }
  }
  __syncthreads();
  const int i1 = (io & 2) ? last_at : nops;
  tile_ops<T, M, false, GEN2Q, NT, SWZ, VEC>(s, ops + i0, i1 - i0, prm);
  if (io & 2) {
    stage_io<T, M, GEN2Q, NT, SWZ, VEC, 1, NTM>(a, base, w, lomask, geo, s, ops, last_at, prm);
  } else if constexpr (VEC) {
    Q buf[QPT];
#pragma unroll
    for (int i = 0; i < QPT; ++i) {
      const int c = tid + i * NT;
      if (c < E / 4) buf[i] = lds_get_quad(s, lds_swz<SWZ>(4 * c));
    }
#pragma unroll
    for (int i = 0; i < QPT; ++i) {
      const int c = tid + i * NT;
      if (c < E / 4) stq<T, NTM>(a + base + tile_offset<T, M>(4 * c, w, lomask, geo), buf[i]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < QPT; ++i) {
      const int c = tid + i * NT;
      if (c < E / 4) stq<T, NTM>(a + base + tile_offset<T, M>(4 * c, w, lomask, geo), lds_get_quad(s, lds_swz<SWZ>(4 * c)));
    }
  }
}

#include "tile_reg.h"

// ---------------------------------------------------------------------------
// K6: reductions (FP64 accumulation).
// ---------------------------------------------------------------------------

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

__device__ __forceinline__ double block_sum(double v) {
  __shared__ double s_part[kBlock / 64];
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) s_part[wave] = v;
  __syncthreads();
  double t = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < kBlock / 64; ++w) t += s_part[w];
  return t;
}

// W consecutive coefficients as FP64, streamed (nontemporal).
template <int W, typename T>
__device__ __forceinline__ void load_sum(const T *p, double (&x)[W]) {
  constexpr int H = W * sizeof(T) > 16 ? 16 / sizeof(T) : W;
  using V = T __attribute__((ext_vector_type(H)));
#pragma unroll
  for (int h = 0; h < W / H; ++h) {
    const V v = __builtin_nontemporal_load(reinterpret_cast<const V *>(p + h * H));
#pragma unroll
    for (int e = 0; e < H; ++e) x[h * H + e] = (double)v[e];
  }
}

// Sums over N coefficients, N a multiple of 4: each thread takes packs of 16
// bytes with the stride of the grid, two in flight.  Bound by HBM (14 qubits:
// FP32, one coefficient per load 282 us, packs 170; FP64 355 and 311, with 32
// bytes a thread 370; more than 1024 workgroups are slower).
constexpr int kSumGrid = 1024;

template <typename T>
__global__ __launch_bounds__(kBlock) void k_sumsq(const T *__restrict__ a, uint64_t packs, double *part) {
  constexpr int W = 16 / sizeof(T);
  double s0 = 0.0, s1 = 0.0;
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  for (; i + step < packs; i += 2 * step) {
    double x[W], y[W];
    load_sum<W>(a + W * i, x);
    load_sum<W>(a + W * (i + step), y);
#pragma unroll
    for (int e = 0; e < W; ++e) {
      s0 += x[e] * x[e];
      s1 += y[e] * y[e];
    }
  }
  if (i < packs) {
    double x[W];
    load_sum<W>(a + W * i, x);
#pragma unroll
    for (int e = 0; e < W; ++e) s0 += x[e] * x[e];
  }
  const double s = block_sum(s0 + s1);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

template <typename T, typename TB>
__global__ __launch_bounds__(kBlock) void k_dot(const T *__restrict__ a, const TB *__restrict__ b,
                                                uint64_t N, double *part) {
  double s = 0.0;
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < N; i += step)
    s += (double)a[i] * b[i];
  s = block_sum(s);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// per block: max |a-b|, sum a*b, sum a*a, sum b*b (columns of gridDim.x).
// Coefficients per load: four, in FP64 against FP64 one (14 qubits: 594 us with
// one and 2048 workgroups, 638 with two and 1024, 734 with four and 4096;
// FP32 against FP32 341 with four, 535 with one).
template <typename TA, typename TB>
struct DiffShape {
  static constexpr bool both64 = sizeof(TA) + sizeof(TB) == 16;
  static constexpr int width = both64 ? 1 : 4, grid = both64 ? 2 * kSumGrid : kSumGrid;
};

template <typename TA, typename TB>
__global__ __launch_bounds__(kBlock) void k_diff(const TA *__restrict__ a, const TB *__restrict__ b, uint64_t packs,
                                                 double *part) {
  constexpr int W = DiffShape<TA, TB>::width;
  double mx = 0.0, ab = 0.0, aa = 0.0, bb = 0.0;
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < packs; i += step) {
    double x[W], y[W];
    load_sum<W>(a + W * i, x);
    load_sum<W>(b + W * i, y);
#pragma unroll
    for (int e = 0; e < W; ++e) {
      mx = fmax(mx, fabs(x[e] - y[e]));
      ab += x[e] * y[e];
      aa += x[e] * x[e];
      bb += y[e] * y[e];
    }
  }
  __shared__ double s_m[kBlock];
  s_m[threadIdx.x] = mx;
  __syncthreads();
  for (int off = kBlock / 2; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) s_m[threadIdx.x] = fmax(s_m[threadIdx.x], s_m[threadIdx.x + off]);
    __syncthreads();
  }
  const double m = s_m[0];
  __syncthreads();
  ab = block_sum(ab);
  __syncthreads();
  aa = block_sum(aa);
  __syncthreads();
  bb = block_sum(bb);
  if (threadIdx.x == 0) {
    const int g = gridDim.x;
    part[blockIdx.x] = m;
    part[g + blockIdx.x] = ab;
    part[2 * g + blockIdx.x] = aa;
    part[3 * g + blockIdx.x] = bb;
  }
}

// The partials of k_diff: out[0] their maximum, out[1..3] their sums.
__global__ __launch_bounds__(kBlock) void k_diff_parts(const double *part, int nparts, double *out) {
  const double *p = part + (size_t)blockIdx.x * nparts;
  if (blockIdx.x == 0) {
    __shared__ double s_m[kBlock];
    double m = 0.0;
    for (int i = threadIdx.x; i < nparts; i += kBlock) m = fmax(m, p[i]);
    s_m[threadIdx.x] = m;
    __syncthreads();
    for (int off = kBlock / 2; off > 0; off >>= 1) {
      if ((int)threadIdx.x < off) s_m[threadIdx.x] = fmax(s_m[threadIdx.x], s_m[threadIdx.x + off]);
      __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = s_m[0];
    return;
  }
  double s = 0.0;
  for (int i = threadIdx.x; i < nparts; i += kBlock) s += p[i];
  s = block_sum(s);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}

__global__ __launch_bounds__(kBlock) void k_sum_parts(const double *part, int nparts, double *out) {
  double s = 0.0;
  for (int i = threadIdx.x; i < nparts; i += kBlock) s += part[i];
  s = block_sum(s);
  if (threadIdx.x == 0) out[0] = s;
}

// Gather the coefficients with measured qubits' components in the basis
// support and I on every other qubit. j's digit t (base 2 or 4, most
// significant first) is measured qubit t.
struct GatherSpec {
  int m;
  int base_log;           // 1 (components {0,k}) or 2 (all four)
  int comp;               // k for base 2
  uint64_t stride[kMaxQubits];
};

template <typename T>
__global__ __launch_bounds__(kBlock) void k_gather(const T *__restrict__ a, uint64_t count, GatherSpec gs,
                                                   double *out) {
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  for (uint64_t j = (uint64_t)blockIdx.x * kBlock + threadIdx.x; j < count; j += step) {
    uint64_t idx = 0;
    for (int t = 0; t < gs.m; ++t) {
      const int sh = gs.base_log * (gs.m - 1 - t);
      const uint64_t d = (j >> sh) & ((1ull << gs.base_log) - 1ull);
      const uint64_t c = gs.base_log == 1 ? (d ? (uint64_t)gs.comp : 0ull) : d;
      idx += c * gs.stride[t];
    }
    out[j] = (double)a[idx];
  }
}

// Gather and the contraction of the last `low` measured digits, in LDS: the
// block's gathered values are those of the leading digits' index blockIdx.x.
// Base 2 (components {I, k}): digit pairs (u, w) -> (u + e w, u - e w) in
// place.  Base 4: values of 4 components -> 2 outcomes, the leading digit of
// the remaining index first, ping-pong between two halves of LDS.  One launch
// instead of a gather and one contraction per digit (latency bound: 16 qubits
// 17 launches of 4.5 us).
constexpr int kProbDigits2 = 12;  // 32 KB of LDS
constexpr int kProbDigits4 = 6;   // 32 KB and 16 KB

template <typename T>
__global__ __launch_bounds__(1024) void k_probs(const T *__restrict__ a, GatherSpec gs, int low, double w1, double w2,
                                                double w3, double *__restrict__ out) {
  __shared__ double s[4096 + 2048];
  const int bl = gs.base_log;
  const uint32_t cnt = 1u << (bl * low);
  uint64_t base = 0;
  for (int t = 0; t < gs.m - low; ++t) {
    const uint64_t d = ((uint64_t)blockIdx.x >> (bl * (gs.m - low - 1 - t))) & ((1u << bl) - 1u);
    base += (bl == 1 ? (d ? (uint64_t)gs.comp : 0ull) : d) * gs.stride[t];
  }
  for (uint32_t j = threadIdx.x; j < cnt; j += blockDim.x) {
    uint64_t idx = base;
    for (int t = 0; t < low; ++t) {
      const uint32_t d = (j >> (bl * (low - 1 - t))) & ((1u << bl) - 1u);
      idx += (bl == 1 ? (d ? (uint64_t)gs.comp : 0ull) : (uint64_t)d) * gs.stride[gs.m - low + t];
    }
    s[j] = (double)a[idx];
  }
  __syncthreads();
  double *src = s;
  if (bl == 1) {
    for (int q = 0; q < low; ++q) {
      for (uint32_t x = threadIdx.x; x < cnt / 2; x += blockDim.x) {
        const uint32_t lo = x & ((1u << q) - 1u), b = ((x >> q) << (q + 1)) | lo;
        const double u = s[b], w = w1 * s[b | (1u << q)];
        s[b] = u + w;
        s[b | (1u << q)] = u - w;
      }
      __syncthreads();
    }
  } else {
    double *dst = s + 4096;
    for (int t = 0; t < low; ++t) {
      // (2^t, 4, post) -> (2^t, 2, post)
      const uint32_t post = 1u << (2 * (low - 1 - t)), total = (2u << t) * post;
      for (uint32_t o = threadIdx.x; o < total / 2; o += blockDim.x) {
        const uint32_t q = o & (post - 1), p = o / post;
        const double *x = src + (size_t)p * 4 * post + q;
        const double u = x[0], w = w1 * x[post] + w2 * x[2 * post] + w3 * x[3 * post];
        dst[(size_t)p * 2 * post + q] = u + w;
        dst[(size_t)p * 2 * post + post + q] = u - w;
      }
      __syncthreads();
      double *const t2 = src;
      src = dst;
      dst = t2;
    }
  }
  const uint32_t no = 1u << low;
  for (uint32_t x = threadIdx.x; x < no; x += blockDim.x) out[(uint64_t)blockIdx.x * no + x] = src[x];
}

// Contraction of up to four leading base-2 digits in registers: column c of
// (2^lead, 2^D, post) values.
template <int D>
__global__ __launch_bounds__(kBlock) void k_probs_lead(double *__restrict__ v, uint64_t cols, uint64_t post, double e) {
  const uint64_t c = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  if (c >= cols) return;
  double *p = v + (c / post) * (post << D) + c % post;
  double x[1 << D];
#pragma unroll
  for (int i = 0; i < (1 << D); ++i) x[i] = p[(uint64_t)i * post];
#pragma unroll
  for (int q = 0; q < D; ++q)
#pragma unroll
    for (int i = 0; i < (1 << D); ++i)
      if (!((i >> q) & 1)) {
        const double u = x[i], w = e * x[i | (1 << q)];
        x[i] = u + w;
        x[i | (1 << q)] = u - w;
      }
#pragma unroll
  for (int i = 0; i < (1 << D); ++i) p[(uint64_t)i * post] = x[i];
}

// One contraction step over a base-4 digit: (pre, 4, post) -> (pre, 2, post),
// the outcomes u + w and u - w of u = in[p, 0, q], w = sum_k wk in[p, k, q].
__global__ __launch_bounds__(kBlock) void k_contract(const double *__restrict__ in, double *__restrict__ out,
                                                     uint64_t pre, uint64_t post, double w1, double w2, double w3) {
  const uint64_t total = pre * post;
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  for (uint64_t o = (uint64_t)blockIdx.x * kBlock + threadIdx.x; o < total; o += step) {
    const uint64_t q = o % post, p = o / post;
    const double *x = in + p * 4 * post + q;
    const double u = x[0], w = w1 * x[post] + w2 * x[2 * post] + w3 * x[3 * post];
    out[p * 2 * post + q] = u + w;
    out[p * 2 * post + post + q] = u - w;
  }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_chop(T *__restrict__ a, uint64_t N, T thr) {
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < N; i += step)
    if (fabs((double)a[i]) < (double)thr) a[i] = T(0);
}

template <typename TS, typename TD>
__global__ __launch_bounds__(kBlock) void k_convert(const TS *__restrict__ s, TD *__restrict__ d, uint64_t N) {
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < N; i += step) d[i] = (TD)s[i];
}

// ---------------------------------------------------------------------------
// K7: Pauli -> matrix conversion.  Per qubit, (I,X,Y,Z) -> (I+Z, X-iY, X+iY,
// I-Z) on complex values; then mu_q = 2 r_q + c_q is scattered to
// (row, col) with qubit 0 the most significant bit.
// ---------------------------------------------------------------------------

// First qubit: real coefficients in, complex values out (out of place).
template <typename TS>
__global__ __launch_bounds__(kBlock) void k_dense_first(const TS *__restrict__ in, double2 *__restrict__ out,
                                                        uint64_t groups, int p) {
  const uint64_t S = pow4(p);
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  for (uint64_t g = (uint64_t)blockIdx.x * kBlock + threadIdx.x; g < groups; g += step) {
    const uint64_t hi = g >> (2 * p), lo = g & (S - 1);
    const uint64_t b = hi * 4 * S + lo;
    const double x0 = (double)in[b], x1 = (double)in[b + S], x2 = (double)in[b + 2 * S], x3 = (double)in[b + 3 * S];
    // mu0 = I + Z; mu1 = X - iY; mu2 = X + iY; mu3 = I - Z
    out[b] = make_double2(x0 + x3, 0.0);
    out[b + S] = make_double2(x1, -x2);
    out[b + 2 * S] = make_double2(x1, x2);
    out[b + 3 * S] = make_double2(x0 - x3, 0.0);
  }
}

// Every other qubit, in place on the complex buffer: each thread owns the
// four entries of its group.
__global__ __launch_bounds__(kBlock) void k_dense_pass(double2 *__restrict__ buf, uint64_t groups, int p) {
  const uint64_t S = pow4(p);
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  for (uint64_t g = (uint64_t)blockIdx.x * kBlock + threadIdx.x; g < groups; g += step) {
    const uint64_t hi = g >> (2 * p), lo = g & (S - 1);
    const uint64_t b = hi * 4 * S + lo;
    const double2 x0 = buf[b], x1 = buf[b + S], x2 = buf[b + 2 * S], x3 = buf[b + 3 * S];
    buf[b] = make_double2(x0.x + x3.x, x0.y + x3.y);
    buf[b + S] = make_double2(x1.x + x2.y, x1.y - x2.x);
    buf[b + 2 * S] = make_double2(x1.x - x2.y, x1.y + x2.x);
    buf[b + 3 * S] = make_double2(x0.x - x3.x, x0.y - x3.y);
  }
}

__device__ __forceinline__ uint64_t spread_bits(uint64_t x) {
  // bit i -> bit 2i (x < 2^32)
  x &= 0xffffffffull;
  x = (x | (x << 16)) & 0x0000ffff0000ffffull;
  x = (x | (x << 8)) & 0x00ff00ff00ff00ffull;
  x = (x | (x << 4)) & 0x0f0f0f0f0f0f0f0full;
  x = (x | (x << 2)) & 0x3333333333333333ull;
  x = (x | (x << 1)) & 0x5555555555555555ull;
  return x;
}

// Output entries [o0, o0 + count) of the row-major 2^n x 2^n matrix: entry
// (row, col) is the buffer value at the bit-interleaved index
// sum_q (2 r_q + c_q) 4^p(q).
__global__ __launch_bounds__(kBlock) void k_dense_scatter(const double2 *__restrict__ b, double2 *__restrict__ out,
                                                          int n, uint64_t o0, uint64_t count) {
  const uint64_t dim = 1ull << n;
  const uint64_t step = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < count; i += step) {
    const uint64_t o = o0 + i;
    const uint64_t row = o >> n, col = o & (dim - 1);
    out[i] = b[(spread_bits(row) << 1) | spread_bits(col)];
  }
}

}  // namespace

namespace {

// ---------------------------------------------------------------------------
// K8: whole-circuit kernel for small registers (n <= 7).  One workgroup holds
// one circuit's entire state (4^n coefficients, at most 128 KB in FP64) in
// LDS, applies its operations (tile ops over all n digits; TOP_ALLQ applies
// one 1q map to every qubit, the per-level memory noise), then writes the
// Z-basis ensemble probabilities 2^n values and its start / end GPU clock.
// ---------------------------------------------------------------------------

enum { TOP_ALLQ = 5 };

struct BatchCirc {
  int32_t n, nops;
  int64_t op_off;   // first TileOp
  int64_t out_off;  // first probability
  double err;       // measurement polarisation retention
};

__device__ __forceinline__ void stamp_now(uint64_t *where) { *where = wall_clock64(); }

__global__ void k_stamp(uint64_t *where) { stamp_now(where); }

template <typename T>
__global__ __launch_bounds__(1024) void k_circuit_lds(const BatchCirc *__restrict__ circs, const TileOp *__restrict__ allops,
                                                      const T *__restrict__ prm, double *__restrict__ probs,
                                                      uint64_t *__restrict__ stamps) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *s = reinterpret_cast<T *>(smem_raw);
  const BatchCirc c = circs[blockIdx.x];
  const int n = c.n;
  const int E = 1 << (2 * n);
  const int tid = threadIdx.x, nt = blockDim.x;
  if (tid == 0) stamp_now(&stamps[2 * blockIdx.x]);
  const T amp = (T)ldexp(1.0, -n);
  for (int i = tid; i < E; i += nt) {
    // |0...0>: 2^-n on indices whose digits are all I or Z
    const uint32_t lo = (uint32_t)i & 0x55555555u, hi = ((uint32_t)i >> 1) & 0x55555555u;
    s[i] = (lo ^ hi) ? T(0) : amp;
  }
  __syncthreads();
  const TileOp *ops = allops + c.op_off;
  for (int oi = 0; oi < c.nops; ++oi) {
    const TileOp op = ops[oi];
    const T *pv = prm + op.param;
    if (op.kind == TOP_1Q || op.kind == TOP_ALLQ) {
      const int j0 = op.kind == TOP_1Q ? op.d[0] : 0;
      const int j1 = op.kind == TOP_1Q ? op.d[0] + 1 : n;
      for (int j = j0; j < j1; ++j) {
        const int st = 1 << (2 * j);
        for (int g = tid; g < E / 4; g += nt) {
          const int b = ins_zero(g, j);
          const T x0 = s[b], x1 = s[b + st], x2 = s[b + 2 * st], x3 = s[b + 3 * st];
          s[b + st] = pv[0] * x0 + pv[1] * x1 + pv[2] * x2 + pv[3] * x3;
          s[b + 2 * st] = pv[4] * x0 + pv[5] * x1 + pv[6] * x2 + pv[7] * x3;
          s[b + 3 * st] = pv[8] * x0 + pv[9] * x1 + pv[10] * x2 + pv[11] * x3;
        }
        __syncthreads();
      }
      continue;
    }
    if (op.kind == TOP_CX || op.kind == TOP_2Q) {
      const int jc = op.d[0], jt = op.d[1];
      const int jl = min(jc, jt), jh = max(jc, jt);
      const int sc = 1 << (2 * jc), stt = 1 << (2 * jt);
      for (int g = tid; g < E / 16; g += nt) {
        const int b = ins_zero(ins_zero(g, jl), jh);
        T v[4][4];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
          for (int t = 0; t < 4; ++t) v[a][t] = s[b + a * sc + t * stt];
        if (op.kind == TOP_CX) {
          Scale16<T> sv;
#pragma unroll
          for (int q = 0; q < 16; ++q) sv.s[q] = op.k ? pv[q] : T(1);
          cx_map<T, T, true, true>(v, sv);
#pragma unroll
          for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int t = 0; t < 4; ++t)
              if (a | t) s[b + a * sc + t * stt] = v[a][t];
        } else {
#pragma unroll
          for (int r = 1; r < 16; ++r) {
            T acc = T(0);
#pragma unroll
            for (int q = 0; q < 16; ++q) acc += pv[16 * r + q] * v[q >> 2][q & 3];
            s[b + (r >> 2) * sc + (r & 3) * stt] = acc;
          }
        }
      }
    }
    __syncthreads();
  }
  // Z ensemble: gather the {I,Z}^n sub-lattice into the free LDS after the
  // state (2^n values), contract one qubit at a time in place (FP64).
  double *v = reinterpret_cast<double *>(smem_raw + (size_t)E * sizeof(T));
  const int M = 1 << n;
  for (int x = tid; x < M; x += nt) {
    int idx = 0;
    for (int q = 0; q < n; ++q)  // bit q of x -> qubit n-1-q -> position q
      if ((x >> q) & 1) idx |= 3 << (2 * q);
    v[x] = (double)s[idx];
  }
  __syncthreads();
  for (int q = 0; q < n; ++q) {  // butterfly on bit q: (u, w) -> (u + e w, u - e w)
    for (int x = tid; x < M / 2; x += nt) {
      const int lo = x & ((1 << q) - 1);
      const int b = ((x >> q) << (q + 1)) | lo;
      const double u = v[b], w = v[b | (1 << q)];
      v[b] = u + c.err * w;
      v[b | (1 << q)] = u - c.err * w;
    }
    __syncthreads();
  }
  // outcome b: bit of qubit k is bit (n-1-k) of b (qubit 0 most significant);
  // in v, qubit k is bit n-1-k as well, so the order already matches
  for (int x = tid; x < M; x += nt) probs[c.out_off + x] = v[x];
  __syncthreads();
  if (tid == 0) stamp_now(&stamps[2 * blockIdx.x + 1]);
}

// ---------------------------------------------------------------------------
// K8 (HBM tier): batched circuits whose state lives in HBM.
//
// Each circuit is a chain of passes over its own state in one arena:
//   BP_INIT   write |0...0> (2^-n on every index whose digits are I or Z),
//   BP_TILE   one 6-digit tile pass (the tile operations of a fused block,
//             or a single gate / memory-noise group as a one-pass block),
//   BP_PROBS  gather the {I,Z}^n sub-lattice (2^n values), Walsh-Hadamard in
//             LDS (FP64), write the Z-ensemble probabilities.
// A pass is split into items of consecutive tiles.  Round r holds pass r of
// every circuit that has one; the items of a round are independent (distinct
// circuits, or distinct tiles of one pass), and one launch per round works
// through them with a grid-stride loop.  Rounds follow each other on one
// stream, so a pass sees the previous pass's writes through the kernel
// boundary: no workgroup ever waits for another.
// ---------------------------------------------------------------------------

enum { BP_INIT = 0, BP_TILE = 1, BP_PROBS = 2 };

struct BatchPass {
  TileGeom geo;       // BP_TILE: the pass's tile (6 digits, or 7 in FP32)
  int32_t kind;
  int32_t circ;       // HBM-tier circuit index (clock stamps)
  int32_t n;          // register size
  int32_t nops;       // BP_TILE: tile operations
  int32_t io;         // BP_TILE: stage_io bits (first / last stage reads / writes HBM)
  int32_t last_at;    // BP_TILE: header index of the last operation
  int64_t top_off;    // BP_TILE: first tile operation (register-resident: first record word)
  int64_t val_off;    // BP_TILE, register-resident: first value
  int32_t reg_stages; // BP_TILE: stages of the register-resident form, 0 in the LDS form
  RegGeom rgeo;
  int64_t state_off;  // first coefficient of the circuit's state in the arena
  int64_t out_off;    // BP_PROBS: first probability
  double err;         // BP_PROBS: measurement polarisation retention
};

struct BatchItem {
  uint32_t pass;    // index into the pass table
  uint32_t tile0;   // first tile (BP_INIT: first 4096-coefficient chunk)
  uint32_t ntiles;
  uint32_t pad;
};

constexpr int kQueueThreads = 256;
constexpr int kQueueTile = 6;          // tile digits of HBM-tier passes
constexpr int kQueueMaxQubits = 12;    // 2^12 FP64 probabilities fill the LDS buffer
constexpr int kQueueLdsBytes = 32768;  // one FP64 6-digit tile, or 2^12 FP64 values
// FP32 passes whose 6-digit tile would leave runs of 4^2 coefficients take
// 7-digit tiles (64 KB of LDS, 512 threads, as the one-tile kernel), run by
// a second launch per round over those items only.
constexpr int kQueueTile7 = 7;
constexpr int kQueueThreads7 = 512;
template <int M>
struct QueueShape {
  static constexpr int threads = M == kQueueTile7 ? kQueueThreads7 : kQueueThreads;
  static constexpr int lds = M == kQueueTile7 ? 65536 : kQueueLdsBytes;
};

template <typename T, bool SWZ, int M>
__device__ __forceinline__ void queue_tiles(T *s, T *a, const BatchPass &bp, uint32_t t0, uint32_t nt,
                                            const TileOp *__restrict__ tops, const T *__restrict__ prm) {
  constexpr int NT = QueueShape<M>::threads;
  constexpr int E = 1 << (2 * M);
  constexpr int QPT = E / 4 / NT;
  constexpr bool VEC = E / NT >= 32;
  // 7-digit passes hold single-qubit and CX members only (the host refuses
  // others): the 16x16 member's registers would spill at 128 per lane
  constexpr bool GEN2Q = M != kQueueTile7;
  static_assert(E * sizeof(T) <= QueueShape<M>::lds, "the tile fits the round kernel's LDS");
  using Q = Pack<T, 4>;
  const int tid = threadIdx.x;
  const int w = bp.geo.w;
  const int lomask = (1 << (2 * w)) - 1;
  const TileOp *ops = tops + bp.top_off;
  for (uint32_t tile = t0; tile < t0 + nt; ++tile) {
    uint64_t base = 0, r = tile;
    for (int j = 0; j < bp.geo.nr; ++j) {
      base |= (r & 3ull) << (2 * bp.geo.rpos[j]);
      r >>= 2;
    }
    // the first and last stage read and write HBM themselves where
    // stage_io allows (bp.io), as in the one-tile kernel
    if ((bp.io & 3) == 3 && bp.last_at == 0) {
      stage_io<T, M, GEN2Q, NT, SWZ, VEC, 2, false>(a, base, w, lomask, bp.geo, s, ops, 0, prm);
      continue;
    }
    int i0 = 0;
    if (bp.io & 1) {
      stage_io<T, M, GEN2Q, NT, SWZ, VEC, 0, false>(a, base, w, lomask, bp.geo, s, ops, 0, prm);
      i0 = 1 + ops[0].k;
    } else {
      Q buf[QPT];
#pragma unroll
      for (int i = 0; i < QPT; ++i)
        buf[i] = ldp<Q>(a + base + tile_offset<T, M>(4 * (tid + i * NT), w, lomask, bp.geo));
#pragma unroll
      for (int i = 0; i < QPT; ++i) lds_put_quad(s, lds_swz<SWZ>(4 * (tid + i * NT)), buf[i]);
    }
    __syncthreads();
    const int i1 = (bp.io & 2) ? bp.last_at : bp.nops;
    tile_ops<T, M, false, GEN2Q, NT, SWZ>(s, ops + i0, i1 - i0, prm);
    if (bp.io & 2) {
      stage_io<T, M, GEN2Q, NT, SWZ, VEC, 1, false>(a, base, w, lomask, bp.geo, s, ops, bp.last_at, prm);
    } else {
#pragma unroll
      for (int i = 0; i < QPT; ++i) {
        const int c = tid + i * NT;
        stp(a + base + tile_offset<T, M>(4 * c, w, lomask, bp.geo), lds_get_quad(s, lds_swz<SWZ>(4 * c)));
      }
    }
    __syncthreads();  // LDS reads of this tile before the next tile's writes
  }
}

// The M-digit tile items [i0, i0 + gridDim.x) of one round: one workgroup
// per item of one tile, without the round kernel's loops, so the registers
// are those of the one-tile kernel (in the grid-stride round kernel the tile
// code sat at the 106-SGPR limit and the 7-digit form spilled to scratch).
// Waves per SIMD: at least 4 in FP32 and 2 in FP64 (87 and 154 VGPRs with the
// register-resident form: 5 and 3); the 6-digit LDS form is left for registers of 6 qubits and dense two-qubit
// maps, the 7-digit one (two 64 KB workgroups of 8 waves per CU) for tiles
// that do not hold the three lowest positions.
template <typename T, int M>
__global__ __launch_bounds__(QueueShape<M>::threads) __attribute__((amdgpu_waves_per_eu(
    sizeof(T) == 4 ? 4 : 2))) void k_batch_tile(const BatchPass *__restrict__ passes,
                                                                          const BatchItem *__restrict__ items,
                                                                          uint32_t i0,
                                                                          const TileOp *__restrict__ tops,
                                                                          const uint32_t *__restrict__ recs,
                                                                          const T *__restrict__ prm,
                                                                          T *__restrict__ arena) {
  constexpr int LDS = M == kQueueTile7 ? 1 << (2 * M) : std::max(1 << (2 * M), RegShape<T>::lds);
  __shared__ __align__(32) T s[LDS];
  const BatchItem it = items[i0 + blockIdx.x];
  const BatchPass &bp = passes[it.pass];
  T *a = arena + bp.state_off;
  if constexpr (M != kQueueTile7) {
    if (bp.reg_stages) {
      const RegStage *st = reinterpret_cast<const RegStage *>(recs + bp.top_off);
      reg_tile<T, false>(a, s, bp.rgeo, it.tile0, st, bp.reg_stages,
                         reinterpret_cast<const uint32_t *>(st + bp.reg_stages), prm + bp.val_off);
      return;
    }
  }
  if (bp.geo.ident) queue_tiles<T, false, M>(s, a, bp, it.tile0, 1, tops, prm);
  else queue_tiles<T, true, M>(s, a, bp, it.tile0, 1, tops, prm);
}

// The INIT and PROBS items [i0, i1) of one round, grid-stride over
// workgroups.
template <typename T>
__global__ __launch_bounds__(kQueueThreads) void k_batch_round(const BatchPass *__restrict__ passes,
                                                               const BatchItem *__restrict__ items, uint32_t i0,
                                                               uint32_t i1, const TileOp *__restrict__ tops,
                                                               const T *__restrict__ prm, T *__restrict__ arena,
                                                               double *__restrict__ probs,
                                                               uint64_t *__restrict__ stamps) {
  __shared__ __align__(32) unsigned char raw[kQueueLdsBytes];
  const int tid = threadIdx.x;
  for (uint32_t t = i0 + blockIdx.x; t < i1; t += gridDim.x) {
    const BatchItem it = items[t];
    const BatchPass &bp = passes[it.pass];
    T *a = arena + bp.state_off;
    if (bp.kind == BP_INIT) {
      if (tid == 0 && it.tile0 == 0) stamp_now(&stamps[2 * bp.circ]);
      const T amp = (T)ldexp(1.0, -bp.n);
      const uint64_t c0 = (uint64_t)it.tile0 << (2 * kQueueTile);
      const uint64_t c1 = c0 + ((uint64_t)it.ntiles << (2 * kQueueTile));
      for (uint64_t i = c0 + 4 * tid; i < c1; i += 4 * kQueueThreads) {
        Pack<T, 4> q;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const uint64_t x = i + c;
          const uint64_t lo = x & 0x5555555555555555ull, hi = (x >> 1) & 0x5555555555555555ull;
          q.v[c] = (lo ^ hi) ? T(0) : amp;
        }
        stp(a + i, q);
      }
    } else {
      // Z ensemble: bit q of x is the Z/I choice of qubit n-1-q (position q);
      // the butterfly on bit q applies (u, w) -> (u + e w, u - e w), and the
      // outcome index has qubit 0 as its most significant bit, as v does
      double *v = reinterpret_cast<double *>(raw);
      const int n = bp.n, nv = 1 << n;
      for (int x = tid; x < nv; x += kQueueThreads) {
        uint64_t idx = 0;
        for (int q = 0; q < n; ++q)
          if ((x >> q) & 1) idx |= 3ull << (2 * q);
        v[x] = (double)a[idx];
      }
      __syncthreads();
      for (int q = 0; q < n; ++q) {
        for (int x = tid; x < nv / 2; x += kQueueThreads) {
          const int lo = x & ((1 << q) - 1);
          const int b = ((x >> q) << (q + 1)) | lo;
          const double u = v[b], wv = v[b | (1 << q)];
          v[b] = u + bp.err * wv;
          v[b | (1 << q)] = u - bp.err * wv;
        }
        __syncthreads();
      }
      for (int x = tid; x < nv; x += kQueueThreads) probs[bp.out_off + x] = v[x];
      if (tid == 0) stamp_now(&stamps[2 * bp.circ + 1]);
    }
    __syncthreads();  // the LDS buffer is free before the next item
  }
}

}  // namespace

// ===========================================================================
// Host side
// ===========================================================================

struct ProfSlot {
  uint64_t launches = 0;
  double ms = 0.0;
};

struct ProfPending {
  hipEvent_t a, b;
  int fam;
};

// A program image from pinned host memory (see enqueue_image).
__global__ __launch_bounds__(kBlock) void k_image(uint4 *__restrict__ dst, const uint4 *__restrict__ src,
                                                  uint32_t packs) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i < packs) dst[i] = src[i];
}

// A fused pass parsed from its parameter record (see DM_OP_FUSED in dmsim.h).
struct FusedPass {
  int m = 0;
  TileGeom geo;
  std::vector<TileOp> ops;     // param offsets relative to this pass's values
  std::vector<double> vals;    // values in kernel layout (FP64; converted at upload)
  bool reg = false;            // register-resident form (reg_geo, recs) instead of geo and ops
  RegGeom reg_geo;
  bool whole = false;          // reg, on a whole state of up to 6 qubits (k_state_reg, reg_whole)
  RegWhole reg_whole;
  int reg_stages = 0;
  int plain = -1;              // stands for this operation of the program, run by its own kernel
  std::vector<uint32_t> recs;  // its device records: the stages, then the members' kinds
  // device records as 32-bit words
  size_t rec_words() const { return reg ? recs.size() : ops.size() * (sizeof(TileOp) / 4); }
  void put_recs(std::vector<uint32_t> *out) const {
    const size_t at = out->size();
    out->resize(at + rec_words());
    if (rec_words())
      memcpy(out->data() + at, reg ? (const void *)recs.data() : (const void *)ops.data(), rec_words() * 4);
  }
};

struct dm_state {
  int n = 0;
  int dtype = DM_FP64;
  uint64_t N = 0;
  int device = 0;
  int cu_count = 256;
  void *d_a = nullptr;
  hipStream_t stream = nullptr;
  bool owns_stream = true;
  bool batched = false;  // a circuit of a batch that fills the CUs (host-side planning only)
  // scratch
  double *d_red = nullptr;      // reduction partials + results
  size_t red_cap = 0;           // doubles
  void *d_mat = nullptr;        // program image: tile-operation records, block matrices (storage dtype)
  size_t mat_cap = 0;           // bytes
  // the image on its way to d_mat: small ones and the first larger ones in
  // pageable memory, then in pinned memory
  std::vector<char> page_img;
  void *h_img = nullptr;
  size_t img_cap = 0;           // bytes
  int large_images = 0;         // larger ones without the pinned buffer
  hipEvent_t img_ev = nullptr;  // that upload's end
  bool img_busy = false;
  double *d_aux = nullptr;      // gathered vectors / overlap operand
  size_t aux_cap = 0;           // bytes
  // memory noise with a thermal feed as tile passes: the passes, and their
  // records and values on the device, for the last (f, p, g)
  std::vector<FusedPass> mn_passes;
  std::vector<size_t> mn_top_off, mn_val_off;
  void *d_mn = nullptr;
  size_t mn_cap = 0;
  double mn_key[3] = {0.0, 0.0, -1.0};
  // profiling
  bool prof = false;
  int prof_depth = 0;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  ProfSlot slots[kFamilies];
  std::vector<ProfPending> pending;      // recorded, not yet resolved
  std::vector<hipEvent_t> spare_events;  // reusable
  hipEvent_t cur_a = nullptr;
};

namespace {

// One thread per work unit: for streaming passes a full grid measured faster
// on gfx950 than a capped grid-stride launch.  The kernels keep 64-bit
// grid-stride loops; the cap (2^22 workgroups = 2^30 work-items) keeps a
// launch below the 2^32 work-item limit of one grid dimension.
int grid_for(const dm_state *h, uint64_t units) {
  (void)h;
  const uint64_t want = (units + kBlock - 1) / kBlock;
  return (int)std::max<uint64_t>(1, std::min<uint64_t>(want, 1ull << 22));
}

int ensure(void **p, size_t *cap, size_t bytes) {
  if (*cap >= bytes) return DM_OK;
  if (*p) hipFree(*p);
  *p = nullptr;
  *cap = 0;
  HIP_TRY(hipMalloc(p, bytes));
  *cap = bytes;
  return DM_OK;
}

int check_handle(const dm_state *h) {
  if (!h) return fail(DM_ERR_ARG, "null handle");
  if (!h->d_a) return fail(DM_ERR_STATE, "handle has no device state");
  return DM_OK;
}

int check_qubit(const dm_state *h, int q) {
  if (q < 0 || q >= h->n) return fail(DM_ERR_ARG, "qubit %d out of range for %d qubits", q, h->n);
  return DM_OK;
}

hipEvent_t take_event(dm_state *h) {
  if (!h->spare_events.empty()) {
    hipEvent_t e = h->spare_events.back();
    h->spare_events.pop_back();
    return e;
  }
  hipEvent_t e = nullptr;
  if (hipEventCreate(&e) != hipSuccess) return nullptr;
  return e;
}

// Brackets the outermost library operation with a pair of HIP events on the
// handle's stream (nested scopes of composite operations fold into the outer
// one).  Nothing synchronises here; dm_profile_read resolves the pairs.
struct ProfScope {
  dm_state *h;
  int fam;
  bool outer;
  hipEvent_t a = nullptr;
  ProfScope(dm_state *h_, int fam_) : h(h_), fam(fam_), outer(h_->prof_depth++ == 0) {
    if (h->prof && outer) {
      a = take_event(h);
      if (a) hipEventRecord(a, h->stream);
    }
  }
  ~ProfScope() {
    h->prof_depth--;
    if (!h->prof || !outer || !a) return;
    hipEvent_t b = take_event(h);
    if (!b) return;
    hipEventRecord(b, h->stream);
    h->pending.push_back({a, b, fam});
  }
};

int resolve_profile(dm_state *h) {
  if (h->pending.empty()) return DM_OK;
  HIP_TRY(hipStreamSynchronize(h->stream));
  for (auto &pp : h->pending) {
    float ms = 0.f;
    hipEventElapsedTime(&ms, pp.a, pp.b);
    h->slots[pp.fam].launches += 1;
    h->slots[pp.fam].ms += ms;
    h->spare_events.push_back(pp.a);
    h->spare_events.push_back(pp.b);
  }
  h->pending.clear();
  return DM_OK;
}

int last_launch(const char *what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(DM_ERR_HIP, "%s launch failed: %s", what, hipGetErrorString(e));
  return DM_OK;
}

template <typename T>
int launch_1q(dm_state *h, int q, const double *R) {
  const int p = h->n - 1 - q;
  bool use_i = R[0] != 0.0 || R[4] != 0.0 || R[8] != 0.0;
  Rows3<T> m = make_rows3<T>(R);
  T *a = static_cast<T *>(h->d_a);
  constexpr int W = 16 / sizeof(T);
  ProfScope ps(h, 0);
  if (p == 0) {
    const uint64_t groups = h->N / 4;
    if (use_i)
      hipLaunchKernelGGL((k_1q_p0<T, true>), dim3(grid_for(h, groups)), dim3(kBlock), 0, h->stream, a, groups, m);
    else
      hipLaunchKernelGGL((k_1q_p0<T, false>), dim3(grid_for(h, groups)), dim3(kBlock), 0, h->stream, a, groups, m);
  } else {
    const uint64_t S = pow4(p);
    const uint64_t units = h->N / 4 / W;
    int sh = 2 * p - (W == 2 ? 1 : 2);
    const dim3 grid(grid_for(h, units));
    if (p >= 2) {  // runs of >= 16 coefficients: nontemporal
      if (use_i) hipLaunchKernelGGL((k_1q_wide<T, true, true>), grid, dim3(kBlock), 0, h->stream, a, units, sh, S, m);
      else hipLaunchKernelGGL((k_1q_wide<T, false, true>), grid, dim3(kBlock), 0, h->stream, a, units, sh, S, m);
    } else {
      if (use_i) hipLaunchKernelGGL((k_1q_wide<T, true, false>), grid, dim3(kBlock), 0, h->stream, a, units, sh, S, m);
      else hipLaunchKernelGGL((k_1q_wide<T, false, false>), grid, dim3(kBlock), 0, h->stream, a, units, sh, S, m);
    }
  }
  return last_launch("k_1q");
}

template <typename T, bool CTRL_HI, bool SCALED>
int launch_cx_t(dm_state *h, int ph, int pl, const Scale16<T> &sc) {
  T *a = static_cast<T *>(h->d_a);
  constexpr int W = 16 / sizeof(T);
  const uint64_t Sh = pow4(ph), Sl = pow4(pl);
  const int sh_mid = 2 * (ph - pl - 1);
  if (pl == 0) {
    const uint64_t groups = h->N / 16;
    hipLaunchKernelGGL((k_cx_p0<T, CTRL_HI, SCALED>), dim3(grid_for(h, groups)), dim3(kBlock), 0, h->stream, a,
                       groups, sh_mid, Sh, sc);
  } else {
    const uint64_t units = h->N / 16 / W;
    const int sh_lo = 2 * pl - (W == 2 ? 1 : 2);
    if (pl >= 2)  // runs of >= 16 coefficients: nontemporal
      hipLaunchKernelGGL((k_cx_wide<T, CTRL_HI, SCALED, true>), dim3(grid_for(h, units)), dim3(kBlock), 0, h->stream,
                         a, units, sh_lo, sh_mid, Sh, Sl, sc);
    else
      hipLaunchKernelGGL((k_cx_wide<T, CTRL_HI, SCALED, false>), dim3(grid_for(h, units)), dim3(kBlock), 0,
                         h->stream, a, units, sh_lo, sh_mid, Sh, Sl, sc);
  }
  return last_launch("k_cx");
}

template <typename T>
int launch_cx(dm_state *h, int c, int t, const double *scale16) {
  const int pc = h->n - 1 - c, pt = h->n - 1 - t;
  const bool ctrl_hi = pc > pt;
  const int ph = std::max(pc, pt), pl = std::min(pc, pt);
  Scale16<T> sc;
  bool scaled = false;
  for (int i = 0; i < 16; ++i) {
    sc.s[i] = scale16 ? (T)scale16[i] : T(1);
    if (scale16 && scale16[i] != 1.0 && i != 0) scaled = true;
  }
  ProfScope ps(h, 1);
  if (ctrl_hi) {
    return scaled ? launch_cx_t<T, true, true>(h, ph, pl, sc) : launch_cx_t<T, true, false>(h, ph, pl, sc);
  }
  return scaled ? launch_cx_t<T, false, true>(h, ph, pl, sc) : launch_cx_t<T, false, false>(h, ph, pl, sc);
}

template <typename T>
int launch_2q(dm_state *h, int qa, int qb, const double *R) {
  const int pa = h->n - 1 - qa, pb = h->n - 1 - qb;
  const int ph = std::max(pa, pb), pl = std::min(pa, pb);
  // pair index in position order (i_hi, i_lo); R uses (i_qa, i_qb)
  Mat16<T> M;
  uint32_t rowmask = 0;
  for (int r = 0; r < 16; ++r) {
    const int rh = r >> 2, rl = r & 3;
    const int ra = pa > pb ? rh : rl, rb = pa > pb ? rl : rh;
    const int rsrc = 4 * ra + rb;
    bool ident = true;
    for (int c = 0; c < 16; ++c) {
      const int ch = c >> 2, cl = c & 3;
      const int ca = pa > pb ? ch : cl, cb = pa > pb ? cl : ch;
      const double v = R[16 * rsrc + 4 * ca + cb];
      M.m[r][c] = (T)v;
      if (v != (r == c ? 1.0 : 0.0)) ident = false;
    }
    if (!ident) rowmask |= 1u << r;
  }
  const uint64_t groups = h->N / 16;
  const int sh_lo = 2 * pl, sh_mid = 2 * (ph - pl - 1);
  ProfScope ps(h, 2);
  hipLaunchKernelGGL((k_2q_dense<T>), dim3(grid_for(h, groups)), dim3(kBlock), 0, h->stream,
                     static_cast<T *>(h->d_a), groups, sh_lo, sh_mid, pow4(ph), pow4(pl), M, rowmask);
  return last_launch("k_2q_dense");
}

template <typename T, int M>
int launch_tile_maps(dm_state *h, const int *pos, const double (*A)[4][4]) {
  TileMaps<T, M> tm;
  for (int j = 0; j < M; ++j) {
    tm.pos[j] = pos[j];
    for (int r = 0; r < 4; ++r)
      for (int c = 0; c < 4; ++c) tm.A[j][r][c] = (T)A[j][r][c];
  }
  const uint64_t units = h->N >> (2 * M);
  hipLaunchKernelGGL((k_tile_maps<T, M>), dim3(grid_for(h, units)), dim3(kBlock), 0, h->stream,
                     static_cast<T *>(h->d_a), units, tm);
  return last_launch("k_tile_maps");
}

template <typename T>
int launch_memory_noise_tiles(dm_state *h, double f, double p, double g);

template <typename T>
int launch_memory_noise(dm_state *h, double f, double p, double g) {
  const double od = sqrt(g) * f;
  const double dd = (1 - g) * (2 * p - 1);
  ProfScope ps(h, 3);
  if (dd != 0.0 && h->n >= 6) return launch_memory_noise_tiles<T>(h, f, p, g);
  if (dd == 0.0) {
    constexpr int W = 16 / sizeof(T);
    const uint64_t units = h->N / W;
    hipLaunchKernelGGL((k_diag_pow<T>), dim3(grid_for(h, units)), dim3(kBlock), 0, h->stream,
                       static_cast<T *>(h->d_a), units, h->n, od, g);
    return last_launch("k_diag_pow");
  }
  double A[3][4][4];
  for (int j = 0; j < 3; ++j) {
    memset(A[j], 0, sizeof(A[j]));
    A[j][0][0] = 1.0;
    A[j][1][1] = od;
    A[j][2][2] = od;
    A[j][3][3] = g;
    A[j][3][0] = dd;
  }
  // position 0 (the last qubit): contiguous quads, the vectorised 1q kernel
  {
    const double R[12] = {0, od, 0, 0, 0, 0, od, 0, dd, 0, 0, g};
    int rc = launch_1q<T>(h, h->n - 1, R);
    if (rc) return rc;
  }
  int p0 = 1;
  while (p0 < h->n) {
    const int m = std::min(3, h->n - p0);
    int pos[3] = {p0, p0 + 1, p0 + 2};
    int rc = m == 3 ? launch_tile_maps<T, 3>(h, pos, A)
                    : m == 2 ? launch_tile_maps<T, 2>(h, pos, A) : launch_tile_maps<T, 1>(h, pos, A);
    if (rc) return rc;
    p0 += m;
  }
  return DM_OK;
}

template <typename T>
int launch_diag_tab(dm_state *h, const double *tab_by_pos, bool write_only, double scale) {
  Tab4 tab;
  memset(&tab, 0, sizeof(tab));
  memcpy(tab.t, tab_by_pos, sizeof(double) * 4 * h->n);
  ProfScope ps(h, write_only ? 7 : 4);
  if (sizeof(T) == 8 && !write_only && h->n >= 12) {
    const uint64_t units = h->N / 2;
    hipLaunchKernelGGL(k_diag_units, dim3(grid_for(h, units)), dim3(kBlock), 0, h->stream,
                       static_cast<double *>(h->d_a), units, h->n, tab, scale);
    return last_launch("k_diag_units");
  }
  const int low = std::min(h->n, h->n <= 10 ? kTabDigits - 1 : kTabDigits);
  const uint64_t chunks = h->N >> (2 * low);
  // several chunks a workgroup, so that the LDS table is a small part of it
  const dim3 grid((unsigned)std::min<uint64_t>(chunks, 8192));
  const bool nt = h->N * sizeof(T) > (256ull << 20);
  T *a = static_cast<T *>(h->d_a);
#define DIAG_TAB(WO, NT) \
  hipLaunchKernelGGL((k_diag_tab<T, WO, NT>), grid, dim3(kBlock), 0, h->stream, a, chunks, low, h->n, tab, scale)
  if (write_only) {
    if (nt) DIAG_TAB(true, true);
    else DIAG_TAB(true, false);
  } else {
    if (nt) DIAG_TAB(false, true);
    else DIAG_TAB(false, false);
  }
#undef DIAG_TAB
  return last_launch("k_diag_tab");
}

template <typename T, int K, int L>
int launch_block_t(dm_state *h, const int *pos_sorted, const T *dST) {
  BlockGeom geo;
  memset(&geo, 0, sizeof(geo));
  geo.n = h->n;
  bool inblk[kMaxQubits] = {false};
  for (int j = 0; j < K; ++j) {
    geo.pos[j] = pos_sorted[j];
    inblk[pos_sorted[j]] = true;
  }
  int nl = 0;
  for (int p = 0; p < h->n && nl < L; ++p)
    if (!inblk[p]) {
      geo.lpos[nl++] = p;
      inblk[p] = true;
    }
  if (nl < L) return fail(DM_ERR_ARG, "block needs at least %d qubits", K + L);
  geo.nr = 0;
  for (int p = 0; p < h->n; ++p)
    if (!inblk[p]) geo.rpos[geo.nr++] = p;
  geo.tiles = 1ull << (2 * geo.nr);
  const int grid = (int)std::min<uint64_t>(geo.tiles, (uint64_t)h->cu_count * 8);
  hipLaunchKernelGGL((k_block_mfma<T, K, L>), dim3(grid), dim3(kBlock), 0, h->stream, static_cast<T *>(h->d_a),
                     dST, geo);
  return last_launch("k_block_mfma");
}

// Block matrix in kernel order: S is indexed by sum_j i_{qubits[j]} 4^j; the
// kernel's row digit j is the j-th ascending position.  Writes ST[col][row]
// (rows*rows values of T) and the ascending positions.
template <typename T>
void prep_block_matrix(int n, const int *qubits, int k, const double *S, T *st, int *pos_sorted) {
  const int rows = 1 << (2 * k);
  int pos[4], order[4];
  for (int j = 0; j < k; ++j) {
    pos[j] = n - 1 - qubits[j];
    order[j] = j;
  }
  std::sort(order, order + k, [&](int x, int y) { return pos[x] < pos[y]; });
  for (int j = 0; j < k; ++j) pos_sorted[j] = pos[order[j]];
  std::vector<int> remap(rows);
  for (int r = 0; r < rows; ++r) {
    int src = 0;
    for (int j = 0; j < k; ++j) src |= ((r >> (2 * j)) & 3) << (2 * order[j]);
    remap[r] = src;
  }
  for (int r = 0; r < rows; ++r)
    for (int c = 0; c < rows; ++c) st[(size_t)c * rows + r] = (T)S[(size_t)remap[r] * rows + remap[c]];
}

template <typename T>
int launch_block_dev(dm_state *h, int k, const int *pos_sorted, const T *dST) {
  ProfScope ps(h, k == 4 ? 8 : 5);
  if (k == 3) return launch_block_t<T, 3, 3>(h, pos_sorted, dST);
  if (k == 4) return launch_block_t<T, 4, 2>(h, pos_sorted, dST);
  return fail(DM_ERR_ARG, "block size k=%d not supported (3 or 4)", k);
}

template <typename T>
int launch_block(dm_state *h, const int *qubits, int k, const double *S) {
  const int rows = 1 << (2 * k);
  std::vector<T> st((size_t)rows * rows);
  int pos_sorted[4];
  prep_block_matrix<T>(h->n, qubits, k, S, st.data(), pos_sorted);
  int rc = ensure(&h->d_mat, &h->mat_cap, st.size() * sizeof(T));
  if (rc) return rc;
  // synchronous copy: the staging vector is released on return, and the
  // previous block kernel reading d_mat has to finish first
  HIP_TRY(hipStreamSynchronize(h->stream));
  HIP_TRY(hipMemcpy(h->d_mat, st.data(), st.size() * sizeof(T), hipMemcpyHostToDevice));
  return launch_block_dev<T>(h, k, pos_sorted, static_cast<const T *>(h->d_mat));
}

int reserve_red(dm_state *h, size_t doubles) {
  return ensure(reinterpret_cast<void **>(&h->d_red), &h->red_cap, doubles * sizeof(double));
}

template <typename T>
int do_sumsq(dm_state *h, double *out) {
  const uint64_t packs = h->N / (16 / sizeof(T));
  const int grid = std::min(grid_for(h, packs), kSumGrid);
  int rc = reserve_red(h, (size_t)grid + 8);
  if (rc) return rc;
  ProfScope ps(h, 6);
  hipLaunchKernelGGL((k_sumsq<T>), dim3(grid), dim3(kBlock), 0, h->stream, static_cast<const T *>(h->d_a), packs,
                     h->d_red);
  hipLaunchKernelGGL(k_sum_parts, dim3(1), dim3(kBlock), 0, h->stream, h->d_red, grid, h->d_red + grid);
  rc = last_launch("k_sumsq");
  if (rc) return rc;
  HIP_TRY(hipMemcpyAsync(out, h->d_red + grid, sizeof(double), hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  return DM_OK;
}

template <typename T>
int do_dot(dm_state *h, const double *d_b, double *out) {
  const int grid = std::min(grid_for(h, h->N), 4096);
  int rc = reserve_red(h, (size_t)grid + 8);
  if (rc) return rc;
  ProfScope ps(h, 6);
  hipLaunchKernelGGL((k_dot<T, double>), dim3(grid), dim3(kBlock), 0, h->stream, static_cast<const T *>(h->d_a),
                     d_b, h->N, h->d_red);
  hipLaunchKernelGGL(k_sum_parts, dim3(1), dim3(kBlock), 0, h->stream, h->d_red, grid, h->d_red + grid);
  rc = last_launch("k_dot");
  if (rc) return rc;
  HIP_TRY(hipMemcpyAsync(out, h->d_red + grid, sizeof(double), hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  return DM_OK;
}

// Host <-> device copies and dot products over the coefficients [off, off +
// count), the host side in type H (double or float).  Equal types copy
// directly; otherwise each chunk of at most kStageBytes passes through the
// handle's staging buffer and is converted on the device.  Nothing here
// allocates more than one chunk, so a 17-qubit state streams through a few
// hundred megabytes of device memory.
constexpr uint64_t kStageBytes = 256ull << 20;

template <typename T, typename H>
int copy_range(dm_state *h, uint64_t off, uint64_t count, H *host, bool to_host) {
  T *a = static_cast<T *>(h->d_a) + off;
  if (std::is_same<T, H>::value) {
    HIP_TRY(hipMemcpyAsync(to_host ? (void *)host : (void *)a, to_host ? (const void *)a : (const void *)host,
                           count * sizeof(T), to_host ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice, h->stream));
    HIP_TRY(hipStreamSynchronize(h->stream));
    return last_launch("copy_range");
  }
  const uint64_t chunk = kStageBytes / sizeof(H);
  HIP_TRY(hipStreamSynchronize(h->stream));  // the staging buffer may still be read by earlier work
  if (int rc = ensure(reinterpret_cast<void **>(&h->d_aux), &h->aux_cap, std::min(count, chunk) * sizeof(H)))
    return rc;
  H *stage = reinterpret_cast<H *>(h->d_aux);
  for (uint64_t i = 0; i < count; i += chunk) {
    const uint64_t c = std::min(chunk, count - i);
    if (to_host) {
      hipLaunchKernelGGL((k_convert<T, H>), dim3(grid_for(h, c)), dim3(kBlock), 0, h->stream, a + i, stage, c);
      HIP_TRY(hipMemcpyAsync(host + i, stage, c * sizeof(H), hipMemcpyDeviceToHost, h->stream));
    } else {
      HIP_TRY(hipMemcpyAsync(stage, host + i, c * sizeof(H), hipMemcpyHostToDevice, h->stream));
      hipLaunchKernelGGL((k_convert<H, T>), dim3(grid_for(h, c)), dim3(kBlock), 0, h->stream, stage, a + i, c);
    }
    if (int rc = last_launch("k_convert")) return rc;
  }
  HIP_TRY(hipStreamSynchronize(h->stream));
  return DM_OK;
}

template <typename T, typename H>
int dot_range(dm_state *h, uint64_t off, uint64_t count, const H *host, double *out) {
  const T *a = static_cast<const T *>(h->d_a) + off;
  const uint64_t chunk = kStageBytes / sizeof(H);
  HIP_TRY(hipStreamSynchronize(h->stream));
  if (int rc = ensure(reinterpret_cast<void **>(&h->d_aux), &h->aux_cap, std::min(count, chunk) * sizeof(H)))
    return rc;
  H *stage = reinterpret_cast<H *>(h->d_aux);
  const int grid = 2048;
  if (int rc = reserve_red(h, (size_t)grid + 8)) return rc;
  double total = 0.0;
  for (uint64_t i = 0; i < count; i += chunk) {
    const uint64_t c = std::min(chunk, count - i);
    HIP_TRY(hipMemcpyAsync(stage, host + i, c * sizeof(H), hipMemcpyHostToDevice, h->stream));
    const int g = std::min(grid_for(h, c), grid);
    hipLaunchKernelGGL((k_dot<T, H>), dim3(g), dim3(kBlock), 0, h->stream, a + i, stage, c, h->d_red);
    hipLaunchKernelGGL(k_sum_parts, dim3(1), dim3(kBlock), 0, h->stream, h->d_red, g, h->d_red + grid);
    if (int rc = last_launch("k_dot")) return rc;
    double part = 0.0;
    HIP_TRY(hipMemcpyAsync(&part, h->d_red + grid, sizeof(double), hipMemcpyDeviceToHost, h->stream));
    HIP_TRY(hipStreamSynchronize(h->stream));
    total += part;
  }
  *out = total;
  return DM_OK;
}

template <typename T>
int do_probabilities(dm_state *h, const int *qubits, int m, char basis, const double *nvec, double err,
                     double *out) {
  GatherSpec gs;
  memset(&gs, 0, sizeof(gs));
  gs.m = m;
  double w[3] = {err, 0, 0};  // outcomes u + w.x and u - w.x of a digit's components (u, x)
  if (basis == 'N') {
    gs.base_log = 2;
    for (int k = 0; k < 3; ++k) w[k] = nvec[k] * err;
  } else {
    gs.base_log = 1;
    gs.comp = basis == 'X' ? 1 : basis == 'Y' ? 2 : 3;
  }
  for (int t = 0; t < m; ++t) gs.stride[t] = pow4(h->n - 1 - qubits[t]);
  const uint64_t count = 1ull << (gs.base_log * m);
  const uint64_t outn = 1ull << m;
  // aux holds two ping-pong buffers of `count` doubles
  int rc = ensure(reinterpret_cast<void **>(&h->d_aux), &h->aux_cap, 2 * count * sizeof(double));
  if (rc) return rc;
  double *buf0 = h->d_aux, *buf1 = h->d_aux + count;
  ProfScope ps(h, 6);
  double *src = buf0, *dst = buf1;
  if (gs.base_log == 1 || m <= kProbDigits4) {
    const int low = gs.base_log == 1 ? std::min(m, kProbDigits2) : m;
    const int threads = std::max(64, std::min(1024, 1 << std::max(0, gs.base_log * low - 2)));
    hipLaunchKernelGGL((k_probs<T>), dim3(1u << (m - low)), dim3(threads), 0, h->stream,
                       static_cast<const T *>(h->d_a), gs, low, w[0], w[1], w[2], buf0);
    for (int done = low; done < m;) {
      const int d = std::min(4, m - done);
      const uint64_t cols = outn >> d, post = 1ull << done;
      const dim3 grid((unsigned)((cols + kBlock - 1) / kBlock));
      switch (d) {
        case 1: hipLaunchKernelGGL((k_probs_lead<1>), grid, dim3(kBlock), 0, h->stream, buf0, cols, post, err); break;
        case 2: hipLaunchKernelGGL((k_probs_lead<2>), grid, dim3(kBlock), 0, h->stream, buf0, cols, post, err); break;
        case 3: hipLaunchKernelGGL((k_probs_lead<3>), grid, dim3(kBlock), 0, h->stream, buf0, cols, post, err); break;
        default: hipLaunchKernelGGL((k_probs_lead<4>), grid, dim3(kBlock), 0, h->stream, buf0, cols, post, err); break;
      }
      done += d;
    }
  } else {
    hipLaunchKernelGGL((k_gather<T>), dim3(grid_for(h, count)), dim3(kBlock), 0, h->stream,
                       static_cast<const T *>(h->d_a), count, gs, buf0);
    for (int t = 0; t < m; ++t) {
      const uint64_t pre = 1ull << t, post = pow4(m - 1 - t);
      hipLaunchKernelGGL(k_contract, dim3(grid_for(h, pre * post)), dim3(kBlock), 0, h->stream, src, dst, pre, post,
                         w[0], w[1], w[2]);
      std::swap(src, dst);
    }
  }
  rc = last_launch("k_probs");
  if (rc) return rc;
  HIP_TRY(hipMemcpyAsync(out, src, outn * sizeof(double), hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  // marginal over the unmeasured qubits: each contributes a factor 2 (sum of
  // its two outcome rows on the identity component)
  const double fac = ldexp(1.0, h->n - m);
  for (uint64_t i = 0; i < outn; ++i) out[i] *= fac;
  return DM_OK;
}

// Largest staging chunk of the dense output (bytes): the n per-qubit passes
// run in place on one complex buffer of 4^n entries, then the scatter writes
// the row-major matrix through this chunk to the host.
constexpr uint64_t kDenseChunkBytes = 1ull << 31;

template <typename T>
int do_to_dense(dm_state *h, double *out_c128) {
  const uint64_t N = h->N;
  const size_t bytes = N * sizeof(double2);
  const uint64_t chunk = std::min<uint64_t>(N, kDenseChunkBytes / sizeof(double2));
  double2 *buf = nullptr, *stage = nullptr;
  HIP_TRY(hipMallocAsync(reinterpret_cast<void **>(&buf), bytes, h->stream));
  hipError_t e1 = hipMallocAsync(reinterpret_cast<void **>(&stage), chunk * sizeof(double2), h->stream);
  if (e1 != hipSuccess) {
    hipFreeAsync(buf, h->stream);
    hipStreamSynchronize(h->stream);
    return fail(DM_ERR_HIP, "dense output of %d qubits: device buffer of %.1f GB: %s", h->n, bytes / 1e9,
                hipGetErrorString(e1));
  }
  const uint64_t groups = N / 4;
  ProfScope ps(h, 6);
  // qubit order 0..n-1, i.e. position n-1 down to 0 (the per-qubit maps commute)
  for (int q = 0; q < h->n; ++q) {
    const int p = h->n - 1 - q;
    if (q == 0)
      hipLaunchKernelGGL((k_dense_first<T>), dim3(grid_for(h, groups)), dim3(kBlock), 0, h->stream,
                         static_cast<const T *>(h->d_a), buf, groups, p);
    else
      hipLaunchKernelGGL(k_dense_pass, dim3(grid_for(h, groups)), dim3(kBlock), 0, h->stream, buf, groups, p);
  }
  int rc = last_launch("k_dense");
  for (uint64_t o0 = 0; rc == DM_OK && o0 < N; o0 += chunk) {
    const uint64_t cnt = std::min<uint64_t>(chunk, N - o0);
    hipLaunchKernelGGL(k_dense_scatter, dim3(grid_for(h, cnt)), dim3(kBlock), 0, h->stream, buf, stage, h->n, o0,
                       cnt);
    rc = last_launch("k_dense_scatter");
    if (rc) break;
    hipError_t e = hipMemcpyAsync(reinterpret_cast<double2 *>(out_c128) + o0, stage, cnt * sizeof(double2),
                                  hipMemcpyDeviceToHost, h->stream);
    if (e != hipSuccess) rc = fail(DM_ERR_HIP, "dense download failed: %s", hipGetErrorString(e));
  }
  hipFreeAsync(buf, h->stream);
  hipFreeAsync(stage, h->stream);
  HIP_TRY(hipStreamSynchronize(h->stream));
  return rc;
}

int param_count(const dm_state *h, const dm_op &op) {
  switch (op.kind) {
    case DM_OP_1Q: return 12;
    case DM_OP_CX: return 0;
    case DM_OP_CX_SCALED: return 16;
    case DM_OP_2Q: return 256;
    case DM_OP_BLOCK: return 1 << (4 * op.k);
    case DM_OP_MEMORY_NOISE: return 3;
    case DM_OP_DIAG: return 4 * h->n;
    case DM_OP_FUSED: return 0;  // variable length, checked by the parser
    default: return -1;
  }
}

int validate_op(const dm_state *h, const dm_op &op, int i, int64_t nparams) {
  const int need = param_count(h, op);
  if (need < 0) return fail(DM_ERR_ARG, "op %d: unknown kind %d", i, op.kind);
  int nq = 0;
  switch (op.kind) {
    case DM_OP_1Q: nq = 1; break;
    case DM_OP_CX: case DM_OP_CX_SCALED: case DM_OP_2Q: nq = 2; break;
    case DM_OP_BLOCK:
      if (op.k != 3 && op.k != 4) return fail(DM_ERR_ARG, "op %d: block size %d not supported", i, op.k);
      if (h->n < op.k + (op.k == 3 ? 3 : 2)) return fail(DM_ERR_ARG, "op %d: block too large for %d qubits", i, h->n);
      nq = op.k;
      break;
    default: nq = 0;
  }
  for (int j = 0; j < nq; ++j) {
    if (op.qubits[j] < 0 || op.qubits[j] >= h->n)
      return fail(DM_ERR_ARG, "op %d: qubit %d out of range for %d qubits", i, op.qubits[j], h->n);
    for (int m = 0; m < j; ++m)
      if (op.qubits[m] == op.qubits[j]) return fail(DM_ERR_ARG, "op %d: repeated qubit %d", i, op.qubits[j]);
  }
  if (need > 0 && (op.param < 0 || op.param + need > nparams))
    return fail(DM_ERR_ARG, "op %d: parameters [%lld, %lld) outside the %lld given", i, (long long)op.param,
                (long long)(op.param + need), (long long)nparams);
  return DM_OK;
}

// Stages.  An operation applied on its own costs one LDS round trip of the
// whole tile; operations whose digits fit in two tile digits are gathered
// into stages that apply them in registers, one round trip per stage.  An
// operation joins the first stage, at or after the last stage that touches
// its digits, whose digit set stays within two digits (it commutes with
// every later stage, which acts on other digits); otherwise it opens a new
// stage at the end.  Single-qubit operations that end up alone on their
// digit become one product PTM, run as a stage with digit 0 (or digit 3 when
// the digit is 0).  A dense operation is a stage of its own and stays a
// TOP_DENSE record.  Every other record of the result is a TOP_STAGE header
// followed by its members.
void group_stages(FusedPass *fp) {
  struct Stage {
    unsigned mask;
    std::vector<int> mem;
    bool dense;
  };
  std::vector<Stage> st;
  const int nops = (int)fp->ops.size();
  for (int i = 0; i < nops; ++i) {
    const TileOp &op = fp->ops[i];
    const int nd = op.kind == TOP_1Q ? 1 : op.kind == TOP_DENSE ? op.k : 2;
    unsigned D = 0;
    for (int x = 0; x < nd; ++x) D |= 1u << op.d[x];
    int j = -1;
    for (int k = 0; k < (int)st.size(); ++k)
      if (st[k].mask & D) j = k;
    int best = -1;
    if (op.kind != TOP_DENSE)
      for (int k = std::max(j, 0); k < (int)st.size() && best < 0; ++k)
        if (!st[k].dense && __builtin_popcount(st[k].mask | D) <= 2) best = k;
    if (best < 0) {
      st.push_back(Stage{D, {i}, op.kind == TOP_DENSE});
    } else {
      st[best].mask |= D;
      st[best].mem.push_back(i);
    }
  }
  // The one-tile kernel fuses the first and the last stage with the HBM copy
  // when their digits allow it (stage_io_ok).  A stage that shares no digit
  // with any stage before it may move to the front, one that shares none
  // with any stage after it to the back (it commutes with the others).
  auto io_ok = [&](const Stage &x) {
    if (x.dense) return false;
    TileOp hd;
    memset(&hd, 0, sizeof(hd));
    if (__builtin_popcount(x.mask) == 1) {
      const int d = __builtin_ctz(x.mask);
      hd.d[1] = d == 0 ? 3 : d;
    } else {
      hd.d[0] = __builtin_ctz(x.mask);
      hd.d[1] = 31 - __builtin_clz(x.mask);
    }
    return stage_io_ok(hd);
  };
  const int ns = (int)st.size();
  if (ns > 1 && !io_ok(st[0])) {
    unsigned before = 0;
    for (int k = 0; k < ns; ++k) {
      if (!(st[k].mask & before) && io_ok(st[k])) {
        std::rotate(st.begin(), st.begin() + k, st.begin() + k + 1);
        break;
      }
      before |= st[k].mask;
    }
  }
  if (ns > 2 && !io_ok(st[ns - 1])) {
    unsigned after = 0;
    for (int k = ns - 1; k >= 1; --k) {
      if (!(st[k].mask & after) && io_ok(st[k])) {
        std::rotate(st.begin() + k, st.begin() + k + 1, st.end());
        break;
      }
      after |= st[k].mask;
    }
  }
  std::vector<TileOp> out;
  out.reserve(nops + st.size());
  for (const Stage &s : st) {
    if (s.dense) {
      out.push_back(fp->ops[s.mem[0]]);
      continue;
    }
    TileOp hd;
    memset(&hd, 0, sizeof(hd));
    hd.kind = TOP_STAGE;
    if (__builtin_popcount(s.mask) == 1) {
      // P = R_last ... R_first over the components (I, X, Y, Z); each R has
      // the identity's first row and rows X, Y, Z from the operation
      TileOp op = fp->ops[s.mem[0]];
      if (s.mem.size() > 1) {
        double P[4][4] = {{1, 0, 0, 0}, {0, 1, 0, 0}, {0, 0, 1, 0}, {0, 0, 0, 1}};
        for (int i : s.mem) {
          double R[4][4] = {{1, 0, 0, 0}};
          const double *r = &fp->vals[fp->ops[i].param];
          for (int c = 0; c < 3; ++c)
            for (int y = 0; y < 4; ++y) R[c + 1][y] = r[4 * c + y];
          double Q[4][4];
          for (int x = 0; x < 4; ++x)
            for (int y = 0; y < 4; ++y) {
              double acc = 0.0;
              for (int z = 0; z < 4; ++z) acc += R[x][z] * P[z][y];
              Q[x][y] = acc;
            }
          memcpy(P, Q, sizeof(P));
        }
        op.param = (int32_t)fp->vals.size();
        for (int c = 1; c < 4; ++c)
          for (int y = 0; y < 4; ++y) fp->vals.push_back(P[c][y]);
      }
      const int d = op.d[0];
      hd.k = 1;
      hd.d[0] = 0;
      hd.d[1] = d == 0 ? 3 : d;
      out.push_back(hd);
      out.push_back(op);
      continue;
    }
    hd.k = (int32_t)s.mem.size();
    hd.d[0] = __builtin_ctz(s.mask);
    hd.d[1] = 31 - __builtin_clz(s.mask);
    out.push_back(hd);
    for (int i : s.mem) out.push_back(fp->ops[i]);
  }
  for (TileOp &op : out) {
    if (op.kind == TOP_1Q) {
      const double *r = &fp->vals[op.param];
      if (r[0] == 0.0 && r[4] == 0.0 && r[8] == 0.0) op.kind = TOP_1QU;
    } else if (op.kind == TOP_CX && op.k == 0) {
      op.k = 1;
      op.param = (int32_t)fp->vals.size();
      fp->vals.insert(fp->vals.end(), 16, 1.0);
    }
  }
  fp->ops.swap(out);
}

// A 7-digit tile: the given positions (at most 7) completed with the lowest
// others.  False if the positions 0-2 are not all in it.
struct RegTile {
  int tpos[kRegTile], rpos[kMaxQubits], digit[kMaxQubits], nr;
};

bool reg_tile_of(int n, const int *pos, int count, RegTile *t) {
  bool in[kMaxQubits] = {false};
  for (int j = 0; j < count; ++j) in[pos[j]] = true;
  for (int p = 0; p < n && count < kRegTile; ++p)
    if (!in[p]) {
      in[p] = true;
      ++count;
    }
  if (!in[0] || !in[1] || !in[2]) return false;
  int nt = 0;
  t->nr = 0;
  for (int p = 0; p < n; ++p) {
    if (in[p]) {
      t->digit[p] = nt;
      t->tpos[nt++] = p;
    } else {
      t->rpos[t->nr++] = p;
    }
  }
  return true;
}

void set_reg(FusedPass *fp, RegPlan &&rp, const RegTile &t) {
  fp->reg = true;
  fp->reg_geo = reg_geom(rp, t.tpos, t.rpos, t.nr);
  fp->reg_stages = rp.ns;
  fp->recs = std::move(rp.words);
  fp->vals = std::move(rp.vals);
  fp->ops.clear();
}

// The register-resident form (k_tile_reg) of a parsed pass, its tile
// completed to 7 digits with the lowest other positions, where that is the
// faster one; false leaves the pass as it is.  It takes single-qubit and CX
// operations in a tile that holds the positions 0-2 (64 consecutive
// coefficients per access).  The grid is one workgroup of 256 threads per
// tile, so 18 qubits are the most that fit the 2^32 work items of a launch.
// From 12 qubits on it is faster for FP64 passes (16 qubits, one / 8 / 16
// pairs of a single-qubit map and a CX on three digits: 12.0 / 12.6 / 16.4 ms
// against 13.1 / 15.5 / 24.8) and for FP32 passes inside the last-level cache
// (13 qubits, 7-32 maps, CX and scales: 93-171 us against 107-197).  Above it an FP32
// pass of few operations is bound by HBM in either form, and the persistent
// tile-in-LDS kernel walks the state at least as well (16 qubits, 33 passes
// of 3-11 maps, CX and scales: 6.59 ms each in LDS against 6.60; single ones on positions
// 8-12 up to 1.6 ms less); passes of 12 and more take 6.77 ms in
// registers against 7.99.  Below 12 qubits, a launch is a few workgroups per CU
// and its latency counts: the tile-in-LDS kernel's 6-digit tiles fill more
// CUs, and in FP32 the operations in order need too many redistributions (300
// gates on 9 / 11 qubits, matching, learned: 437 / 494 us in LDS against 463 /
// 518).  FP64 passes of many operations per redistribution gain on 7 digits,
// whose LDS form is one workgroup a CU (same circuits, 7 / 9 qubits: 360 / 458
// us against 278 / 420), and on fewer digits from 11 qubits on (greedy, 800
// against 769 us; 9 qubits 523 against 553).
// A batch's passes run side by side; with 256 tiles and more between them
// (h->batched) throughput counts at every register size (7 qubits, FP32, 328
// circuits 797 -> 755 us, 49 circuits 431 -> 468).
bool plan_reg(const dm_state *h, FusedPass *fp) {
  if (h->n < kRegTile || h->n > 18) return false;
  const bool few = h->n < 12 && !h->batched;
  const bool light = h->dtype == DM_FP32 && h->N * 4 > (256ull << 20);
  if (few && (h->dtype == DM_FP32 || fp->ops.size() < 12 || (fp->m < 7 && h->n < 11))) return false;
  for (const TileOp &op : fp->ops)
    if (op.kind != TOP_1Q && op.kind != TOP_CX) return false;
  RegTile t;
  if (!reg_tile_of(h->n, fp->geo.tpos, fp->m, &t)) return false;
  // FP32 keeps the order of operations of the tile-in-LDS form, and with it
  // every rounding: a state does not depend on which form ran.  FP64 may
  // reorder what commutes (differences of 1e-15).
  const bool ordered = h->dtype == DM_FP32;
  std::vector<TileOp> ops;
  std::vector<double> vals;
  if (ordered) {
    FusedPass staged;
    staged.ops = fp->ops;
    staged.vals = fp->vals;
    group_stages(&staged);
    for (const TileOp &op : staged.ops)
      if (op.kind != TOP_STAGE) ops.push_back(op);
    vals = std::move(staged.vals);
  } else {
    ops = fp->ops;
    vals = fp->vals;
  }
  for (TileOp &op : ops)
    for (int x = 0; x < (op.kind == TOP_CX ? 2 : 1); ++x) op.d[x] = t.digit[fp->geo.tpos[op.d[x]]];
  RegPlan rp;
  if (ordered) {
    const std::vector<RegItem<double>> items = reg_items_in_order(ops, vals);
    if (light && items.size() < 12) return false;
    reg_plan(items, kRegTile, true, true, &rp);
  } else {
    reg_plan(reg_items(ops, vals, kRegTile), kRegTile, true, false, &rp);
  }
  if (few && ops.size() < 4 * (size_t)rp.ns) return false;
  set_reg(fp, std::move(rp), t);
  return true;
}

// The passes that replace the run, or none if one kernel per operation is
// expected to be as fast (plain_pass_cost).
template <typename T>
std::vector<FusedPass> fuse_plain_run(const dm_state *h, const PlainRun &run, const dm_op *ops) {
  std::vector<FusedPass> out;
  const int n = h->n;
  if (run.total < 2) return out;
  if (plain_pass_cost(n, 1) >= run.kernels) return out;
  if (n <= 6) {
    RegPlan rp;
    reg_plan(reg_items(run.ops, run.vals, 6), 6, false, false, &rp);
    FusedPass fp;
    fp.reg = fp.whole = true;
    memset(&fp.reg_whole, 0, sizeof(fp.reg_whole));
    fp.reg_whole.n = n;
    fp.reg_whole.ns = rp.ns;
    for (int j = 0; j < 3; ++j) {
      fp.reg_whole.fr[j] = rp.first.r[j];
      fp.reg_whole.fl[j] = rp.first.l[j];
      fp.reg_whole.lr[j] = rp.last.r[j];
      fp.reg_whole.ll[j] = rp.last.l[j];
    }
    fp.reg_stages = rp.ns;
    fp.recs = std::move(rp.words);
    fp.vals = std::move(rp.vals);
    out.push_back(std::move(fp));
    return out;
  }
  const std::vector<std::vector<int>> blocks = plain_blocks(n, run);
  if (plain_pass_cost(n, blocks.size()) >= run.kernels) return out;
  for (const std::vector<int> &b : blocks) {
    FusedPass fp;
    if (b.size() == 1 && run.count[b[0]] == 1 && ops[run.src[b[0]]].kind != DM_OP_MEMORY_NOISE) {
      fp.plain = run.src[b[0]];  // its own kernel
      out.push_back(std::move(fp));
      continue;
    }
    int tpos[kRegTile], count = 0;
    uint32_t used = 7u;
    for (int i : b) used |= (1u << run.ops[i].d[0]) | (run.ops[i].kind == TOP_CX ? 1u << run.ops[i].d[1] : 0u);
    for (int pos = 0; pos < n; ++pos)
      if ((used >> pos) & 1) tpos[count++] = pos;
    RegTile t;
    reg_tile_of(n, tpos, count, &t);
    std::vector<TileOp> tops;
    for (int i : b) {
      TileOp op = run.ops[i];
      op.d[0] = t.digit[op.d[0]];
      if (op.kind == TOP_CX) op.d[1] = t.digit[op.d[1]];
      tops.push_back(op);
    }
    RegPlan rp;
    reg_plan(reg_items(tops, run.vals, kRegTile), kRegTile, true, false, &rp);
    set_reg(&fp, std::move(rp), t);
    out.push_back(std::move(fp));
  }
  return out;
}

// Geometry of a tile: the positions in it, its digits and the others.
void tile_geometry(int n, int m, const bool *intile, FusedPass *fp, int *digit_of_pos) {
  memset(&fp->geo, 0, sizeof(fp->geo));
  fp->m = m;
  fp->geo.m = m;
  int j = 0;
  for (int pos = 0; pos < n; ++pos)
    if (intile[pos]) {
      digit_of_pos[pos] = j;
      fp->geo.tpos[j++] = pos;
    } else {
      fp->geo.rpos[fp->geo.nr++] = pos;
    }
  int w = 0;
  while (w < m && fp->geo.tpos[w] == w) ++w;
  fp->geo.w = w;
  fp->geo.tiles = 1ull << (2 * fp->geo.nr);
}

// The lowest position outside joins the tile.
void widen_tile(int n, FusedPass *fp) {
  bool intile[kMaxQubits] = {false};
  int pos[8], digit_of_pos[kMaxQubits];
  for (int j = 0; j < fp->m; ++j) intile[pos[j] = fp->geo.tpos[j]] = true;
  int low = 0;
  while (intile[low]) ++low;
  intile[low] = true;
  tile_geometry(n, fp->m + 1, intile, fp, digit_of_pos);
  for (TileOp &op : fp->ops)
    for (int x = 0; x < (op.kind == TOP_1Q ? 1 : op.kind == TOP_DENSE ? op.k : 2); ++x)
      op.d[x] = digit_of_pos[pos[op.d[x]]];
}

// With `run`, a record of single-qubit and CX operations joins it instead and
// leaves *fp without operations.
int parse_fused(const dm_state *h, const double *p, int64_t avail, int opi, FusedPass *fp, bool allow_reg = false,
                PlainRun *run = nullptr) {
  int64_t at = 0;
  auto next = [&](double *out) -> bool {
    if (at >= avail) return false;
    *out = p[at++];
    return true;
  };
  auto next_int = [&](int *out) -> bool {
    double v;
    if (!next(&v) || v != (double)(int)v) return false;
    *out = (int)v;
    return true;
  };
  int m = 0, nq = 0;
  if (!next_int(&m) || m < 5 || m > 7) return fail(DM_ERR_ARG, "op %d: fused tile size must be 5, 6 or 7", opi);
  if (h->n < m) return fail(DM_ERR_ARG, "op %d: fused tile of %d qubits on %d qubits", opi, m, h->n);
  if (!next_int(&nq) || nq < 0 || nq > m) return fail(DM_ERR_ARG, "op %d: bad fused qubit count", opi);
  bool intile[kMaxQubits] = {false};
  int count = 0;
  for (int i = 0; i < nq; ++i) {
    int q;
    if (!next_int(&q) || q < 0 || q >= h->n) return fail(DM_ERR_ARG, "op %d: bad fused qubit", opi);
    const int pos = h->n - 1 - q;
    if (!intile[pos]) {
      intile[pos] = true;
      ++count;
    }
  }
  for (int pos = 0; pos < h->n && count < m; ++pos)
    if (!intile[pos]) {
      intile[pos] = true;
      ++count;
    }
  if (!intile[0]) return fail(DM_ERR_ARG, "op %d: fused tile must hold the last qubit's position", opi);
  int digit_of_pos[kMaxQubits];
  tile_geometry(h->n, m, intile, fp, digit_of_pos);
  int nsub = 0;
  if (!next_int(&nsub) || nsub < 0) return fail(DM_ERR_ARG, "op %d: bad fused op count", opi);
  for (int i = 0; i < nsub; ++i) {
    int kind, kq, nv, qs[4];
    if (!next_int(&kind) || !next_int(&kq) || kq < 0 || kq > 4)
      return fail(DM_ERR_ARG, "op %d.%d: bad fused sub-op header", opi, i);
    for (int x = 0; x < 4; ++x)
      if (!next_int(&qs[x])) return fail(DM_ERR_ARG, "op %d.%d: bad fused sub-op qubits", opi, i);
    if (!next_int(&nv) || nv < 0 || at + nv > avail) return fail(DM_ERR_ARG, "op %d.%d: bad value count", opi, i);
    TileOp op;
    memset(&op, 0, sizeof(op));
    op.kind = kind;
    op.k = kq;
    for (int x = 0; x < kq; ++x) {
      if (qs[x] < 0 || qs[x] >= h->n || !intile[h->n - 1 - qs[x]])
        return fail(DM_ERR_ARG, "op %d.%d: qubit %d is not in the fused tile", opi, i, qs[x]);
      op.d[x] = digit_of_pos[h->n - 1 - qs[x]];
      for (int y = 0; y < x; ++y)
        if (qs[y] == qs[x]) return fail(DM_ERR_ARG, "op %d.%d: repeated qubit", opi, i);
    }
    int want = -1;
    if (kind == TOP_1Q && kq == 1) want = 12;
    else if (kind == TOP_CX && kq == 2) want = (nv == 16) ? 16 : 0;
    else if (kind == TOP_2Q && kq == 2) want = 256;
    else if (kind == TOP_DENSE && (kq == 3 || kq == 4) && m == 6) want = 1 << (4 * kq);
    if (want < 0 || nv != want) return fail(DM_ERR_ARG, "op %d.%d: bad fused sub-op (kind %d, %d qubits, %d values)",
                                           opi, i, kind, kq, nv);
    if (kind == TOP_CX) op.k = (nv == 16) ? 1 : 0;
    op.param = (int32_t)fp->vals.size();
    const double *v = p + at;
    if (kind == TOP_2Q) {
      for (int r = 0; r < 16; ++r)
        for (int c = 0; c < 16; ++c)
          if (r == 0 && v[c] != (c == 0 ? 1.0 : 0.0))
            return fail(DM_ERR_ARG, "op %d.%d: two-qubit PTM is not trace preserving", opi, i);
    }
    if (kind == TOP_DENSE) {
      const int rows = 1 << (2 * kq);
      for (int c = 0; c < rows; ++c)
        for (int r = 0; r < rows; ++r) fp->vals.push_back(v[(size_t)r * rows + c]);  // transposed
    } else {
      fp->vals.insert(fp->vals.end(), v, v + nv);
    }
    at += nv;
    fp->ops.push_back(op);
  }
  if (run) {
    for (const TileOp &op : fp->ops)
      if (op.kind != TOP_1Q && op.kind != TOP_CX) return DM_OK;
    for (TileOp op : fp->ops) {
      for (int x = 0; x < (op.kind == TOP_CX ? 2 : 1); ++x) op.d[x] = fp->geo.tpos[op.d[x]];
      push_plain(op, fp->vals.data() + op.param, op.kind == TOP_1Q ? 12 : op.k ? 16 : 0, opi, run);
    }
    fp->ops.clear();
    return DM_OK;
  }
  if (allow_reg && plan_reg(h, fp)) return DM_OK;
  // Tiles of short runs on states above the last-level cache: the workgroups
  // of a small tile are so many, and ask HBM for so short pieces at once, that
  // a larger tile is faster whatever its operations need.  Two passes each:
  // 14 qubits FP64, 5 / 6 digits 5.8 / 2.5 ms; 16 qubits FP32, runs of 4^2 in
  // 6 digits / 4^3 in 7 digits 19-21 / 13 ms.  (The matrix-core operations
  // take 6 digits.)
  if (fp->m == 5 && h->n >= 13) widen_tile(h->n, fp);
  if (h->dtype == DM_FP32 && fp->m == 6 && h->n >= 14 && fp->geo.w < 3) {
    bool dense = false;
    for (const TileOp &op : fp->ops) dense = dense || op.kind == TOP_DENSE;
    if (!dense) widen_tile(h->n, fp);
  }
  m = fp->m;
  // LDS layout.  The 64 banks (4 bytes each) are LDS index bits 0-5, tile
  // digits 0-2.  Stages on digits 3 and up, and stages on digit 0 and a
  // digit >= 3 (one quad access per component), fall on distinct banks in
  // the identity layout.  A pass with any other stage (digit 1 or 2 without
  // digit 0, or digit 0 with digit 1 or 2), whose lanes would hit each bank
  // 4 or 16 times (measured on MI355X: a CX on digits 0 and 1 costs 3.5x a
  // CX on digits 3 and 4), stores the tile swizzled (lds_swz, bank fields
  // [d0, d1^d3, d2^d4]) and gives each stage an order of its free digits
  // whose first ones cover distinct fields: d0, then d1 (else d3), then d2
  // (else d4), then the rest ascending.  Matrix-core passes keep the
  // identity layout.
  group_stages(fp);
  bool dense = false, swz = false;
  for (size_t i = 0; i < fp->ops.size(); ++i) {
    const TileOp &op = fp->ops[i];
    dense = dense || op.kind == TOP_DENSE;
    if (op.kind != TOP_STAGE) continue;
    swz = swz || (op.d[0] == 0 ? op.d[1] < 3 : op.d[0] < 3);
    i += op.k;  // members run in registers
  }
  swz = swz && !dense;
  fp->geo.ident = swz ? 0 : 1;
  // group orders of the stage headers (members run in registers)
  if (swz)
    for (TileOp &op : fp->ops) {
      if (op.kind != TOP_STAGE) continue;
      bool busy[8] = {false};
      busy[op.d[0]] = busy[op.d[1]] = true;
      int ord[8], nf = 0;
      auto take = [&](int d) {
        if (d < m && !busy[d]) {
          busy[d] = true;
          ord[nf++] = d;
          return true;
        }
        return false;
      };
      take(0);
      if (!take(1)) take(3);
      if (!take(2)) take(4);
      for (int d = 0; d < m; ++d) take(d);
      int packed = 0;
      for (int k = 0; k < nf; ++k) packed |= ord[k] << (3 * k);
      op.lanes = packed;
    }
  for (TileOp &op : fp->ops) {
    if (op.kind != TOP_STAGE) continue;
    bool busy[8] = {false};
    busy[0] = busy[op.d[0]] = busy[op.d[1]] = true;
    int ord[8], nf = 0;
    auto take = [&](int d) {
      if (d < m && !busy[d]) {
        busy[d] = true;
        ord[nf++] = d;
        return true;
      }
      return false;
    };
    if (!take(1)) take(3);
    if (!take(2)) take(4);
    for (int d = 1; d < m; ++d) take(d);
    int packed = 0;
    for (int k = 0; k < nf; ++k) packed |= ord[k] << (3 * k);
    op.qlanes = packed;
  }
  return DM_OK;
}

// Workgroups of one tile-program variant that fit on a CU at once (registers,
// LDS, waves), from the runtime's occupancy calculator; cached per variant.
template <typename T, int MM, bool D, bool G, int NTH, bool L>
int tile_resident_per_cu() {
  static int cached = 0;
  if (cached == 0) {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_tile_prog<T, MM, D, G, NTH, L>, NTH, 0) != hipSuccess ||
        nb < 1)
      nb = 1;
    cached = nb;
  }
  return cached;
}


template <typename T, int MM, bool G, int NTH, bool L>
int stream_resident_per_cu() {
  static int cached = 0;
  if (cached == 0) {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_tile_stream<T, MM, G, NTH, L>, NTH, 0) != hipSuccess ||
        nb < 1)
      nb = 1;
    cached = nb;
  }
  return cached;
}

// stage_io bits of a pass (bit 0: its first operation is a stage that can
// read HBM itself, bit 1: its last one can write HBM; stage_io_ok) and the
// header index of its last operation.
int stage_io_flags(const FusedPass &fp, int *last) {
  const int nops = (int)fp.ops.size();
  int last_stage = 0, io = 0;
  for (int i = 0; i < nops; i += fp.ops[i].kind == TOP_STAGE ? 1 + fp.ops[i].k : 1) last_stage = i;
  if (nops > 0 && fp.ops[0].kind == TOP_STAGE && stage_io_ok(fp.ops[0])) io |= 1;
  if (nops > 0 && fp.ops[last_stage].kind == TOP_STAGE && stage_io_ok(fp.ops[last_stage])) io |= 2;
  *last = last_stage;
  return io;
}

template <typename T>
int launch_fused(dm_state *h, const FusedPass &fp, const uint32_t *d_recs, const T *d_vals) {
  ProfScope ps(h, 9);
  if (fp.reg) {
    const RegStage *st = reinterpret_cast<const RegStage *>(d_recs);
    const uint32_t *mem = reinterpret_cast<const uint32_t *>(st + fp.reg_stages);
    if constexpr (sizeof(T) == 8) {
      if (fp.whole) {  // (FP64 programs only)
        hipLaunchKernelGGL((k_state_reg<T>), dim3(1), dim3(64), 0, h->stream, static_cast<T *>(h->d_a), fp.reg_whole,
                           st, mem, d_vals);
        return last_launch("k_state_reg");
      }
    }
    // states above the 256 MB of the last-level cache stream with
    // nontemporal accesses (16 qubits, FP32: 6.0 against 6.4 ms a pass), the
    // others stay in it from pass to pass with plain ones (13 qubits, FP32,
    // 256 MB: 71 against 93 us)
    const bool nt = h->N * sizeof(T) > (256ull << 20);
    if (nt)
      hipLaunchKernelGGL((k_tile_reg<T, true>), dim3(fp.reg_geo.tiles), dim3(kRegThreads), 0, h->stream,
                         static_cast<T *>(h->d_a), fp.reg_geo, st, fp.reg_stages, mem, d_vals);
    else
      hipLaunchKernelGGL((k_tile_reg<T, false>), dim3(fp.reg_geo.tiles), dim3(kRegThreads), 0, h->stream,
                         static_cast<T *>(h->d_a), fp.reg_geo, st, fp.reg_stages, mem, d_vals);
    return last_launch("k_tile_reg");
  }
  const TileOp *d_ops = reinterpret_cast<const TileOp *>(d_recs);
  const int nops = (int)fp.ops.size();
  bool dense = false, gen = false;
  for (const TileOp &op : fp.ops) {
    dense = dense || op.kind == TOP_DENSE;
    gen = gen || op.kind == TOP_2Q;
  }
  T *a = static_cast<T *>(h->d_a);
  // the one-tile kernel fuses the first and the last stage with the HBM
  // copy where their group order suits both HBM and LDS
  int last_stage = 0;
  const int io = stage_io_flags(fp, &last_stage);
  // FP64 7-digit one-tile passes (1024 threads): the HBM-side stages of the
  // 16-byte form (stages on digit 0) ran slower than the staging copy
  // (16 qubits: 17.7 against 15.0 ms), those of the other forms faster
  int io_no_quad = io;
  if ((io & 1) && fp.ops[0].d[0] == 0) io_no_quad &= ~1;
  if ((io & 2) && fp.ops[last_stage].d[0] == 0) io_no_quad &= ~2;
  // one variant per feature set keeps the register footprint of the common
  // 1q + CX passes small; 7-qubit tiles (64 / 128 KB of LDS) use 512 threads
  // Grid shape, from 16-qubit sweeps on MI355X:
  //  - FP32, runs of >= 4^3 coefficients, at least 28 waves of the
  //    one-tile kernel resident per CU (6-digit tiles: 64 VGPRs, 8
  //    workgroups of 256 threads; 7-digit tiles stay below, their 64 KB of
  //    LDS allows 2): k_tile_stream, one tile per workgroup in tile order
  //    (the hardware overlaps the load, LDS and store phases of different
  //    workgroups);
  //  - FP64 6-digit tiles over runs of >= 4^3: k_tile_stream with plain
  //    accesses (110 VGPRs, 4 waves per SIMD; k_tile_prog's 146-162 leave
  //    3); FP64 7-digit tiles over such runs (without 16x16 members): the
  //    same with 1024 threads (113 VGPRs, 4 waves per SIMD in the one
  //    128 KB workgroup per CU, against 2 for the persistent kernel of 512,
  //    which spills at 1024);
  //  - other runs of >= 4^3 with 2 or more resident workgroups per CU:
  //    k_tile_prog with one tile per workgroup, whose loads all issue before
  //    the LDS writes; in FP32, where k_tile_prog's registers leave one
  //    resident workgroup and k_tile_stream's leave two, k_tile_stream;
  //  - otherwise (runs of 4^2, whose neighbouring tiles share HBM lines, or
  //    one resident workgroup per CU): persistent workgroups that prefetch
  //    their next tile, 8 (resp. 4) per resident slot, with consecutive
  //    tiles kept on one XCD.  FP32 6-digit tiles at 13 qubits (256 MB) keep
  //    to four workgroups a CU, where their registers allow five: four
  //    16x16 maps 427 us a pair of passes with four, 453 with five (12
  //    qubits, inside the cache, 4 % the other way).
  // FP32 tiles over runs of >= 4^3 load and store nontemporally (FP64
  // passes measured 1.3x slower with the hint).
  // Measured and rejected for FP32 7-digit tiles over runs of 4^3: the
  // persistent prefetching kernel (one resident workgroup per CU: 1.56x the
  // headline pass time) and one-tile workgroups of 1024 threads (64 VGPRs,
  // 8 waves per SIMD: 1.36x).
#define TILE_LAUNCH_L(MM, D, G, NTH, L)                                                                          \
  do {                                                                                                           \
    const int per_cu = tile_resident_per_cu<T, MM, D, G, NTH, L>();                                             \
    /* one workgroup per tile only where tiles x NTH work items fit a grid */                                 \
    const bool long_runs = fp.geo.w >= 3 && fp.geo.tiles * (uint64_t)NTH <= 0xffffffffull;                    \
    const int s_cu = D ? 0 : stream_resident_per_cu<T, MM, G, NTH, L>();                                        \
    if (long_runs && !D && sizeof(T) == 4 && (s_cu * NTH / 64 >= 28 || (per_cu < 2 && s_cu >= 2))) {            \
      hipLaunchKernelGGL((k_tile_stream<T, MM, G, NTH, L>), dim3((unsigned)fp.geo.tiles), dim3(NTH), 0,          \
                         h->stream, a, fp.geo, d_ops, nops, d_vals, io, last_stage);                             \
      break;                                                                                                     \
    }                                                                                                            \
    if constexpr (sizeof(T) == 8 && (MM == 6 || NTH == 1024) && !D) {                                            \
      if (long_runs) {                                                                                           \
        hipLaunchKernelGGL((k_tile_stream<T, MM, G, NTH, L, false>), dim3((unsigned)fp.geo.tiles), dim3(NTH), 0, \
                           h->stream, a, fp.geo, d_ops, nops, d_vals, MM == 7 ? io_no_quad : io, last_stage);    \
        break;                                                                                                   \
      }                                                                                                          \
    }                                                                                                            \
    const bool full = long_runs && per_cu >= 2;                                                                  \
    /* FP32 6-digit tiles of short runs at 13 qubits: four workgroups a CU, held by 33 KB of LDS each */       \
    const bool four = !full && sizeof(T) == 4 && MM == 6 && h->n >= 13 && per_cu > 4;                            \
    const size_t pad = four ? (33 << 10) - (sizeof(T) << (2 * MM)) : 0;                                          \
    const uint64_t slots = (uint64_t)h->cu_count * (four ? 4 : per_cu) * (per_cu >= 2 ? 8 : 4);                 \
    uint64_t g = full ? fp.geo.tiles : std::min<uint64_t>(fp.geo.tiles, slots);                                 \
    if (!full && g >= 8) g -= g % 8;                                                                             \
    hipLaunchKernelGGL((k_tile_prog<T, MM, D, G, NTH, L>), dim3((unsigned)g), dim3(NTH), pad, h->stream, a,     \
                       fp.geo, d_ops, nops, d_vals, (full ? 0 : 1) | (sizeof(T) == 4 && fp.geo.w >= 3 ? 2 : 0)); \
  } while (0)
#define TILE_LAUNCH(MM, D, G, NTH)               \
  do {                                           \
    if (fp.geo.ident) TILE_LAUNCH_L(MM, D, G, NTH, false); \
    else TILE_LAUNCH_L(MM, D, G, NTH, true);     \
  } while (0)
  if (fp.m == 7 && gen) TILE_LAUNCH(7, false, true, 512);
  else if (fp.m == 7 && sizeof(T) == 8 && fp.geo.w >= 3) TILE_LAUNCH(7, false, false, 1024);
  else if (fp.m == 7) TILE_LAUNCH(7, false, false, 512);
  else if (fp.m == 6 && dense) TILE_LAUNCH_L(6, true, true, 256, false);
  else if (fp.m == 6 && gen) TILE_LAUNCH(6, false, true, 256);
  else if (fp.m == 6) TILE_LAUNCH(6, false, false, 256);
  else if (gen) TILE_LAUNCH(5, false, true, 256);
  else TILE_LAUNCH(5, false, false, 256);
#undef TILE_LAUNCH_L
#undef TILE_LAUNCH
  return last_launch("k_tile_prog");
}

// Memory noise with a thermal feed, d = (1-g)(2p-1) != 0 (the z component
// of every qubit takes d a_I, so the channel is not diagonal), as tile
// passes of the 1-qubit channel R = [X: od x; Y: od y; Z: g z + d a_I] on
// every position: the first pass holds positions 0 .. m-1 (runs of 4^m
// coefficients), each further pass the three lowest positions (runs of 4^3)
// and m - 3 new ones; m = 6 in FP64 (32 KB of LDS), 7 in FP32 (64 KB).
// 1 + ceil((n - m) / (m - 3)) passes, against 1 + ceil((n - 1) / 3) for
// 3-qubit register tiles.  The passes and their device records are kept per
// handle for the last (f, p, g).
template <typename T>
int launch_memory_noise_tiles(dm_state *h, double f, double p, double g) {
  const int n = h->n;
  const int m = sizeof(T) == 4 && n >= 7 ? 7 : 6;
  if (!(h->mn_key[0] == f && h->mn_key[1] == p && h->mn_key[2] == g)) {
    const double od = sqrt(g) * f, dd = (1 - g) * (2 * p - 1);
    const double R[12] = {0, od, 0, 0, 0, 0, od, 0, dd, 0, 0, g};
    std::vector<FusedPass> passes;
    auto add_pass = [&](int lo, int hi) -> int {  // channel on positions [lo, hi); tile filled from position 0
      std::vector<double> rec = {(double)m, (double)(hi - lo)};
      for (int pos = lo; pos < hi; ++pos) rec.push_back(n - 1 - pos);
      rec.push_back(hi - lo);
      for (int pos = lo; pos < hi; ++pos) {
        const double head[7] = {(double)TOP_1Q, 1.0, (double)(n - 1 - pos), 0, 0, 0, 12.0};
        rec.insert(rec.end(), head, head + 7);
        rec.insert(rec.end(), R, R + 12);
      }
      FusedPass fp;
      if (int rc = parse_fused(h, rec.data(), (int64_t)rec.size(), 0, &fp, true)) return rc;
      passes.push_back(std::move(fp));
      return DM_OK;
    };
    if (int rc = add_pass(0, std::min(n, m))) return rc;
    for (int lo = m; lo < n; lo += m - 3)
      if (int rc = add_pass(lo, std::min(n, lo + m - 3))) return rc;
    // device image: [records of every pass | values (T)], values 256-byte aligned
    std::vector<uint32_t> tops;
    std::vector<T> vals;
    std::vector<size_t> top_off, val_off;
    for (const FusedPass &fp : passes) {
      top_off.push_back(tops.size());
      val_off.push_back(vals.size());
      fp.put_recs(&tops);
      for (double v : fp.vals) vals.push_back((T)v);
    }
    const size_t vals_at = (tops.size() * 4 + 255) & ~(size_t)255;
    const size_t bytes = vals_at + vals.size() * sizeof(T);
    HIP_TRY(hipStreamSynchronize(h->stream));  // earlier passes may still read the old image
    if (int rc = ensure(&h->d_mn, &h->mn_cap, bytes)) return rc;
    HIP_TRY(hipMemcpy(h->d_mn, tops.data(), tops.size() * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(static_cast<char *>(h->d_mn) + vals_at, vals.data(), vals.size() * sizeof(T),
                      hipMemcpyHostToDevice));
    for (size_t &o : val_off) o = vals_at + o * sizeof(T);
    h->mn_passes = std::move(passes);
    h->mn_top_off = std::move(top_off);
    h->mn_val_off = std::move(val_off);
    h->mn_key[0] = f;
    h->mn_key[1] = p;
    h->mn_key[2] = g;
  }
  for (size_t i = 0; i < h->mn_passes.size(); ++i) {
    const uint32_t *d_ops = static_cast<const uint32_t *>(h->d_mn) + h->mn_top_off[i];
    const T *d_vals = reinterpret_cast<const T *>(static_cast<const char *>(h->d_mn) + h->mn_val_off[i]);
    if (int rc = launch_fused<T>(h, h->mn_passes[i], d_ops, d_vals)) return rc;
  }
  return DM_OK;
}

// A program split into a host phase (stage: validate, parse the fused
// passes, lay out every tile-operation record and block matrix in one host
// image), an upload phase (the image into device memory) and a launch phase
// that only enqueues kernels on the handle's stream (so it can be captured in
// a graph).  The device image is [tile-operation records | values (T)], the
// values starting at a 256-byte boundary.
struct Prepared {
  std::vector<dm_op> ops;
  const double *params = nullptr;      // the caller's (a Prepared lives for one call)
  std::vector<FusedPass> fused;
  std::vector<int> fused_of;
  std::vector<size_t> offs, top_off;
  std::vector<int> pos;
  std::vector<uint32_t> tops;          // host image: records (32-bit words)
  std::vector<unsigned char> values;   // host image: values, storage type
  size_t vals_at = 0;                  // byte offset of the values in the image
  const void *d_mat = nullptr;         // device values (after upload)
  const void *d_ops = nullptr;         // device records (after upload)
  size_t image_bytes() const { return vals_at + values.size(); }
};

// `in_registers` false: no runs of single operations and no register-resident
// passes, whose image is larger where passes have few operations (one map on
// position 0, FP64: three stage records and a spare member, 504 bytes against
// 168).
template <typename T>
int stage_program(dm_state *h, const dm_op *ops, int nops, const double *params, int64_t nparams, Prepared *pp,
                  bool in_registers = true) {
  pp->params = nparams > 0 ? params : nullptr;
  pp->ops.clear();
  pp->fused.clear();
  pp->fused_of.clear();
  for (int i = 0; i < nops; ++i)
    if (int rc = validate_op(h, ops[i], i, nparams)) return rc;
  size_t pool = 0;
  auto add_fused = [&](const dm_op &op, FusedPass &&fp) {
    pool += fp.vals.size();
    pp->ops.push_back(op);
    pp->fused_of.push_back((int)pp->fused.size());
    pp->fused.push_back(std::move(fp));
  };
  const bool runs = sizeof(T) == 8 && in_registers && h->n <= 18;
  int one_by_one = 0;  // operations before this one have been found not to gain as a run
  int counted = 0;     // operations before this one have been counted
  for (int i = 0; i < nops; ++i) {
    auto fused_args = [&](int j) {
      return ops[j].param < 0 || ops[j].param >= nparams ? fail(DM_ERR_ARG, "op %d: bad parameter offset", j) : DM_OK;
    };
    if (runs && i >= counted) {
      // operations that may form runs; too few of them are not even collected
      double most = 0.0;
      uint32_t used = 0;
      for (counted = i; counted < nops && (plain_op(ops[counted]) || (h->n <= 6 && ops[counted].kind == DM_OP_FUSED));
           ++counted) {
        most += plain_kernels(h->n, ops[counted], params);
        used |= plain_positions(h->n, ops[counted]);
      }
      if (plain_pass_cost(h->n, least_blocks(used)) >= most) one_by_one = counted;
    }
    if (runs && i >= one_by_one) {
      PlainRun run;
      int e = i;
      for (; e < nops; ++e) {
        if (plain_op(ops[e])) {
          add_plain(h->n, ops[e], params, e, &run);
          continue;
        }
        if (h->n > 6 || ops[e].kind != DM_OP_FUSED) break;
        FusedPass fp;
        const int before = run.total;
        if (int rc = fused_args(e)) return rc;
        if (int rc = parse_fused(h, params + ops[e].param, nparams - ops[e].param, e, &fp, false, &run)) return rc;
        if (!fp.ops.empty()) break;
        if (run.total > before) run.kernels += plain_kernels(h->n, ops[e], params);
      }
      settle_all(h->n, &run);
      std::vector<FusedPass> fps = fuse_plain_run<T>(h, run, ops);
      dm_op synth;
      memset(&synth, 0, sizeof(synth));
      synth.kind = DM_OP_FUSED;
      for (FusedPass &fp : fps) {
        if (fp.plain < 0) {
          add_fused(synth, std::move(fp));
          continue;
        }
        pp->ops.push_back(ops[fp.plain]);
        pp->fused_of.push_back(-1);
      }
      if (!fps.empty()) {
        i = e - 1;
        continue;
      }
      one_by_one = e;
    }
    if (ops[i].kind == DM_OP_FUSED) {
      if (int rc = fused_args(i)) return rc;
      FusedPass fp;
      if (int rc = parse_fused(h, params + ops[i].param, nparams - ops[i].param, i, &fp, in_registers)) return rc;
      add_fused(ops[i], std::move(fp));
      continue;
    }
    if (ops[i].kind == DM_OP_BLOCK) pool += (size_t)1 << (4 * ops[i].k);
    pp->ops.push_back(ops[i]);
    pp->fused_of.push_back(-1);
  }
  ops = pp->ops.data();
  nops = (int)pp->ops.size();
  pp->offs.assign(nops, 0);
  pp->pos.assign(4 * (size_t)nops, 0);
  pp->top_off.assign(pp->fused.size(), 0);
  // Tile operations are gathered for every fused pass, also when no pass
  // has parameter values (noiseless CX only): the kernels read them from
  // the records.
  pp->tops.clear();
  pp->values.resize(pool * sizeof(T));
  T *staging = reinterpret_cast<T *>(pp->values.data());
  size_t off = 0;
  for (int i = 0; i < nops; ++i) {
    if (ops[i].kind == DM_OP_BLOCK) {
      prep_block_matrix<T>(h->n, ops[i].qubits, ops[i].k, params + ops[i].param, staging + off,
                           &pp->pos[4 * (size_t)i]);
      pp->offs[i] = off;
      off += (size_t)1 << (4 * ops[i].k);
    } else if (ops[i].kind == DM_OP_FUSED) {
      FusedPass &fp = pp->fused[pp->fused_of[i]];
      pp->offs[i] = off;
      for (double v : fp.vals) staging[off++] = (T)v;
      pp->top_off[pp->fused_of[i]] = pp->tops.size();
      fp.put_recs(&pp->tops);
    }
  }
  pp->vals_at = (pp->tops.size() * 4 + 255) & ~(size_t)255;
  return DM_OK;
}

// Copies the host image to dev (the caller owns dev, at least
// image_bytes() long) after the handle's earlier work, which may still read
// the previous image there, has finished.
int upload_image(dm_state *h, Prepared *pp, void *dev) {
  if (pp->tops.empty() && pp->values.empty()) return DM_OK;
  HIP_TRY(hipStreamSynchronize(h->stream));
  if (!pp->tops.empty())
    HIP_TRY(hipMemcpy(dev, pp->tops.data(), pp->tops.size() * 4, hipMemcpyHostToDevice));
  if (!pp->values.empty())
    HIP_TRY(hipMemcpy(static_cast<char *>(dev) + pp->vals_at, pp->values.data(), pp->values.size(),
                      hipMemcpyHostToDevice));
  pp->d_ops = dev;
  pp->d_mat = static_cast<const char *>(dev) + pp->vals_at;
  return DM_OK;
}

// The same in stream order, from a host copy that
// the handle keeps until the upload has ended: nothing waits for the device
// unless the previous image is still on its way.  Passes walk their records
// one after another, so what counts is where the image lies afterwards: a
// kernel's copy is in the caches, a copy engine's is not (a dependent walk:
// 126-199 ns a 64-byte line against 372; a pass of 300 operations on 6 qubits,
// FP32, 162 us against 197).
// - Up to kSmallImage the runtime copies with a kernel, also from pageable
//   memory (2.7-8 us a call; pinning a buffer costs 17-110 us with its first
//   touch, and as much again when it is freed).
// - Larger ones up to kKernelImage go in pieces of that size while a handle
//   has had only a few of them (8 us a piece), as pinning would cost a program
//   that runs once more than it saves; then k_image copies them from a pinned
//   buffer (64 KB: 13.5 us against the engine's 10.5; 1 MB: 37 against 28).
// - Above, the engine; the first few wait for the stream.
// `pin` false: no buffer is pinned (images above kKernelImage wait).
constexpr size_t kSmallImage = 16 << 10, kKernelImage = 256 << 10;
constexpr int kUnpinnedImages = 3;

int enqueue_image(dm_state *h, Prepared *pp, void *dev, bool pin) {
  const size_t bytes = pp->image_bytes();
  if (bytes == 0) return DM_OK;
  bool pinned = bytes > kSmallImage;
  if (pinned && (!pin || h->large_images < kUnpinnedImages)) {
    h->large_images += pin;
    if (bytes > kKernelImage) return upload_image(h, pp, dev);
    pinned = false;
  }
  if (h->img_busy) {
    HIP_TRY(hipEventSynchronize(h->img_ev));
    h->img_busy = false;
  }
  if (!h->img_ev) HIP_TRY(hipEventCreateWithFlags(&h->img_ev, hipEventDisableTiming));
  if (pinned && h->img_cap < bytes) {
    if (h->h_img) hipHostFree(h->h_img);
    h->h_img = nullptr;
    h->img_cap = 0;
    const size_t cap = std::max<size_t>(2 * bytes, 64 << 10);
    if (hipHostMalloc(&h->h_img, cap, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      h->h_img = nullptr;
      return upload_image(h, pp, dev);
    }
    h->img_cap = cap;
  }
  if (!pinned && h->page_img.size() < bytes) h->page_img.resize(bytes);
  char *img = pinned ? static_cast<char *>(h->h_img) : h->page_img.data();
  if (!pp->tops.empty()) memcpy(img, pp->tops.data(), pp->tops.size() * 4);
  if (!pp->values.empty()) memcpy(img + pp->vals_at, pp->values.data(), pp->values.size());
  if (pinned && bytes <= kKernelImage) {
    const size_t packs = (bytes + 15) / 16;  // (both buffers hold a multiple of 16)
    hipLaunchKernelGGL(k_image, dim3((unsigned)((packs + kBlock - 1) / kBlock)), dim3(kBlock), 0, h->stream,
                       static_cast<uint4 *>(dev), reinterpret_cast<const uint4 *>(img), (uint32_t)packs);
    if (int rc = last_launch("k_image")) return rc;
  } else {
    const size_t piece = pinned ? bytes : kSmallImage;
    for (size_t at = 0; at < bytes; at += piece)
      HIP_TRY(hipMemcpyAsync(static_cast<char *>(dev) + at, img + at, std::min(piece, bytes - at),
                             hipMemcpyHostToDevice, h->stream));
  }
  HIP_TRY(hipEventRecord(h->img_ev, h->stream));
  h->img_busy = true;
  pp->d_ops = dev;
  pp->d_mat = static_cast<const char *>(dev) + pp->vals_at;
  return DM_OK;
}

// Stage, then upload into the handle's own buffer (grown with hipMalloc).
template <typename T>
int prepare_program(dm_state *h, const dm_op *ops, int nops, const double *params, int64_t nparams, Prepared *pp) {
  if (int rc = stage_program<T>(h, ops, nops, params, nparams, pp)) return rc;
  if (pp->tops.empty() && pp->values.empty()) return DM_OK;
  const size_t bytes = (pp->image_bytes() + 15) & ~(size_t)15;  // (k_image copies 16 at a time)
  if (h->mat_cap < bytes) HIP_TRY(hipStreamSynchronize(h->stream));  // the old buffer may be in use
  if (int rc = ensure(&h->d_mat, &h->mat_cap, bytes)) return rc;
  return enqueue_image(h, pp, h->d_mat, true);
}

template <typename T>
int launch_program(dm_state *h, const Prepared &pp) {
  const T *dmat = static_cast<const T *>(pp.d_mat);
  for (size_t i = 0; i < pp.ops.size(); ++i) {
    const dm_op &op = pp.ops[i];
    const double *pv = pp.params ? pp.params + op.param : nullptr;
    int rc = DM_OK;
    switch (op.kind) {
      case DM_OP_1Q: rc = launch_1q<T>(h, op.qubits[0], pv); break;
      case DM_OP_CX: rc = launch_cx<T>(h, op.qubits[0], op.qubits[1], nullptr); break;
      case DM_OP_CX_SCALED: rc = launch_cx<T>(h, op.qubits[0], op.qubits[1], pv); break;
      case DM_OP_2Q: rc = launch_2q<T>(h, op.qubits[0], op.qubits[1], pv); break;
      case DM_OP_BLOCK: rc = launch_block_dev<T>(h, op.k, &pp.pos[4 * i], dmat + pp.offs[i]); break;
      case DM_OP_FUSED: {
        const int f = pp.fused_of[i];
        rc = launch_fused<T>(h, pp.fused[f], static_cast<const uint32_t *>(pp.d_ops) + pp.top_off[f],
                             dmat + pp.offs[i]);
        break;
      }
      case DM_OP_MEMORY_NOISE:
        if (!(pv[0] == 1.0 && pv[2] == 1.0)) rc = launch_memory_noise<T>(h, pv[0], pv[1], pv[2]);
        break;
      case DM_OP_DIAG: {
        double tab[4 * kMaxQubits];
        for (int p = 0; p < h->n; ++p)
          for (int c = 0; c < 4; ++c) tab[4 * p + c] = pv[4 * (h->n - 1 - p) + c];
        rc = launch_diag_tab<T>(h, tab, false, 1.0);
        break;
      }
      default: rc = fail(DM_ERR_ARG, "op %zu: unknown kind", i);
    }
    if (rc) return rc;
  }
  return DM_OK;
}

template <typename T>
int run_program(dm_state *h, const dm_op *ops, int nops, const double *params, int64_t nparams) {
  Prepared pp;
  if (int rc = prepare_program<T>(h, ops, nops, params, nparams, &pp)) return rc;
  return launch_program<T>(h, pp);
}

}  // namespace

// Program image of dm_run_program_noalloc: one fixed array per device, held
// until the process ends.  In host code `scratch` names a host-side stand-in,
// not device memory; its device address comes from hipGetSymbolAddress
// (scratch_address), once per device.
constexpr size_t kNoAllocScratchBytes = 8u << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {nullptr};

// Device address of `scratch` on `device`, looked up on the first call for
// that device with that device current (the caller's device is restored).
int scratch_address(int device, void **out) {
  if (device < 0 || device >= kMaxDevices) return fail(DM_ERR_ARG, "device %d out of range", device);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    int cur = 0;
    HIP_TRY(hipGetDevice(&cur));
    if (cur != device) HIP_TRY(hipSetDevice(device));
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (cur != device) hipSetDevice(cur);
    if (e != hipSuccess || !p)
      return fail(DM_ERR_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", device, hipGetErrorString(e));
    g_scratch_ptr[device] = p;
  }
  *out = g_scratch_ptr[device];
  return DM_OK;
}

// dm_run_program with the program image in the device's fixed scratch array
// instead of the handle's growable buffer: stage on the host, refuse an
// image larger than the array, copy it there behind the handle's earlier work
// on its stream, enqueue the same kernels.
template <typename T>
int run_program_noalloc(dm_state *h, const dm_op *ops, int nops, const double *params, int64_t nparams) {
  Prepared pp;
  if (int rc = stage_program<T>(h, ops, nops, params, nparams, &pp)) return rc;
  // a larger image of the register-resident forms is not what a program may
  // be refused for
  if (pp.image_bytes() > kNoAllocScratchBytes)
    if (int rc = stage_program<T>(h, ops, nops, params, nparams, &pp, false)) return rc;
  if (pp.image_bytes() > kNoAllocScratchBytes)
    return fail(DM_ERR_ARG, "program image of %zu bytes exceeds the %zu-byte scratch of dm_run_program_noalloc",
                pp.image_bytes(), kNoAllocScratchBytes);
  if (!pp.tops.empty() || !pp.values.empty()) {
    void *dev = nullptr;
    if (int rc = scratch_address(h->device, &dev)) return rc;
    if (int rc = enqueue_image(h, &pp, dev, false)) return rc;
  }
  return launch_program<T>(h, pp);
}

}  // namespace

// A batch of independent circuits run together (see dm_batch_create).
struct dm_batch {
  int dtype = DM_FP64;
  int ncirc = 0;
  std::vector<int> nq;
  std::vector<int64_t> prob_off;
  int64_t nprobs = 0;
  std::vector<double> err;
  // circuits held entirely in one workgroup, in the order: in registers up to 6
  // qubits and 7 qubits, in LDS up to 6 qubits (of at most lds6_width) and 7
  std::vector<int> small;
  int nreg6 = 0, nreg7 = 0, nlds6 = 0, nlds7 = 0, lds6_width = 0;
  void *d_rcircs = nullptr, *d_rrecs = nullptr, *d_rvals = nullptr;
  void *d_circs = nullptr, *d_tops = nullptr, *d_vals = nullptr;
  int lds_threads = 256;
  // HBM tier: the states in one arena, the pass table, the items in round
  // order (round r: pass r of every circuit), and the tile operations and
  // values of every pass
  std::vector<int> large;
  void *d_arena = nullptr, *d_passes = nullptr, *d_items = nullptr, *d_qtops = nullptr, *d_qvals = nullptr;
  void *d_recs = nullptr;             // records of the register-resident passes
  std::vector<uint32_t> round_start;  // items of round r: [round_start[r], round_start[r + 1])
  // round r: INIT and PROBS items [round_start[r], split[r][0]), tile items of
  // 6-digit records [split[r][0], split[r][1]), of 7-digit records in the
  // register-resident form [split[r][1], split[r][2]) and in the LDS form
  // [split[r][2], round_start[r + 1]); one tile per tile item
  struct Split {
    uint32_t at[3];
  };
  std::vector<Split> split;
  // groups of circuits (rounds [group_start[g], group_start[g + 1])) in
  // several chains, one stream each
  std::vector<uint32_t> group_start;
  std::vector<int> group_chain;
  int nchains = 0;
  uint32_t nitems = 0;
  int64_t npasses = 0;
  int queue_grid = 0;  // resident workgroups of k_batch_round on the device
  hipStream_t master = nullptr, side = nullptr;
  hipEvent_t fork = nullptr, join = nullptr, ev0 = nullptr, ev1 = nullptr;
  // a round's tile launches run beside its INIT / PROBS launch
  hipStream_t side6 = nullptr, side7 = nullptr;  // also the streams of the second and third chain
  hipEvent_t forkr = nullptr, join6 = nullptr, join7 = nullptr;
  double *d_probs = nullptr;
  uint64_t *d_stamps = nullptr;  // start / end clock per circuit: LDS tier first, then the HBM tier
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  double clock_khz = 1.0e5;
  int64_t launches = 0;  // kernel launches one run enqueues
};

namespace {

// Tile ops of a small circuit: every position is a tile digit (digit j = position j).
int small_circuit_ops(int n, const dm_op *ops, int nops, const double *params, int64_t nparams, int ci,
                      std::vector<TileOp> *tops, std::vector<double> *vals) {
  auto digit = [&](int q) { return n - 1 - q; };
  auto push = [&](int kind, int k, const int *qs, const double *v, int nv) {
    TileOp op;
    memset(&op, 0, sizeof(op));
    op.kind = kind;
    op.k = k;
    for (int x = 0; x < 4; ++x) op.d[x] = qs ? digit(qs[x] < 0 ? 0 : qs[x]) : 0;
    op.param = (int32_t)vals->size();
    vals->insert(vals->end(), v, v + nv);
    tops->push_back(op);
  };
  dm_state probe;
  probe.n = n;
  for (int i = 0; i < nops; ++i) {
    const dm_op &op = ops[i];
    if (int rc = validate_op(&probe, op, i, nparams)) return rc;
    const double *pv = params + op.param;
    int qs[4] = {op.qubits[0], op.qubits[1], op.qubits[2], op.qubits[3]};
    switch (op.kind) {
      case DM_OP_1Q: push(TOP_1Q, 1, qs, pv, 12); break;
      case DM_OP_CX: push(TOP_CX, 0, qs, pv, 0); break;
      case DM_OP_CX_SCALED: push(TOP_CX, 1, qs, pv, 16); break;
      case DM_OP_2Q: {
        for (int c = 0; c < 16; ++c)
          if (pv[c] != (c == 0 ? 1.0 : 0.0))
            return fail(DM_ERR_ARG, "circuit %d op %d: two-qubit PTM is not trace preserving", ci, i);
        push(TOP_2Q, 2, qs, pv, 256);
        break;
      }
      case DM_OP_MEMORY_NOISE: {
        const double f = pv[0], p = pv[1], g = pv[2];
        if (f == 1.0 && g == 1.0) break;
        const double od = sqrt(g) * f, dd = (1 - g) * (2 * p - 1);
        const double R[12] = {0, od, 0, 0, 0, 0, od, 0, dd, 0, 0, g};
        push(TOP_ALLQ, n, nullptr, R, 12);
        break;
      }
      case DM_OP_FUSED: {
        // the whole register is the tile: inline the sub-operations
        // (record: m, nq, q..., nsub, then (kind, kq, q0..q3, nv, v...) each)
        int64_t at = op.param;
        const double *p = params;
        if (at + 2 > nparams) return fail(DM_ERR_ARG, "circuit %d op %d: truncated fused record", ci, i);
        const int nq = (int)p[at + 1];
        at += 2 + nq;
        if (nq < 0 || at + 1 > nparams) return fail(DM_ERR_ARG, "circuit %d op %d: truncated fused record", ci, i);
        const int nsub = (int)p[at++];
        for (int j = 0; j < nsub; ++j) {
          if (at + 7 > nparams) return fail(DM_ERR_ARG, "circuit %d op %d: truncated fused record", ci, i);
          const int kind = (int)p[at], kq = (int)p[at + 1];
          int sq[4] = {(int)p[at + 2], (int)p[at + 3], (int)p[at + 4], (int)p[at + 5]};
          const int nv = (int)p[at + 6];
          at += 7;
          if (nv < 0 || at + nv > nparams) return fail(DM_ERR_ARG, "circuit %d op %d: bad fused values", ci, i);
          if (kq < 0 || kq > 4) return fail(DM_ERR_ARG, "circuit %d op %d: bad fused sub-op size %d", ci, i, kq);
          for (int x = 0; x < kq; ++x)
            if (sq[x] < 0 || sq[x] >= n) return fail(DM_ERR_ARG, "circuit %d op %d: bad qubit", ci, i);
          if (kind == TOP_1Q && kq == 1 && nv == 12) push(TOP_1Q, 1, sq, p + at, 12);
          else if (kind == TOP_CX && kq == 2 && (nv == 0 || nv == 16)) push(TOP_CX, nv ? 1 : 0, sq, p + at, nv);
          else if (kind == TOP_2Q && kq == 2 && nv == 256) push(TOP_2Q, 2, sq, p + at, 256);
          else return fail(DM_ERR_ARG, "circuit %d op %d: sub-op kind %d not supported in LDS circuits", ci, i, kind);
          at += nv;
        }
        break;
      }
      default:
        return fail(DM_ERR_ARG, "circuit %d op %d: kind %d not supported in LDS circuits", ci, i, op.kind);
    }
  }
  return DM_OK;
}

// The register-resident program of a small circuit; *fits false (and no
// error) if it holds operations that form does not take.  FP64: memory noise
// and single-qubit maps between two CX gates on a qubit become one map.
// FP32: every operation on its own and in order, as the LDS kernel rounds; on
// fewer than 7 qubits that many redistributions cost more than the LDS
// kernel's passes (49 circuits of 6 qubits and 40-150 gates, memory noise
// after each: 1109 us against 604; 7 qubits 1454 against 1749).  Planning
// takes the host 24 us an FP64 circuit of 6 qubits and 95 gates with noise
// after each (a run of 49: 645 -> 165 us) and 100 us an FP32 one of 7 qubits
// and 60 gates (200 circuits of 2-7 qubits: 3.5 ms once, a run 2.07 -> 1.05).
template <typename T>
int small_circuit_plan(int n, const dm_op *ops, int nops, const double *params, int64_t nparams, int ci, bool *fits,
                       RegPlan *rp) {
  *fits = false;
  if (sizeof(T) == 4 && n < kRegTile) return DM_OK;
  std::vector<TileOp> tops;
  std::vector<double> vals;
  if (int rc = small_circuit_ops(n, ops, nops, params, nparams, ci, &tops, &vals)) return rc;
  for (const TileOp &op : tops)
    if (op.kind == TOP_2Q) return DM_OK;
  const int m = n == 7 ? 7 : 6;
  if (sizeof(T) == 8) {
    PlainRun run;
    for (const TileOp &op : tops) {
      const double *v = vals.data() + op.param;
      if (op.kind == TOP_ALLQ) run.levels.push_back({v[1], v[11], v[8], 0});
      else push_plain(op, v, op.kind == TOP_1Q ? 12 : op.k ? 16 : 0, 0, &run);
    }
    settle_all(n, &run);
    reg_plan(reg_items(run.ops, run.vals, m), m, false, false, rp);
  } else {
    std::vector<TileOp> flat;
    flat.reserve(tops.size() * (n + 1) / 2);
    for (const TileOp &op : tops) {
      if (op.kind != TOP_ALLQ) {
        flat.push_back(op);
        continue;
      }
      TileOp one = op;
      one.kind = TOP_1Q;
      one.k = 1;
      for (one.d[0] = 0; one.d[0] < n; ++one.d[0]) flat.push_back(one);
    }
    reg_plan(reg_items_in_order(flat, vals), m, false, true, rp);
  }
  *fits = true;
  return DM_OK;
}

size_t lds_bytes(int n, int dtype) {
  return ((size_t)1 << (2 * n)) * (dtype == DM_FP64 ? 8 : 4) + ((size_t)1 << n) * 8;
}

// The tile pass of one plain operation (a 1q / CX / 2q PTM): a one-operation
// fused record over its qubits, parsed like any fused pass.
int plain_op_pass(const dm_state *h, int kind, int kq, const int *qs, const double *v, int nv, int opi,
                  FusedPass *fp) {
  std::vector<double> rec = {(double)kQueueTile, (double)kq};
  for (int x = 0; x < kq; ++x) rec.push_back(qs[x]);
  rec.push_back(1.0);
  rec.push_back(kind);
  rec.push_back(kq);
  for (int x = 0; x < 4; ++x) rec.push_back(x < kq ? qs[x] : 0);
  rec.push_back(nv);
  rec.insert(rec.end(), v, v + nv);
  return parse_fused(h, rec.data(), (int64_t)rec.size(), opi, fp, true);
}

// The 6-digit tile passes of one program operation of an HBM-tier circuit.
// Memory noise becomes one 1-qubit channel per qubit, positions 0-5 in the
// first pass and 5 more per further pass.
int queue_op_passes(const dm_state *h, const dm_op &op, const double *params, int64_t nparams, int ci, int i,
                    std::vector<FusedPass> *out) {
  if (int rc = validate_op(h, op, i, nparams)) return rc;
  const double *pv = params + op.param;
  FusedPass fp;
  int rc = DM_OK;
  switch (op.kind) {
    case DM_OP_1Q: rc = plain_op_pass(h, TOP_1Q, 1, op.qubits, pv, 12, i, &fp); break;
    case DM_OP_CX: rc = plain_op_pass(h, TOP_CX, 2, op.qubits, pv, 0, i, &fp); break;
    case DM_OP_CX_SCALED: rc = plain_op_pass(h, TOP_CX, 2, op.qubits, pv, 16, i, &fp); break;
    case DM_OP_2Q: rc = plain_op_pass(h, TOP_2Q, 2, op.qubits, pv, 256, i, &fp); break;
    case DM_OP_FUSED: {
      if (op.param < 0 || op.param >= nparams) return fail(DM_ERR_ARG, "circuit %d op %d: bad parameter offset", ci, i);
      rc = parse_fused(h, params + op.param, nparams - op.param, i, &fp, true);
      if (rc) return rc;
      if (fp.m != kQueueTile && !(fp.m == kQueueTile7 && h->dtype == DM_FP32))
        return fail(DM_ERR_ARG, "circuit %d op %d: batched circuits take %d-digit fused tiles (or %d in FP32), not %d",
                    ci, i, kQueueTile, kQueueTile7, fp.m);
      for (const TileOp &t : fp.ops) {
        if (t.kind == TOP_DENSE) return fail(DM_ERR_ARG, "circuit %d op %d: dense tile operations are not batched", ci, i);
        if (t.kind == TOP_2Q && fp.m == kQueueTile7)
          return fail(DM_ERR_ARG, "circuit %d op %d: batched %d-digit passes take single-qubit and CX operations only",
                      ci, i, kQueueTile7);
      }
      break;
    }
    case DM_OP_MEMORY_NOISE: {
      const double f = pv[0], p = pv[1], g = pv[2];
      if (f == 1.0 && g == 1.0) return DM_OK;
      const double od = sqrt(g) * f, dd = (1 - g) * (2 * p - 1);
      const double R[12] = {0, od, 0, 0, 0, 0, od, 0, dd, 0, 0, g};
      for (int lo = 0; lo < h->n; lo = (lo == 0 ? kQueueTile : lo + kQueueTile - 1)) {
        const int hi = std::min(h->n, lo == 0 ? kQueueTile : lo + kQueueTile - 1);
        std::vector<double> rec = {(double)kQueueTile, (double)(hi - lo)};
        for (int pos = lo; pos < hi; ++pos) rec.push_back(h->n - 1 - pos);
        rec.push_back(hi - lo);
        for (int pos = lo; pos < hi; ++pos) {
          const double head[7] = {(double)TOP_1Q, 1.0, (double)(h->n - 1 - pos), 0, 0, 0, 12.0};
          rec.insert(rec.end(), head, head + 7);
          rec.insert(rec.end(), R, R + 12);
        }
        FusedPass mp;
        if (int r2 = parse_fused(h, rec.data(), (int64_t)rec.size(), i, &mp, true)) return r2;
        out->push_back(std::move(mp));
      }
      return DM_OK;
    }
    default:
      return fail(DM_ERR_ARG, "circuit %d op %d: kind %d is not batched", ci, i, op.kind);
  }
  if (rc) return rc;
  out->push_back(std::move(fp));
  return DM_OK;
}

template <typename T>
int enqueue_batch(dm_batch *b) {
  HIP_TRY(hipEventRecord(b->fork, b->master));
  HIP_TRY(hipStreamWaitEvent(b->side, b->fork, 0));
  // whole circuits on the side stream; without an HBM tier those of 7 qubits
  // beside them on the master stream, as either kind rarely fills the chip (a
  // stream of their own costs a batch 0.8 ms when it is destroyed)
  constexpr bool SEQ = sizeof(T) == 4;
  hipStream_t side7 = b->nitems ? b->side : b->master;
  if (b->nreg7) {
    hipLaunchKernelGGL((k_circuit_reg<T, 7, SEQ>), dim3(b->nreg7), dim3(RegCircShape<7>::threads), 0, side7,
                       static_cast<const RegCirc *>(b->d_rcircs) + b->nreg6, static_cast<const uint32_t *>(b->d_rrecs),
                       static_cast<const T *>(b->d_rvals), b->d_probs, b->d_stamps + 2 * (size_t)b->nreg6);
    if (int rc = last_launch("k_circuit_reg")) return rc;
  }
  if constexpr (!SEQ) {
    if (b->nreg6) {
      hipLaunchKernelGGL((k_circuit_reg<T, 6, SEQ>), dim3(b->nreg6), dim3(RegCircShape<6>::threads), 0, b->side,
                         static_cast<const RegCirc *>(b->d_rcircs), static_cast<const uint32_t *>(b->d_rrecs),
                         static_cast<const T *>(b->d_rvals), b->d_probs, b->d_stamps);
      if (int rc = last_launch("k_circuit_reg")) return rc;
    }
  }
  const int reg = b->nreg6 + b->nreg7;
  auto in_lds = [&](int first, int count, int width, hipStream_t st) -> int {
    if (!count) return DM_OK;
    hipLaunchKernelGGL((k_circuit_lds<T>), dim3(count), dim3(b->lds_threads), lds_bytes(width, b->dtype), st,
                       static_cast<const BatchCirc *>(b->d_circs) + first, static_cast<const TileOp *>(b->d_tops),
                       static_cast<const T *>(b->d_vals), b->d_probs, b->d_stamps + 2 * (size_t)(reg + first));
    return last_launch("k_circuit_lds");
  };
  if (int rc = in_lds(0, b->nlds6, b->lds6_width, b->side)) return rc;
  if (int rc = in_lds(b->nlds6, b->nlds7, 7, side7)) return rc;
  // HBM tier.  One group: its rounds in order on the master stream; a round's
  // INIT / PROBS items (master), tile items of 6-digit records (side6) and of
  // 7-digit ones (side7: the register-resident form, then the LDS form) belong
  // to distinct circuits, and where a round has more than one of these they
  // run side by side, forked from and joined back into master.  Several
  // groups: each one's launches in order on its chain's stream (master, side6,
  // side7), forked from master once and joined back at the end.
  const BatchPass *passes = static_cast<const BatchPass *>(b->d_passes);
  const BatchItem *items = static_cast<const BatchItem *>(b->d_items);
  const TileOp *tops = static_cast<const TileOp *>(b->d_qtops);
  const uint32_t *recs = static_cast<const uint32_t *>(b->d_recs);
  const T *vals = static_cast<const T *>(b->d_qvals);
  T *arena = static_cast<T *>(b->d_arena);
  auto ends = [&](uint32_t i0, uint32_t i1, hipStream_t st) -> int {
    if (i1 <= i0) return DM_OK;
    const int grid = (int)std::min<uint32_t>(i1 - i0, (uint32_t)b->queue_grid);
    hipLaunchKernelGGL((k_batch_round<T>), dim3(grid), dim3(kQueueThreads), 0, st, passes, items, i0, i1, tops, vals,
                       arena, b->d_probs, b->d_stamps + 2 * b->small.size());
    return last_launch("k_batch_round");
  };
  auto tiles = [&](uint32_t i0, uint32_t i1, hipStream_t st) -> int {
    if (i1 <= i0) return DM_OK;
    hipLaunchKernelGGL((k_batch_tile<T, kQueueTile>), dim3(i1 - i0), dim3(kQueueThreads), 0, st, passes, items, i0,
                       tops, recs, vals, arena);
    return last_launch("k_batch_tile");
  };
  auto tiles7 = [&](uint32_t i0, uint32_t i1, hipStream_t st) -> int {
    if constexpr (sizeof(T) == 4) {
      if (i1 <= i0) return DM_OK;
      hipLaunchKernelGGL((k_batch_tile<float, kQueueTile7>), dim3(i1 - i0), dim3(kQueueThreads7), 0, st, passes, items,
                         i0, tops, recs, vals, arena);
      return last_launch("k_batch_tile");
    }
    return DM_OK;
  };
  if (b->nchains > 1) {
    hipStream_t streams[3] = {b->master, b->side6, b->side7};
    HIP_TRY(hipEventRecord(b->forkr, b->master));
    for (int c = 1; c < b->nchains; ++c) HIP_TRY(hipStreamWaitEvent(streams[c], b->forkr, 0));
    for (size_t g = 0; g + 1 < b->group_start.size(); ++g) {
      hipStream_t st = streams[b->group_chain[g]];
      for (uint32_t r = b->group_start[g]; r < b->group_start[g + 1]; ++r) {
        const uint32_t *at = b->split[r].at;
        if (int rc = ends(b->round_start[r], at[0], st)) return rc;
        if (int rc = tiles(at[0], at[1], st)) return rc;
        if (int rc = tiles(at[1], at[2], st)) return rc;
        if (int rc = tiles7(at[2], b->round_start[r + 1], st)) return rc;
      }
    }
    hipEvent_t joins[3] = {nullptr, b->join6, b->join7};
    for (int c = 1; c < b->nchains; ++c) {
      HIP_TRY(hipEventRecord(joins[c], streams[c]));
      HIP_TRY(hipStreamWaitEvent(b->master, joins[c], 0));
    }
  } else {
    for (size_t r = 0; r + 1 < b->round_start.size(); ++r) {
      const uint32_t i0 = b->round_start[r], i6 = b->split[r].at[0], i7 = b->split[r].at[1], i8 = b->split[r].at[2],
                     i1 = b->round_start[r + 1];
      const bool t6 = i7 > i6, t7 = i1 > i7;
      // one kind of items stays on master; otherwise fork and join
      const bool fork = (i6 > i0) + t6 + t7 > 1;
      hipStream_t s6 = fork ? b->side6 : b->master, s7 = fork ? b->side7 : b->master;
      if (fork) {
        HIP_TRY(hipEventRecord(b->forkr, b->master));
        if (t6) HIP_TRY(hipStreamWaitEvent(b->side6, b->forkr, 0));
        if (t7) HIP_TRY(hipStreamWaitEvent(b->side7, b->forkr, 0));
      }
      if (int rc = ends(i0, i6, b->master)) return rc;
      if (int rc = tiles(i6, i7, s6)) return rc;
      if (int rc = tiles(i7, i8, s7)) return rc;
      if (int rc = tiles7(i8, i1, s7)) return rc;
      if (fork && t6) {
        HIP_TRY(hipEventRecord(b->join6, b->side6));
        HIP_TRY(hipStreamWaitEvent(b->master, b->join6, 0));
      }
      if (fork && t7) {
        HIP_TRY(hipEventRecord(b->join7, b->side7));
        HIP_TRY(hipStreamWaitEvent(b->master, b->join7, 0));
      }
    }
  }
  HIP_TRY(hipEventRecord(b->join, b->side));
  HIP_TRY(hipStreamWaitEvent(b->master, b->join, 0));
  return DM_OK;
}

}  // namespace

namespace dmsim_internal {
int set_error(int code, const char *msg) {
  snprintf(g_err, sizeof(g_err), "%s", msg);
  return code;
}
}  // namespace dmsim_internal

// ===========================================================================
// C ABI
// ===========================================================================

extern "C" int dm_batch_destroy(dm_batch *b);

template <typename T>
static int batch_create_t(dm_batch *b, const int64_t *op_start, const dm_op *ops, const double *params,
                          int64_t nparams, int lds_max_qubits, int items_per_pass) {
  int cu = 256, dev = 0;
  {
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
      cu = prop.multiProcessorCount;
    int khz = 0;
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) == hipSuccess && khz > 0)
      b->clock_khz = khz;
  }
  // LDS circuits grouped by width (probabilities stay in circuit order)
  std::vector<BatchCirc> circs;
  std::vector<TileOp> tops;
  std::vector<double> vals;
  // register-resident: circuits of single-qubit maps, CX and memory noise,
  // the longest first
  std::vector<RegCirc> rcircs;
  std::vector<uint32_t> rrecs;
  std::vector<T> rvals;
  std::vector<char> in_reg(b->ncirc, 0);
  {
    struct Planned {
      int c;
      RegPlan rp;
    };
    std::vector<Planned> planned[2];
    for (int c = 0; c < b->ncirc; ++c) {
      if (b->nq[c] > lds_max_qubits) continue;
      Planned p;
      p.c = c;
      bool fits = false;
      if (int rc = small_circuit_plan<T>(b->nq[c], ops + op_start[c], (int)(op_start[c + 1] - op_start[c]), params,
                                         nparams, c, &fits, &p.rp))
        return rc;
      if (!fits) continue;
      in_reg[c] = 1;
      planned[b->nq[c] == 7].push_back(std::move(p));
    }
    for (auto &list : planned)
      std::stable_sort(list.begin(), list.end(),
                       [](const Planned &x, const Planned &y) { return x.rp.vals.size() > y.rp.vals.size(); });
    b->nreg6 = (int)planned[0].size();
    b->nreg7 = (int)planned[1].size();
    for (auto &list : planned)
      for (Planned &p : list) {
        RegCirc rc;
        memset(&rc, 0, sizeof(rc));
        rc.n = b->nq[p.c];
        rc.ns = p.rp.ns;
        rc.st_off = (int64_t)rrecs.size();
        rc.val_off = (int64_t)rvals.size();
        rc.out_off = b->prob_off[p.c];
        rc.err = b->err[p.c];
        for (int j = 0; j < 3; ++j) {
          rc.fr[j] = p.rp.first.r[j];
          rc.fl[j] = p.rp.first.l[j];
          rc.lr[j] = p.rp.last.r[j];
          rc.ll[j] = p.rp.last.l[j];
        }
        rc.fw = p.rp.first.w;
        rc.lw = p.rp.last.w;
        rrecs.insert(rrecs.end(), p.rp.words.begin(), p.rp.words.end());
        rvals.insert(rvals.end(), p.rp.vals.begin(), p.rp.vals.end());
        rcircs.push_back(rc);
        b->small.push_back(p.c);
      }
    b->launches += (b->nreg6 > 0) + (b->nreg7 > 0);
  }
  // in LDS: 7 qubits last, the others widest first in one launch (with one a
  // width, on two streams in turn, a graph of small circuits took 280 us more
  // to set up)
  for (int w : {6, 5, 4, 3, 2, 1, 7}) {
    if (w > lds_max_qubits) continue;
    for (int c = 0; c < b->ncirc; ++c) {
      if (b->nq[c] != w || in_reg[c]) continue;
      ++(w == 7 ? b->nlds7 : b->nlds6);
      if (w < 7) b->lds6_width = std::max(b->lds6_width, w);
      BatchCirc bc;
      bc.n = w;
      bc.op_off = (int64_t)tops.size();
      if (int rc = small_circuit_ops(w, ops + op_start[c], (int)(op_start[c + 1] - op_start[c]), params, nparams, c,
                                     &tops, &vals))
        return rc;
      bc.nops = (int32_t)(tops.size() - bc.op_off);
      bc.out_off = b->prob_off[c];
      bc.err = b->err[c];
      circs.push_back(bc);
      b->small.push_back(c);
    }
  }
  b->launches += (b->nlds6 > 0) + (b->nlds7 > 0);

  // HBM tier: every circuit as INIT, its tile passes, PROBS; states in one arena
  std::vector<BatchPass> passes;
  std::vector<TileOp> qtops;
  std::vector<uint32_t> recs;           // register-resident passes
  std::vector<T> qvals;
  std::vector<std::vector<int>> chain;  // pass-table indices of each HBM circuit, in order
  std::vector<double> work;             // per HBM circuit: bytes moved (ticket order)
  uint64_t arena = 0, tiles = 0;
  for (int c = 0; c < b->ncirc; ++c)
    if (b->nq[c] > lds_max_qubits && b->nq[c] >= kRegTile) tiles += pow4(b->nq[c] - kRegTile);
  for (int c = 0; c < b->ncirc; ++c) {
    if (b->nq[c] <= lds_max_qubits) continue;
    const int j = (int)b->large.size();
    b->large.push_back(c);
    dm_state probe;
    probe.n = b->nq[c];
    probe.dtype = b->dtype;
    probe.N = pow4(probe.n);
    probe.batched = tiles >= (uint64_t)cu;
    BatchPass bp;
    memset(&bp, 0, sizeof(bp));
    bp.circ = j;
    bp.n = probe.n;
    bp.state_off = (int64_t)arena;
    arena += (probe.N + 63) & ~63ull;  // 256-byte aligned states
    std::vector<int> ids;
    bp.kind = BP_INIT;
    ids.push_back((int)passes.size());
    passes.push_back(bp);
    for (int64_t i = op_start[c]; i < op_start[c + 1]; ++i) {
      std::vector<FusedPass> fps;
      if (int rc = queue_op_passes(&probe, ops[i], params, nparams, c, (int)(i - op_start[c]), &fps)) return rc;
      for (FusedPass &fp : fps) {
        BatchPass tp = bp;
        tp.kind = BP_TILE;
        tp.geo = fp.geo;  // (geo.m: the record's tile digits)
        const size_t vbase = qvals.size();
        if (fp.reg) {
          tp.reg_stages = fp.reg_stages;
          tp.rgeo = fp.reg_geo;
          tp.top_off = (int64_t)recs.size();
          tp.val_off = (int64_t)vbase;
          fp.put_recs(&recs);
        } else {
          tp.nops = (int32_t)fp.ops.size();
          int last_at = 0;
          tp.io = stage_io_flags(fp, &last_at);
          tp.last_at = last_at;
          tp.top_off = (int64_t)qtops.size();
        }
        for (TileOp t : fp.ops) {
          t.param += (int32_t)vbase;
          qtops.push_back(t);
        }
        qvals.insert(qvals.end(), fp.vals.begin(), fp.vals.end());
        ids.push_back((int)passes.size());
        passes.push_back(tp);
      }
    }
    bp.kind = BP_PROBS;
    bp.out_off = b->prob_off[c];
    bp.err = b->err[c];
    ids.push_back((int)passes.size());
    passes.push_back(bp);
    work.push_back((double)ids.size() * (double)probe.N);
    chain.push_back(std::move(ids));
  }
  if (qvals.size() > (size_t)INT32_MAX) return fail(DM_ERR_ARG, "batch: too many tile-operation values");
  b->npasses = (int64_t)passes.size();

  // Items in round order: round r of a group holds pass r of every circuit
  // of the group that has one.  Batches of up to 300 MiB of states are one
  // group, the 256 MB last-level cache holds most of it (152 FP32 circuits of
  // 8-10 qubits, 273 MB: 2.4 ms, in groups 3.4; 20 of 11 qubits, 335 MB, one
  // group 2.49, groups 2.32).  Larger ones form groups, most
  // work first, that run one after another in two or three chains (a stream
  // each): all but a state's first pass then read what the pass before left
  // in the cache, and the chains fill each other's launch gaps and tails.
  // 512 circuits of 6-12 qubits, FP32: one group 70.6 ms, groups of 200 MB in
  // one chain 68.4, of 70 MB in three 58.7 (in two 64.8, of 140 MB in three
  // 62.3); 256 circuits, FP64 (134 MB at 12 qubits): one group 57.5 ms, one
  // chain 57.2, two 47.9, three 49.9.
  std::vector<BatchItem> items;
  {
    std::vector<int> order(chain.size());
    for (size_t j = 0; j < order.size(); ++j) order[j] = (int)j;
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return work[x] > work[y]; });
    constexpr uint64_t kCacheBytes = 200ull << 20, kOneGroup = 300ull << 20;
    uint64_t total = 0, largest = 1;
    for (const auto &ids : chain) {
      const uint64_t bytes = pow4(passes[ids[0]].n) * sizeof(T);
      total += bytes;
      largest = std::max(largest, bytes);
    }
    const int chains = total <= kOneGroup ? 1 : largest * 3 <= kCacheBytes ? 3 : 2;
    const uint64_t group_bytes = chains == 1 ? kOneGroup : kCacheBytes / chains;
    std::vector<double> load(chains, 0.0);
    for (size_t g0 = 0; g0 < order.size();) {
      size_t g1 = g0;
      double gw = 0;
      b->group_start.push_back((uint32_t)b->round_start.size());
      uint64_t bytes = 0;
      while (g1 < order.size()) {
        const uint64_t more = pow4(passes[chain[order[g1]][0]].n) * sizeof(T);
        if (g1 > g0 && bytes + more > group_bytes) break;
        bytes += more;
        gw += work[order[g1]];
        ++g1;
      }
      const int lc = (int)(std::min_element(load.begin(), load.end()) - load.begin());
      load[lc] += gw;
      b->group_chain.push_back(lc);
      size_t rounds = 0;
      for (size_t g = g0; g < g1; ++g) rounds = std::max(rounds, chain[order[g]].size());
      for (size_t r = 0; r < rounds; ++r) {
        b->round_start.push_back((uint32_t)items.size());
        dm_batch::Split sp;
        for (int kind = 0; kind < 4; ++kind) {
          if (kind) sp.at[kind - 1] = (uint32_t)items.size();
          for (size_t g = g0; g < g1; ++g) {
            const int j = order[g];
            if (r >= chain[j].size()) continue;
            const int pi = chain[j][r];
            const BatchPass &bp = passes[pi];
            const int k = bp.kind != BP_TILE ? 0 : bp.geo.m != kQueueTile7 ? 1 : bp.reg_stages ? 2 : 3;
            if (k != kind) continue;
            const uint64_t units =
                bp.kind == BP_PROBS ? 1
                                    : pow4(bp.n - (bp.kind == BP_TILE ? (bp.reg_stages ? kRegTile : bp.geo.m) : kQueueTile));
            const uint64_t per = k ? 1 : std::max<uint64_t>(1, (units + items_per_pass - 1) / items_per_pass);
            for (uint64_t t0 = 0; t0 < units; t0 += per) {
              BatchItem it;
              it.pass = (uint32_t)pi;
              it.tile0 = (uint32_t)t0;
              it.ntiles = (uint32_t)std::min<uint64_t>(per, units - t0);
              it.pad = 0;
              items.push_back(it);
            }
            if (items.size() > (size_t)UINT32_MAX / 2) return fail(DM_ERR_ARG, "batch: too many work items");
          }
        }
        b->split.push_back(sp);
      }
      g0 = g1;
    }
    b->group_start.push_back((uint32_t)b->round_start.size());
    b->nchains = std::min(chains, (int)b->group_chain.size());
    if (!b->round_start.empty()) b->round_start.push_back((uint32_t)items.size());
  }
  b->nitems = (uint32_t)items.size();

  HIP_TRY(hipStreamCreateWithFlags(&b->master, hipStreamNonBlocking));
  HIP_TRY(hipStreamCreateWithFlags(&b->side, hipStreamNonBlocking));
  HIP_TRY(hipEventCreateWithFlags(&b->fork, hipEventDisableTiming));
  HIP_TRY(hipEventCreateWithFlags(&b->join, hipEventDisableTiming));
  HIP_TRY(hipStreamCreateWithFlags(&b->side6, hipStreamNonBlocking));
  HIP_TRY(hipStreamCreateWithFlags(&b->side7, hipStreamNonBlocking));
  HIP_TRY(hipEventCreateWithFlags(&b->forkr, hipEventDisableTiming));
  HIP_TRY(hipEventCreateWithFlags(&b->join6, hipEventDisableTiming));
  HIP_TRY(hipEventCreateWithFlags(&b->join7, hipEventDisableTiming));
  HIP_TRY(hipEventCreate(&b->ev0));
  HIP_TRY(hipEventCreate(&b->ev1));
  auto upload = [](void **dst, const void *src, size_t bytes) -> int {
    HIP_TRY(hipMalloc(dst, std::max<size_t>(bytes, 16)));
    if (bytes) HIP_TRY(hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice));
    return DM_OK;
  };
  if (!rcircs.empty()) {
    if (int rc = upload(&b->d_rcircs, rcircs.data(), rcircs.size() * sizeof(RegCirc))) return rc;
    if (int rc = upload(&b->d_rrecs, rrecs.data(), rrecs.size() * 4)) return rc;
    if (int rc = upload(&b->d_rvals, rvals.data(), rvals.size() * sizeof(T))) return rc;
  }
  if (!circs.empty()) {
    std::vector<T> tv(vals.begin(), vals.end());
    if (int rc = upload(&b->d_circs, circs.data(), circs.size() * sizeof(BatchCirc))) return rc;
    if (int rc = upload(&b->d_tops, tops.data(), tops.size() * sizeof(TileOp))) return rc;
    if (int rc = upload(&b->d_vals, tv.data(), tv.size() * sizeof(T))) return rc;
    size_t need = 0;
    for (auto &bc : circs) need = std::max(need, lds_bytes(bc.n, b->dtype));
    HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_circuit_lds<T>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)need));
  }
  if (b->nitems) {
    HIP_TRY(hipMalloc(&b->d_arena, arena * sizeof(T)));
    if (int rc = upload(&b->d_passes, passes.data(), passes.size() * sizeof(BatchPass))) return rc;
    if (int rc = upload(&b->d_items, items.data(), items.size() * sizeof(BatchItem))) return rc;
    if (int rc = upload(&b->d_qtops, qtops.data(), qtops.size() * sizeof(TileOp))) return rc;
    if (int rc = upload(&b->d_qvals, qvals.data(), qvals.size() * sizeof(T))) return rc;
    if (int rc = upload(&b->d_recs, recs.data(), recs.size() * 4)) return rc;
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_batch_round<T>, kQueueThreads, 0) != hipSuccess ||
        per_cu < 1)
      per_cu = 1;
    b->queue_grid = cu * per_cu;
    for (size_t r = 0; r + 1 < b->round_start.size(); ++r)
      b->launches += (b->split[r].at[0] > b->round_start[r]) + (b->split[r].at[1] > b->split[r].at[0]) +
                     (b->split[r].at[2] > b->split[r].at[1]) + (b->round_start[r + 1] > b->split[r].at[2]);
  }
  HIP_TRY(hipMalloc(&b->d_probs, std::max<int64_t>(1, b->nprobs) * sizeof(double)));
  HIP_TRY(hipMalloc(&b->d_stamps, 2 * (size_t)b->ncirc * sizeof(uint64_t)));
  HIP_TRY(hipDeviceSynchronize());
  return DM_OK;
}

constexpr int kHostParts = 256;  // (FP64, 8 qubits: 25 us against 27)

template <typename TA, typename TB>
static int diff_t(dm_state *a, dm_state *b, double *out4) {
  using Shape = DiffShape<TA, TB>;
  const uint64_t packs = a->N / Shape::width;
  const int grid = std::min(grid_for(a, packs), Shape::grid);
  if (int rc = reserve_red(a, 4 * (size_t)grid + 8)) return rc;
  HIP_TRY(hipStreamSynchronize(b->stream));
  hipLaunchKernelGGL((k_diff<TA, TB>), dim3(grid), dim3(kBlock), 0, a->stream, static_cast<const TA *>(a->d_a),
                     static_cast<const TB *>(b->d_a), packs, a->d_red);
  if (grid > kHostParts) {
    double *res = a->d_red + 4 * (size_t)grid;
    hipLaunchKernelGGL(k_diff_parts, dim3(4), dim3(kBlock), 0, a->stream, a->d_red, grid, res);
    if (int rc = last_launch("k_diff")) return rc;
    HIP_TRY(hipMemcpyAsync(out4, res, 4 * sizeof(double), hipMemcpyDeviceToHost, a->stream));
    HIP_TRY(hipStreamSynchronize(a->stream));
    return DM_OK;
  }
  // few partials: their sums are cheaper here than by a second launch
  if (int rc = last_launch("k_diff")) return rc;
  double part[4 * kHostParts];
  HIP_TRY(hipMemcpyAsync(part, a->d_red, 4 * (size_t)grid * sizeof(double), hipMemcpyDeviceToHost, a->stream));
  HIP_TRY(hipStreamSynchronize(a->stream));
  for (int c = 0; c < 4; ++c) {
    out4[c] = 0.0;
    for (int i = 0; i < grid; ++i) {
      const double p = part[c * grid + i];
      out4[c] = c ? out4[c] + p : std::max(out4[c], p);
    }
  }
  return DM_OK;
}

#define DISPATCH(h, fn, ...) ((h)->dtype == DM_FP64 ? fn<double>(__VA_ARGS__) : fn<float>(__VA_ARGS__))

extern "C" {

int dm_last_error(char *buf, size_t len) {
  if (!buf || len == 0) return DM_ERR_ARG;
  snprintf(buf, len, "%s", g_err);
  return DM_OK;
}

int dm_device_info(int device, int *n_devices, int *cu_count, uint64_t *hbm_bytes) {
  int nd = 0;
  HIP_TRY(hipGetDeviceCount(&nd));
  if (n_devices) *n_devices = nd;
  if (device < 0 || device >= nd) return fail(DM_ERR_ARG, "device %d not present (%d visible)", device, nd);
  hipDeviceProp_t prop;
  HIP_TRY(hipGetDeviceProperties(&prop, device));
  if (cu_count) *cu_count = prop.multiProcessorCount;
  if (hbm_bytes) *hbm_bytes = (uint64_t)prop.totalGlobalMem;
  return DM_OK;
}

int dm_create(int n_qubits, int dtype, dm_state **out) {
  if (!out) return fail(DM_ERR_ARG, "null output pointer");
  *out = nullptr;
  if (n_qubits < 1 || n_qubits > kMaxQubits)
    return fail(DM_ERR_ARG, "number of qubits %d outside [1, %d]", n_qubits, kMaxQubits);
  if (dtype != DM_FP64 && dtype != DM_FP32) return fail(DM_ERR_ARG, "unknown dtype %d", dtype);
  dm_state *h = new dm_state();
  h->n = n_qubits;
  h->dtype = dtype;
  h->N = pow4(n_qubits);
  hipError_t e = hipGetDevice(&h->device);
  if (e == hipSuccess) {
    hipDeviceProp_t prop;
    e = hipGetDeviceProperties(&prop, h->device);
    if (e == hipSuccess) h->cu_count = prop.multiProcessorCount;
  }
  if (e == hipSuccess) e = hipStreamCreate(&h->stream);
  const size_t es = dtype == DM_FP64 ? sizeof(double) : sizeof(float);
  if (e == hipSuccess) e = hipMalloc(&h->d_a, h->N * es);
  if (e == hipSuccess) e = hipEventCreate(&h->ev0);
  if (e == hipSuccess) e = hipEventCreate(&h->ev1);
  if (e != hipSuccess) {
    const int rc = fail(DM_ERR_HIP, "dm_create(%d qubits, %s): %s", n_qubits, dtype ? "fp32" : "fp64",
                        hipGetErrorString(e));
    dm_destroy(h);
    return rc;
  }
  *out = h;
  return DM_OK;
}

int dm_destroy(dm_state *h) {
  if (!h) return DM_OK;
  if (h->stream) hipStreamSynchronize(h->stream);
  if (h->d_a) hipFree(h->d_a);
  if (h->d_red) hipFree(h->d_red);
  if (h->d_mat) hipFree(h->d_mat);
  if (h->h_img) hipHostFree(h->h_img);
  if (h->img_ev) hipEventDestroy(h->img_ev);
  if (h->d_aux) hipFree(h->d_aux);
  if (h->d_mn) hipFree(h->d_mn);
  if (h->ev0) hipEventDestroy(h->ev0);
  if (h->ev1) hipEventDestroy(h->ev1);
  for (auto &pp : h->pending) {
    hipEventDestroy(pp.a);
    hipEventDestroy(pp.b);
  }
  for (auto e : h->spare_events) hipEventDestroy(e);
  if (h->stream && h->owns_stream) hipStreamDestroy(h->stream);
  delete h;
  return DM_OK;
}

int dm_num_qubits(const dm_state *h, int *n) {
  if (!h || !n) return fail(DM_ERR_ARG, "null argument");
  *n = h->n;
  return DM_OK;
}

int dm_dtype(const dm_state *h, int *dtype) {
  if (!h || !dtype) return fail(DM_ERR_ARG, "null argument");
  *dtype = h->dtype;
  return DM_OK;
}

int dm_device_ptr(const dm_state *h, void **ptr) {
  if (int rc = check_handle(h)) return rc;
  if (!ptr) return fail(DM_ERR_ARG, "null argument");
  *ptr = h->d_a;
  return DM_OK;
}

int dm_init_product(dm_state *h, const double *per_qubit4, double scale) {
  if (int rc = check_handle(h)) return rc;
  if (!per_qubit4) return fail(DM_ERR_ARG, "null per-qubit vectors");
  // table row p = position p = qubit n-1-p
  double tab[4 * kMaxQubits];
  for (int p = 0; p < h->n; ++p)
    for (int c = 0; c < 4; ++c) tab[4 * p + c] = per_qubit4[4 * (h->n - 1 - p) + c];
  return DISPATCH(h, launch_diag_tab, h, tab, true, scale);
}

int dm_upload(dm_state *h, const double *host) {
  if (int rc = check_handle(h)) return rc;
  if (!host) return fail(DM_ERR_ARG, "null host buffer");
  ProfScope ps(h, 7);
  if (h->dtype == DM_FP64) {
    HIP_TRY(hipMemcpyAsync(h->d_a, host, h->N * sizeof(double), hipMemcpyHostToDevice, h->stream));
  } else {
    double *tmp = nullptr;
    HIP_TRY(hipMallocAsync(reinterpret_cast<void **>(&tmp), h->N * sizeof(double), h->stream));
    HIP_TRY(hipMemcpyAsync(tmp, host, h->N * sizeof(double), hipMemcpyHostToDevice, h->stream));
    hipLaunchKernelGGL((k_convert<double, float>), dim3(grid_for(h, h->N)), dim3(kBlock), 0, h->stream, tmp,
                       static_cast<float *>(h->d_a), h->N);
    HIP_TRY(hipFreeAsync(tmp, h->stream));
  }
  HIP_TRY(hipStreamSynchronize(h->stream));
  return last_launch("upload");
}

static int download_impl(dm_state *h, double *host) {
  if (h->dtype == DM_FP64) {
    HIP_TRY(hipMemcpyAsync(host, h->d_a, h->N * sizeof(double), hipMemcpyDeviceToHost, h->stream));
  } else {
    double *tmp = nullptr;
    HIP_TRY(hipMallocAsync(reinterpret_cast<void **>(&tmp), h->N * sizeof(double), h->stream));
    hipLaunchKernelGGL((k_convert<float, double>), dim3(grid_for(h, h->N)), dim3(kBlock), 0, h->stream,
                       static_cast<const float *>(h->d_a), tmp, h->N);
    HIP_TRY(hipMemcpyAsync(host, tmp, h->N * sizeof(double), hipMemcpyDeviceToHost, h->stream));
    HIP_TRY(hipFreeAsync(tmp, h->stream));
  }
  HIP_TRY(hipStreamSynchronize(h->stream));
  return last_launch("download");
}

int dm_download(dm_state *h, double *host) {
  if (int rc = check_handle(h)) return rc;
  if (!host) return fail(DM_ERR_ARG, "null host buffer");
  return download_impl(h, host);
}

int dm_download_chop(dm_state *h, double thr, double *host) {
  if (int rc = check_handle(h)) return rc;
  if (!host) return fail(DM_ERR_ARG, "null host buffer");
  if (thr > 0) {
    if (h->dtype == DM_FP64)
      hipLaunchKernelGGL((k_chop<double>), dim3(grid_for(h, h->N)), dim3(kBlock), 0, h->stream,
                         static_cast<double *>(h->d_a), h->N, thr);
    else
      hipLaunchKernelGGL((k_chop<float>), dim3(grid_for(h, h->N)), dim3(kBlock), 0, h->stream,
                         static_cast<float *>(h->d_a), h->N, (float)thr);
  }
  return download_impl(h, host);
}

int dm_read_coeffs(dm_state *h, const uint64_t *index, int k, double *out) {
  if (int rc = check_handle(h)) return rc;
  if (k < 0 || (k > 0 && (!index || !out))) return fail(DM_ERR_ARG, "bad index list");
  const size_t es = h->dtype == DM_FP64 ? 8 : 4;
  for (int i = 0; i < k; ++i) {
    if (index[i] >= h->N) return fail(DM_ERR_ARG, "coefficient index %llu out of range", (unsigned long long)index[i]);
    if (h->dtype == DM_FP64) {
      HIP_TRY(hipMemcpyAsync(out + i, static_cast<char *>(h->d_a) + index[i] * es, es, hipMemcpyDeviceToHost,
                             h->stream));
    } else {
      float f = 0.f;
      HIP_TRY(hipMemcpyAsync(&f, static_cast<char *>(h->d_a) + index[i] * es, es, hipMemcpyDeviceToHost, h->stream));
      HIP_TRY(hipStreamSynchronize(h->stream));
      out[i] = f;
    }
  }
  HIP_TRY(hipStreamSynchronize(h->stream));
  return DM_OK;
}

int dm_apply_1q(dm_state *h, int q, const double R[12]) {
  if (int rc = check_handle(h)) return rc;
  if (int rc = check_qubit(h, q)) return rc;
  if (!R) return fail(DM_ERR_ARG, "null matrix");
  return DISPATCH(h, launch_1q, h, q, R);
}

int dm_apply_cx(dm_state *h, int control, int target, const double *scale16) {
  if (int rc = check_handle(h)) return rc;
  if (control == target || control < 0 || target < 0 || control >= h->n || target >= h->n)
    return fail(DM_ERR_ARG, "Qubit Labels out of bound in CX Gate (%d, %d; n=%d)", control, target, h->n);
  return DISPATCH(h, launch_cx, h, control, target, scale16);
}

int dm_apply_2q(dm_state *h, int qa, int qb, const double R[256]) {
  if (int rc = check_handle(h)) return rc;
  if (qa == qb || qa < 0 || qb < 0 || qa >= h->n || qb >= h->n)
    return fail(DM_ERR_ARG, "bad qubit pair (%d, %d; n=%d)", qa, qb, h->n);
  if (!R) return fail(DM_ERR_ARG, "null matrix");
  return DISPATCH(h, launch_2q, h, qa, qb, R);
}

int dm_memory_noise(dm_state *h, double f, double p, double g) {
  if (int rc = check_handle(h)) return rc;
  if (f == 1.0 && g == 1.0) return DM_OK;  // identity (up to the sign of zeros)
  return DISPATCH(h, launch_memory_noise, h, f, p, g);
}

int dm_apply_diag(dm_state *h, const double *tab4n) {
  if (int rc = check_handle(h)) return rc;
  if (!tab4n) return fail(DM_ERR_ARG, "null table");
  double tab[4 * kMaxQubits];
  for (int p = 0; p < h->n; ++p)
    for (int c = 0; c < 4; ++c) tab[4 * p + c] = tab4n[4 * (h->n - 1 - p) + c];
  return DISPATCH(h, launch_diag_tab, h, tab, false, 1.0);
}

int dm_apply_block(dm_state *h, const int *qubits, int k, const double *S) {
  if (int rc = check_handle(h)) return rc;
  if (!qubits || !S) return fail(DM_ERR_ARG, "null argument");
  if (k != 3 && k != 4) return fail(DM_ERR_ARG, "block size k=%d not supported (3 or 4)", k);
  for (int j = 0; j < k; ++j) {
    if (int rc = check_qubit(h, qubits[j])) return rc;
    for (int i = 0; i < j; ++i)
      if (qubits[i] == qubits[j]) return fail(DM_ERR_ARG, "repeated qubit %d in block", qubits[j]);
  }
  const int L = (k == 3) ? 3 : 2;
  if (h->n < k + L) return fail(DM_ERR_ARG, "block of %d qubits needs n >= %d (n=%d)", k, k + L, h->n);
  return DISPATCH(h, launch_block, h, qubits, k, S);
}

int dm_probabilities(dm_state *h, const int *qubits, int m, char basis, const double *nvec, double err,
                     double *out) {
  if (int rc = check_handle(h)) return rc;
  if (m < 1 || m > h->n || !qubits || !out) return fail(DM_ERR_ARG, "bad measured-qubit list");
  if (basis != 'X' && basis != 'Y' && basis != 'Z' && basis != 'N') return fail(DM_ERR_ARG, "bad basis '%c'", basis);
  if (basis == 'N' && !nvec) return fail(DM_ERR_ARG, "basis N needs a direction");
  if (basis == 'N' && m > 13) return fail(DM_ERR_ARG, "basis N gathers 4^m values; m=%d too large", m);
  for (int t = 0; t < m; ++t) {
    if (int rc = check_qubit(h, qubits[t])) return rc;
    if (t && qubits[t] <= qubits[t - 1]) return fail(DM_ERR_ARG, "measured qubits must be ascending");
  }
  return DISPATCH(h, do_probabilities, h, qubits, m, basis, nvec, err, out);
}

int dm_trace_purity(dm_state *h, double *tr, double *purity) {
  if (int rc = check_handle(h)) return rc;
  if (tr) {
    uint64_t zero = 0;
    double a0 = 0;
    if (int rc = dm_read_coeffs(h, &zero, 1, &a0)) return rc;
    *tr = ldexp(a0, h->n);
  }
  if (purity) {
    double s = 0;
    if (int rc = DISPATCH(h, do_sumsq, h, &s)) return rc;
    *purity = ldexp(s, h->n);
  }
  return DM_OK;
}

int dm_overlap(dm_state *h, const double *other_host, double *out) {
  if (int rc = check_handle(h)) return rc;
  if (!other_host || !out) return fail(DM_ERR_ARG, "null argument");
  double *d_b = nullptr;
  HIP_TRY(hipMallocAsync(reinterpret_cast<void **>(&d_b), h->N * sizeof(double), h->stream));
  hipError_t e = hipMemcpyAsync(d_b, other_host, h->N * sizeof(double), hipMemcpyHostToDevice, h->stream);
  int rc = DM_OK;
  if (e != hipSuccess) rc = fail(DM_ERR_HIP, "overlap upload failed: %s", hipGetErrorString(e));
  double s = 0;
  if (rc == DM_OK) rc = DISPATCH(h, do_dot, h, d_b, &s);
  hipFreeAsync(d_b, h->stream);
  HIP_TRY(hipStreamSynchronize(h->stream));
  if (rc == DM_OK) *out = ldexp(s, h->n);
  return rc;
}

static int check_range(const dm_state *h, uint64_t offset, uint64_t count, int host_dtype, const void *host) {
  if (int rc = check_handle(h)) return rc;
  if (host_dtype != DM_FP64 && host_dtype != DM_FP32) return fail(DM_ERR_ARG, "unknown host dtype %d", host_dtype);
  if (offset > h->N || count > h->N - offset)
    return fail(DM_ERR_ARG, "range [%llu, +%llu) outside the %llu coefficients", (unsigned long long)offset,
                (unsigned long long)count, (unsigned long long)h->N);
  if (count && !host) return fail(DM_ERR_ARG, "null host buffer");
  return DM_OK;
}

#define STATE_DISPATCH(fn, H, ...) ((h)->dtype == DM_FP64 ? fn<double, H>(__VA_ARGS__) : fn<float, H>(__VA_ARGS__))

int dm_download_range(dm_state *h, uint64_t offset, uint64_t count, int host_dtype, void *host) {
  if (int rc = check_range(h, offset, count, host_dtype, host)) return rc;
  if (!count) return DM_OK;
  ProfScope ps(h, 7);
  if (host_dtype == DM_FP64)
    return STATE_DISPATCH(copy_range, double, h, offset, count, static_cast<double *>(host), true);
  return STATE_DISPATCH(copy_range, float, h, offset, count, static_cast<float *>(host), true);
}

int dm_upload_range(dm_state *h, uint64_t offset, uint64_t count, int host_dtype, const void *host) {
  if (int rc = check_range(h, offset, count, host_dtype, host)) return rc;
  if (!count) return DM_OK;
  ProfScope ps(h, 7);
  if (host_dtype == DM_FP64)
    return STATE_DISPATCH(copy_range, double, h, offset, count,
                          const_cast<double *>(static_cast<const double *>(host)), false);
  return STATE_DISPATCH(copy_range, float, h, offset, count, const_cast<float *>(static_cast<const float *>(host)),
                        false);
}

int dm_dot_range(dm_state *h, uint64_t offset, uint64_t count, int host_dtype, const void *host, double *sum) {
  if (int rc = check_range(h, offset, count, host_dtype, host)) return rc;
  if (!sum) return fail(DM_ERR_ARG, "null output");
  *sum = 0.0;
  if (!count) return DM_OK;
  if (host_dtype == DM_FP64)
    return STATE_DISPATCH(dot_range, double, h, offset, count, static_cast<const double *>(host), sum);
  return STATE_DISPATCH(dot_range, float, h, offset, count, static_cast<const float *>(host), sum);
}
#undef STATE_DISPATCH

int dm_to_dense(dm_state *h, double *out_c128) {
  if (int rc = check_handle(h)) return rc;
  if (!out_c128) return fail(DM_ERR_ARG, "null output");
  return DISPATCH(h, do_to_dense, h, out_c128);
}

int dm_run_program(dm_state *h, const dm_op *ops, int nops, const double *params, int64_t nparams) {
  if (int rc = check_handle(h)) return rc;
  if (nops < 0 || (nops > 0 && !ops)) return fail(DM_ERR_ARG, "bad op list");
  if (nparams < 0 || (nparams > 0 && !params)) return fail(DM_ERR_ARG, "bad parameter array");
  return DISPATCH(h, run_program, h, ops, nops, params, nparams);
}

int dm_run_program_noalloc(dm_state *h, const dm_op *ops, int nops, const double *params, int64_t nparams) {
  if (int rc = check_handle(h)) return rc;
  if (nops < 0 || (nops > 0 && !ops)) return fail(DM_ERR_ARG, "bad op list");
  if (nparams < 0 || (nparams > 0 && !params)) return fail(DM_ERR_ARG, "bad parameter array");
  return DISPATCH(h, run_program_noalloc, h, ops, nops, params, nparams);
}

int dm_batch_destroy(dm_batch *b) {
  if (!b) return DM_OK;
  if (b->master) hipStreamSynchronize(b->master);
  if (b->side) hipStreamSynchronize(b->side);
  if (b->side6) hipStreamSynchronize(b->side6);
  if (b->side7) hipStreamSynchronize(b->side7);
  if (b->exec) hipGraphExecDestroy(b->exec);
  if (b->graph) hipGraphDestroy(b->graph);
  for (void *p : {b->d_circs, b->d_tops, b->d_vals, b->d_arena, b->d_passes, b->d_items, b->d_qtops, b->d_qvals, b->d_recs,
                  b->d_rcircs, b->d_rrecs, b->d_rvals, (void *)b->d_probs, (void *)b->d_stamps})
    if (p) hipFree(p);
  for (hipEvent_t e : {b->fork, b->join, b->ev0, b->ev1, b->forkr, b->join6, b->join7})
    if (e) hipEventDestroy(e);
  for (hipStream_t st : {b->side, b->side6, b->side7, b->master})
    if (st) hipStreamDestroy(st);
  delete b;
  return DM_OK;
}

int dm_batch_create(int dtype, int ncirc, const int *n_qubits, const int64_t *op_start, const dm_op *ops,
                    const double *params, int64_t nparams, const double *meas_err, int lds_max_qubits,
                    int lds_threads, int items_per_pass, dm_batch **out) {
  if (!out) return fail(DM_ERR_ARG, "null output pointer");
  *out = nullptr;
  if (dtype != DM_FP64 && dtype != DM_FP32) return fail(DM_ERR_ARG, "unknown dtype %d", dtype);
  if (ncirc < 1 || !n_qubits || !op_start || !meas_err) return fail(DM_ERR_ARG, "bad circuit list");
  if (lds_threads != 256 && lds_threads != 512 && lds_threads != 1024)
    return fail(DM_ERR_ARG, "lds_threads must be 256, 512 or 1024");
  if (lds_max_qubits < kQueueTile - 1 || lds_max_qubits > 7)
    return fail(DM_ERR_ARG, "lds_max_qubits must lie in [%d, 7]", kQueueTile - 1);
  if (items_per_pass < 1 || items_per_pass > 65536) return fail(DM_ERR_ARG, "items_per_pass must lie in [1, 65536]");
  if (nparams < 0 || (nparams > 0 && !params)) return fail(DM_ERR_ARG, "bad parameter array");
  for (int c = 0; c < ncirc; ++c) {
    if (n_qubits[c] < 1 || n_qubits[c] > kQueueMaxQubits)
      return fail(DM_ERR_ARG, "circuit %d: %d qubits outside [1, %d]", c, n_qubits[c], kQueueMaxQubits);
    if (op_start[c + 1] < op_start[c] || (op_start[c + 1] > op_start[c] && !ops))
      return fail(DM_ERR_ARG, "circuit %d: bad op range", c);
  }
  dm_batch *b = new dm_batch();
  b->dtype = dtype;
  b->ncirc = ncirc;
  b->lds_threads = lds_threads;
  for (int c = 0; c < ncirc; ++c) {
    b->nq.push_back(n_qubits[c]);
    b->prob_off.push_back(b->nprobs);
    b->nprobs += (int64_t)1 << n_qubits[c];
    b->err.push_back(meas_err[c]);
  }
  const int rc = dtype == DM_FP64
                     ? batch_create_t<double>(b, op_start, ops, params, nparams, lds_max_qubits, items_per_pass)
                     : batch_create_t<float>(b, op_start, ops, params, nparams, lds_max_qubits, items_per_pass);
  if (rc) {
    dm_batch_destroy(b);
    return rc;
  }
  *out = b;
  return DM_OK;
}

int dm_batch_info(const dm_batch *b, int64_t *hbm_circuits, int64_t *passes, int64_t *items, int64_t *launches) {
  if (!b) return fail(DM_ERR_ARG, "null batch");
  if (hbm_circuits) *hbm_circuits = (int64_t)b->large.size();
  if (passes) *passes = b->npasses;
  if (items) *items = b->nitems;
  if (launches) *launches = b->launches;
  return DM_OK;
}

int dm_batch_run(dm_batch *b, int use_graph, double *probs_out, double *circuit_us, double *total_ms) {
  if (!b) return fail(DM_ERR_ARG, "null batch");
  if (use_graph && !b->exec) {
    HIP_TRY(hipStreamBeginCapture(b->master, hipStreamCaptureModeThreadLocal));
    const int rc = b->dtype == DM_FP64 ? enqueue_batch<double>(b) : enqueue_batch<float>(b);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(b->master, &g);
    if (rc) {
      if (g) hipGraphDestroy(g);
      return rc;
    }
    if (e != hipSuccess) return fail(DM_ERR_HIP, "batch capture: %s", hipGetErrorString(e));
    b->graph = g;
    HIP_TRY(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
  }
  HIP_TRY(hipEventRecord(b->ev0, b->master));
  if (use_graph) {
    HIP_TRY(hipGraphLaunch(b->exec, b->master));
  } else {
    const int rc = b->dtype == DM_FP64 ? enqueue_batch<double>(b) : enqueue_batch<float>(b);
    if (rc) return rc;
  }
  HIP_TRY(hipEventRecord(b->ev1, b->master));
  HIP_TRY(hipEventSynchronize(b->ev1));
  float ms = 0.f;
  HIP_TRY(hipEventElapsedTime(&ms, b->ev0, b->ev1));
  if (total_ms) *total_ms = ms;
  if (probs_out) HIP_TRY(hipMemcpy(probs_out, b->d_probs, b->nprobs * sizeof(double), hipMemcpyDeviceToHost));
  if (circuit_us) {
    std::vector<uint64_t> st(2 * (size_t)b->ncirc);
    HIP_TRY(hipMemcpy(st.data(), b->d_stamps, st.size() * sizeof(uint64_t), hipMemcpyDeviceToHost));
    // stamps are stored LDS-tier circuits first, then HBM-tier circuits; report in circuit order
    std::vector<int> order(b->small);
    order.insert(order.end(), b->large.begin(), b->large.end());
    for (size_t j = 0; j < order.size(); ++j)
      circuit_us[order[j]] = (double)(st[2 * j + 1] - st[2 * j]) / b->clock_khz * 1e3;
  }
  return DM_OK;
}

int dm_compare(dm_state *a, dm_state *b, double *max_abs_diff, double *dot, double *norm2_a, double *norm2_b) {
  if (int rc = check_handle(a)) return rc;
  if (int rc = check_handle(b)) return rc;
  if (a->n != b->n) return fail(DM_ERR_ARG, "states of %d and %d qubits", a->n, b->n);
  double o[4];
  int rc;
  if (a->dtype == DM_FP64 && b->dtype == DM_FP64) rc = diff_t<double, double>(a, b, o);
  else if (a->dtype == DM_FP64) rc = diff_t<double, float>(a, b, o);
  else if (b->dtype == DM_FP64) rc = diff_t<float, double>(a, b, o);
  else rc = diff_t<float, float>(a, b, o);
  if (rc) return rc;
  if (max_abs_diff) *max_abs_diff = o[0];
  if (dot) *dot = o[1];
  if (norm2_a) *norm2_a = o[2];
  if (norm2_b) *norm2_b = o[3];
  return DM_OK;
}

int dm_synchronize(dm_state *h) {
  if (int rc = check_handle(h)) return rc;
  HIP_TRY(hipStreamSynchronize(h->stream));
  return last_launch("stream");
}

int dm_profile(dm_state *h, int enable) {
  if (int rc = check_handle(h)) return rc;
  h->prof = enable != 0;
  return DM_OK;
}

int dm_profile_read(dm_state *h, int family, uint64_t *launches, double *ms) {
  if (int rc = check_handle(h)) return rc;
  if (family < 0 || family >= kFamilies) return fail(DM_ERR_ARG, "bad kernel family %d", family);
  if (int rc = resolve_profile(h)) return rc;
  if (launches) *launches = h->slots[family].launches;
  if (ms) *ms = h->slots[family].ms;
  return DM_OK;
}

int dm_profile_reset(dm_state *h) {
  if (int rc = check_handle(h)) return rc;
  if (int rc = resolve_profile(h)) return rc;
  for (auto &s : h->slots) s = ProfSlot();
  return DM_OK;
}

}  // extern "C"
