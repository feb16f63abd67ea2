// tile_reg.h -- fused tile passes with the tile held in registers (gfx950).
// Included by dmsim.hip.
//
// A workgroup of 256 threads owns a tile of 4^7 coefficients, 64 per thread:
// three tile digits ("register digits") index a thread's 64 values, the four
// others ("lane digits", three, and one "wave digit") say which thread holds
// them.  A stage applies single-qubit maps and CX gates on its three register
// digits without touching LDS; between stages the tile is redistributed
// through LDS once so that the next three digits are in registers.

constexpr int kRegThreads = 256;

struct RegGeom {
  int nr;
  int rpos[kMaxQubits];   // positions enumerating the tiles, ascending
  uint32_t tiles;
  // HBM strides (coefficients) of the register digits and the wave digit in
  // the layouts that load and store the tile; the lane digits are digits 0-2,
  // 64 consecutive coefficients
  uint64_t is[3], iw, os[3], ow;
};

// a * x + c into a register of its own choice: the compiler's two-address
// form would accumulate into c and then copy the result into its place.
__device__ __forceinline__ float reg_fma(float a, float x, float c) {
  float r;
  asm("v_fma_f32 %0, %1, %2, %3" : "=v"(r) : "s"(a), "v"(x), "v"(c));
  return r;
}
__device__ __forceinline__ double reg_fma(double a, double x, double c) {
  double r;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "s"(a), "v"(x), "v"(c));
  return r;
}

// SEQ: products and sums rounded one by one, as k_circuit_lds does; otherwise
// fused multiply-adds, as the tile kernels.
template <typename T, int SLOT, bool AFF, bool SEQ>
__device__ __forceinline__ void reg_1q(T (&v)[64], const T (&pv)[kRegVals]) {
  constexpr int S = 1 << (2 * SLOT);
  constexpr int C = AFF ? 4 : 3;
  T r[3][C];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < C; ++j) r[i][j] = pv[C * i + j];
#pragma unroll
  for (int o = 0; o < 16; ++o) {
    const int b = SLOT == 0 ? 4 * o : SLOT == 1 ? (o & 3) + 16 * (o >> 2) : o;
    const T x0 = v[b], x1 = v[b + S], x2 = v[b + 2 * S], x3 = v[b + 3 * S];
    T t[3];
    if constexpr (SEQ) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const T *q = &r[i][AFF ? 1 : 0];
        t[i] = (AFF ? r[i][0] * x0 + q[0] * x1 : q[0] * x1) + q[1] * x2 + q[2] * x3;
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) v[b + (i + 1) * S] = t[i];
      continue;
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const T *q = &r[i][AFF ? 1 : 0];
      const T first = AFF ? fmad(q[0], x1, r[i][0] * x0) : q[0] * x1;
      t[i] = fmad(q[1], x2, first);
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) v[b + (i + 1) * S] = reg_fma(r[i][AFF ? 3 : 2], x3, t[i]);
  }
}

// In place (v_swap_b32): plain copies would keep a second set of registers
// alive where the members' code paths join (FP64: 196 VGPRs, two waves per
// SIMD, against 154 and three: 15 qubits 81.7 -> 76.9 ms, 10 qubits 366 -> 331
// us).
template <typename T>
__device__ __forceinline__ void reg_swap(T &a, T &b) {
  if constexpr (sizeof(T) == 4) {
    asm("v_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  } else {
    typedef uint32_t U2 __attribute__((ext_vector_type(2)));
    const U2 x = __builtin_bit_cast(U2, a), y = __builtin_bit_cast(U2, b);
    uint32_t xl = x.x, xh = x.y, yl = y.x, yh = y.y;
    asm("v_swap_b32 %0, %1" : "+v"(xl), "+v"(yl));
    asm("v_swap_b32 %0, %1" : "+v"(xh), "+v"(yh));
    a = __builtin_bit_cast(T, U2{xl, xh});
    b = __builtin_bit_cast(T, U2{yl, yh});
  }
}

// CX with control digit slot C and target slot T_ (pairs as cx_map).
template <typename T, int C, int TG>
__device__ __forceinline__ void reg_cx(T (&v)[64]) {
  constexpr int SC = 1 << (2 * C), ST = 1 << (2 * TG), SO = 1 << (2 * (3 - C - TG));
#pragma unroll
  for (int o = 0; o < 4; ++o) {
    auto X = [&](int c, int t) -> T & { return v[o * SO + c * SC + t * ST]; };
    reg_swap(X(0, 2), X(3, 2));
    reg_swap(X(0, 3), X(3, 3));
    reg_swap(X(1, 0), X(1, 1));
    reg_swap(X(1, 2), X(2, 3));
    reg_swap(X(2, 0), X(2, 1));
    reg_swap(X(1, 3), X(2, 2));
    X(1, 3) = -X(1, 3);
    X(2, 2) = -X(2, 2);
  }
}

// The same followed by the pair's scales; the two signs go into their scales
// (the product has the same bits).  A pair that swaps is two products and a
// copy, against a swap, two products and a separate member (13 qubits FP32:
// 2.86 -> 2.70 ms, 16 qubits FP32 504 -> 498 ms).
template <typename T, int C, int TG>
__device__ __forceinline__ void reg_cxd(T (&v)[64], const T (&pv)[kRegVals]) {
  constexpr int SC = 1 << (2 * C), ST = 1 << (2 * TG), SO = 1 << (2 * (3 - C - TG));
  T d[16];
#pragma unroll
  for (int i = 1; i < 16; ++i) d[i] = pv[i];
  d[7] = -d[7];
  d[10] = -d[10];
#pragma unroll
  for (int o = 0; o < 4; ++o) {
    auto X = [&](int i) -> T & { return v[o * SO + (i >> 2) * SC + (i & 3) * ST]; };
    constexpr int pairs[6][2] = {{2, 14}, {3, 15}, {4, 5}, {6, 11}, {8, 9}, {7, 10}};
#pragma unroll
    for (int p = 0; p < 6; ++p) {
      const int i = pairs[p][0], j = pairs[p][1];
      const T t = d[i] * X(j);
      X(j) = d[j] * X(i);
      X(i) = t;
    }
    X(1) *= d[1];
    X(12) *= d[12];
    X(13) *= d[13];
  }
}

template <typename T, int SLOT>
__device__ __forceinline__ void reg_d1(T (&v)[64], const T (&pv)[kRegVals]) {
  constexpr int S = 1 << (2 * SLOT);
  const T d[3] = {pv[0], pv[1], pv[2]};
#pragma unroll
  for (int i = 0; i < 64; ++i) {
    const int c = (i / S) & 3;
    if (c) v[i] *= d[c - 1];
  }
}

template <typename T, int A, int B>
__device__ __forceinline__ void reg_d2(T (&v)[64], const T (&pv)[kRegVals]) {
  constexpr int SA = 1 << (2 * A), SB = 1 << (2 * B);
  T d[16];
#pragma unroll
  for (int i = 1; i < 16; ++i) d[i] = pv[i];
#pragma unroll
  for (int i = 0; i < 64; ++i) {
    const int c = 4 * ((i / SA) & 3) + ((i / SB) & 3);
    if (c) v[i] *= d[c];
  }
}

// The members of a stage in order.  The next member's kind and values are
// loaded (scalar loads) while the current one computes.
template <typename T, bool SEQ>
__device__ __forceinline__ void reg_members(T (&v)[64], const uint32_t *__restrict__ kinds, uint32_t nm,
                                            const T *__restrict__ prm) {
  if (nm == 0) return;
  uint32_t next_kind = kinds[0];
  T next[kRegVals];
#pragma unroll
  for (int i = 0; i < kRegVals; ++i) next[i] = prm[i];
  for (uint32_t q = 0; q < nm; ++q) {
    const uint32_t kind = __builtin_amdgcn_readfirstlane(next_kind);
    T pv[kRegVals];
#pragma unroll
    for (int i = 0; i < kRegVals; ++i) pv[i] = next[i];
    // scalar loads return out of order: wait for this member's values, then
    // start the next one's (the arrays end with one spare member)
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
    next_kind = kinds[q + 1];
    prm += kRegVals;
#pragma unroll
    for (int i = 0; i < kRegVals; ++i) next[i] = prm[i];
    __builtin_amdgcn_sched_barrier(0);
    switch (kind) {
      case RM_U1 + 0: reg_1q<T, 0, false, SEQ>(v, pv); break;
      case RM_U1 + 1: reg_1q<T, 1, false, SEQ>(v, pv); break;
      case RM_U1 + 2: reg_1q<T, 2, false, SEQ>(v, pv); break;
      case RM_A1 + 0: reg_1q<T, 0, true, SEQ>(v, pv); break;
      case RM_A1 + 1: reg_1q<T, 1, true, SEQ>(v, pv); break;
      case RM_A1 + 2: reg_1q<T, 2, true, SEQ>(v, pv); break;
      case RM_CX + 0: reg_cx<T, 0, 1>(v); break;
      case RM_CX + 1: reg_cx<T, 1, 0>(v); break;
      case RM_CX + 2: reg_cx<T, 0, 2>(v); break;
      case RM_CX + 3: reg_cx<T, 2, 0>(v); break;
      case RM_CX + 4: reg_cx<T, 1, 2>(v); break;
      case RM_CX + 5: reg_cx<T, 2, 1>(v); break;
      case RM_D1 + 0: reg_d1<T, 0>(v, pv); break;
      case RM_D1 + 1: reg_d1<T, 1>(v, pv); break;
      case RM_D1 + 2: reg_d1<T, 2>(v, pv); break;
      case RM_D2 + 0: reg_d2<T, 0, 1>(v, pv); break;
      case RM_D2 + 1: reg_d2<T, 0, 2>(v, pv); break;
      case RM_D2 + 2: reg_d2<T, 1, 2>(v, pv); break;
      case RM_CXD + 0: reg_cxd<T, 0, 1>(v, pv); break;
      case RM_CXD + 1: reg_cxd<T, 1, 0>(v, pv); break;
      case RM_CXD + 2: reg_cxd<T, 0, 2>(v, pv); break;
      case RM_CXD + 3: reg_cxd<T, 2, 0>(v, pv); break;
      case RM_CXD + 4: reg_cxd<T, 1, 2>(v, pv); break;
      default: reg_cxd<T, 2, 1>(v, pv); break;
    }
  }
}

// Barrier of the workgroup that orders LDS accesses only: global loads and
// stores stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Redistribution through LDS in phases: phase h moves the coefficients whose
// digit in SLOT (a register digit before and after) lies in the h-th part of
// its range, from and into the same registers, so that a phase needs only
// 1/PH of the tile's bytes of LDS and several workgroups fit a CU.
template <typename T, int M, int SLOT, int PH>
__device__ __forceinline__ void reg_exchange(T (&v)[64], T *s, const RegStage &st, int lane, int wave) {
  constexpr int S = 1 << (2 * SLOT);
  constexpr int IN = 4 / PH;  // digit values per phase
  constexpr uint32_t PART = 1u << (2 * (M - 1));  // coefficients of one digit value
  const uint32_t l0 = lane & 3, l1 = (lane >> 2) & 3, l2 = lane >> 4;
  constexpr uint32_t B = sizeof(T);
  const uint32_t tw = ((l0 * st.wl[0]) ^ (l1 * st.wl[1]) ^ (l2 * st.wl[2]) ^ ((uint32_t)wave * st.ww)) * B;
  const uint32_t tr = ((l0 * st.rl[0]) ^ (l1 * st.rl[1]) ^ (l2 * st.rl[2]) ^ ((uint32_t)wave * st.rw)) * B;
  constexpr int SA = SLOT == 0 ? 1 : 0, SB = SLOT == 2 ? 1 : 2;  // the other slots
  char *c = reinterpret_cast<char *>(s);
#pragma unroll
  for (int h = 0; h < PH; ++h) {
    // addresses are computed anew in each phase: kept over the phases they
    // would cost the registers of another wave (FP32: 88 VGPRs and 5 waves
    // per SIMD against 105 and 4: 13 qubits 2.80 against 2.86 ms, a batch of
    // 512 circuits 58.5 against 60.2 ms)
    uint32_t bw = tw, br = tr;
    asm volatile("" : "+v"(bw), "+v"(br));
    lds_barrier();  // the previous phase has been read
#pragma unroll
    for (int i = 0; i < 64; ++i) {
      const int d = (i / S) & 3;
      if (d / IN != h) continue;
      const uint32_t o = ((((i >> (2 * SA)) & 3) * st.wr[SA]) ^ (((i >> (2 * SB)) & 3) * st.wr[SB])) * B;
      *reinterpret_cast<T *>(c + (bw ^ o) + (d % IN) * PART * B) = v[i];
    }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < 64; ++i) {
      const int d = (i / S) & 3;
      if (d / IN != h) continue;
      const uint32_t o = ((((i >> (2 * SA)) & 3) * st.rr[SA]) ^ (((i >> (2 * SB)) & 3) * st.rr[SB])) * B;
      v[i] = *reinterpret_cast<const T *>(c + (br ^ o) + (d % IN) * PART * B);
    }
  }
}

template <typename T, bool NTM>
__device__ __forceinline__ T reg_load(const T *p, uint32_t off) {
  const T *q = reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + off);
  return NTM ? __builtin_nontemporal_load(q) : *q;
}
template <typename T, bool NTM>
__device__ __forceinline__ void reg_store(T *p, uint32_t off, T x) {
  T *q = reinterpret_cast<T *>(reinterpret_cast<char *>(p) + off);
  if (NTM) __builtin_nontemporal_store(x, q);
  else *q = x;
}

// Phases of a redistribution: 32 KB of LDS (FP32 two phases, FP64 four).
template <typename T>
struct RegShape {
  static constexpr int phases = sizeof(T) == 4 ? 2 : 4;
  static constexpr int lds = (1 << (2 * kRegTile)) / phases;  // coefficients
};

// The stages of a program on the tile in v (the first one's layout).
template <typename T, int M, int PH, bool SEQ>
__device__ __forceinline__ void reg_stages(T (&v)[64], T *s, const RegStage *__restrict__ st, int ns,
                                           const uint32_t *__restrict__ kinds, const T *__restrict__ prm, int lane,
                                           int wave) {
  for (int k = 0; k < ns; ++k) {
    const RegStage sg = st[k];
    if (k) {
      if (sg.slot == 0) reg_exchange<T, M, 0, PH>(v, s, sg, lane, wave);
      else if (sg.slot == 1) reg_exchange<T, M, 1, PH>(v, s, sg, lane, wave);
      else reg_exchange<T, M, 2, PH>(v, s, sg, lane, wave);
    }
    reg_members<T, SEQ>(v, kinds + sg.mem, sg.nm, prm + (size_t)sg.mem * kRegVals);
  }
}

template <typename T, bool NTM>
__device__ __forceinline__ void reg_tile(T *__restrict__ a, T *s, const RegGeom &geo, uint32_t tile,
                                         const RegStage *__restrict__ st, int ns, const uint32_t *__restrict__ kinds,
                                         const T *__restrict__ prm) {
  constexpr int PH = RegShape<T>::phases;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint64_t base = 0;
  {
    uint32_t r = tile;
    for (int j = 0; j < geo.nr; ++j) {
      base |= (uint64_t)(r & 3u) << (2 * geo.rpos[j]);
      r >>= 2;
    }
  }
  const uint32_t loff = lane * (uint32_t)sizeof(T);
  T v[64];
  {
    const T *p = a + base + wave * geo.iw;
#pragma unroll
    for (int i = 0; i < 64; ++i)
      v[i] = reg_load<T, NTM>(p + (i & 3) * geo.is[0] + ((i >> 2) & 3) * geo.is[1] + (i >> 4) * geo.is[2], loff);
  }
  reg_stages<T, kRegTile, PH, false>(v, s, st, ns, kinds, prm, lane, wave);
  {
    T *p = a + base + wave * geo.ow;
    // (a 32-bit offset of its own, so that the stores take a scalar base)
    uint32_t soff = loff;
    asm volatile("" : "+v"(soff));
#pragma unroll
    for (int i = 0; i < 64; ++i)
      reg_store<T, NTM>(p + (i & 3) * geo.os[0] + ((i >> 2) & 3) * geo.os[1] + (i >> 4) * geo.os[2], soff, v[i]);
  }
}

template <typename T, bool NTM>
__global__ __launch_bounds__(kRegThreads, sizeof(T) == 4 ? 5 : 3) void k_tile_reg(T *__restrict__ a, RegGeom geo,
                                                             const RegStage *__restrict__ st, int ns,
                                                             const uint32_t *__restrict__ kinds,
                                                             const T *__restrict__ prm) {
  __shared__ __align__(16) T s[RegShape<T>::lds];
  // Workgroups go to the 8 XCDs in turn.  Streaming from HBM (NTM: at least
  // 4^6 tiles), an XCD takes 64 consecutive tiles, whose low digits run over
  // consecutive addresses, so that its requests fall on fewer DRAM pages:
  // 16 qubits FP32 519 -> 504 ms, 15 qubits FP64 84.2 -> 81.7 ms; 32 to 256
  // tiles measured the same.  States inside the last-level cache lose a
  // little by it (13 qubits FP32 2.83 -> 2.87 ms) and keep the plain order.
  uint32_t t = blockIdx.x;
  if (NTM) t = (t & ~511u) + (t % 8) * 64 + (t / 8) % 64;
  reg_tile<T, NTM>(a, s, geo, t, st, ns, kinds, prm);
}

// A whole circuit of up to M qubits (6: one wave; 7: four) in registers, from
// |0...0> to the Z-ensemble probabilities: its program is one list of stages.
// Qubits fewer than 6 leave digits that no operation touches; only their
// component 0 is initialised and read.  What bounds it is one circuit's
// serial chain of members and redistributions: a circuit is one workgroup.
// 512 circuits of 2-7 qubits and 50-300 gates, memory noise after every gate,
// FP64: 8.2 ms one workgroup a circuit in LDS (an LDS round trip per gate and
// per qubit's noise, the widths one after another) -> 0.62 ms.
struct RegCirc {
  int32_t n, ns;
  int64_t st_off;   // first record word
  int64_t val_off;  // first value
  int64_t out_off;  // first probability
  double err;       // measurement polarisation retention
  // digits of the register slots, lanes and waves in the first and the last
  // stage's layout
  int32_t fr[3], fl[3], fw, lr[3], ll[3], lw;
};

template <int M>
struct RegCircShape {
  static constexpr int threads = M == 7 ? 256 : 64;
  static constexpr int phases = 2;
};

template <typename T, int M, bool SEQ>
__global__ __launch_bounds__(RegCircShape<M>::threads, 2) void k_circuit_reg(const RegCirc *__restrict__ circs,
                                                                             const uint32_t *__restrict__ recs,
                                                                             const T *__restrict__ prm,
                                                                             double *__restrict__ probs,
                                                                             uint64_t *__restrict__ stamps) {
  constexpr int PH = RegCircShape<M>::phases;
  constexpr int NT = RegCircShape<M>::threads;
  __shared__ __align__(16) T s[(1 << (2 * M)) / PH];
  const RegCirc c = circs[blockIdx.x];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = M == 7 ? __builtin_amdgcn_readfirstlane(tid >> 6) : 0;
  if (tid == 0) stamps[2 * blockIdx.x] = wall_clock64();
  const RegStage *st = reinterpret_cast<const RegStage *>(recs + c.st_off);
  // components of a digit with a value: I and Z of a qubit, 0 of the others
  auto ok = [&](int digit, int x) { return ((digit < c.n ? 9 : 1) >> x) & 1; };
  auto lanes_ok = [&](const int32_t *l, int32_t w) {
    return ok(l[0], lane & 3) && ok(l[1], (lane >> 2) & 3) && ok(l[2], lane >> 4) && (M != 7 || ok(w, wave));
  };
  T v[64];
  {
    const T amp = lanes_ok(c.fl, c.fw) ? (T)ldexp(1.0, -c.n) : T(0);
#pragma unroll
    for (int i = 0; i < 64; ++i)
      v[i] = ok(c.fr[0], i & 3) && ok(c.fr[1], (i >> 2) & 3) && ok(c.fr[2], i >> 4) ? amp : T(0);
  }
  reg_stages<T, M, PH, SEQ>(v, s, st, c.ns, reinterpret_cast<const uint32_t *>(st + c.ns), prm + c.val_off, lane,
                            wave);
  __syncthreads();  // the last redistribution has been read
  // Z ensemble: bit q of an index is the I / Z choice of digit q (qubit
  // n-1-q), which is the order of the outcomes too
  double *z = reinterpret_cast<double *>(s);
  if (lanes_ok(c.ll, c.lw)) {
    const int hi = ((lane & 3) ? 1 << c.ll[0] : 0) | ((lane & 12) ? 1 << c.ll[1] : 0) |
                   ((lane & 48) ? 1 << c.ll[2] : 0) | (M == 7 && wave ? 1 << c.lw : 0);
#pragma unroll
    for (int i = 0; i < 64; ++i)
      if ((i & 3) % 3 == 0 && ((i >> 2) & 3) % 3 == 0 && (i >> 4) % 3 == 0)
        if (ok(c.lr[0], i & 3) && ok(c.lr[1], (i >> 2) & 3) && ok(c.lr[2], i >> 4))
          z[hi | ((i & 3) ? 1 << c.lr[0] : 0) | ((i & 12) ? 1 << c.lr[1] : 0) | ((i & 48) ? 1 << c.lr[2] : 0)] =
              (double)v[i];
  }
  __syncthreads();
  const int nv = 1 << c.n;
  for (int q = 0; q < c.n; ++q) {  // butterfly on bit q: (u, w) -> (u + e w, u - e w)
    for (int x = tid; x < nv / 2; x += NT) {
      const int lo = x & ((1 << q) - 1);
      const int b = ((x >> q) << (q + 1)) | lo;
      const double u = z[b], w = z[b | (1 << q)];
      z[b] = u + c.err * w;
      z[b | (1 << q)] = u - c.err * w;
    }
    __syncthreads();
  }
  for (int x = tid; x < nv; x += NT) probs[c.out_off + x] = z[x];
  if (tid == 0) stamps[2 * blockIdx.x + 1] = wall_clock64();
}

// A run of operations on a whole state of up to 6 qubits: one wave, loaded
// and stored in the layouts of the first and the last stage.  Latency bound.
struct RegWhole {
  int32_t n, ns;
  int32_t fr[3], fl[3], lr[3], ll[3];
};

template <typename T>
__global__ __launch_bounds__(64, 2) void k_state_reg(T *__restrict__ a, RegWhole w, const RegStage *__restrict__ st,
                                                     const uint32_t *__restrict__ kinds,
                                                     const T *__restrict__ prm) {
  constexpr int M = 6, PH = RegCircShape<M>::phases;
  __shared__ __align__(16) T s[(1 << (2 * M)) / PH];
  const int lane = threadIdx.x;
  // digits from n on do not exist: only their component 0 is in the state
  auto at = [&](int digit, int x, bool &in) -> uint32_t {
    in = in && (digit < w.n || x == 0);
    return (uint32_t)x << (2 * digit);
  };
  T v[64];
  {
    bool lin = true;
    const uint32_t lo = at(w.fl[0], lane & 3, lin) + at(w.fl[1], (lane >> 2) & 3, lin) + at(w.fl[2], lane >> 4, lin);
#pragma unroll
    for (int i = 0; i < 64; ++i) {
      bool in = lin;
      const uint32_t o = lo + at(w.fr[0], i & 3, in) + at(w.fr[1], (i >> 2) & 3, in) + at(w.fr[2], i >> 4, in);
      v[i] = in ? a[o] : T(0);
    }
  }
  reg_stages<T, M, PH, false>(v, s, st, w.ns, kinds, prm, lane, 0);
  {
    bool lin = true;
    const uint32_t lo = at(w.ll[0], lane & 3, lin) + at(w.ll[1], (lane >> 2) & 3, lin) + at(w.ll[2], lane >> 4, lin);
#pragma unroll
    for (int i = 0; i < 64; ++i) {
      bool in = lin;
      const uint32_t o = lo + at(w.lr[0], i & 3, in) + at(w.lr[1], (i >> 2) & 3, in) + at(w.lr[2], i >> 4, in);
      if (in) a[o] = v[i];
    }
  }
}

// HBM strides of a tile's load and store layouts.
inline RegGeom reg_geom(const RegPlan &rp, const int *tpos, const int *rpos, int nr) {
  RegGeom geo;
  memset(&geo, 0, sizeof(geo));
  geo.nr = nr;
  for (int j = 0; j < nr; ++j) geo.rpos[j] = rpos[j];
  geo.tiles = 1u << (2 * nr);
  for (int j = 0; j < 3; ++j) {
    geo.is[j] = pow4(tpos[rp.first.r[j]]);
    geo.os[j] = pow4(tpos[rp.last.r[j]]);
  }
  geo.iw = pow4(tpos[rp.first.w]);
  geo.ow = pow4(tpos[rp.last.w]);
  return geo;
}
