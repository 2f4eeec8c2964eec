// Device pieces shared by the SSD walks (ssd_walk.hip: fp32 products;
// ssd_walk_bf16.hip: bf16 products): a wave's work unit, its staged operands
// and the state in registers.
#pragma once

#include "ssd_dev.h"

#include <type_traits>

namespace tssm {
namespace {

constexpr double kWalkFloor = -4096; // log2 decay of one step, clamped: 2^-4096 is 0 either way

// Lane i of each 16-lane row gets lane i - n (row_shr), 0.0 before the row.
template <int CTRL>
__device__ inline double dpp_shr_f64(double v) {
  const u32x2 w = __builtin_bit_cast(u32x2, v);
  u32x2 r;
  r[0] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w[0], CTRL, 0xf, 0xf, true);
  r[1] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w[1], CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, r);
}

// What a wave works on.  Waves of one (batch, segment) share the 128-byte
// lines of dt, so with enough (batch, segment) groups their workgroups are
// numbered onto one XCD (blockIdx mod 8).
struct WalkUnit {
  uint32_t b, h, row, seg;
  int p0;
  bool on;
};
__device__ inline WalkUnit walk_unit(const SsdArgs& a, uint32_t npg, uint32_t nseg, int pw,
                                     bool by_xcd) {
  const uint32_t wv = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t per = a.H * npg;  // waves per (batch, segment)
  const uint32_t groups = a.rows / a.H * nseg;
  uint32_t g, u;
  if (by_xcd) {
    const uint32_t wgs = (per + 3) / 4, idx = blockIdx.x >> 3;
    g = (idx / wgs) * 8 + (blockIdx.x & 7);
    u = (idx % wgs) * 4 + wv;
  } else {
    const uint32_t w = blockIdx.x * 4 + wv;
    g = w / per;
    u = w - g * per;
  }
  WalkUnit o;
  o.on = g < groups && u < per;
  o.b = g / nseg;
  o.seg = g - o.b * nseg;
  o.h = u / npg;
  o.p0 = (int)(u - o.h * npg) * pw;
  o.row = o.b * a.H + o.h;
  return o;
}

typedef f32x4 mfma_acc;
__device__ inline mfma_acc mfma4(float a, float b, mfma_acc c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Workgroups of 4 waves for `groups` (batch, segment) pairs of `per` waves.
inline dim3 walk_grid(int64_t groups, int64_t per, int* by_xcd) {
  // an uneven split over the XCDs costs more than sharing dt's lines gains
  *by_xcd = groups % 8 == 0 || groups >= 64;
  return *by_xcd ? dim3((unsigned)(8 * cdiv64(groups, 8) * cdiv64(per, 4)))
                 : dim3((unsigned)cdiv64(groups * per, 4));
}

// Orders a wave's LDS writes before its other lanes' reads (the LDS itself
// runs a wave's accesses in order: no instruction).
__device__ inline void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One staged operand: Q rows (steps) of 16 WB columns.  In LDS a row takes
// 16 bytes more than its columns, so that the rows c of a vector read and the
// rows 4 j + r of an element read fall on different banks.
template <typename T, int WB, bool VEC, int Q>
struct WalkTile {
  static constexpr int E = (int)sizeof(T), W = 16 * WB, kStride = W * E + 16;
  static constexpr int kBytes = Q * kStride;
  static constexpr int VE = VEC ? 16 / E : 1;  // elements of one access
  static constexpr int NP = W / VE;            // accesses of a row
  static constexpr int K = (Q * NP + 63) / 64;
  typedef std::conditional_t<VEC, uint32_t, uint64_t> off_t;
  typedef std::conditional_t<VEC, u32x4, uint32_t> raw_t;
  struct Regs {
    raw_t v[K];
  };
  off_t off[K];
  int lim;  // columns that exist (the others are zero)
  static __device__ inline int row_of(int lane, int k) { return (lane + 64 * k) / NP % Q; }
  static __device__ inline int col_of(int lane, int k) { return (lane + 64 * k) % NP * VE; }
  // Byte offsets from the block's first row; rows past `last` re-read it.
  __device__ inline void rows(int lane, int64_t stride, int last) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int r = row_of(lane, k), c = col_of(lane, k);
      off[k] = (off_t)(r < last ? r : last) * (off_t)stride + (off_t)((c < lim ? c : 0) * E);
    }
  }
  __device__ inline void load(Regs& g, const char* base) const {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if constexpr (VEC) g.v[k] = *reinterpret_cast<const u32x4*>(base + off[k]);
      else if constexpr (E == 4) g.v[k] = *reinterpret_cast<const uint32_t*>(base + off[k]);
      else g.v[k] = *reinterpret_cast<const uint16_t*>(base + off[k]);
    }
  }
  // Columns past lim and rows past `n` are stored as zero.
  __device__ inline void store(Regs& g, char* lds, int lane, bool edge, int n) const {
    if (edge) {
#pragma unroll
      for (int k = 0; k < K; ++k)
        g.v[k] &= row_of(lane, k) < n && col_of(lane, k) < lim ? ~0u : 0u;
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      char* p = lds + row_of(lane, k) * kStride + col_of(lane, k) * E;
      if constexpr (VEC) *reinterpret_cast<u32x4*>(p) = g.v[k];
      else if constexpr (E == 4) *reinterpret_cast<uint32_t*>(p) = g.v[k];
      else *reinterpret_cast<uint16_t*>(p) = (uint16_t)g.v[k];
    }
  }
  static __device__ inline float get(const char* lds, int row, int col) {
    return ldf(reinterpret_cast<const T*>(lds + row * kStride + col * E));
  }
  static __device__ inline void get4(const char* lds, int row, int col, float* o) {
    ld_lanes<T, 4>(reinterpret_cast<const T*>(lds + row * kStride + col * E), o);
  }
};

// The operands of a wave: a block in LDS, the next one's loads in flight.
template <typename T, int PB, int NB, bool VEC, bool OUT, int Q>
struct WalkIn {
  typedef WalkTile<T, PB, VEC, Q> TX;
  typedef WalkTile<T, NB, VEC, Q> TN;
  static constexpr int kX = 0, kB = TX::kBytes, kC = kB + TN::kBytes;
  static constexpr int kBytes = OUT ? kC + TN::kBytes : kC;
  // the registers of one block's loads
  struct Regs {
    typename TX::Regs x;
    typename TN::Regs B, C;
    float dt;
  };
  TX x;
  TN B, C;
  const char *px, *pB, *pC, *pd;  // (batch, head) bases
  int64_t L, sx, sB, sC, sdt;     // row strides in bytes
  typename TX::off_t od;
  bool edge;                      // some columns do not exist
  int lane;
  __device__ inline void rows(int last) {
    const int c = lane & (Q - 1);
    x.rows(lane, sx, last);
    B.rows(lane, sB, last);
    if constexpr (OUT) C.rows(lane, sC, last);
    od = (typename TX::off_t)(c < last ? c : last) * (typename TX::off_t)sdt;
  }
  __device__ inline void init(const SsdArgs& a, const WalkUnit& u, int N, int ln) {
    lane = ln;
    px = reinterpret_cast<const char*>(reinterpret_cast<const T*>(a.x) + u.b * a.sx_b +
                                       u.h * a.sx_h + u.p0);
    pB = reinterpret_cast<const char*>(reinterpret_cast<const T*>(a.B) + u.b * a.sB_b +
                                       u.h * a.sB_h);
    pC = reinterpret_cast<const char*>(reinterpret_cast<const T*>(a.C) + u.b * a.sC_b +
                                       u.h * a.sC_h);
    pd = reinterpret_cast<const char*>(a.dt + u.b * a.sdt_b + u.h * a.sdt_h);
    L = a.L;
    sx = a.sx_l * (int64_t)sizeof(T);
    sB = a.sB_l * (int64_t)sizeof(T);
    sC = a.sC_l * (int64_t)sizeof(T);
    sdt = a.sdt_l * 4;
    x.lim = (int)a.P - u.p0 < TX::W ? (int)a.P - u.p0 : TX::W;
    B.lim = C.lim = N;
    edge = x.lim < TX::W || N < TN::W;
    rows(Q - 1);
  }
  // First row of the block at t0 (the last row for a block past the end);
  // keeps the offsets inside the sequence.
  __device__ inline int64_t row0(int64_t t0) {
    const int64_t tb = t0 < L ? t0 : L - 1;
    if (tb + Q > L) rows((int)(L - 1 - tb));
    return tb;
  }
  __device__ inline void load(Regs& g, int64_t t0) {
    const int64_t tb = row0(t0);
    g.dt = *reinterpret_cast<const float*>(pd + tb * sdt + od);
    x.load(g.x, px + tb * sx);
    B.load(g.B, pB + tb * sB);
    if constexpr (OUT) C.load(g.C, pC + tb * sC);
  }
  // The loaded block, whose first step is t0, into LDS; returns the dt of step
  // t0 + lane % Q (0 past the end).
  __device__ inline float stage(Regs& g, char* lds, int64_t t0) const {
    const int64_t left = L - t0;
    const int n = left < Q ? (left > 0 ? (int)left : 0) : Q;
    const bool e = edge || n < Q;
    wave_lds_order();  // after the reads of the block before
    x.store(g.x, lds + kX, lane, e, n);
    B.store(g.B, lds + kB, lane, e, n);
    if constexpr (OUT) C.store(g.C, lds + kC, lane, e, n);
    wave_lds_order();
    return (lane & (Q - 1)) < n ? g.dt : 0.0f;
  }
};

// H^T[i][q] reg r  <->  S[p][n], n = 16 i + 4 j + r, p = p0 + 16 q + c.
template <int PB, int NB>
__device__ inline void walk_put(float* S, const mfma_acc (&H)[NB][PB], int p0, int P, int N, int c,
                                int j) {
#pragma unroll
  for (int q = 0; q < PB; ++q) {
    const int p = p0 + 16 * q + c;
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int n0 = 16 * i + 4 * j;
      if (p < P && n0 < N) {
#pragma unroll
        for (int r = 0; r < 4; ++r) S[(int64_t)p * N + n0 + r] = H[i][q][r];
      }
    }
  }
}

// The inverse: a wave's slice of a [P][N] state (zero if S is null).  Loads
// first (lanes past P or N re-read the slice's start), zeroes by mask: the
// compiler turns a select on a loaded value into a branch around the load,
// which then waits for it alone.
template <int PB, int NB>
__device__ inline void walk_get(mfma_acc (&H)[NB][PB], const float* S, int p0, int P, int N, int c,
                                int j) {
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int q = 0; q < PB; ++q) H[i][q] = mfma_acc{0.0f, 0.0f, 0.0f, 0.0f};
  if (!S) return;
#pragma unroll
  for (int q = 0; q < PB; ++q)
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int p = p0 + 16 * q + c, n0 = 16 * i + 4 * j;
      const float* hp = S + (int64_t)(p < P ? p : 0) * N + (n0 < N ? n0 : 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) H[i][q][r] = hp[r];
    }
#pragma unroll
  for (int q = 0; q < PB; ++q)
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const uint32_t m = p0 + 16 * q + c < P && 16 * i + 4 * j < N ? ~0u : 0u;
#pragma unroll
      for (int r = 0; r < 4; ++r) H[i][q][r] = __uint_as_float(__float_as_uint(H[i][q][r]) & m);
    }
}

}  // namespace
}  // namespace tssm
