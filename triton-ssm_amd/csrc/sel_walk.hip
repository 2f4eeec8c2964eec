// Mamba-1 selective scan in one sweep over time, for problems whose (batch,
// channel, state) lanes fill the chip within a short sequence: each lane owns one
// state h[b, d, n] and walks the whole sequence, so nothing is computed twice and
// no chunk state or output makes a second trip through memory.
//
//   h' = h + (ab - 1)(h + B x / a)  (ZOH)  or  ab h + B dt x  (Euler),
//   ab = exp2(dt a log2 e);   y_t[d] = sum_n C_t[n] h[d, n] + D[d] x_t[d]
//
// (discretize_kernel.py:16-57 followed by ssm_scan.py:239-264, summed over n;
// the update is the three-pass scan's, sel_update in selective_dev.h.)
//
// A workgroup takes 16 consecutive channels of one batch and all N states:
// wave w the states 4 w .. 4 w + 3, lane 16 j + c state 4 w + j of channel c.
// Steps go in tiles of TS: the tile's x, B, C and dt are staged in LDS
// transposed ([channel or state][step]), so a lane reads four steps at once;
// the next tile's loads are in flight meanwhile.  The products C h of four
// steps are summed over a wave's four states by lane swaps (3 swaps and 3 adds
// give lane j the sum of step j), the waves' sums meet in LDS and leave with
// the skip term, once per tile.
//
// What bounds it: vector issue, and below two waves a SIMD the latency of one
// wave's instructions: 37 ns a step with one wave a SIMD, 51 with two, 97 with four
// (N = 16), so it wins where the passes' 25 us of launches and second trips weigh
// more than its steps.  y is rounded once: error against float64 in bf16 1.7e-3,
// with the passes 2.1e-3.
#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "common.h"
#include "selective.h"

namespace tssm {
namespace {

struct SelWalkArgs {
  const void* x;
  const float* dt;
  const float* A_log;
  const void* B;
  const void* C;
  const float* D;
  const float* h0;
  void* y;
  float* h_last;
  int64_t L, Dc;
  int64_t sx_b, sx_l, sdt_b, sdt_l, sdt_d, sB_b, sB_l, sC_b, sC_l, sy_b, sy_l;
  uint32_t groups, total, per_xcd;  // channel groups of a batch; workgroups; of an XCD
};

constexpr int kSwCh = 16;  // channels of a workgroup

// Four steps' values of one column, as the lane that stages them loads them.
// Offsets are bytes from the tile's first row.
template <typename T>
struct SwQuad {
  uint32_t off[4];
  float v[4];
  __device__ inline void rows(int t, int64_t stride, int col, int last) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      off[i] = ((uint32_t)min(t + i, last) * (uint32_t)stride + (uint32_t)col) *
               (uint32_t)sizeof(T);
  }
  __device__ inline void load(const T* base) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      v[i] = ldf(reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + off[i]));
  }
  // steps t .. t + 3 to LDS, zero from `n` on (by mask: the compiler would put
  // the load behind a branch for a select)
  __device__ inline void store(float* s, int t, int n) const {
    f32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = __uint_as_float(__float_as_uint(v[i]) & (t + i < n ? ~0u : 0u));
    *reinterpret_cast<f32x4*>(s + t) = o;
  }
};

// Sums over the four 16-lane rows of p[0..3]: row j gets the sum of p[j].
__device__ inline float row_sums(const float* p) {
  const auto s32 = [](float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                    false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  };
  const float u = s32(p[0], p[2]), v = s32(p[1], p[3]);
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(u), __float_as_uint(v), false,
                                                  false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <typename T, int DISC, int NW, bool DTS, bool TAU, bool HAS_D>
__global__ __launch_bounds__(64 * NW) void sel_walk_kernel(SelWalkArgs a) {
  static_assert(!TAU || DTS, "timestamps only when shared by the channels");
  constexpr int N = 4 * NW, TH = 64 * NW, TS = NW <= 4 ? 64 : 32, ROW = TS + 4;
  constexpr int QX = kSwCh * TS / 4, KX = (QX + TH - 1) / TH;  // quads of x (and dt)
  constexpr int QN = N * TS / 4, KN = (QN + TH - 1) / TH;      // quads of B and of C
  __shared__ __align__(16) float sX[kSwCh][ROW], sB[N][ROW], sC[N][ROW];
  __shared__ __align__(16) float sDt[DTS ? 1 : kSwCh][ROW];
  __shared__ __align__(16) float sY[NW][kSwCh][ROW];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, j = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t unit = (blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3);
  if (unit >= a.total) return;
  const uint32_t b = unit / a.groups;
  const int64_t d0 = (int64_t)(unit - b * a.groups) * kSwCh;
  const int nd = (int)(a.Dc - d0 < kSwCh ? a.Dc - d0 : kSwCh);  // channels that exist
  const T* xb = static_cast<const T*>(a.x) + b * a.sx_b + d0;
  const T* Bb = static_cast<const T*>(a.B) + b * a.sB_b;
  const T* Cb = static_cast<const T*>(a.C) + b * a.sC_b;
  const float* db = a.dt + b * a.sdt_b + (DTS ? 0 : d0 * a.sdt_d);
  T* yb = static_cast<T*>(a.y) + b * a.sy_b + d0;

  SwQuad<T> qx[KX], qb[KN], qc[KN];
  SwQuad<float> qd[DTS ? 1 : KX];
  // quad k of this thread: column and first step (threads past the last quad
  // repeat an earlier one and store nothing)
  auto xcol = [&](int k) { return (tid + TH * k) % QX % kSwCh; };
  auto xt = [&](int k) { return (tid + TH * k) % QX / kSwCh * 4; };
  auto ncol = [&](int k) { return (tid + TH * k) % QN % N; };
  auto nt = [&](int k) { return (tid + TH * k) % QN / N * 4; };
  auto rows = [&](int last) {
#pragma unroll
    for (int k = 0; k < KX; ++k) {
      const int col = min(xcol(k), nd - 1);
      qx[k].rows(xt(k), a.sx_l, col, last);
      if constexpr (!DTS) {
        qd[k].rows(xt(k), a.sdt_l, 0, last);
#pragma unroll
        for (int i = 0; i < 4; ++i) qd[k].off[i] += (uint32_t)col * (uint32_t)a.sdt_d * 4u;
      }
    }
#pragma unroll
    for (int k = 0; k < KN; ++k) {
      qb[k].rows(nt(k), a.sB_l, ncol(k), last);
      qc[k].rows(nt(k), a.sC_l, ncol(k), last);
    }
  };
  float dts = 0.0f, dts_prev = 0.0f;
  auto load = [&](int64_t t0) {
    const int64_t tb = t0 < a.L ? t0 : a.L - 1;
    if (tb + TS > a.L) rows((int)(a.L - 1 - tb));
#pragma unroll
    for (int k = 0; k < KX; ++k) qx[k].load(xb + tb * a.sx_l);
    if constexpr (DTS) {
      const int64_t t = tb + (tid & (TS - 1)) < a.L ? tb + (tid & (TS - 1)) : a.L - 1;
      dts = db[t * a.sdt_l];
      if constexpr (TAU) dts_prev = db[(t > 0 ? t - 1 : 0) * a.sdt_l];
    } else {
#pragma unroll
      for (int k = 0; k < KX; ++k) qd[k].load(db + tb * a.sdt_l);
    }
#pragma unroll
    for (int k = 0; k < KN; ++k) qb[k].load(Bb + tb * a.sB_l);
#pragma unroll
    for (int k = 0; k < KN; ++k) qc[k].load(Cb + tb * a.sC_l);
  };
  // the loaded tile, whose first step is t0, to LDS (zero past the end)
  auto stage = [&](int64_t t0) {
    const int n = (int)(a.L - t0 < TS ? (a.L > t0 ? a.L - t0 : 0) : TS);
#pragma unroll
    for (int k = 0; k < KX; ++k)
      if (KX * TH == QX || tid + TH * k < QX) qx[k].store(sX[xcol(k)], xt(k), n);
    if constexpr (DTS) {
      float v = dts;
      if constexpr (TAU) v -= t0 + tid > 0 ? dts_prev : 0.0f;
      if (tid < TS) sDt[0][tid] = tid < n ? v : 0.0f;
    } else {
#pragma unroll
      for (int k = 0; k < KX; ++k)
        if (KX * TH == QX || tid + TH * k < QX) qd[k].store(sDt[xcol(k)], xt(k), n);
    }
#pragma unroll
    for (int k = 0; k < KN; ++k)
      if (KN * TH == QN || tid + TH * k < QN) {
        qb[k].store(sB[ncol(k)], nt(k), n);
        qc[k].store(sC[ncol(k)], nt(k), n);
      }
  };

  rows(TS - 1);
  load(0);
  const int64_t dl = d0 + min(c, nd - 1);  // lanes past Dc compute its last channel
  const int nl = 4 * w + j;
  const float al = a.A_log[dl * N + nl] * kLog2e;
  const float a2 = -__builtin_amdgcn_exp2f(al) * kLog2e, ia = -__builtin_amdgcn_exp2f(-al);
  const int64_t hid = (b * a.Dc + dl) * N + nl;
  float h = a.h0 ? a.h0[hid] : 0.0f;
  float Dd[HAS_D ? KX : 1];
  if constexpr (HAS_D) {
#pragma unroll
    for (int k = 0; k < KX; ++k) Dd[k] = a.D[d0 + min(xcol(k), nd - 1)];
  }
  const float *px = sX[c], *pb = sB[nl], *pc = sC[nl], *pd = DTS ? sDt[0] : sDt[DTS ? 0 : c];
  float* py = &sY[w][c][j];
  for (int64_t t0 = 0; t0 < a.L; t0 += TS) {
    stage(t0);
    float xs[KX][4];
#pragma unroll
    for (int k = 0; k < KX; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i) xs[k][i] = qx[k].v[i];
    __syncthreads();
    load(t0 + TS);
    const int left = (int)(a.L - t0 < TS ? a.L - t0 : TS);
    const int ng = (left + 3) / 4;  // groups of four steps
    struct Four {
      f32x4 x, B, C, dt;
    };
    auto read = [&](int k) {
      const int o = 4 * min(k, TS / 4 - 1);
      return Four{*reinterpret_cast<const f32x4*>(px + o), *reinterpret_cast<const f32x4*>(pb + o),
                  *reinterpret_cast<const f32x4*>(pc + o), *reinterpret_cast<const f32x4*>(pd + o)};
    };
    // What a group needs that does not depend on h, formed one group ahead so
    // that the wave always has independent instructions between the links of
    // the chain through h.
    struct Pre {
      float e[4], u[4], C[4];
    };
    auto ahead = [&](const Four& q, Pre& o, int i) {
      const float ab = __builtin_amdgcn_exp2f(q.dt[i] * a2);
      if constexpr (DISC == TSSM_DISC_ZOH) {
        o.e[i] = ab - 1.0f;
        o.u[i] = q.B[i] * q.x[i];
      } else {
        o.e[i] = ab;
        o.u[i] = q.B[i] * (q.dt[i] * q.x[i]);
      }
      o.C[i] = q.C[i];
    };
    auto step = [&](const Pre& o, int i) {
      if constexpr (DISC == TSSM_DISC_ZOH) {
        const float hb = __builtin_fmaf(ia, o.u[i], h);
        h = __builtin_fmaf(o.e[i], hb, h);
      } else {
        h = __builtin_fmaf(o.e[i], h, o.u[i]);
      }
      return o.C[i] * h;
    };
    Four raw = read(0);
    Pre pre;
#pragma unroll
    for (int i = 0; i < 4; ++i) ahead(raw, pre, i);
    raw = read(1);
    // 16 steps at a time.  Past the end e is 0 or 1 and u 0, which keeps a finite
    // h; the last tile keeps h by a select, so that an infinite one stays too.
    auto walk = [&](auto last) {
      for (int kb = 0; kb < ng; kb += 4) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
          const int k = kb + kk;
          const Four nxt = read(k + 2);
          Pre po;
          float pr[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float h0 = h;
            pr[i] = step(pre, i);
            if constexpr (decltype(last)::value) h = 4 * k + i < left ? h : h0;
            ahead(raw, po, i);
          }
          py[4 * k] = row_sums(pr);
          pre = po;
          raw = nxt;
        }
      }
    };
    if (left < TS)
      walk(std::true_type());
    else
      walk(std::false_type());
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KX; ++k) {
      if (KX * TH != QX && tid + TH * k >= QX) continue;
      const int col = xcol(k), t = xt(k);
      f32x4 s = *reinterpret_cast<const f32x4*>(&sY[0][col][t]);
#pragma unroll
      for (int v = 1; v < NW; ++v) s += *reinterpret_cast<const f32x4*>(&sY[v][col][t]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float yv = HAS_D ? __builtin_fmaf(Dd[HAS_D ? k : 0], xs[k][i], s[i]) : s[i];
        if (col < nd && t + i < left) stf(yb + (t0 + t + i) * a.sy_l + col, yv);
      }
    }
  }
  if (a.h_last && c < nd) a.h_last[hid] = h;
}

template <typename T, int DISC, int NW, bool DTS, bool TAU>
int launch_d(const SelWalkArgs& a, hipStream_t s) {
  const dim3 grid(8 * a.per_xcd), block(64 * NW);
  if (a.D)
    hipLaunchKernelGGL((sel_walk_kernel<T, DISC, NW, DTS, TAU, true>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((sel_walk_kernel<T, DISC, NW, DTS, TAU, false>), grid, block, 0, s, a);
  return launch_status();
}
template <typename T, int DISC, int NW>
int launch_dt(bool dts, bool tau, const SelWalkArgs& a, hipStream_t s) {
  if (!dts) return launch_d<T, DISC, NW, false, false>(a, s);
  return tau ? launch_d<T, DISC, NW, true, true>(a, s) : launch_d<T, DISC, NW, true, false>(a, s);
}
template <typename T, int DISC>
int launch_n(int64_t N, bool dts, bool tau, const SelWalkArgs& a, hipStream_t s) {
  return N == 8 ? launch_dt<T, DISC, 2>(dts, tau, a, s) : launch_dt<T, DISC, 4>(dts, tau, a, s);
}
template <typename T>
int launch_t(int disc, int64_t N, bool dts, bool tau, const SelWalkArgs& a, hipStream_t s) {
  return disc == TSSM_DISC_ZOH ? launch_n<T, TSSM_DISC_ZOH>(N, dts, tau, a, s)
                               : launch_n<T, TSSM_DISC_EULER>(N, dts, tau, a, s);
}

}  // namespace

// The lines below are fits to measured times (us, fp32; the passes are slower in
// bf16, the walk is not): a step of the walk costs by how many of its workgroups a
// CU holds, the passes by states updated.
//   B=16 D=256 N=16 (1 workgroup a CU), passes -> walk: L=300 34.0 -> 15.3, 640
//   45.1 -> 26.5, 1000 45.3 -> 40.9, 1600 66.5 -> 61.0; bf16 39.8 -> 15.2, 54.2 ->
//   26.6, 55.7 -> 40.0, 75.6 -> 60.6, and at L=2000 85.6 -> 81.6.
//   B=16 D=128 N=16 (half of the CUs): L=640 39.8 -> 25.9, 1000 41.1 -> 40.1, 1600
//   43.9 -> 60.2.  B=16 D=512 N=16 (2): L=1000 70.2 -> 53.6.  B=16 D=1024 (4): L=300
//   63.9 -> 32.2.  N=8, B=16 D=256: L=300 24.0 -> 15.1, 800 30.3 -> 34.0.
// N = 32 has no passes; against the one-launch scan the walk measured 0.7 to 1.5x
// without a clear line, so it is not offered there.
bool sel_walk_ok(int64_t nbatch, int64_t L, int64_t Dc, int64_t N, bool dt_shared,
                 int64_t sx_l, int64_t sdt_l, int64_t sdt_d, int64_t sB_l, int64_t sC_l) {
  if (!(N == 8 || N == 16)) return false;
  const int64_t groups = nbatch * cdiv64(Dc, kSwCh);
  // byte offsets within a tile in 32 bits
  const int64_t far = (sx_l | sdt_l | sB_l | sC_l | (dt_shared ? 0 : sdt_d * kSwCh)) >> 22;
  if (groups >= (int64_t)1 << 26 || far != 0) return false;
  const double rounds = (double)cdiv64(groups, 256);
  const double step = N == 16 ? fmax(0.037, 0.0255 * rounds)
                              : (rounds == 1 ? 0.0375 : fmax(0.052, 0.0145 * rounds));
  const double updates = 1e-6 * (double)nbatch * (double)L * (double)(Dc * N);
  const double passes = N == 16 ? 26.0 + 0.336 * updates : 18.0 + 0.38 * updates;
  return 4.0 + step * (double)L < passes;
}

int sel_walk_launch(int dtype, int disc, bool dt_shared, bool tau, const SelPtrs& p,
                    int64_t nbatch, int64_t L, int64_t Dc, int64_t N, int64_t sx_b, int64_t sx_l,
                    int64_t sdt_b, int64_t sdt_l, int64_t sdt_d, int64_t sB_b, int64_t sB_l,
                    int64_t sC_b, int64_t sC_l, int64_t sy_b, int64_t sy_l, hipStream_t s) {
  SelWalkArgs a;
  a.x = p.x; a.dt = p.dt; a.A_log = p.A_log; a.B = p.B; a.C = p.C; a.D = p.D; a.h0 = p.h0;
  a.y = p.y; a.h_last = p.h_last;
  a.L = L; a.Dc = Dc;
  a.sx_b = sx_b; a.sx_l = sx_l; a.sdt_b = sdt_b; a.sdt_l = sdt_l; a.sdt_d = sdt_d;
  a.sB_b = sB_b; a.sB_l = sB_l; a.sC_b = sC_b; a.sC_l = sC_l; a.sy_b = sy_b; a.sy_l = sy_l;
  a.groups = (uint32_t)cdiv64(Dc, kSwCh);
  a.total = (uint32_t)(nbatch * a.groups);
  a.per_xcd = (a.total + 7) / 8;
  switch (dtype) {
    case TSSM_BF16: return launch_t<bf16_t>(disc, N, dt_shared, tau, a, s);
    default: return launch_t<float>(disc, N, dt_shared, tau, a, s);
  }
}

}  // namespace tssm
