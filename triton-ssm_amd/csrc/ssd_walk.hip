// SSD selective scan with fp32 matrix products, for every operand form the
// bf16 kernels of ssd.hip and ssd_walk_bf16.hip do not take (fp32 and fp16,
// bf16 at other head dims and state sizes, any alignment).
//
// One wave owns (row, 16 PB channels, time segment) and walks its segment in
// 16-step blocks with its slice of the state in registers.  With cum_t the
// inclusive sum of log2 decay over a block and coef_s the input coefficient:
//   G[s][t]   = B_s . C_t
//   M[s][t]   = G[s][t] 2^(cum_t - cum_s) coef_s           (s <= t, else 0)
//   Y^T[p][t] = 2^cum_t sum_n H[p][n] C_t[n] + sum_s x_s[p] M[s][t]
//   H^T[n][p] = 2^cum_e H^T[n][p] + sum_s 2^(cum_e - cum_s) coef_s B_s[n] x_s[p]
// all on v_mfma_f32_16x16x4_f32 (fp32 products and sums, no operand split).
// Its operands take one value per lane, lane l = 16 j + c holding row or
// column c at k = j, and its result holds rows 4 j + r of column c: a result
// is the next product's operand where that product runs over k = 4 j + r.  G
// feeds the x product and H^T feeds the C product that way, with no data moved
// between lanes.  x, B and C are staged through LDS (a wave's own region, one
// block; the next one's loads are in flight meanwhile): loads cover whole rows
// in 16-byte pieces, and the reads take B both by step (G: lane 16 j + c row c)
// and by state column (the update: column 16 i + c).  Operands loaded straight from memory in their lane order, with
// neighbouring lanes on different rows, cost the first-level cache ~1000
// accesses a block instead of ~160, and twice the waves then ran slower (75
// against 66 us); two blocks in LDS leave room for one wave a SIMD (105
// against 79 us at B=2 L=8000 H=16).
//
// The log2 decays are summed in fp64: within a block they may reach hundreds
// while the differences that matter are near zero, and an fp32 sum would put
// 1e-5 of error on those weights (y of the fp32 layer with P = N = 64 stays
// within 1e-7 of float64, as the step-by-step recurrence did).
//
// What bounds it: the matrix unit, then the vector instructions around it.  A
// 16-step block takes 4 NB (1 + 2 PB) + 4 PB products of 32 cycles (88 at N = 64
// and 32 channels); at one wave a SIMD these are 45% of the block's cycles and
// nothing overlaps them, at two 60%.  fp32 B=2 L=4000 H=16 P=N=64: 335 -> 67 us
// (passes 16 + 7 + 44) against the step-by-step passes this replaced, whose
// lanes each carried N states; B=8 L=4096 H=16: 608 -> 184 us; fp16 B=8 L=2048
// H=24 P=64 N=32: 385 -> 88 us; B=1 L=16 H=1 (launch-bound): 29.7 -> 24.5 us.
//
// Segments: pass 1 (ssd_walk_state_kernel) forms the end state and the decay
// of each segment but the last, last block first, stopping where the decay
// has underflowed to exactly zero; ssd_walk_prefix_kernel turns them into
// entry states; ssd_walk_out_kernel writes the outputs.  One segment takes the last
// kernel alone.
#include "ssd_walk_dev.h"

namespace tssm {
namespace {

constexpr int kWalkQ = 16;  // steps per block

// The step scalars of one block.  Lane 16 j + c: cum, coef of step c; cs, cf
// those of steps 4 j + r; cum_e the sum over the block (uniform).
struct WalkScalars {
  double cum, cum_e, cs[4];
  float cf[4];
};
__device__ inline WalkScalars walk_scalars(float d, float a2, double a2d, bool zoh, int j) {
  WalkScalars o;
  const float y = d * a2;
  const float coef = zoh ? phi1_from_exp(y * 0.6931471805599453f, exp2_fast(y)) * d : d;
  double l = (double)d * a2d;
  l = l < kWalkFloor ? kWalkFloor : l;
  l += dpp_shr_f64<0x111>(l);
  l += dpp_shr_f64<0x112>(l);
  l += dpp_shr_f64<0x114>(l);
  l += dpp_shr_f64<0x118>(l);
  o.cum = l;
  const u32x2 w = __builtin_bit_cast(u32x2, l);
  u32x2 e;
  e[0] = (uint32_t)__builtin_amdgcn_readlane((int)w[0], 15);
  e[1] = (uint32_t)__builtin_amdgcn_readlane((int)w[1], 15);
  o.cum_e = __builtin_bit_cast(double, e);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int src = 4 * (4 * j + r);
    u32x2 s;
    s[0] = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)w[0]);
    s[1] = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)w[1]);
    o.cs[r] = __builtin_bit_cast(double, s);
    o.cf[r] = __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(coef)));
  }
  return o;
}

// H^T += sum_s w_s B_s x_s^T over one block, w[r] the weight of step 4 j + r,
// xv its channels 16 q + c.
template <typename In, int PB, int NB>
__device__ inline void walk_update(mfma_acc (&H)[NB][PB], const char* lds, const float (&xv)[4][PB],
                                   const float* w, int c, int j) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const float wb = w[r] * In::TN::get(lds + In::kB, 4 * j + r, 16 * i + c);
#pragma unroll
      for (int q = 0; q < PB; ++q) H[i][q] = mfma4(wb, xv[r][q], H[i][q]);
    }
  }
}

// Pass 1: end state from zero and decay of segment seg < nseg - 1.
template <typename T, int PB, int NB, bool VEC>
__global__ __launch_bounds__(256) void ssd_walk_state_kernel(SsdArgs a, int N, uint32_t npg,
                                                             uint32_t nsub, uint32_t segb, int zoh,
                                                             int by_xcd) {
  typedef WalkIn<T, PB, NB, VEC, false, kWalkQ> In;
  __shared__ __align__(16) char s_in[4][In::kBytes];
  const int lane = threadIdx.x & 63, c = lane & 15, j = lane >> 4;
  const WalkUnit u = walk_unit(a, npg, nsub, 16 * PB, by_xcd != 0);
  if (!u.on) return;
  char* lds = &s_in[threadIdx.x >> 6][0];
  In in;
  in.init(a, u, N, lane);
  // blocks from the last (segments before the last hold segb whole blocks)
  const int64_t t_first = (int64_t)u.seg * segb * kWalkQ;
  auto at = [&](int k) { return t_first + (int64_t)(k > 0 ? k : 0) * kWalkQ; };
  typename In::Regs in_flight;
  in.load(in_flight, at((int)segb - 1));
  const float a2 = -expf(a.A_log[u.h]) * kLog2e;
  const double a2d = -exp((double)a.A_log[u.h]) * 1.4426950408889634;
  mfma_acc H[NB][PB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int q = 0; q < PB; ++q) H[i][q] = mfma_acc{0.0f, 0.0f, 0.0f, 0.0f};
  double lsum = 0.0;  // log2 decay of the blocks already taken (the later ones)
  for (int kb = (int)segb - 1; kb >= 0; --kb) {
    const float d = in.stage(in_flight, lds, at(kb));
    in.load(in_flight, at(kb - 1));
    float xv[4][PB];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int q = 0; q < PB; ++q) xv[r][q] = In::TX::get(lds + In::kX, 4 * j + r, 16 * q + c);
    const WalkScalars s = walk_scalars(d, a2, a2d, zoh != 0, j);
    lsum += s.cum_e;
    float w[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) w[r] = exp2_fast((float)(lsum - s.cs[r])) * s.cf[r];
    walk_update<In, PB, NB>(H, lds, xv, w, c, j);
    if (exp2_fast((float)lsum) == 0.0f) break;  // uniform: every earlier weight is zero too
  }
  const int64_t PN = (int64_t)a.P * N;
  const int64_t unit = (int64_t)u.row * (nsub + 1) + u.seg;
  walk_put<PB, NB>(a.chunkX + unit * PN, H, u.p0, (int)a.P, N, c, j);
  if (u.p0 == 0 && lane == 0) a.chunkA[unit] = exp2_fast((float)lsum);
}

// The outputs of one segment from its entry state.
template <typename T, int PB, int NB, bool VEC, bool HAS_D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void ssd_walk_out_kernel(
    SsdArgs a, int N, uint32_t npg, uint32_t nseg, uint32_t segb, int zoh, int by_xcd) {
  typedef WalkIn<T, PB, NB, VEC, true, kWalkQ> In;
  __shared__ __align__(16) char s_in[4][In::kBytes];
  const int lane = threadIdx.x & 63, c = lane & 15, j = lane >> 4;
  const int P = (int)a.P;
  const WalkUnit u = walk_unit(a, npg, nseg, 16 * PB, by_xcd != 0);
  if (!u.on) return;
  char* lds = &s_in[threadIdx.x >> 6][0];
  In in;
  in.init(a, u, N, lane);
  const int64_t nblk = (a.L + kWalkQ - 1) / kWalkQ;
  const int64_t blk0 = (int64_t)u.seg * segb;
  const int64_t blk1 = blk0 + segb < nblk ? blk0 + segb : nblk;
  typename In::Regs in_flight;
  in.load(in_flight, blk0 * kWalkQ);
  const float a2 = -expf(a.A_log[u.h]) * kLog2e;
  const double a2d = -exp((double)a.A_log[u.h]) * 1.4426950408889634;
  const int64_t PN = (int64_t)P * N;
  const float* hin = nseg > 1 ? a.chunkX + ((int64_t)u.row * nseg + u.seg) * PN
                              : (a.h0 ? a.h0 + (int64_t)u.row * PN : nullptr);
  mfma_acc H[NB][PB];
  walk_get<PB, NB>(H, hin, u.p0, P, N, c, j);
  // outputs: lane (c = step, j) holds channels po + 16 q + r
  const int po = u.p0 + 4 * j;
  T* yp = reinterpret_cast<T*>(a.y) + u.b * a.sy_b + u.h * a.sy_h + po;
  float dv[HAS_D ? PB : 1][4];
  if constexpr (HAS_D) {
#pragma unroll
    for (int q = 0; q < PB; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int p = po + 16 * q + r;
        dv[q][r] = a.D[u.h * P + (p < P ? p : 0)];
      }
  }
  for (int64_t blk = blk0; blk < blk1; ++blk) {
    const int64_t t = blk * kWalkQ + c;
    const float d = in.stage(in_flight, lds, blk * kWalkQ);
    in.load(in_flight, (blk + 1) * kWalkQ);
    const WalkScalars s = walk_scalars(d, a2, a2d, zoh != 0, j);
    mfma_acc g = {0.0f, 0.0f, 0.0f, 0.0f}, y[PB];
#pragma unroll
    for (int q = 0; q < PB; ++q) y[q] = mfma_acc{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      float bv[4], cv[4];
      In::TN::get4(lds + In::kB, c, 16 * i + 4 * j, bv);
      In::TN::get4(lds + In::kC, c, 16 * i + 4 * j, cv);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        g = mfma4(bv[r], cv[r], g);
#pragma unroll
        for (int q = 0; q < PB; ++q) y[q] = mfma4(H[i][q][r], cv[r], y[q]);
      }
    }
    float xv[4][PB];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int q = 0; q < PB; ++q) xv[r][q] = In::TX::get(lds + In::kX, 4 * j + r, 16 * q + c);
    const float et = exp2_fast((float)s.cum);
    float m[4], w[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float v = g[r] * (exp2_fast((float)(s.cum - s.cs[r])) * s.cf[r]);
      m[r] = __uint_as_float(__float_as_uint(v) & (4 * j + r <= c ? ~0u : 0u));
      w[r] = exp2_fast((float)(s.cum_e - s.cs[r])) * s.cf[r];
    }
#pragma unroll
    for (int q = 0; q < PB; ++q) {
#pragma unroll
      for (int r = 0; r < 4; ++r) y[q][r] *= et;
    }
    // A step that is not finite must not reach earlier steps through 0 * inf:
    // then each output step takes the product over its own past only.
    float z = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int q = 0; q < PB; ++q) z = __builtin_fmaf(xv[r][q], 0.0f, z);
    if (__ballot(z != 0.0f) == 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int q = 0; q < PB; ++q) y[q] = mfma4(xv[r][q], m[r], y[q]);
    } else {
#pragma unroll 1
      for (int tt = 0; tt < kWalkQ; ++tt) {
#pragma unroll
        for (int q = 0; q < PB; ++q) {
          mfma_acc part = y[q];
#pragma unroll
          for (int r = 0; r < 4; ++r) part = mfma4(4 * j + r <= tt ? xv[r][q] : 0.0f, m[r], part);
#pragma unroll
          for (int r = 0; r < 4; ++r) y[q][r] = c == tt ? part[r] : y[q][r];
        }
      }
    }
    const float dec = exp2_fast((float)s.cum_e);
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int q = 0; q < PB; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) H[i][q][r] *= dec;
    walk_update<In, PB, NB>(H, lds, xv, w, c, j);
    if (N < 16 * NB) {  // padded columns stay zero whatever x holds
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int q = 0; q < PB; ++q)
#pragma unroll
          for (int r = 0; r < 4; ++r) H[i][q][r] = 4 * j + r < N ? H[i][q][r] : 0.0f;
    }
#pragma unroll
    for (int q = 0; q < PB; ++q) {
      float yv[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) yv[r] = y[q][r];
      if constexpr (HAS_D) {
        float xd[4];
        In::TX::get4(lds + In::kX, c, 16 * q + 4 * j, xd);
#pragma unroll
        for (int r = 0; r < 4; ++r) yv[r] = __builtin_fmaf(dv[q][r], xd[r], yv[r]);
      }
      if (t < a.L) {
        if constexpr (VEC) {
          if (po + 16 * q < P) st_lanes<T, 4>(yp + t * a.sy_l + 16 * q, yv);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (po + 16 * q + r < P) stf(yp + t * a.sy_l + 16 * q + r, yv[r]);
        }
      }
    }
  }
  if (a.h_last && u.seg == nseg - 1)
    walk_put<PB, NB>(a.h_last + (int64_t)u.row * PN, H, u.p0, P, N, c, j);
}

// Entry states from end states, in place: thread (row, state entry) walks the
// segments, S <- A S + X, from h0 or zero.
constexpr int kWalkBatch = 32;  // segments loaded at once
__global__ __launch_bounds__(256) void ssd_walk_prefix_kernel(SsdArgs a, uint32_t nseg,
                                                              int64_t PN) {
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = id / PN, e = id - row * PN;
  if (row >= (int64_t)a.rows) return;
  float S = a.h0 ? a.h0[row * PN + e] : 0.0f;
  float* X = a.chunkX + row * nseg * PN + e;
  const float* A = a.chunkA + row * nseg;
  for (uint32_t s0 = 0; s0 < nseg; s0 += kWalkBatch) {
    float xs[kWalkBatch], as[kWalkBatch];
#pragma unroll
    for (int k = 0; k < kWalkBatch; ++k) {
      // the last segment has no end state: its slot is only written
      const uint32_t sc = min(s0 + k, nseg - 2);
      xs[k] = X[(int64_t)sc * PN];
      as[k] = A[sc];
    }
#pragma unroll
    for (int k = 0; k < kWalkBatch; ++k) {
      if (s0 + k < nseg) {
        X[(int64_t)(s0 + k) * PN] = S;
        S = __builtin_fmaf(as[k], S, xs[k]);
      }
    }
  }
}

}  // namespace

void launch_ssd_walk_prefix(uint32_t nseg, int64_t PN, hipStream_t s, const SsdArgs& a) {
  hipLaunchKernelGGL(ssd_walk_prefix_kernel, dim3((unsigned)cdiv64(a.rows * PN, 256)), dim3(256), 0,
                     s, a, nseg, PN);
}

namespace {

struct WalkPlan {
  int pb;
  uint32_t npg, nseg, segb;
};

// Channels per wave (16 or 32) and time segments, the cheapest by a count of
// what was measured at P = N = 64 fp32: a block takes a SIMD 40 cycles per
// matrix product and 1500 more (one wave alone 1200 longer) at about 2.2 GHz;
// 1024 SIMDs share the waves; segments add pass 1, the prefix and two launches
// (kWalkSegUs).  32 channels form G once where 16 form it twice (2.45 against
// 2 x 1.6 us a block with the SIMDs full); 64 channels leave room for one
// wave a SIMD, with nothing to run beside its products (5.0 against 2 x 2.45
// us), and are not built.
constexpr double kWalkSegUs = 14;
WalkPlan walk_plan(int64_t rows, int64_t P, int N, int64_t L, int64_t max_seg, int max_pb) {
  const int nb = N <= 16 ? 1 : N / 16;
  const int64_t nblk = cdiv64(L, kWalkQ);
  WalkPlan best{1, 1, 1, 1};
  double best_us = 1e30;
  for (int pb = 1; pb <= max_pb && (pb == 1 || P > 16); pb *= 2) {
    const int64_t npg = cdiv64(P, 16 * pb);
    const double full = (40.0 * (4 * nb * (1 + 2 * pb) + 4 * pb) + 1500) / 2200;
    for (int m = 0; m <= 4; ++m) {  // one segment, or m waves a SIMD
      int64_t want = m ? 1024 * m / (rows * npg) : 1;
      if (want > max_seg) want = max_seg;
      if (want > nblk) want = nblk;
      if (want < 1) want = 1;
      const int64_t segb = cdiv64(nblk, want), nseg = cdiv64(nblk, segb);
      const double share = (double)cdiv64(rows * npg * nseg, 1024) * full;
      const double us = segb * (share > full + 0.55 ? share : full + 0.55) +
                        (nseg > 1 ? kWalkSegUs : 0.0);
      if (us < best_us) {
        best_us = us;
        best = WalkPlan{pb, (uint32_t)npg, (uint32_t)nseg, (uint32_t)segb};
      }
    }
  }
  return best;
}

template <typename T, int PB, int NB, bool VEC>
int launch_walk(const WalkPlan& pl, int disc, int N, hipStream_t s, SsdArgs a) {
  a.chunkA = a.chunkX + (int64_t)a.rows * pl.nseg * a.P * N;
  const int64_t per = (int64_t)a.H * pl.npg, nbatch = a.rows / a.H;
  const int zoh = disc == TSSM_DISC_ZOH;
  auto grid = [&](int64_t nseg, int* by_xcd) { return walk_grid(nbatch * nseg, per, by_xcd); };
  int bx = 0;
  if (pl.nseg > 1) {
    const dim3 g1 = grid(pl.nseg - 1, &bx);
    hipLaunchKernelGGL((ssd_walk_state_kernel<T, PB, NB, VEC>), g1, dim3(256), 0, s, a, N, pl.npg,
                       pl.nseg - 1, pl.segb, zoh, bx);
    launch_ssd_walk_prefix(pl.nseg, (int64_t)a.P * N, s, a);
  }
  const dim3 g3 = grid(pl.nseg, &bx);
  if (a.D)
    hipLaunchKernelGGL((ssd_walk_out_kernel<T, PB, NB, VEC, true>), g3, dim3(256), 0, s, a, N,
                       pl.npg, pl.nseg, pl.segb, zoh, bx);
  else
    hipLaunchKernelGGL((ssd_walk_out_kernel<T, PB, NB, VEC, false>), g3, dim3(256), 0, s, a, N,
                       pl.npg, pl.nseg, pl.segb, zoh, bx);
  return launch_status();
}

template <typename T, int NB>
int launch_walk_n(int disc, int N, hipStream_t s, const SsdArgs& a) {
  // vector accesses of 16 bytes, 16 rows' byte offsets in 32 bits
  const int64_t strides = a.sx_b | a.sx_l | a.sx_h | a.sB_b | a.sB_l | a.sB_h | a.sC_b | a.sC_l |
                          a.sC_h | (int64_t)a.P;
  const bool vec = strides % (int64_t)(16 / sizeof(T)) == 0 && aligned(a.x, 16) &&
                   aligned(a.B, 16) && aligned(a.C, 16) && aligned(a.y, 4 * sizeof(T)) &&
                   ((a.sy_b | a.sy_l | a.sy_h) & 3) == 0 &&
                   ((a.sx_l | a.sB_l | a.sC_l | a.sdt_l) >> 25) == 0;
  // a segment takes one state (end, then entry) and one decay of the
  // workspace, which holds two states and a decay per chunk
  const int64_t PN = (int64_t)a.P * N, max_seg = (int64_t)a.nchunks * (2 * PN + 1) / (PN + 1);
  const WalkPlan pl =
      walk_plan((int64_t)a.rows, (int64_t)a.P, N, a.L, max_seg, vec ? 2 : 1);
  if (!vec) return launch_walk<T, 1, NB, false>(pl, disc, N, s, a);
  return pl.pb == 2 ? launch_walk<T, 2, NB, true>(pl, disc, N, s, a)
                    : launch_walk<T, 1, NB, true>(pl, disc, N, s, a);
}

template <typename T>
int launch_walk_t(int disc, int N, hipStream_t s, const SsdArgs& a) {
  if (N <= 16) return launch_walk_n<T, 1>(disc, N, s, a);
  if (N == 32) return launch_walk_n<T, 2>(disc, N, s, a);
  return launch_walk_n<T, 4>(disc, N, s, a);
}

}  // namespace

int launch_ssd_walk(int dtype, int disc, int N, hipStream_t s, const SsdArgs& a) {
  switch (dtype) {
    case TSSM_BF16: return launch_walk_t<bf16_t>(disc, N, s, a);
    case TSSM_F16: return launch_walk_t<f16_t>(disc, N, s, a);
    default: return launch_walk_t<float>(disc, N, s, a);
  }
}

}  // namespace tssm
