// SSD selective scan, bf16 with N = 64 and P a multiple of 16, on the bf16 matrix
// cores: the walk of ssd_walk.hip with 32-step blocks and K = 32 products.
//
// A unit is (row, 32 channels, time segment).  In the state pass one wave owns a
// unit; in the output pass a workgroup of 8 waves takes 8 blocks of it at a time:
// each wave forms its block's share of the state, the shares meet in LDS, and the
// fold of them leaves every wave the state its block starts from.  A wave's share
// is in registers (fp32, H^T: lane 16 j + c holds columns 16 i + 4 j + r of channel
// 16 q + c).  A block is two halves of 16 steps; with cum_t the inclusive sum
// of log2 decay within step t's half, tot_b a half's sum and coef_s the input
// coefficient,
//   u_t = 2^(cum_t - tot/2)   v_s = 2^(tot/2 - cum_s) coef_s   (diagonal blocks)
//   w_s = 2^(tot - cum_s) coef_s   e_t = 2^cum_t               (across halves)
//   y_t (half 0) = u_t (2^(tot0/2) H.C_t + sum_s (B_s.C_t) v_s x_s)
//   y_t (half 1) = u_t (2^(tot1/2) (2^tot0 H.C_t + sum_{half 0} (B_s.C_t) w_s x_s)
//                       + sum_{s <= t} (B_s.C_t) v_s x_s)
//   H' = 2^(tot0 + tot1) H + sum_s w_s 2^(tot of the later half) x_s B_s
// Every factor stays within 2^+-64 while a half decays by at most 2^-128
// (kW16Factored); a block with a half beyond that takes its diagonal weights
// element by element.  w comes from sums taken backwards (W16Steps).  x, B and C
// enter the products exactly; operands formed in fp32 (weighted Gram blocks,
// weighted x, the state) are split into bf16 hi + lo and multiplied twice, as in
// the other bf16 kernels.
//
// No operand is transposed by instructions: Gram blocks and the state come out
// of one product in the layout the next one takes (the order of k is free, so
// lane group j's eight k-values are its rows 4 j .. 4 j + 3 of two tiles), and
// the operands that run over steps (x for the outputs, x and B for the update)
// are read from row-major LDS by ds_read_b64_tr_b16.
//
// Bound by the chain of dependent phases with one workgroup (two waves a SIMD) on a
// CU, not by HBM: B=8 L=4096 H=16 P=N=64 takes 88.4 us with 271 MB moved (the one-pass
// kernel it replaced: 100.8), about 53 at a copy's rate.  A super-block of 8 x 32
// steps costs a wave 10,350 cycles, no phase over a fifth of them.
// B=1 L=65536 H=8: 119.8 - 123.8 us a call by box (before 139 - 144).  16 channels a
// wave measured 115 - 129 us on the first shape, 12 waves a workgroup 118 (spills).
//
// x that is not finite is rare.  The wave that finds some in its block (a dot
// product with zero of the loaded registers, 8 instructions) takes it through
// products of its own, each output step over its own past, so that steps before it
// stay as they are (88.5 us without, 88.4 with).  It makes its channel's state NaN.
//
// The hi/lo operands keep 16 bits, which y's rounding hides and the fp32 final
// state does not: 2.2e-6 of float64 on it, where fp32 products give 1e-7.  So bf16
// at other head dims and state sizes, whose state is formed in fp32 throughout, is
// not taken here, though N = 32 would run in 55 us instead of 104 (B=8 L=4096 H=16
// P=64).
#include "ssd_walk_dev.h"

namespace tssm {
namespace {

constexpr int kW16Q = 32;  // steps per block
constexpr int NB = 4;      // column tiles of 16: N = 64
// Most sub-segments whose end states the output pass folds into entry states
// itself; more take the prefix pass.  Folding reads eight states where decays
// forget and 16 rounds of eight at worst, the prefix pass 10-18 us either way.
constexpr int64_t kW16Fold = 128;

// Largest log2 decay of a half whose diagonal weights are formed as u_t v_s.  A
// weighted Gram value B_s.C_t v_s may be 2^+-64 off its final size, is split into
// bf16 hi and lo and summed with x: it must neither reach 2^128 (with 2^+-120 a half
// of 2^-232 gave inf from B.C of a few hundred) nor lose its lo part, 2^-16 of it, at
// 2^-126 (with 2^+-120 steps of 1e-4 before a long gap were off by their own size).
// B=8 L=4096 H=16 P=N=64: 87.9 us with 2^+-120, 88.4 with 2^+-64.
constexpr float kW16Factored = -128.0f;

typedef __attribute__((address_space(3))) s16x4_t* lds_s16x4;

// Four rows (steps r0 .. r0 + 3, r0 = 4 j + 16 a) of column col0 + c, for lane
// 16 j + c.  The transposing read takes a 16-lane group's 8-byte pieces as
// 4 rows x 16 columns and hands each lane a column.
template <typename Tile>
__device__ inline s16x4_t read_cols(const char* lds, int a, int col0, int c, int j) {
  const char* p = lds + (16 * a + 4 * j + (c >> 2)) * Tile::kStride + (col0 + 4 * (c & 3)) * 2;
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (lds_s16x4)(uintptr_t)(const __attribute__((address_space(3))) char*)p);
}
// Eight state columns of one row: 32 m + 4 j .. + 3 and 32 m + 16 + 4 j .. + 3.
template <typename Tile>
__device__ inline bf16x8_t read_row(const char* lds, int row, int m, int j) {
  const char* p = lds + row * Tile::kStride + (32 * m + 4 * j) * 2;
  const uint2 a = *reinterpret_cast<const uint2*>(p);
  const uint2 b = *reinterpret_cast<const uint2*>(p + 32);
  return as_bf16x8(u32x4{a.x, a.y, b.x, b.y});
}

__device__ inline bf16x8_t join(uint2 a, uint2 b) { return as_bf16x8(u32x4{a.x, a.y, b.x, b.y}); }
__device__ inline s16x4_t as_s16x4(uint2 v) { return __builtin_bit_cast(s16x4_t, v); }

// Four floats as packed bf16 hi and lo parts.
__device__ inline void split4(const float* v, uint2& hi, uint2& lo) {
  hi.x = pk_bf16(v[0], v[1]);
  hi.y = pk_bf16(v[2], v[3]);
  lo.x = pk_bf16(v[0] - bf16_lo(hi.x), v[1] - bf16_hi(hi.x));
  lo.y = pk_bf16(v[2] - bf16_lo(hi.y), v[3] - bf16_hi(hi.y));
}

// Whether any of a block's x is not finite (uniform), from the registers it was
// loaded into: x . 0 is zero or NaN.
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
template <typename Regs>
__device__ inline bool any_not_finite(const Regs& x) {
  const bf16x2_t zero = {};
  float z[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (const u32x4 v : x.v)
#pragma unroll
    for (int k = 0; k < 4; ++k)
      z[k] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, (uint32_t)v[k]), zero,
                                             z[k], false);
  return __ballot((z[0] + z[1]) + (z[2] + z[3]) != 0.0f) != 0;
}
// x split into its finite values, which stay, and the others, which are moved to
// xb (zero elsewhere): a product with zero weights, of steps before them, must
// not meet them.
template <int PB>
__device__ inline void take_not_finite(s16x4_t (&xc)[2][PB], s16x4_t (&xb)[2][PB]) {
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int q = 0; q < PB; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const short v = xc[a][q][r];
        const bool f = (v & 0x7f80) != 0x7f80;
        xb[a][q][r] = f ? (short)0 : v;
        xc[a][q][r] = f ? v : (short)0;
      }
}
// x of rows r0 .. r0 + 3, zero after row `last`.
__device__ inline s16x4_t past_only(s16x4_t x, int r0, int last) {
  s16x4_t o;
#pragma unroll
  for (int r = 0; r < 4; ++r) o[r] = r0 + r <= last ? x[r] : (short)0;
  return o;
}
__device__ inline mfma_acc mfma16(s16x4_t x, uint2 m, mfma_acc acc) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(x, as_s16x4(m), acc, 0, 0, 0);
}

// One block's step quantities: lane l stands for step l % 32.  The log2 decays
// are summed in fp32 over 16 steps at most, forwards for the outputs and, for the
// state, backwards: 2^(tot - cum) after a long gap would keep the gap's rounding
// (1e-4 on the state after steps of 700; with `after` 3e-6).  kW16Floor: one step's
// decay is 0 either way, and what follows it keeps its bits.
constexpr float kW16Floor = -256.0f;
struct W16Steps {
  float cum, tot0, tot1;  // within the step's half; the halves' sums (uniform)
  float after;            // of the half's steps after this one
  float coef;
};
__device__ inline float lane_f32(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ inline W16Steps w16_steps(float d, float a2, bool zoh) {
  W16Steps o;
  const float y = d * a2;
  o.coef = zoh ? phi1_from_exp(y * 0.6931471805599453f, exp2_fast(y)) * d : d;
  float l = y < kW16Floor ? kW16Floor : y;
  float r = dpp_in<0x101, 0xf>(l);  // row_shl:1
  r += dpp_in<0x101, 0xf>(r);
  r += dpp_in<0x102, 0xf>(r);
  r += dpp_in<0x104, 0xf>(r);
  r += dpp_in<0x108, 0xf>(r);
  o.after = r;
  l += dpp_in<0x111, 0xf>(l);
  l += dpp_in<0x112, 0xf>(l);
  l += dpp_in<0x114, 0xf>(l);
  l += dpp_in<0x118, 0xf>(l);
  o.cum = l;
  o.tot0 = lane_f32(l, 15);
  o.tot1 = lane_f32(l, 31);
  return o;
}

// H^T += sum_s w_s B_s x_s^T over the block's 32 steps: w the LDS weights,
// xc the x columns read_cols gave for (half a, channel block q).
template <typename In, int PB>
__device__ inline void w16_update(mfma_acc (&H)[NB][PB], const char* lds, const float* w,
                                  const s16x4_t (&xc)[2][PB], int c, int j) {
  bf16x8_t xh[PB], xl[PB];
  f32x4 wv[2];
#pragma unroll
  for (int a = 0; a < 2; ++a) wv[a] = *reinterpret_cast<const f32x4*>(w + 16 * a + 4 * j);
#pragma unroll
  for (int q = 0; q < PB; ++q) {
    uint2 h[2], l[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const uint2 xv = __builtin_bit_cast(uint2, xc[a][q]);
      const float v[4] = {bf16_lo(xv.x) * wv[a][0], bf16_hi(xv.x) * wv[a][1],
                          bf16_lo(xv.y) * wv[a][2], bf16_hi(xv.y) * wv[a][3]};
      split4(v, h[a], l[a]);
    }
    xh[q] = join(h[0], h[1]);
    xl[q] = join(l[0], l[1]);
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const bf16x8_t bt =
        join(__builtin_bit_cast(uint2, read_cols<typename In::TN>(lds + In::kB, 0, 16 * i, c, j)),
             __builtin_bit_cast(uint2, read_cols<typename In::TN>(lds + In::kB, 1, 16 * i, c, j)));
#pragma unroll
    for (int q = 0; q < PB; ++q) {
      H[i][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bt, xh[q], H[i][q], 0, 0, 0);
      H[i][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bt, xl[q], H[i][q], 0, 0, 0);
    }
  }
}

// Pass 1: end state from zero and decay of each of the `nsub` sub-segments (segb
// blocks) before the last segment, last block first, stopping once the decay
// has underflowed to exactly zero.
template <int PB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void
ssd_walk16_state_kernel(SsdArgs a, uint32_t npg, uint32_t nsub, uint32_t segb, int zoh,
                        int by_xcd) {
  typedef WalkIn<bf16_t, PB, NB, true, false, kW16Q> In;
  __shared__ __align__(16) char s_in[4][In::kBytes];
  __shared__ __align__(16) float s_w[4][kW16Q];
  const int lane = threadIdx.x & 63, c = lane & 15, j = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const WalkUnit u = walk_unit(a, npg, nsub, 16 * PB, by_xcd != 0);
  if (!u.on) return;
  char* lds = &s_in[wv][0];
  float* w = s_w[wv];
  In in;
  in.init(a, u, 16 * NB, lane);
  const int64_t t_first = (int64_t)u.seg * segb * kW16Q;
  auto at = [&](int k) { return t_first + (int64_t)(k > 0 ? k : 0) * kW16Q; };
  typename In::Regs g0, g1;  // two blocks in flight: a block's products are short
  in.load(g0, at((int)segb - 1));
  in.load(g1, at((int)segb - 2));
  const float a2 = -expf(a.A_log[u.h]) * kLog2e;
  mfma_acc H[NB][PB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int q = 0; q < PB; ++q) H[i][q] = mfma_acc{0.0f, 0.0f, 0.0f, 0.0f};
  float lsum = 0.0f;  // log2 decay of the blocks already taken (the later ones)
  auto step = [&](typename In::Regs& g, int kb) {
    const float d = in.stage(g, lds, at(kb));
    in.load(g, at(kb - 2));
    const W16Steps s = w16_steps(d, a2, zoh != 0);
    const float later = (lane & 16) ? lsum : lsum + s.tot1;
    if (lane < kW16Q) w[lane] = exp2_fast(later + s.after) * s.coef;
    wave_lds_order();
    s16x4_t xc[2][PB];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < PB; ++q)
        xc[h][q] = read_cols<typename In::TX>(lds + In::kX, h, 16 * q, c, j);
    w16_update<In, PB>(H, lds, w, xc, c, j);
    lsum += s.tot0 + s.tot1;
    return exp2_fast(lsum) != 0.0f;  // uniform; at 0 every earlier weight is zero too
  };
  for (int kb = (int)segb - 1; kb >= 0; kb -= 2)
    if (!step(g0, kb) || kb == 0 || !step(g1, kb - 1)) break;
  const int64_t PN = (int64_t)a.P * (16 * NB);
  const int64_t unit = (int64_t)u.row * (nsub + 1) + u.seg;  // a slot per sub-segment and one more
  walk_put<PB, NB>(a.chunkX + unit * PN, H, u.p0, (int)a.P, 16 * NB, c, j);
  if (u.p0 == 0 && lane == 0) a.chunkA[unit] = exp2_fast(lsum);
}

// One block's per-step weights in LDS.
struct __align__(16) W16Weights {
  float u[kW16Q], v[kW16Q], w[kW16Q], wu[kW16Q];
  float cum[kW16Q];
};

// The outputs of one segment.  A workgroup of kW16Waves waves takes (row, 16 PB
// channels, segment) and walks it in super-blocks of kW16Waves blocks, wave w
// its w-th: each wave forms its block's own share of the state (from zero), the
// shares meet in LDS, and the thread that owns four entries of the state folds
// the blocks in order, leaving every block's entry state (split hi/lo) where
// its share was; then each wave forms its block's outputs.  So a row's blocks
// run side by side with one read of the inputs.  A wave's region in LDS holds
// its staged block, then (every operand taken into registers) the state.
constexpr int kW16Waves = 8;
template <int PB, bool HAS_D>
__global__ __launch_bounds__(64 * kW16Waves) __attribute__((amdgpu_waves_per_eu(2))) void
ssd_walk16_out_kernel(SsdArgs a, uint32_t npg, uint32_t nseg, uint32_t segb, uint32_t m, int zoh) {
  typedef WalkIn<bf16_t, PB, NB, true, true, kW16Q> In;
  typedef typename In::TN TN;
  typedef typename In::TX TX;
  constexpr int M = NB / 2, N = 16 * NB;   // K = 32 products over the columns
  constexpr int kRow = 4 * N + 16;         // a channel's state in LDS, bytes
  static_assert(16 * PB * kRow <= In::kBytes, "the state fits the staged block's region");
  __shared__ __align__(16) char s_in[kW16Waves][In::kBytes];
  __shared__ W16Weights s_sc[kW16Waves][2];  // this super-block's and the next one's
  __shared__ float s_dec[2][kW16Waves];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, j = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int P = (int)a.P;
  // the workgroups of one (batch, segment), whose heads share the 128-byte
  // lines of dt, on one XCD (blockIdx mod 8) where their number allows
  const uint32_t per = a.H * npg, groups = a.rows / a.H * nseg;
  uint32_t g, v;
  if (groups % 8 == 0) {
    const uint32_t k = blockIdx.x >> 3;
    g = k / per * 8 + (blockIdx.x & 7);
    v = k % per;
  } else {
    g = blockIdx.x / per;
    v = blockIdx.x - g * per;
  }
  WalkUnit u;
  u.on = true;
  u.b = g / nseg;
  u.seg = g - u.b * nseg;
  u.h = v / npg;
  u.p0 = (int)(v - u.h * npg) * 16 * PB;
  u.row = u.b * a.H + u.h;
  char* lds = &s_in[wv][0];
  const int64_t blk0 = (int64_t)u.seg * segb;
  const int64_t t_end = (blk0 + segb) * kW16Q < a.L ? (blk0 + segb) * kW16Q : a.L;
  In in;
  in.init(a, u, N, lane);
  in.L = t_end;  // steps from the segment's end on count as past the sequence
  typename In::Regs in_flight;
  int64_t t0 = (blk0 + wv) * kW16Q;
  in.load(in_flight, t0);
  // dt is loaded two super-blocks ahead: its weights are formed one ahead
  auto load_dt = [&](int64_t t) {
    t += lane & (kW16Q - 1);
    return *reinterpret_cast<const float*>(in.pd + (t < t_end ? t : t_end - 1) * in.sdt);
  };
  auto live_dt = [&](float d, int64_t t) { return t + (lane & (kW16Q - 1)) < t_end ? d : 0.0f; };
  constexpr int64_t kSuper = kW16Waves * kW16Q;
  float d_next = load_dt(t0 + kSuper);
  const float a2 = -expf(a.A_log[u.h]) * kLog2e;
  // the thread's state entries: channel op, columns 4 on .. + 3
  const int op = tid / (4 * NB), on = tid % (4 * NB);
  const bool own = op < 16 * PB;
  const bool real = own && u.p0 + op < P;
  const int64_t PN = (int64_t)P * N;
  const int64_t oe = real ? (int64_t)(u.p0 + op) * N + 4 * on : 0;
  float S[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  // slots: a row's sub-segments (m a segment) and one more
  const uint32_t nslot = (nseg - 1) * m + 1, slot = u.seg * m;
  const float* X = a.chunkX + (int64_t)u.row * nslot * PN + oe;
  if (nslot > kW16Fold) {
#pragma unroll
    for (int r = 0; r < 4; ++r) S[r] = X[slot * PN + r];
  } else {
    // the sub-segments before this segment, latest first and eight at a time,
    // until their decays' product is exactly zero
    const float* A = a.chunkA + (int64_t)u.row * nslot;
    float dec = 1.0f;
    for (int s = (int)slot - 1; s >= 0 && dec != 0.0f; s -= 8) {
      float x[8][4], ad[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int sk = s - k > 0 ? s - k : 0;
        ad[k] = A[sk];
#pragma unroll
        for (int r = 0; r < 4; ++r) x[k][r] = X[sk * PN + r];
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        if (s - k >= 0 && dec != 0.0f) {
#pragma unroll
          for (int r = 0; r < 4; ++r) S[r] = __builtin_fmaf(dec, x[k][r], S[r]);
          dec *= ad[k];
        }
      }
    }
    if (a.h0 && dec != 0.0f) {
      const float* h = a.h0 + (int64_t)u.row * PN + oe;
#pragma unroll
      for (int r = 0; r < 4; ++r) S[r] = __builtin_fmaf(dec, h[r], S[r]);
    }
  }
  // outputs: lane (c = step of a half, j) holds channels po + 16 q + r
  const int po = u.p0 + 4 * j;
  bf16_t* yp = reinterpret_cast<bf16_t*>(a.y) + u.b * a.sy_b + u.h * a.sy_h + po;
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
  auto weights = [&](float d, int b) {
    const W16Steps s = w16_steps(d, a2, zoh != 0);
    const bool fac = s.tot0 >= kW16Factored && s.tot1 >= kW16Factored;  // uniform in the wave
    W16Weights& k = s_sc[wv][b];
    if (lane < kW16Q) {
      const float tot = lane < 16 ? s.tot0 : s.tot1;
      const float wl = exp2_fast(s.after) * s.coef;
      k.u[lane] = exp2_fast(fac ? s.cum - 0.5f * tot : s.cum);
      k.v[lane] = fac ? exp2_fast(0.5f * tot - s.cum) * s.coef : s.coef;
      k.w[lane] = wl;
      // to the block's end, for the state
      k.wu[lane] = lane < 16 ? exp2_fast(s.tot1 + s.after) * s.coef : wl;
      k.cum[lane] = s.cum;
    }
    if (lane == 0) s_dec[b][wv] = exp2_fast(s.tot0 + s.tot1);
    return s;
  };
  W16Steps s = weights(live_dt(in_flight.dt, t0), 0);
  int buf = 0;
  for (int64_t tb = blk0 * kW16Q; tb < t_end; tb += kSuper, t0 += kSuper, buf ^= 1) {
    const bool bad = any_not_finite(in_flight.x);
    in.stage(in_flight, lds, t0);
    const W16Weights& sc = s_sc[wv][buf];
    const bool fac = s.tot0 >= kW16Factored && s.tot1 >= kW16Factored;
    // every operand of the block into registers, and what needs no state
    s16x4_t xc[2][PB];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < PB; ++q) xc[h][q] = read_cols<TX>(lds + In::kX, h, 16 * q, c, j);
    mfma_acc H[NB][PB];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int q = 0; q < PB; ++q) H[i][q] = mfma_acc{0.0f, 0.0f, 0.0f, 0.0f};
    w16_update<In, PB>(H, lds, sc.wu, xc, c, j);
    // the next block's loads, a part at a time: eight waves issuing all of
    // theirs at once wait on each other
    const int64_t tn = in.row0(t0 + kSuper);
    in.x.load(in_flight.x, in.px + tn * in.sx);
    in.B.load(in_flight.B, in.pB + tn * in.sB);
    bf16x8_t cf[2][M];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int m = 0; m < M; ++m) cf[t][m] = read_row<TN>(lds + In::kC, 16 * t + c, m, j);
    // Gram blocks: half 0 with itself, half 0 against half 1, half 1 with itself
    mfma_acc g00 = {0.0f, 0.0f, 0.0f, 0.0f}, g01 = g00, g11 = g00;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const bf16x8_t b0 = read_row<TN>(lds + In::kB, c, m, j);
      const bf16x8_t b1 = read_row<TN>(lds + In::kB, 16 + c, m, j);
      g00 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b0, cf[0][m], g00, 0, 0, 0);
      g01 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b0, cf[1][m], g01, 0, 0, 0);
      g11 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b1, cf[1][m], g11, 0, 0, 0);
    }
    in.C.load(in_flight.C, in.pC + tn * in.sC);
    uint2 xd[HAS_D ? 2 : 1][PB];
    if constexpr (HAS_D) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int q = 0; q < PB; ++q)
          xd[t][q] = *reinterpret_cast<const uint2*>(lds + In::kX + (16 * t + c) * TX::kStride +
                                                     (16 * q + 4 * j) * 2);
    }
    s16x4_t xb[2][PB];
    if (__builtin_expect(bad, false)) take_not_finite(xc, xb);  // (the share has it already)
    wave_lds_order();
#pragma unroll
    for (int q = 0; q < PB; ++q)
#pragma unroll
      for (int i = 0; i < NB; ++i)
        *reinterpret_cast<f32x4*>(lds + (16 * q + c) * kRow + (4 * i + j) * 16) = H[i][q];
    __syncthreads();
    if (own) {
      char* e = &s_in[0][0] + op * kRow + on * 16;
#pragma unroll
      for (int w = 0; w < kW16Waves; ++w) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(e + w * In::kBytes);
        const float dec = s_dec[buf][w];
        uint2 hi, lo;
        split4(S, hi, lo);
        *reinterpret_cast<u32x4*>(e + w * In::kBytes) = u32x4{hi.x, hi.y, lo.x, lo.y};
#pragma unroll
        for (int r = 0; r < 4; ++r) S[r] = __builtin_fmaf(dec, S[r], x[r]);
      }
    }
    // weighted Gram blocks, while the states settle
    const f32x4 v0 = *reinterpret_cast<const f32x4*>(&sc.v[4 * j]);
    const f32x4 v1 = *reinterpret_cast<const f32x4*>(&sc.v[16 + 4 * j]);
    const f32x4 w0 = *reinterpret_cast<const f32x4*>(&sc.w[4 * j]);
    const float u0 = sc.u[c], u1 = sc.u[16 + c];
    float m00[4], m01[4], m11[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      m00[r] = g00[r] * v0[r];
      m01[r] = g01[r] * w0[r];
      m11[r] = g11[r] * v1[r];
    }
    if (!fac) {
      // the diagonal blocks' weights element by element
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        m00[r] *= exp2_fast(sc.cum[c] - sc.cum[4 * j + r]);
        m11[r] *= exp2_fast(sc.cum[16 + c] - sc.cum[16 + 4 * j + r]);
      }
    }
    // masks as bits: a select would put the weights behind a branch
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t k = 4 * j + r <= c ? ~0u : 0u;
      m00[r] = __uint_as_float(__float_as_uint(m00[r]) & k);
      m11[r] = __uint_as_float(__float_as_uint(m11[r]) & k);
    }
    uint2 h00, l00, h01, l01, h11, l11;
    split4(m00, h00, l00);
    split4(m01, h01, l01);
    split4(m11, h11, l11);
    // fac: y = u (2^(tot/2) carried + diagonal);  else y = e carried + diagonal,
    // with u holding e
    const float dec0 = exp2_fast(s.tot0);
    const float z0 = fac ? exp2_fast(0.5f * s.tot0) : u0;
    const float z1 = fac ? exp2_fast(0.5f * s.tot1) : u1;
    const float f0 = fac ? u0 : 1.0f, f1 = fac ? u1 : 1.0f;
    // the next super-block's weights
    s = weights(live_dt(d_next, t0 + kSuper), buf ^ 1);
    d_next = load_dt(t0 + 2 * kSuper);
    __syncthreads();
    mfma_acc y[2][PB];
#pragma unroll
    for (int q = 0; q < PB; ++q) {
      y[0][q] = y[1][q] = mfma_acc{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const char* hp = lds + (16 * q + c) * kRow + (8 * m + j) * 16;
        const u32x4 e0 = *reinterpret_cast<const u32x4*>(hp);
        const u32x4 e1 = *reinterpret_cast<const u32x4*>(hp + 64);
        const bf16x8_t hh = as_bf16x8(u32x4{e0[0], e0[1], e1[0], e1[1]});
        const bf16x8_t hl = as_bf16x8(u32x4{e0[2], e0[3], e1[2], e1[3]});
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          y[t][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hh, cf[t][m], y[t][q], 0, 0, 0);
          y[t][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hl, cf[t][m], y[t][q], 0, 0, 0);
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        y[0][q][r] *= z0;
        y[1][q][r] *= dec0;
      }
      y[1][q] = mfma16(xc[0][q], h01, y[1][q]);
      y[1][q] = mfma16(xc[0][q], l01, y[1][q]);
      y[0][q] = mfma16(xc[0][q], h00, y[0][q]);
      y[0][q] = mfma16(xc[0][q], l00, y[0][q]);
#pragma unroll
      for (int r = 0; r < 4; ++r) y[1][q][r] *= z1;
      y[1][q] = mfma16(xc[1][q], h11, y[1][q]);
      y[1][q] = mfma16(xc[1][q], l11, y[1][q]);
    }
    if (__builtin_expect(bad, false)) {  // each output step's own past of the x kept apart
#pragma unroll
      for (int q = 0; q < PB; ++q) {
        y[1][q] = mfma16(xb[0][q], h01, y[1][q]);
#pragma unroll 1
        for (int tt = 0; tt < 16; ++tt) {
          const mfma_acc p0 = mfma16(past_only(xb[0][q], 4 * j, tt), h00, y[0][q]);
          const mfma_acc p1 = mfma16(past_only(xb[1][q], 4 * j, tt), h11, y[1][q]);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            y[0][q][r] = c == tt ? p0[r] : y[0][q][r];
            y[1][q][r] = c == tt ? p1[r] : y[1][q][r];
          }
        }
      }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int64_t tt = t0 + 16 * t + c;
      const float f = t == 0 ? f0 : f1;
#pragma unroll
      for (int q = 0; q < PB; ++q) {
        float yv[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) yv[r] = f * y[t][q][r];
        if constexpr (HAS_D) {
          const float xv[4] = {bf16_lo(xd[t][q].x), bf16_hi(xd[t][q].x), bf16_lo(xd[t][q].y),
                               bf16_hi(xd[t][q].y)};
#pragma unroll
          for (int r = 0; r < 4; ++r) yv[r] = __builtin_fmaf(dv[q][r], xv[r], yv[r]);
        }
        if (tt < t_end && po + 16 * q < P)
          *reinterpret_cast<uint2*>(yp + tt * a.sy_l + 16 * q) =
              make_uint2(pk_bf16(yv[0], yv[1]), pk_bf16(yv[2], yv[3]));
      }
    }
  }
  if (a.h_last && u.seg == nseg - 1 && real) {
    float* h = a.h_last + (int64_t)u.row * PN + oe;
#pragma unroll
    for (int r = 0; r < 4; ++r) h[r] = S[r];
  }
}

// Time segments: as many as fill every CU once, each of at least one super-block,
// and one only where two super-blocks hold the sequence (a segment costs pass 1 over
// its end, a launch, and its state twice through memory: B=1 H=2 P=64 L=500 11.7 us
// in one, 13.6 in two, 18.3 with slow decays; L=700 15.6 and 15.4 in one, 13.4 and
// 18.5 in three).  Super-blocks are counted up: counted down they left segments of
// two and half the CUs idle (L=2000 17.6 us, slow decays 22.1; with eight of one
// 13.9 and 18.7).  No more than the output pass folds while two super-blocks each
// suffice (B=1 H=1 P=32 L=40000 23.7 us with the prefix pass, slow decays 27.9;
// folded 17.5 and 29.7); beyond, longer segments lose more than the prefix pass takes
// (L=100000, slow decays: 49 us folded, 40).
// Pass 1 takes a segment in m sub-segments of at least kW16MinSub blocks, up to two of
// its waves a SIMD: with slow decays it walks all of them (B=1 L=65536 H=8 P=N=64, slow
// decays: 190 us with m = 1, 132 with m = 8), and no more of them than the output pass
// folds itself (B=1 L=100000 H=1: 53 us with 389 and the prefix pass, 30 with 98; slow
// decays 59 and 53).
constexpr int64_t kW16StateWaves = 2048, kW16MinSub = 8;
template <int PB>
int launch_walk16(int disc, hipStream_t s, SsdArgs a) {
  const int64_t PN = (int64_t)a.P * (16 * NB), nblk = cdiv64(a.L, kW16Q);
  const int64_t npg = cdiv64(a.P, 16 * PB);
  const int64_t units = (int64_t)a.rows * npg;
  // a slot takes one state and one decay of the workspace, which holds two
  // states and a decay per chunk
  const int64_t cap = (int64_t)a.nchunks * (2 * PN + 1) / (PN + 1);
  const int64_t by_len = nblk <= 2 * kW16Waves ? 1 : cdiv64(nblk, kW16Waves);
  int64_t nseg = 256 / units;
  nseg = nseg < cap ? nseg : cap;
  nseg = nseg < by_len ? nseg : by_len;
  if (nseg > kW16Fold && nblk <= 2 * kW16Waves * kW16Fold) nseg = kW16Fold;
  if (nseg < 1) nseg = 1;
  // whole super-blocks
  const int64_t segb = cdiv64(cdiv64(nblk, nseg), kW16Waves) * kW16Waves;
  nseg = cdiv64(nblk, segb);
  int64_t m = 1;
  while (segb % (2 * m) == 0 && segb / (2 * m) >= kW16MinSub &&
         units * (nseg - 1) * 2 * m <= kW16StateWaves && (nseg - 1) * 2 * m + 1 <= cap &&
         (nseg - 1) * 2 * m + 1 <= kW16Fold)
    m *= 2;
  const int64_t nslot = (nseg - 1) * m + 1;
  a.chunkA = a.chunkX + (int64_t)a.rows * nslot * PN;
  const int64_t per = (int64_t)a.H * npg, nbatch = a.rows / a.H;
  const int zoh = disc == TSSM_DISC_ZOH;
  if (nseg > 1) {
    int bx = 0;
    const dim3 g1 = walk_grid(nbatch * (nslot - 1), per, &bx);
    hipLaunchKernelGGL((ssd_walk16_state_kernel<PB>), g1, dim3(256), 0, s, a, (uint32_t)npg,
                       (uint32_t)(nslot - 1), (uint32_t)(segb / m), zoh, bx);
    if (nslot > kW16Fold) launch_ssd_walk_prefix((uint32_t)nslot, PN, s, a);
  }
  const dim3 g3((unsigned)(nbatch * nseg * per));
  if (a.D)
    hipLaunchKernelGGL((ssd_walk16_out_kernel<PB, true>), g3, dim3(64 * kW16Waves), 0, s, a,
                       (uint32_t)npg, (uint32_t)nseg, (uint32_t)segb, (uint32_t)m, zoh);
  else
    hipLaunchKernelGGL((ssd_walk16_out_kernel<PB, false>), g3, dim3(64 * kW16Waves), 0, s, a,
                       (uint32_t)npg, (uint32_t)nseg, (uint32_t)segb, (uint32_t)m, zoh);
  return launch_status();
}

}  // namespace

int launch_ssd_walk_bf16(int disc, hipStream_t s, const SsdArgs& a) {
  return a.P > 16 ? launch_walk16<2>(disc, s, a) : launch_walk16<1>(disc, s, a);
}

}  // namespace tssm
