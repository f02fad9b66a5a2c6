// The triangle multiplication's factor and output backwards, each with its products in one pass (gfx950; the
// output's is below).  The factor projections' backward, for 16-bit pairs with 64 < C, H <= 128 and positions a
// multiple of 32, without a mask gradient:
//
//   value, gate = xn W^T + b (recomputed), d_proj = the gate's backward of the factor gradients
//   d_xn += d_proj W        d_W = d_proj^T xn        d_b = column sums of d_proj
//
// The [4H][R] projection gradient is the largest tensor of the backward (268 MB for a 512 x 512 pair of 128
// channels): written by the factor backward and read by two GEMMs it cost 151 + 88 + 80 us there, against
// the 335 MB (70 us) of the tensors that must move.  Here it stays in the workgroup: 3 MFMA products per
// 32-token tile out of one resident copy of W, 150 us in all (and 15 us more of partial sums).  A tile's
// steps follow each other between barriers, so the matrix cores (a third of the time), the vector unit (40%)
// and the LDS (half) add up rather than overlap; 41 us of it is MFMA time at the peak rate.
//
// Where it serves: the whole d_W (256 KB of float32) in the accumulators and W in LDS want 65 to 128 channels
// on both sides (64 would leave half of the waves without channels); a mask gradient needs sums over the
// channels, which the separate factor backward makes.
//
// One workgroup of 8 waves per CU walks a run of tiles.  W (512 x 128, 128 KB of LDS) is read as rows (the
// projections) and transposed (d_xn).  Wave w owns channels 32 (w % 4) .. + 31 of factor w / 4, value and
// gate: its d_proj values come out of the accumulators in the order in which the LDS transpose read
// delivers xn's tokens, so they are the A operand of d_W = d_proj^T xn as they are (128 accumulator
// registers for the whole run).  For d_xn they are exchanged through LDS ([channel][token]); wave (cg, kh)
// sums factor kh's channels into columns 32 cg .. + 31, and the two halves meet through LDS in float32.
// The remaining 32 KB of LDS hold in turn: xn, mask and the previous tile's half sums (phase 1), the exchange
// (phase 2).  The next tile's xn and factor gradients are in registers meanwhile.
#include <algorithm>

#include "attn_fast_common.h"
#include "trimul_kernels.h"

namespace oops {

using namespace fast;

namespace {

constexpr int kTok = 32;     // tokens per tile
constexpr int kWide = 128;   // C and H, padded
constexpr int kGradWgs = 256;
// At least this many tiles per workgroup: a tile takes about 5 us of one CU, a workgroup's 256 KB partial of
// d_W 0.1 us of the whole card's memory, which balance near three tiles for a pair of 128 x 128.
constexpr int kGradMinTiles = 3;

struct FactorGradArgs {
  const void* xn;      // [R][c_row]
  const void* w;       // [4H][c_row]
  const float* bias;   // [4H] or null
  const float* mask;   // [R] or null
  const void* gf;      // [2][G][H][P]
  void* d_xn;          // [R][C], added to
  float* w_parts;      // [run][4H][C]
  float* b_parts;      // [run][4H]
  int64_t rows, positions, groups, runs;
  int C, H, c_row, tpw;
};

// 16-byte chunk swizzle of a 64-element row.  Both reads of a tile spread over all LDS banks: the 16 rows of
// a row-fragment read (same chunk) take every slot, and so do the 8 rows x 4 chunks of a transposed read
// (whose rows r .. r + 7 would meet in half of the banks if the swizzle were (row / 2) % 8).
__device__ __forceinline__ int wide_off(int row, int col) {
  const int s = ((row << 1) & 4) | ((row >> 2) & 3);
  return row * 64 + (((col >> 3) ^ s) << 3) + (col & 7);
}
__device__ __forceinline__ TrLane wide_tr_lane(int lane, int c0) {
  const int j = lane & 15, grp = lane >> 4;
  const int col = c0 + ((grp & 1) << 4) + ((j & 3) << 2), row = ((grp >> 1) << 2) + (j >> 2);
  return TrLane{wide_off(row, col) - c0, wide_off(row + 8, col) - c0};
}

template <typename T>
__device__ __forceinline__ float lo_half(uint32_t u) {
  return (float)__builtin_bit_cast(T, (uint16_t)u);
}
template <typename T>
__device__ __forceinline__ float hi_half(uint32_t u) {
  return (float)__builtin_bit_cast(T, (uint16_t)(u >> 16));
}

// inverse of trade16: p[2q], p[2q + 1] hold the lane's entries 8q + 4 g2 + (0, 1), (2, 3)
__device__ __forceinline__ void untrade16(uint4 lo, uint4 hi, uint32_t (&p)[8]) {
  const auto y0 = __builtin_amdgcn_permlane32_swap(lo.x, lo.z, false, false);
  const auto y1 = __builtin_amdgcn_permlane32_swap(lo.y, lo.w, false, false);
  const auto y2 = __builtin_amdgcn_permlane32_swap(hi.x, hi.z, false, false);
  const auto y3 = __builtin_amdgcn_permlane32_swap(hi.y, hi.w, false, false);
  p[0] = y0[0], p[1] = y1[0], p[2] = y2[0], p[3] = y3[0];
  p[4] = y0[1], p[5] = y1[1], p[6] = y2[1], p[7] = y3[1];
}

template <typename T, bool MASKED>
__global__ __launch_bounds__(512, 2) void trimul_factor_grad_kernel(FactorGradArgs a) {
  using E = Elem<T>;
  using Frag = typename E::Frag;
  constexpr int M = 4 * kWide;
  __shared__ __attribute__((aligned(16))) T w_lds[M * kWide];  // panels of 64 columns [m][64]
  __shared__ __attribute__((aligned(16))) T x_lds[M * kTok];   // exchange [m][32 tokens], or:
  float* const half_lds = reinterpret_cast<float*>(x_lds);     //   bytes 0 .. 16 K: half sums of d_xn
  T* const xn_lds = x_lds + 8192;                              //   16 K .. 24 K: xn tile, 64-column panels [32][64]
  float* const mask_lds = reinterpret_cast<float*>(x_lds + 12288);  // 24 K ..: mask of the tile

  const int64_t run = xcd_tile(blockIdx.x, gridDim.x, 0);
  if (run >= a.runs) return;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lq = lane & 31, g2 = lane >> 5;
  const int hi4 = wave >> 2, lo4 = wave & 3;  // (factor, channel group), later (k half, column group)
  const int H = a.H, C = a.C, K = a.c_row;
  const int64_t P = a.positions;
  const int64_t tiles = a.rows / kTok, tile0 = run * a.tpw;
  const int count = (int)(tiles - tile0 < a.tpw ? tiles - tile0 : a.tpw);

  // W: row m = 256 factor + 128 (gate) + channel; rows past H and columns past c_row are zeros
  {
    const __amdgpu_buffer_rsrc_t wr = make_rsrc(a.w, (uint32_t)(4 * H * K * 2));
#pragma unroll
    for (int j = 0; j < M * kWide / 8 / 512; ++j) {
      const int id = tid + 512 * j, m = id >> 4, c = (id & 15) * 8, ch = m & 127;
      const uint4 u = buffer_load16(wr, ch < H && c < K ? (uint32_t)((((m >> 7) * H + ch) * K + c) * 2) : kOut);
      *reinterpret_cast<uint4*>(&w_lds[(c >> 6) * M * 64 + wide_off(m, c & 63)]) = u;
    }
  }

  const int ch = 32 * lo4 + lq;  // this lane's channel of factor hi4
  const bool ch_ok = ch < H;
  const int m_val = 256 * hi4 + ch;  // its value row; the gate's is 128 further
  const float bv = a.bias && ch_ok ? a.bias[hi4 * 2 * H + ch] : 0.f;
  const float bg = a.bias && ch_ok ? -a.bias[hi4 * 2 * H + H + ch] * kLog2e : 0.f;
  float bsum_v = 0.f, bsum_g = 0.f;
  f32x16 gv[4], gg[4];  // d_W of the wave's value and gate channels, columns 32 n ..
#pragma unroll
  for (int n = 0; n < 4; ++n) gv[n] = gg[n] = f32x16{};

  // next tile in registers: 16 bytes of xn, one mask value, 16 tokens of the lane's factor gradient
  const int x_row = tid >> 4, x_col = (tid & 15) * 8;
  T* const x_dst = xn_lds + (x_col >> 6) * kTok * 64 + wide_off(x_row, x_col & 63);
  int64_t g_next = tile0 * kTok / P;
  int64_t p_next = tile0 * kTok - g_next * P;
  uint4 xr = make_uint4(0, 0, 0, 0), dlo, dhi;
  float mr = 0.f;
  auto load_tile = [&](int it) {
    const int64_t r0 = (tile0 + it) * kTok;
    const bool live = it < count;
    const T* xp = static_cast<const T*>(a.xn);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(xp + (live ? r0 * K : 0), live ? (uint32_t)(kTok * K * 2) : 0u);
    xr = buffer_load16(rs, x_col < K ? (uint32_t)((x_row * K + x_col) * 2) : kOut);
    if constexpr (MASKED) mr = a.mask[live ? r0 + (tid & 31) : 0];
    const T* gp = static_cast<const T*>(a.gf);
    const bool ok = live && ch_ok;
    const T* src = gp + (ok ? ((hi4 * a.groups + g_next) * H + ch) * P + p_next + 16 * g2 : 0);
    dlo = *reinterpret_cast<const uint4*>(src);
    dhi = *reinterpret_cast<const uint4*>(src + 8);
    if (!ok) dlo = dhi = make_uint4(0, 0, 0, 0);
    p_next += kTok;
    if (p_next >= P) p_next -= P, ++g_next;
  };
  load_tile(0);

  f32x16 dacc;
  uint4 xlo, xhi;  // d_xn before this pass: 16 columns of the lane's token (half 0)
  const int c0 = 32 * lo4 + 16 * g2;
  // d_xn of tile it: this half's sums, the other's, and the values that are there, rounded once
  auto finish = [&](int it) {
    T* row = static_cast<T*>(a.d_xn) + ((tile0 + it) * kTok + lq) * C;
    uint32_t old[8], p[8];
    untrade16(xlo, xhi, old);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 h = *reinterpret_cast<const float4*>(half_lds + ((lo4 * 4 + q) * 64 + lane) * 4);
      p[2 * q] = pack2<T>(dacc[4 * q] + h.x + lo_half<T>(old[2 * q]), dacc[4 * q + 1] + h.y + hi_half<T>(old[2 * q]));
      p[2 * q + 1] = pack2<T>(dacc[4 * q + 2] + h.z + lo_half<T>(old[2 * q + 1]),
                              dacc[4 * q + 3] + h.w + hi_half<T>(old[2 * q + 1]));
    }
    uint4 lo, hi;
    trade16(p, lo, hi);
    if (c0 < C) *reinterpret_cast<uint4*>(row + c0) = lo;
    if (c0 + 8 < C) *reinterpret_cast<uint4*>(row + c0 + 8) = hi;
  };

  for (int it = 0; it < count; ++it) {
    *reinterpret_cast<uint4*>(x_dst) = xr;
    if (MASKED && tid < 32) mask_lds[tid] = mr;
    const uint4 clo = dlo, chi = dhi;
    lds_barrier();  // xn, mask and the previous tile's half sums are written (and W, the first time)
    if (hi4 == 0 && it > 0) finish(it - 1);
    load_tile(it + 1);

    // each SIMD holds one wave of either half: one half's MFMAs first, so that the other's run beside its
    // arithmetic
    if (hi4 == 0) __builtin_amdgcn_s_setprio(2);
    // ---- projections: lane = channel, entry 4q + i = token 8q + 4 g2 + i
    f32x16 av, ag;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const int col = (16 * ks & 63) + 8 * g2;
      const Frag xf = lds_frag<T>(xn_lds + (ks >> 2) * kTok * 64 + wide_off(lq, col));
      const T* wp = w_lds + (ks >> 2) * M * 64;
      av = E::mma(xf, lds_frag<T>(wp + wide_off(m_val, col)), ks == 0 ? f32x16{} : av);
      ag = E::mma(xf, lds_frag<T>(wp + wide_off(m_val + 128, col)), ks == 0 ? f32x16{} : ag);
    }
    __builtin_amdgcn_s_setprio(0);
    uint32_t d[8], pv[8], pg[8];
    untrade16(clo, chi, d);
    const TrLane t0 = wide_tr_lane(lane, 0), t1 = wide_tr_lane(lane, 32);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float4 keep = make_float4(1.f, 1.f, 1.f, 1.f);
      if constexpr (MASKED) keep = *reinterpret_cast<const float4*>(mask_lds + 8 * q + 4 * g2);
      const float k4[4] = {keep.x, keep.y, keep.z, keep.w};
      float o[4], og[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = av[4 * q + i] + bv;
        const float s = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(__builtin_fmaf(ag[4 * q + i], -kLog2e, bg)));
        const uint32_t u = d[2 * q + (i >> 1)];
        const float dk = ((i & 1) ? hi_half<T>(u) : lo_half<T>(u)) * k4[i];
        o[i] = dk * s;
        og[i] = dk * (v * s) * (1.f - s);
      }
      // the bias gradient sums the float32 values (before their rounding to the dtype)
      bsum_v += (o[0] + o[1]) + (o[2] + o[3]);
      bsum_g += (og[0] + og[1]) + (og[2] + og[3]);
      pv[2 * q] = pack2<T>(o[0], o[1]), pv[2 * q + 1] = pack2<T>(o[2], o[3]);
      pg[2 * q] = pack2<T>(og[0], og[1]), pg[2 * q + 1] = pack2<T>(og[2], og[3]);
      // ---- d_W += d_proj^T xn, 16 tokens at a time (beside the next entries' arithmetic)
      if (q & 1) {
        const int ks = q >> 1;
        const Frag fv = __builtin_bit_cast(Frag, make_uint4(pv[4 * ks], pv[4 * ks + 1], pv[4 * ks + 2], pv[4 * ks + 3]));
        const Frag fg = __builtin_bit_cast(Frag, make_uint4(pg[4 * ks], pg[4 * ks + 1], pg[4 * ks + 2], pg[4 * ks + 3]));
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          const Frag xf = lds_read_tr_frag_sw<T>(xn_lds + (n >> 1) * kTok * 64 + 16 * ks * 64 + 32 * (n & 1),
                                                 (n & 1) ? t1 : t0);
          gv[n] = E::mma(fv, xf, gv[n]);
          gg[n] = E::mma(fg, xf, gg[n]);
        }
      }
    }


    // ---- exchange: [m][32 tokens]
    uint4 vlo, vhi, glo, ghi;
    trade16(pv, vlo, vhi);
    trade16(pg, glo, ghi);
    lds_barrier();  // every wave is done with xn, mask and the half sums
    *reinterpret_cast<uint4*>(&x_lds[swz_off<32>(m_val, 16 * g2)]) = vlo;
    *reinterpret_cast<uint4*>(&x_lds[swz_off<32>(m_val, 16 * g2 + 8)]) = vhi;
    *reinterpret_cast<uint4*>(&x_lds[swz_off<32>(m_val + 128, 16 * g2)]) = glo;
    *reinterpret_cast<uint4*>(&x_lds[swz_off<32>(m_val + 128, 16 * g2 + 8)]) = ghi;
    lds_barrier();  // exchange written
    if (hi4 == 0) {
      const T* row = static_cast<const T*>(a.d_xn) + ((tile0 + it) * kTok + lq) * C;
      xlo = *reinterpret_cast<const uint4*>(row + (c0 < C ? c0 : 0));
      xhi = *reinterpret_cast<const uint4*>(row + (c0 + 8 < C ? c0 + 8 : 0));
    }

    // ---- d_xn: columns 32 lo4 .., factor hi4's 256 channels; lane = token
    const TrLane tw = lo4 & 1 ? t1 : t0, te = tr_lane<32>(lane, 0);
    const T* wt = w_lds + (lo4 >> 1) * M * 64 + 256 * hi4 * 64 + 32 * (lo4 & 1);
    const T* et = x_lds + 256 * hi4 * 32;
#pragma unroll
    for (int ks = 0; ks < 16; ++ks)
      dacc = E::mma(lds_read_tr_frag_sw<T>(wt + 16 * ks * 64, tw), lds_read_tr_frag_sw<T>(et + 16 * ks * 32, te),
                    ks == 0 ? f32x16{} : dacc);
    lds_barrier();  // every wave is done with the exchange
    if (hi4 == 1) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<float4*>(half_lds + ((lo4 * 4 + q) * 64 + lane) * 4) =
            make_float4(dacc[4 * q], dacc[4 * q + 1], dacc[4 * q + 2], dacc[4 * q + 3]);
    }
  }
  lds_barrier();
  if (hi4 == 0) finish(count - 1);

  // partials: gv[n] / gg[n] lane (lq, g2) holds channels 32 lo4 + 8q + 4 g2 + i, column 32 n + lq
  float* wp = a.w_parts + run * 4 * H * C + (int64_t)hi4 * 2 * H * C;
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const int c = 32 * n + lq;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int h = 32 * lo4 + 8 * q + 4 * g2 + i;
        if (h < H && c < C) {
          wp[(int64_t)h * C + c] = gv[n][4 * q + i];
          wp[(int64_t)(H + h) * C + c] = gg[n][4 * q + i];
        }
      }
  }
  bsum_v += __shfl_xor(bsum_v, 32);
  bsum_g += __shfl_xor(bsum_g, 32);
  if (a.b_parts && g2 == 0 && ch_ok) {
    float* bp = a.b_parts + run * 4 * H + hi4 * 2 * H + ch;
    bp[0] = bsum_v;
    bp[H] = bsum_g;
  }
}

// ------------------------------------------------------------------ gated output
// The backward of out = value * sigmoid(gate), value = nrm Wo^T + bo, gate = xn Wg^T + bg, with its products,
// in one pass over the rows (16-bit, 64 < C, H <= 128):
//
//   g_value = d_out s            d_nrm = g_value Wo     d_Wo = g_value^T nrm    d_bo = column sums
//   g_gate = d_out value s (1 - s)  d_xn = g_gate Wg    d_Wg = g_gate^T xn      d_bg = column sums
//
// As separate launches (the elementwise backward with the recomputed projections, then one pass per gradient
// for its products) the 512 x 512 pair of 128 channels took 98 + 2 x 48 us and 740 MB; the tensors that must
// move are 335 MB (68 us), and this kernel takes 86 us.  The scheme is the one above with both weights (2 x 32 KB) in LDS: wave (grp, th)
// owns channels 32 grp .. + 31 of the tile's tokens 32 th .. + 31; d_out comes through the transposed read in
// the accumulators' order.  The tiles (64 tokens) come by direct-to-LDS loads one tile ahead, the exchange
// takes the place of its tile's inputs.  The two token halves' weight gradients meet in LDS at the end.
constexpr int kOutTok = 64;

struct OutputGradArgs {
  const void* nrm;   // [R][h_row]
  const void* xn;    // [R][c_row]
  const void* wo;    // [C][h_row]
  const void* wg;    // [C][c_row]
  const float* bo;
  const float* bg;
  const void* gout;  // [R][C], or [n * n][C] of a padded pair
  void* d_nrm;       // [R][H]
  void* d_xn;        // [R][C]
  float* wo_parts;   // [run][C][H]
  float* wg_parts;   // [run][C][C]
  float* b_parts;    // [2][run][C]
  int64_t rows, runs;
  int C, H, c_row, h_row, tpw;
  uint32_t n, n_pad;  // padded pair: sides of the pair and of the grid of the rows (else 0)
};

template <typename T>
__global__ __launch_bounds__(512, 2) void trimul_output_grads_kernel(OutputGradArgs a) {
  using E = Elem<T>;
  using Frag = typename E::Frag;
  constexpr int RT = kOutTok, TILE = RT * kWide, WT = kWide * kWide;
  // wo, wg; two slots of nrm, xn and d_out tiles (a slot's first 32 KB are its tile's exchange [256 m][64 tokens]
  // afterwards); at the end a token half's weight gradients
  __shared__ __attribute__((aligned(16))) T lds[2 * WT + 6 * TILE];
  static_assert(sizeof(lds) >= (4 * 128 * 64 + 2 * kWide) * sizeof(float), "final sums");
  T* const wo_l = lds;
  T* const wg_l = lds + WT;

  const int64_t run = xcd_tile(blockIdx.x, gridDim.x, 0);
  if (run >= a.runs) return;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lq = lane & 31, g2 = lane >> 5;
  const int grp = wave & 3, th = wave >> 2;
  const int C = a.C, H = a.H;
  const int64_t R = a.rows;
  const int64_t tiles = (R + RT - 1) / RT, tile0 = run * a.tpw;
  const int count = (int)(tiles - tile0 < a.tpw ? tiles - tile0 : a.tpw);

  {
    const __amdgpu_buffer_rsrc_t r1 = make_rsrc(a.wo, (uint32_t)(C * a.h_row * 2));
    const __amdgpu_buffer_rsrc_t r2 = make_rsrc(a.wg, (uint32_t)(C * a.c_row * 2));
#pragma unroll
    for (int j = 0; j < WT / 8 / 512; ++j) {
      const int id = tid + 512 * j, m = id >> 4, c = (id & 15) * 8;
      const int o = (c >> 6) * kWide * 64 + wide_off(m, c & 63);
      const uint4 u1 = buffer_load16(r1, m < C && c < a.h_row ? (uint32_t)((m * a.h_row + c) * 2) : kOut);
      const uint4 u2 = buffer_load16(r2, m < C && c < a.c_row ? (uint32_t)((m * a.c_row + c) * 2) : kOut);
      *reinterpret_cast<uint4*>(&wo_l[o]) = u1;
      *reinterpret_cast<uint4*>(&wg_l[o]) = u2;
    }
  }

  const int ch = 32 * grp + lq;  // this lane's channel
  const float bv = a.bo && ch < C ? a.bo[ch] : 0.f;
  const float bg = a.bg && ch < C ? -a.bg[ch] * kLog2e : 0.f;
  float bsum_v = 0.f, bsum_g = 0.f;
  f32x16 gv[4], gg[4];  // d_Wo and d_Wg of the wave's channels, columns 32 n ..
#pragma unroll
  for (int n = 0; n < 4; ++n) gv[n] = gg[n] = f32x16{};

  // tile it's rows into its slot by direct-to-LDS loads (rows past R: zeros): this lane's row and columns of
  // the wave's two 1 KB pieces of each input
  int d_row[2], d_col[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int slot = (wave * 2 + k) * 64 + lane;
    d_row[k] = (slot >> 3) % RT;
    d_col[k] = (slot / (RT * 8)) * 64 + (wide_off(d_row[k], (slot & 7) * 8) - d_row[k] * 64);
  }
  auto request = [&](int it) {
    const int64_t r0 = (tile0 + it) * RT;
    const int64_t left = it < count ? R - r0 : 0;
    const int nrows = (int)(left < RT ? left : RT);
    const int64_t base = nrows ? r0 : 0;
    const u32x4 s1 = rsrc_words(static_cast<const T*>(a.nrm) + base * a.h_row, (uint32_t)(nrows * a.h_row * 2));
    const u32x4 s2 = rsrc_words(static_cast<const T*>(a.xn) + base * a.c_row, (uint32_t)(nrows * a.c_row * 2));
    // d_out rows: of the tile, or of the pair's cells from the tile's first grid row on
    int64_t u0 = base;
    uint32_t u_bytes = (uint32_t)(nrows * C * 2), i0 = 0;
    if (a.n) {
      i0 = (uint32_t)base / a.n_pad;
      const bool in = nrows && i0 < a.n;
      u0 = in ? (int64_t)i0 * a.n : 0;
      u_bytes = in ? (uint32_t)(((int64_t)a.n * a.n - u0) * C * 2) : 0u;
    }
    const u32x4 s3 = rsrc_words(static_cast<const T*>(a.gout) + u0 * C, u_bytes);
    T* const at = lds + 2 * WT + (it & 1) * 3 * TILE + wave * 1024;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int r = d_row[k], c = d_col[k];
      const bool ok = r < nrows;
      dma16_asm(s1, at + 512 * k, ok && c < a.h_row ? (uint32_t)((r * a.h_row + c) * 2) : kOut, 0);
      dma16_asm(s2, at + TILE + 512 * k, ok && c < a.c_row ? (uint32_t)((r * a.c_row + c) * 2) : kOut, 0);
      uint32_t u = (uint32_t)r;
      bool live = ok && c < C;
      if (a.n) {
        const uint32_t p = (uint32_t)base + (uint32_t)r, i = p / a.n_pad, j = p - i * a.n_pad;
        u = (i - i0) * a.n + j;
        live = live && i < a.n && j < a.n;
      }
      dma16_asm(s3, at + 2 * TILE + 512 * k, live ? (u * (uint32_t)C + (uint32_t)c) * 2 : kOut, 0);
    }
  };
  vmem_wait_all();  // no compiler-visible load outstanding once the requests start
  request(0);

  const TrLane t0 = wide_tr_lane(lane, 0), t1 = wide_tr_lane(lane, 32);
  const TrLane tg = grp & 1 ? t1 : t0, tt = th ? t1 : t0;
  const int c0 = 32 * grp + 16 * g2;
  for (int it = 0; it < count; ++it) {
    // tile it has arrived (four stores per iteration were issued after its request)
    if (it > 0)
      vmem_wait<4>();
    else
      vmem_wait<0>();
    lds_barrier();  // the tile (and the weights) are written; every wave is done with the other slot
    request(it + 1);
    T* const nrm_l = lds + 2 * WT + (it & 1) * 3 * TILE;
    T* const xn_l = nrm_l + TILE;
    T* const do_l = xn_l + TILE;
    T* const ex_l = nrm_l;
    const int64_t r0 = (tile0 + it) * RT + 32 * th;  // this wave's tokens

    // ---- projections: lane = channel, entry 4q + i = token 8q + 4 g2 + i.  Each SIMD holds one wave of
    // either token half: one half's MFMAs first, so that the other's run beside its arithmetic
    if (th == 0) __builtin_amdgcn_s_setprio(2);
    f32x16 av, ag;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const int col = (16 * ks & 63) + 8 * g2;
      const int xo = (ks >> 2) * RT * 64 + wide_off(32 * th + lq, col), wo = (ks >> 2) * kWide * 64 + wide_off(ch, col);
      av = E::mma(lds_frag<T>(nrm_l + xo), lds_frag<T>(wo_l + wo), ks == 0 ? f32x16{} : av);
      ag = E::mma(lds_frag<T>(xn_l + xo), lds_frag<T>(wg_l + wo), ks == 0 ? f32x16{} : ag);
    }
    __builtin_amdgcn_s_setprio(0);
    uint32_t pv[8], pg[8];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int slab = (32 * th + 16 * ks) * 64;
      const Frag df = lds_read_tr_frag_sw<T>(do_l + (grp >> 1) * RT * 64 + slab + 32 * (grp & 1), tg);
#pragma unroll
      for (int qq = 0; qq < 2; ++qq) {
        const int q = 2 * ks + qq;
        float o[4], og[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float v = av[4 * q + i] + bv, d = (float)df[4 * qq + i];
          const float s = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(__builtin_fmaf(ag[4 * q + i], -kLog2e, bg)));
          o[i] = d * s;
          og[i] = d * v * s * (1.f - s);
        }
        bsum_v += (o[0] + o[1]) + (o[2] + o[3]);
        bsum_g += (og[0] + og[1]) + (og[2] + og[3]);
        pv[2 * q] = pack2<T>(o[0], o[1]), pv[2 * q + 1] = pack2<T>(o[2], o[3]);
        pg[2 * q] = pack2<T>(og[0], og[1]), pg[2 * q + 1] = pack2<T>(og[2], og[3]);
      }
      // ---- d_Wo += g_value^T nrm, d_Wg += g_gate^T xn
      const Frag fv = __builtin_bit_cast(Frag, make_uint4(pv[4 * ks], pv[4 * ks + 1], pv[4 * ks + 2], pv[4 * ks + 3]));
      const Frag fg = __builtin_bit_cast(Frag, make_uint4(pg[4 * ks], pg[4 * ks + 1], pg[4 * ks + 2], pg[4 * ks + 3]));
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const int at = (n >> 1) * RT * 64 + slab + 32 * (n & 1);
        gv[n] = E::mma(fv, lds_read_tr_frag_sw<T>(nrm_l + at, (n & 1) ? t1 : t0), gv[n]);
        gg[n] = E::mma(fg, lds_read_tr_frag_sw<T>(xn_l + at, (n & 1) ? t1 : t0), gg[n]);
      }
    }
    // ---- exchange: [m][64 tokens], m = channel (value), 128 + channel (gate)
    lds_barrier();  // every wave is done with the inputs
    uint4 lo, hi;
    trade16(pv, lo, hi);
    *reinterpret_cast<uint4*>(&ex_l[wide_off(ch, 32 * th + 16 * g2)]) = lo;
    *reinterpret_cast<uint4*>(&ex_l[wide_off(ch, 32 * th + 16 * g2 + 8)]) = hi;
    trade16(pg, lo, hi);
    *reinterpret_cast<uint4*>(&ex_l[wide_off(kWide + ch, 32 * th + 16 * g2)]) = lo;
    *reinterpret_cast<uint4*>(&ex_l[wide_off(kWide + ch, 32 * th + 16 * g2 + 8)]) = hi;
    lds_barrier();  // exchange written

    // ---- d_nrm and d_xn: columns 32 grp .., tokens 32 th ..; lane = token
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const T* wt = (k ? wg_l : wo_l) + (grp >> 1) * kWide * 64 + 32 * (grp & 1);
      const T* et = ex_l + k * kWide * 64 + 32 * th;
      f32x16 acc;
#pragma unroll
      for (int ks = 0; ks < 8; ++ks)
        acc = E::mma(lds_read_tr_frag_sw<T>(wt + 16 * ks * 64, tg), lds_read_tr_frag_sw<T>(et + 16 * ks * 64, tt),
                     ks == 0 ? f32x16{} : acc);
      uint32_t p[8];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        p[2 * q] = pack2<T>(acc[4 * q], acc[4 * q + 1]);
        p[2 * q + 1] = pack2<T>(acc[4 * q + 2], acc[4 * q + 3]);
      }
      trade16(p, lo, hi);
      const int width = k ? C : H;
      const int64_t left = R - r0;
      const int nrows = (int)(left < 0 ? 0 : left < 32 ? left : 32);
      const __amdgpu_buffer_rsrc_t ds =
          make_rsrc(static_cast<T*>(k ? a.d_xn : a.d_nrm) + (nrows ? r0 : 0) * width, (uint32_t)(nrows * width * 2));
      const uint32_t off = (uint32_t)((lq * width + c0) * 2);
      buffer_store16(ds, lq < nrows && c0 < width ? off : kOut, lo);
      buffer_store16(ds, lq < nrows && c0 + 8 < width ? off + 16 : kOut, hi);
    }
  }

  // the second token half's sums through LDS (32 KB per channel group, then the bias sums)
  vmem_wait_all();  // the last request has landed
  __syncthreads();
  float* const red = reinterpret_cast<float*>(lds) + grp * 128 * 64;
  float* const bred = reinterpret_cast<float*>(lds) + 4 * 128 * 64;
  bsum_v += __shfl_xor(bsum_v, 32);
  bsum_g += __shfl_xor(bsum_g, 32);
  if (th == 1) {
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        red[(16 * n + e) * 64 + lane] = gv[n][e];
        red[(64 + 16 * n + e) * 64 + lane] = gg[n][e];
      }
    if (g2 == 0) bred[ch] = bsum_v, bred[kWide + ch] = bsum_g;
  }
  __syncthreads();
  if (th == 0) {
    float* op = a.wo_parts + run * C * H;
    float* gp = a.wg_parts + run * C * C;
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const int c = 32 * n + lq;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = 32 * grp + 8 * q + 4 * g2 + i, e = 4 * q + i;
          if (m < C && c < H) op[(int64_t)m * H + c] = gv[n][e] + red[(16 * n + e) * 64 + lane];
          if (m < C && c < C) gp[(int64_t)m * C + c] = gg[n][e] + red[(64 + 16 * n + e) * 64 + lane];
        }
    }
    if (g2 == 0 && ch < C) {
      a.b_parts[run * C + ch] = bsum_v + bred[ch];
      a.b_parts[(a.runs + run) * C + ch] = bsum_g + bred[kWide + ch];
    }
  }
}

struct GradRuns {
  int tpw;
  int64_t runs;
};
GradRuns grad_runs(const oops_trimul_geometry& g, int tokens) {
  const int64_t tiles = (g.groups * g.positions + tokens - 1) / tokens;
  const int64_t tpw = std::max<int64_t>(kGradMinTiles, (tiles + kGradWgs - 1) / kGradWgs);
  return {(int)tpw, (tiles + tpw - 1) / tpw};
}

}  // namespace

int64_t trimul_factor_grad_parts(const oops_trimul_geometry& g) {
  if (g.dtype != OOPS_BF16 && g.dtype != OOPS_F16) return 0;
  if (g.hidden <= 64 || g.hidden > kWide || g.c_row <= 64 || g.c_row > kWide || g.channels % 8 || g.c_row % 8) return 0;
  if (g.groups < 1 || g.positions < kTok || g.positions % kTok) return 0;
  return grad_runs(g, kTok).runs;
}

hipError_t launch_trimul_factor_grad(const oops_trimul_geometry& g, const void* normalized, const void* weight,
                                     const float* bias, const float* mask, const void* grad_factors, void* grad_xn,
                                     float* w_parts, float* b_parts, hipStream_t stream) {
  FactorGradArgs a{};
  a.xn = normalized, a.w = weight, a.bias = bias, a.mask = mask, a.gf = grad_factors;
  a.d_xn = grad_xn, a.w_parts = w_parts, a.b_parts = b_parts;
  a.rows = g.groups * g.positions, a.positions = g.positions, a.groups = g.groups;
  a.C = g.channels, a.H = g.hidden, a.c_row = (int)g.c_row;
  const GradRuns pl = grad_runs(g, kTok);
  a.tpw = pl.tpw, a.runs = pl.runs;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)xcd_grid(a.runs, 0)), dim3(512), 0, stream, a);
    return hipGetLastError();
  };
  if (g.dtype == OOPS_BF16)
    return mask ? go(trimul_factor_grad_kernel<__bf16, true>) : go(trimul_factor_grad_kernel<__bf16, false>);
  if (g.dtype == OOPS_F16)
    return mask ? go(trimul_factor_grad_kernel<_Float16, true>) : go(trimul_factor_grad_kernel<_Float16, false>);
  return hipErrorInvalidValue;
}

int64_t trimul_output_grads_parts(const oops_trimul_geometry& g) {
  if (g.dtype != OOPS_BF16 && g.dtype != OOPS_F16) return 0;
  if (g.hidden <= 64 || g.hidden > kWide || g.channels <= 64 || g.channels > kWide) return 0;
  if (g.channels % 8 || g.hidden % 8 || g.c_row != g.channels || g.h_row != g.hidden) return 0;
  if (g.groups < 1 || g.positions < 1 || g.groups * g.positions >= (int64_t(1) << 31)) return 0;
  return grad_runs(g, kOutTok).runs;
}

hipError_t launch_trimul_output_grads(const oops_trimul_geometry& g, int64_t n, int64_t n_pad, const void* normalized,
                                      const void* pair_normalized, const void* output_weight, const void* gate_weight,
                                      const float* output_bias, const float* gate_bias, const void* grad_out,
                                      void* grad_normalized, void* grad_xn, float* wo_parts, float* wg_parts,
                                      float* b_parts, hipStream_t stream) {
  OutputGradArgs a{};
  a.nrm = normalized, a.xn = pair_normalized, a.wo = output_weight, a.wg = gate_weight;
  a.bo = output_bias, a.bg = gate_bias, a.gout = grad_out, a.d_nrm = grad_normalized, a.d_xn = grad_xn;
  a.wo_parts = wo_parts, a.wg_parts = wg_parts, a.b_parts = b_parts;
  a.rows = g.groups * g.positions, a.C = g.channels, a.H = g.hidden, a.c_row = (int)g.c_row, a.h_row = (int)g.h_row;
  a.n = (uint32_t)n, a.n_pad = (uint32_t)n_pad;
  const GradRuns pl = grad_runs(g, kOutTok);
  a.tpw = pl.tpw, a.runs = pl.runs;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)xcd_grid(a.runs, 0)), dim3(512), 0, stream, a);
    return hipGetLastError();
  };
  if (g.dtype == OOPS_BF16) return go(trimul_output_grads_kernel<__bf16>);
  if (g.dtype == OOPS_F16) return go(trimul_output_grads_kernel<_Float16>);
  return hipErrorInvalidValue;
}

}  // namespace oops
