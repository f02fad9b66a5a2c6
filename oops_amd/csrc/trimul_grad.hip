// The factor projections' backward of the triangle multiplication in one pass over the tokens (gfx950):
// 16-bit pairs with 64 < C, H <= 128 and positions a multiple of 32, no mask gradient.
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

struct GradRuns {
  int tpw;
  int64_t runs;
};
GradRuns grad_runs(const oops_trimul_geometry& g) {
  const int64_t tiles = g.groups * g.positions / kTok;
  const int64_t tpw = std::max<int64_t>(kGradMinTiles, (tiles + kGradWgs - 1) / kGradWgs);
  return {(int)tpw, (tiles + tpw - 1) / tpw};
}

}  // namespace

int64_t trimul_factor_grad_parts(const oops_trimul_geometry& g) {
  if (g.dtype != OOPS_BF16 && g.dtype != OOPS_F16) return 0;
  if (g.hidden <= 64 || g.hidden > kWide || g.c_row <= 64 || g.c_row > kWide || g.channels % 8 || g.c_row % 8) return 0;
  if (g.groups < 1 || g.positions < kTok || g.positions % kTok) return 0;
  return grad_runs(g).runs;
}

hipError_t launch_trimul_factor_grad(const oops_trimul_geometry& g, const void* normalized, const void* weight,
                                     const float* bias, const float* mask, const void* grad_factors, void* grad_xn,
                                     float* w_parts, float* b_parts, hipStream_t stream) {
  FactorGradArgs a{};
  a.xn = normalized, a.w = weight, a.bias = bias, a.mask = mask, a.gf = grad_factors;
  a.d_xn = grad_xn, a.w_parts = w_parts, a.b_parts = b_parts;
  a.rows = g.groups * g.positions, a.positions = g.positions, a.groups = g.groups;
  a.C = g.channels, a.H = g.hidden, a.c_row = (int)g.c_row;
  const GradRuns pl = grad_runs(g);
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

}  // namespace oops
