// The gated output stage as whole passes over its rows (gfx950, 16-bit operands, C, H*D and O at most 256, or
// at most 384 for few rows):
//
//   forward       out = (round(sigmoid(single Wg^T)) * attention) Wo^T           gate_stage_forward_kernel
//   backward 1    d_gated = d_out Wo, its gate backward, d_Wo = d_out^T gated    row_grad_kernel<GATE>
//   backward 2    d_single = d_logits Wg, d_Wg = d_logits^T single               row_grad_kernel
//
// What bounds them is HBM: at C = H*D = O = 256 the products are 25.8 GFLOP each per 196608 rows (about
// 20 us of MFMA) while every tensor of the stage is 100 MB (20 us per pass).  Each kernel therefore reads
// and writes every row once: the gated rows and their gradient live in LDS and registers only, and the
// backward rebuilds the gated rows from the logits with the forward's roundings (the same bits).
//
// One workgroup of 8 waves per CU walks a run of row tiles.  The weights stay in registers as MFMA operands
// (at 256 x 256 each wave holds a 32-column share: 64 registers per weight), the row tiles come through an
// LDS ring filled by direct-to-LDS loads several tiles ahead, and the weight-gradient sums stay in
// accumulators over the whole run (one float32 partial per workgroup, summed by oops_sum_partials).
// At 196608 rows of 256 channels in bf16, against the separate launches (projection kernel, gate kernels,
// library GEMMs, chunked weight gradients): forward 108 us for 149, backward 1 142 us for 205, backward 2
// 85 us for 119, the stage forward and backward 484 -> 306 us.  Few rows gain from the launches: 128 rows
// forward 50 -> 18 us, forward and backward 256 -> 183 us, so there is no lower limit on the rows (replayed
// from a graph, 384 channels: forward and backward 36 us at 8 rows for 29 of separate launches, 37 for 35 at 64, 38
// for 41 at 128; those launches clear a GEMM workspace with a memset, which does not belong in a graph).  The
// upper limits are the register file's: both 256-wide weights fit beside the forward's accumulators, a 384-wide
// one beside the gradients' (with a few spilled registers).
//
// A tile is stored as 64-column panels [row][64] with XOR-swizzled 16-byte chunks, so that a row-fragment
// read (one operand of X W) and a transposed read (both operands of X^T Y) come from the same copy.
#include <algorithm>
#include <initializer_list>

#include "attn_fast_common.h"
#include "gate_device.h"
#include "gate_kernels.h"

namespace oops {

using namespace fast;

namespace {

constexpr int kStageCols = 128;  // columns of D and of the weight gradient per workgroup (row_grad_kernel)
constexpr int kStageRows = 64;   // rows per tile (row_grad_kernel)
constexpr int kStageWgs = 256;   // workgroups: one per CU
constexpr int kWideCols = 384;   // the largest C, H*D and O
// Past 256 channels the forward streams its weights for every 32 rows, which is right for few rows only: forward
// / forward and backward at 384 channels, replayed from a graph, against the separate launches: 384 rows 11 / 40 us
// for 12 / 41, 2048 rows 11 / 49 for 15 / 68, 16384 rows 23 / 89 us for 35 / 147 (eager, where the host's time is
// most of it: 18 / 175 for 55 / 288 and 22 / 172 for 55 / 328).
constexpr int64_t kWideRows = 16384;
// From 129 to 256 channels the streaming forward serves one tile per CU: one short workgroup each beats the
// prologue of the kernel that keeps the weights (replayed at 256 channels: 8.0 us for 12.1 at 384 rows, 9.2 for 12.9
// at 8192 rows), which walks more rows than that (16.1 for 16384 rows).
constexpr int64_t kStreamRows = kStageWgs * 32;

struct StageArgs {
  const void* x;       // forward: single [rows][kx]; gradients: X [rows][kx]
  const void* w;       // forward: Wg [n][kx]; gradients: W [kx][n]
  const void* w_out;   // forward: Wo [o][n]
  const void* y;       // attention values (forward, GATE) or Y [rows][n]
  const void* logits;  // GATE: logits [rows][n]
  void* d;             // forward: out [rows][o]; GATE: attention gradient [rows][n]; else D [rows][n]
  void* e;             // forward: logits [rows][n] (training); GATE: logit gradient [rows][n]
  float* parts;        // X^T Y partials [run][kx][n]
  int64_t rows, x_row, w_row, w_out_row, y_row, d_row;
  int64_t tiles;  // workgroups with work: runs x column blocks
  uint32_t tokens, groups, a_sb, a_sg, a_st, a_sh, a_bytes;
  int kx, n, o, width;
  int tpw;  // row tiles per run
};

// 16 bytes of a tile: tile row and first column of a direct-to-LDS slot (64-column panels of ROWS rows)
template <int ROWS>
struct Slot {
  int row, col;
  __device__ __forceinline__ explicit Slot(int s) {
    row = (s >> 3) % ROWS;
    col = (s / (ROWS * 8)) * 64 + (((s & 7) ^ swz<64>(row)) << 3);
  }
};
template <int ROWS>
__device__ __forceinline__ int panel_off(int row, int col) {
  return (col >> 6) * ROWS * 64 + swz_off<64>(row, col & 63);
}

// byte offset of row r's attention values (head 0, channel 0); the host checked that the extent is below
// 2^31 bytes
__device__ __forceinline__ uint32_t att_row_bytes(const StageArgs& a, uint32_t r) {
  const uint32_t smp = r / a.tokens, t = r - smp * a.tokens;
  const uint32_t b = smp / a.groups, g = smp - b * a.groups;
  return 2 * (b * a.a_sb + g * a.a_sg + t * a.a_st);
}

// Wait until the tile that was requested NS - 1 iterations ago has arrived: LOADS requests per tile and
// STORES stores per iteration of this wave were issued after it (vector-memory operations complete in
// order), fewer in the first iterations.
template <int NS, int STORES, int LOADS>
__device__ __forceinline__ void wait_tile(int it) {
  if (it >= 3 && NS > 3) return vmem_wait<(NS > 3 ? 3 : 0) * STORES + (NS - 2) * LOADS>();
  if (it >= 2 && NS > 2) return vmem_wait<(NS > 2 ? 2 : 0) * STORES + (NS - 2) * LOADS>();
  if (it >= 1) return vmem_wait<STORES + (NS - 2) * LOADS>();
  vmem_wait<(NS - 2) * LOADS>();
}

// an accumulator tile (lane: MFMA column = tile row, 16 of 32 tile columns) rounded to T as 2 x 8 columns
template <typename T>
__device__ __forceinline__ void round_run(const f32x16& acc, uint4& lo, uint4& hi) {
  uint32_t p[8];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    p[2 * q] = pack2<T>(acc[4 * q], acc[4 * q + 1]);
    p[2 * q + 1] = pack2<T>(acc[4 * q + 2], acc[4 * q + 3]);
  }
  trade16(p, lo, hi);
}

template <typename T>
__device__ __forceinline__ uint4 gate_product(uint4 logits, uint4 att) {
  const T* l = reinterpret_cast<const T*>(&logits);
  const T* v = reinterpret_cast<const T*>(&att);
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    o[i] = pack2<T>(rnd<T>(sigmoid_f(to_f(l[2 * i]))) * to_f(v[2 * i]),
                    rnd<T>(sigmoid_f(to_f(l[2 * i + 1]))) * to_f(v[2 * i + 1]));
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// gate_multiply_backward's steps (with its roundings) and the gated values
template <typename T>
__device__ __forceinline__ void gate_backward_run(uint4 grad, uint4 att, uint4 logits, uint4& d_att, uint4& d_logits,
                                                  uint4& gated) {
  const T* gr = reinterpret_cast<const T*>(&grad);
  const T* av = reinterpret_cast<const T*>(&att);
  const T* lg = reinterpret_cast<const T*>(&logits);
  uint32_t da[4], dl[4], gv[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a2[2], l2[2], g2[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const float d = to_f(gr[2 * i + k]), v = to_f(av[2 * i + k]);
      const float g = rnd<T>(sigmoid_f(to_f(lg[2 * i + k])));
      a2[k] = d * g;
      l2[k] = rnd<T>(rnd<T>(d * v) * rnd<T>(1.0f - g)) * g;
      g2[k] = g * v;
    }
    da[i] = pack2<T>(a2[0], a2[1]);
    dl[i] = pack2<T>(l2[0], l2[1]);
    gv[i] = pack2<T>(g2[0], g2[1]);
  }
  d_att = make_uint4(da[0], da[1], da[2], da[3]);
  d_logits = make_uint4(dl[0], dl[1], dl[2], dl[3]);
  gated = make_uint4(gv[0], gv[1], gv[2], gv[3]);
}

// ------------------------------------------------------------------ forward
// P: C, H*D and O padded (128 or 256; columns past the real ones are read as zeros and not stored).  A tile
// is 8192 / P rows; wave (cg, rg) computes gate channels, then output channels 32 cg .. + 31 of tile rows
// 32 rg .. + 31, the tile row being the MFMA column.  The gated values overwrite the attention values in LDS
// (each element by the lane that read it), where the second product reads them.
template <typename T, int P, bool LOGITS>
__global__ __launch_bounds__(512, 2) void gate_stage_forward_kernel(StageArgs a) {
  using E = Elem<T>;
  using Frag = typename E::Frag;
  constexpr int RT = 8192 / P, TILE = RT * P, KS = P / 16, CG = P / 32, NS = 4;
  constexpr int STORES = LOGITS ? 4 : 2, LOADS = 4;
  __shared__ __attribute__((aligned(16))) T ring[NS][2][TILE];  // single, attention -> gated

  const int64_t wg = xcd_tile(blockIdx.x, gridDim.x, 0);
  if (wg >= a.tiles) return;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lq = lane & 31, g2 = lane >> 5;
  const int cg = wave % CG, rg = wave / CG;
  const int64_t tiles_m = (a.rows + RT - 1) / RT, tile0 = wg * a.tpw;
  const int count = (int)(tiles_m - tile0 < a.tpw ? tiles_m - tile0 : a.tpw);

  // this wave's weight rows as MFMA operands (lane: channel 32 cg + lq, k = 16 ks + 8 g2 ..)
  Frag wg_f[KS], wo_f[KS];
  {
    const int c = 32 * cg + lq;
    const __amdgpu_buffer_rsrc_t r1 = make_rsrc(a.w, (uint32_t)(((a.n - 1) * a.w_row + a.kx) * 2));
    const __amdgpu_buffer_rsrc_t r2 = make_rsrc(a.w_out, (uint32_t)(((a.o - 1) * a.w_out_row + a.n) * 2));
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int k = 16 * ks + 8 * g2;
      wg_f[ks] = __builtin_bit_cast(
          Frag, buffer_load16(r1, c < a.n && k < a.kx ? (uint32_t)((c * a.w_row + k) * 2) : kOut));
      wo_f[ks] = __builtin_bit_cast(
          Frag, buffer_load16(r2, c < a.o && k < a.n ? (uint32_t)((c * a.w_out_row + k) * 2) : kOut));
    }
  }
  vmem_wait_all();  // no compiler-visible load outstanding once the ring's requests start

  // this lane's two slots of each tile
  const Slot<RT> s0(wave * 128 + lane), s1(wave * 128 + 64 + lane);
  auto att_col = [&](int n) { return 2 * ((uint32_t)(n / a.width) * a.a_sh + (uint32_t)(n % a.width)); };
  const uint32_t x0 = s0.col < a.kx ? (uint32_t)((s0.row * a.x_row + s0.col) * 2) : kOut;
  const uint32_t x1 = s1.col < a.kx ? (uint32_t)((s1.row * a.x_row + s1.col) * 2) : kOut;
  const uint32_t y0 = att_col(s0.col), y1 = att_col(s1.col);
  const bool v0 = s0.col < a.n, v1 = s1.col < a.n;
  const u32x4 ys = rsrc_words(a.y, a.a_bytes);
  auto request = [&](int it) {
    const int64_t r0 = (tile0 + it) * RT;
    const int64_t left = it < count ? a.rows - r0 : 0;
    const int nrows = (int)(left < RT ? left : RT);
    const u32x4 xs = rsrc_words(static_cast<const T*>(a.x) + (nrows ? r0 * a.x_row : 0),
                                nrows ? (uint32_t)(((nrows - 1) * a.x_row + a.kx) * 2) : 0u);
    T* xt = ring[it % NS][0] + wave * 1024;
    T* yt = ring[it % NS][1] + wave * 1024;
    const uint32_t r = (uint32_t)r0;
    dma16_asm(xs, xt, s0.row < nrows ? x0 : kOut, 0);
    dma16_asm(xs, xt + 512, s1.row < nrows ? x1 : kOut, 0);
    dma16_asm(ys, yt, v0 && s0.row < nrows ? att_row_bytes(a, r + s0.row) + y0 : kOut, 0);
    dma16_asm(ys, yt + 512, v1 && s1.row < nrows ? att_row_bytes(a, r + s1.row) + y1 : kOut, 0);
  };
#pragma unroll
  for (int it = 0; it < NS - 1; ++it) request(it);

  const int row = 32 * rg + lq, c0 = 32 * cg + 16 * g2;
  for (int it = 0; it < count; ++it) {
    wait_tile<NS, STORES, LOADS>(it);
    lds_barrier();          // tile it written by every wave; every wave is past tile it - 1
    request(it + NS - 1);  // into tile it - 1's slot
    const T* xt = ring[it % NS][0];
    T* yt = ring[it % NS][1];
    const int64_t r0 = (tile0 + it) * RT;
    const int64_t left = a.rows - r0;
    const int nrows = (int)(left < RT ? left : RT);
    uint4 lo, hi;
    {
      f32x16 acc = f32x16{};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        acc = E::mma(wg_f[ks], lds_frag<T>(xt + panel_off<RT>(row, 16 * ks + 8 * g2)), acc);
      round_run<T>(acc, lo, hi);  // the logits of channels c0 .. c0 + 15
    }
    if constexpr (LOGITS) {
      const __amdgpu_buffer_rsrc_t lr = make_rsrc(static_cast<T*>(a.e) + r0 * a.n, (uint32_t)(nrows * a.n * 2));
      const uint32_t off = (uint32_t)((row * a.n + c0) * 2);
      buffer_store16(lr, row < nrows && c0 < a.n ? off : kOut, lo);
      buffer_store16(lr, row < nrows && c0 + 8 < a.n ? off + 16 : kOut, hi);
    }
    uint4* p0 = reinterpret_cast<uint4*>(yt + panel_off<RT>(row, c0));
    uint4* p1 = reinterpret_cast<uint4*>(yt + panel_off<RT>(row, c0 + 8));
    // (columns past H*D stay zero whatever their padded logits are: an infinite `single` makes those NaN)
    *p0 = c0 < a.n ? gate_product<T>(lo, *p0) : make_uint4(0, 0, 0, 0);
    *p1 = c0 + 8 < a.n ? gate_product<T>(hi, *p1) : make_uint4(0, 0, 0, 0);
    lds_barrier();  // gated rows written
    f32x16 acc = f32x16{};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      acc = E::mma(wo_f[ks], lds_frag<T>(yt + panel_off<RT>(row, 16 * ks + 8 * g2)), acc);
    round_run<T>(acc, lo, hi);
    const __amdgpu_buffer_rsrc_t orr = make_rsrc(static_cast<T*>(a.d) + r0 * a.o, (uint32_t)(nrows * a.o * 2));
    const uint32_t off = (uint32_t)((row * a.o + c0) * 2);
    buffer_store16(orr, row < nrows && c0 < a.o ? off : kOut, lo);
    buffer_store16(orr, row < nrows && c0 + 8 < a.o ? off + 16 : kOut, hi);
  }
  vmem_wait_all();  // the ring's last requests land before the LDS is given back
}

constexpr int kWideThreads = kWideCols / 32 * 64;

// All but the last N vector-memory operations of this wave are done (no LDS read moves above it)
template <int N>
__device__ __forceinline__ void own_loads_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// The forward for 129 to 384 channels and few rows (the single representation): one 32-row tile per workgroup, one
// wave per 32 channels.  The weights do not fit in a workgroup's registers or LDS, so each wave streams its own 32
// rows of either in blocks of 64 columns through two LDS slots of its own (direct-to-LDS loads of whole 128-byte
// lines, the next block in flight; no barrier).  That stream bounds it: 590 KB per workgroup.  Fragments loaded
// straight from the rows touch 32 lines per load and made it 19 us at 384 rows of 384 channels for 10.8 now.
template <typename T, bool LOGITS>
__global__ __launch_bounds__(kWideThreads, 3) void gate_stage_wide_kernel(StageArgs a) {
  using E = Elem<T>;
  using Frag = typename E::Frag;
  constexpr int RT = 32, P = kWideCols, BLK = 32 * 64;  // BLK: elements of a weight block
  __shared__ __attribute__((aligned(16))) T x_lds[RT * P];
  __shared__ __attribute__((aligned(16))) T y_lds[RT * P];  // attention -> gated
  __shared__ __attribute__((aligned(16))) T w_lds[kWideThreads / 64][2][BLK];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lq = lane & 31, g2 = lane >> 5;
  const int64_t r0 = (int64_t)blockIdx.x * RT;
  const int nrows = (int)(a.rows - r0 < RT ? a.rows - r0 : RT);
  {
    const u32x4 xs = rsrc_words(static_cast<const T*>(a.x) + r0 * a.x_row, (uint32_t)(((nrows - 1) * a.x_row + a.kx) * 2));
    const u32x4 ys = rsrc_words(a.y, a.a_bytes);
#pragma unroll
    for (int j = 0; j < RT * P / 8 / kWideThreads; ++j) {
      const int at = (wave * 2 + j) * 64;
      const Slot<RT> s(at + lane);
      const bool ok = s.row < nrows;
      dma16_asm(xs, x_lds + at * 8, ok && s.col < a.kx ? (uint32_t)((s.row * a.x_row + s.col) * 2) : kOut, 0);
      dma16_asm(ys, y_lds + at * 8,
                ok && s.col < a.n ? att_row_bytes(a, (uint32_t)r0 + s.row) +
                                        2 * ((uint32_t)(s.col / a.width) * a.a_sh + (uint32_t)(s.col % a.width))
                                  : kOut, 0);
    }
  }
  // block t of the wave's stream: Wg's k blocks, then Wo's (past the last one: zeros, no memory traffic)
  const int t1 = (a.kx + 63) >> 6, t_end = t1 + ((a.n + 63) >> 6);
  auto request = [&](int t) {
    const bool first = t < t1;
    const int rows = first ? a.n : a.o, cols = first ? a.kx : t < t_end ? a.n : 0, k0 = (first ? t : t - t1) * 64;
    const int64_t w_row = first ? a.w_row : a.w_out_row;
    const u32x4 ws = rsrc_words(first ? a.w : a.w_out, (uint32_t)(((rows - 1) * w_row + (first ? a.kx : a.n)) * 2));
#pragma unroll
    for (int j = 0; j < BLK / 512; ++j) {
      const Slot<32> s(j * 64 + lane);
      const int c = 32 * wave + s.row, k = k0 + s.col;
      dma16_asm(ws, &w_lds[wave][t & 1][j * 512], c < rows && k < cols ? (uint32_t)((c * w_row + k) * 2) : kOut, 0);
    }
  };
  constexpr int LOADS = BLK / 512;
  request(0);
  request(1);
  own_loads_wait<2 * LOADS>();
  lds_barrier();  // single and attention rows written

  auto product = [&](const T* tile, int t, int end, uint4& lo, uint4& hi) {
    f32x16 acc = f32x16{};
    for (int k0 = 0; t < end; ++t, k0 += 64) {
      own_loads_wait<LOADS>();  // (the next block may be in flight; stores in between only make this stricter)
      const T* wb = w_lds[wave][t & 1];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        acc = E::mma(lds_frag<T>(wb + panel_off<32>(lq, 16 * ks + 8 * g2)),
                     lds_frag<T>(tile + panel_off<RT>(lq, k0 + 16 * ks + 8 * g2)), acc);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the block has been read
      request(t + 2);
    }
    round_run<T>(acc, lo, hi);
  };
  uint4 lo, hi;
  const int c0 = 32 * wave + 16 * g2;
  product(x_lds, 0, t1, lo, hi);
  if (32 * wave < a.n) {
    if constexpr (LOGITS) {
      const __amdgpu_buffer_rsrc_t lr = make_rsrc(static_cast<T*>(a.e) + r0 * a.n, (uint32_t)(nrows * a.n * 2));
      const uint32_t off = (uint32_t)((lq * a.n + c0) * 2);
      buffer_store16(lr, lq < nrows && c0 < a.n ? off : kOut, lo);
      buffer_store16(lr, lq < nrows && c0 + 8 < a.n ? off + 16 : kOut, hi);
    }
    uint4* p0 = reinterpret_cast<uint4*>(y_lds + panel_off<RT>(lq, c0));
    uint4* p1 = reinterpret_cast<uint4*>(y_lds + panel_off<RT>(lq, c0 + 8));
    // (columns past H*D stay zero whatever their padded logits are: an infinite `single` makes those NaN)
    *p0 = c0 < a.n ? gate_product<T>(lo, *p0) : make_uint4(0, 0, 0, 0);
    *p1 = c0 + 8 < a.n ? gate_product<T>(hi, *p1) : make_uint4(0, 0, 0, 0);
  }
  lds_barrier();  // gated rows written
  product(y_lds, t1, t_end, lo, hi);
  if (32 * wave < a.o) {
    const __amdgpu_buffer_rsrc_t orr = make_rsrc(static_cast<T*>(a.d) + r0 * a.o, (uint32_t)(nrows * a.o * 2));
    const uint32_t off = (uint32_t)((lq * a.o + c0) * 2);
    buffer_store16(orr, lq < nrows && c0 < a.o ? off : kOut, lo);
    buffer_store16(orr, lq < nrows && c0 + 8 < a.o ? off + 16 : kOut, hi);
  }
  vmem_wait_all();  // the last requests land before the LDS is given back
}

// ------------------------------------------------------------------ gradients
// D = X W (the gate's backward applied to it with GATE) and partials of X^T Y (Y = the gated rows with GATE)
// for 128 columns n0 .. n0 + 127 of W, Y, D and all KX (128, 256 or 384, padded like P above) columns of X.
// Wave (cg, rg) computes columns 32 cg .. + 31 of D's tile rows 32 rg .. + 31, and X columns
// (KX / 4) cg .. of X^T Y's columns 64 rg .. + 63.  Splitting the columns over workgroups halves the
// float32 partials (a 256 x 256 partial per CU is 64 MB per launch) and the accumulators; the two
// workgroups of a run are neighbours in one XCD and read the X rows through its L2.
template <typename T, int KX, bool GATE>
__global__ __launch_bounds__(512, 2) void row_grad_kernel(StageArgs a) {
  using E = Elem<T>;
  using Frag = typename E::Frag;
  constexpr int RT = kStageRows, NB = kStageCols, KS = KX / 16, MT = KX / 128;
  constexpr int XT = RT * KX, YT = RT * NB, STAGE = XT + (GATE ? 2 : 1) * YT;  // elements
  constexpr int NS = STAGE * 2 * 4 <= 128 * 1024 ? 4 : STAGE * 2 * 3 <= 160 * 1024 ? 3 : 2;
  constexpr int XL = KX / 64, STORES = GATE ? 4 : 2, LOADS = XL + (GATE ? 4 : 2);
  static_assert(NS * STAGE >= KX * NB, "the ring holds W at the start");
  __shared__ __attribute__((aligned(16))) T ring[NS * STAGE];

  const int64_t wg = xcd_tile(blockIdx.x, gridDim.x, 0);
  if (wg >= a.tiles) return;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lq = lane & 31, g2 = lane >> 5;
  const int cg = wave & 3, rg = wave >> 2;
  const int nb = (a.n + NB - 1) / NB;
  const int n0 = (int)(wg % nb) * NB;
  const int64_t run = wg / nb;
  const int64_t tiles_m = (a.rows + RT - 1) / RT, tile0 = run * a.tpw;
  const int count = (int)(tiles_m - tile0 < a.tpw ? tiles_m - tile0 : a.tpw);

  // W^T fragments (lane: column n0 + 32 cg + lq, k = 16 ks + 8 g2 ..) through the transposed read: row k of
  // each 16 goes to the LDS row that this read returns as k (rows 0-3, 8-11 to the lower half-wave)
  Frag wf[KS];
  {
    const __amdgpu_buffer_rsrc_t wr = make_rsrc(a.w, (uint32_t)(((a.kx - 1) * a.w_row + a.n) * 2));
    uint4 u[KX / 32];
#pragma unroll
    for (int j = 0; j < KX / 32; ++j) {
      const int id = tid + 512 * j, k = id >> 4, c = n0 + (id & 15) * 8;
      u[j] = buffer_load16(wr, k < a.kx && c < a.n ? (uint32_t)((k * a.w_row + c) * 2) : kOut);
    }
#pragma unroll
    for (int j = 0; j < KX / 32; ++j) {
      const int id = tid + 512 * j, k = id >> 4;
      const int r = (k & ~12) | ((k & 8) >> 1) | ((k & 4) << 1);
      *reinterpret_cast<uint4*>(&ring[panel_off<KX>(r, (id & 15) * 8)]) = u[j];
    }
    __syncthreads();
    const TrLane tw = tr_lane<64>(lane, (32 * cg) & 63);
    const T* wp = ring + (cg >> 1) * KX * 64 + ((32 * cg) & 63);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) wf[ks] = lds_read_tr_frag_sw<T>(wp + 16 * ks * 64, tw);
    __syncthreads();
  }

  uint32_t xo[XL];
  int xr[XL];
#pragma unroll
  for (int j = 0; j < XL; ++j) {
    const Slot<RT> s((wave * XL + j) * 64 + lane);
    xr[j] = s.row;
    xo[j] = s.col < a.kx ? (uint32_t)((s.row * a.x_row + s.col) * 2) : kOut;
  }
  uint32_t yo[2], lo_off[2];
  int yr[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const Slot<RT> s((wave * 2 + j) * 64 + lane);
    const int n = n0 + s.col;
    yr[j] = s.row;
    if constexpr (GATE) {
      yo[j] = n < a.n ? 2 * ((uint32_t)(n / a.width) * a.a_sh + (uint32_t)(n % a.width)) : kOut;
      lo_off[j] = n < a.n ? (uint32_t)((s.row * a.n + n) * 2) : kOut;
    } else {
      yo[j] = n < a.n ? (uint32_t)((s.row * a.y_row + n) * 2) : kOut;
    }
  }
  u32x4 att_rs;
  if constexpr (GATE) att_rs = rsrc_words(a.y, a.a_bytes);
  auto request = [&](int it) {
    const int64_t r0 = (tile0 + it) * RT;
    const int64_t left = it < count ? a.rows - r0 : 0;
    const int nrows = (int)(left < RT ? left : RT);
    T* st = ring + (it % NS) * STAGE;
    const u32x4 xs = rsrc_words(static_cast<const T*>(a.x) + (nrows ? r0 * a.x_row : 0),
                                nrows ? (uint32_t)(((nrows - 1) * a.x_row + a.kx) * 2) : 0u);
#pragma unroll
    for (int j = 0; j < XL; ++j) dma16_asm(xs, st + (wave * XL + j) * 512, xr[j] < nrows ? xo[j] : kOut, 0);
    T* yt = st + XT + wave * 1024;
    if constexpr (GATE) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
        dma16_asm(att_rs, yt + 512 * j,
                  yo[j] != kOut && yr[j] < nrows ? att_row_bytes(a, (uint32_t)r0 + yr[j]) + yo[j] : kOut, 0);
      const u32x4 ls = rsrc_words(static_cast<const T*>(a.logits) + (nrows ? r0 * a.n : 0), (uint32_t)(nrows * a.n * 2));
#pragma unroll
      for (int j = 0; j < 2; ++j) dma16_asm(ls, yt + YT + 512 * j, yr[j] < nrows ? lo_off[j] : kOut, 0);
    } else {
      const u32x4 ys = rsrc_words(static_cast<const T*>(a.y) + (nrows ? r0 * a.y_row : 0),
                                  nrows ? (uint32_t)(((nrows - 1) * a.y_row + a.n) * 2) : 0u);
#pragma unroll
      for (int j = 0; j < 2; ++j) dma16_asm(ys, yt + 512 * j, yr[j] < nrows ? yo[j] : kOut, 0);
    }
  };
  vmem_wait_all();
#pragma unroll
  for (int it = 0; it < NS - 1; ++it) request(it);

  f32x16 gacc[MT][2];
#pragma unroll
  for (int i = 0; i < MT; ++i) gacc[i][0] = gacc[i][1] = f32x16{};

  const int row = 32 * rg + lq, c0 = 32 * cg + 16 * g2;  // D: this lane's tile row and 16 columns (from n0)
  for (int it = 0; it < count; ++it) {
    wait_tile<NS, STORES, LOADS>(it);
    lds_barrier();          // tile it written by every wave; every wave is past tile it - 1
    request(it + NS - 1);  // into tile it - 1's slot
    T* st = ring + (it % NS) * STAGE;
    T* yt = st + XT;
    const int64_t r0 = (tile0 + it) * RT;
    const int64_t left = a.rows - r0;
    const int nrows = (int)(left < RT ? left : RT);
    uint4 lo, hi;
    {
      f32x16 acc = f32x16{};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        acc = E::mma(wf[ks], lds_frag<T>(st + panel_off<RT>(row, 16 * ks + 8 * g2)), acc);
      round_run<T>(acc, lo, hi);
    }
    const int n = n0 + c0;
    if constexpr (GATE) {
      const uint32_t bytes = (uint32_t)(nrows * a.n * 2);
      const __amdgpu_buffer_rsrc_t ar = make_rsrc(static_cast<T*>(a.d) + r0 * a.n, bytes);
      const __amdgpu_buffer_rsrc_t er = make_rsrc(static_cast<T*>(a.e) + r0 * a.n, bytes);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        uint4* y = reinterpret_cast<uint4*>(yt + panel_off<RT>(row, c0 + 8 * k));
        const uint4 l = *reinterpret_cast<const uint4*>(yt + YT + panel_off<RT>(row, c0 + 8 * k));
        uint4 da, dl, gated;
        gate_backward_run<T>(k ? hi : lo, *y, l, da, dl, gated);
        *y = gated;
        const uint32_t off = row < nrows && n + 8 * k < a.n ? (uint32_t)((row * a.n + n + 8 * k) * 2) : kOut;
        buffer_store16(ar, off, da);
        buffer_store16(er, off, dl);
        asm volatile("" ::: "memory");  // one run of eight at a time: fewer live registers
      }
      lds_barrier();  // gated rows written
    } else {
      const __amdgpu_buffer_rsrc_t dr =
          make_rsrc(static_cast<T*>(a.d) + r0 * a.d_row, (uint32_t)(((nrows - 1) * a.d_row + a.n) * 2));
      const uint32_t off = (uint32_t)((row * a.d_row + n) * 2);
      buffer_store16(dr, row < nrows && n < a.n ? off : kOut, lo);
      buffer_store16(dr, row < nrows && n + 8 < a.n ? off + 16 : kOut, hi);
    }
    const TrLane t0 = tr_lane<64>(lane, 0), t1 = tr_lane<64>(lane, 32);
#pragma unroll
    for (int ks = 0; ks < RT / 16; ++ks) {
      const T* yp = yt + rg * RT * 64 + 16 * ks * 64;
      const Frag b0 = lds_read_tr_frag_sw<T>(yp, t0), b1 = lds_read_tr_frag_sw<T>(yp + 32, t1);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const int m = (MT * cg + i) * 32;
        const Frag af = lds_read_tr_frag_sw<T>(st + (m >> 6) * RT * 64 + 16 * ks * 64 + (m & 63), (m & 63) ? t1 : t0);
        gacc[i][0] = E::mma(af, b0, gacc[i][0]);
        gacc[i][1] = E::mma(af, b1, gacc[i][1]);
      }
    }
  }

  // partial of X^T Y: lane (lq, g2) of gacc[i][j] holds rows 32 (MT cg + i) + 8q + 4 g2 + k, column
  // n0 + 64 rg + 32 j + lq
  float* gp = a.parts + run * a.kx * a.n;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int n = n0 + 64 * rg + 32 * j + lq;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int m = 32 * (MT * cg + i) + 8 * q + 4 * g2 + k;
          if (m < a.kx && n < a.n) gp[(int64_t)m * a.n + n] = gacc[i][j][4 * q + k];
        }
    }
  vmem_wait_all();  // the ring's last requests land before the LDS is given back
}

struct RunPlan {
  int tpw;
  int64_t runs;
};
RunPlan run_plan(int64_t rows, int tile_rows, int64_t max_runs) {
  const int64_t tiles = (rows + tile_rows - 1) / tile_rows;
  const int64_t tpw = std::max<int64_t>(1, (tiles + max_runs - 1) / max_runs);
  return {(int)tpw, (tiles + tpw - 1) / tpw};
}

template <typename F>
hipError_t by_half(int dtype, F&& f) {
  if (dtype == OOPS_BF16) return f(__bf16{});
  if (dtype == OOPS_F16) return f(_Float16{});
  return hipErrorInvalidValue;
}

// 32-bit byte offsets over a tile's rows and over a weight's rows
bool rows_fit(int64_t stride, int64_t count) { return stride * count * 2 < (int64_t(1) << 31); }

}  // namespace

int64_t row_grad_parts(int dtype, int64_t rows, int64_t k, int64_t n) {
  if (dtype != OOPS_BF16 && dtype != OOPS_F16) return 0;
  if (rows < 1 || rows >= (int64_t(1) << 31) || k < 8 || k > kWideCols || n < 8 || n > kWideCols || k % 8 || n % 8) return 0;
  return run_plan(rows, kStageRows, kStageWgs / ((n + kStageCols - 1) / kStageCols)).runs;
}

bool gate_stage_ok(const oops_gate_geometry& g, int64_t out_channels, int64_t wo_row, const void* single,
                   const void* weight, const void* attention, const void* output_weight) {
  const int64_t n = (int64_t)g.heads * g.width;
  if (row_grad_parts(g.dtype, g.rows, n, g.channels) == 0 || row_grad_parts(g.dtype, g.rows, out_channels, n) == 0)
    return false;
  if (std::max({n, (int64_t)g.channels, out_channels}) > 256 && g.rows > kWideRows) return false;
  if (g.width % 8 || g.a_sd != 1 || g.s_row % 8 || g.w_row % 8 || wo_row % 8) return false;
  int64_t extent = g.width;
  const int64_t sizes[4] = {g.rows / (g.tokens * g.groups), g.groups, g.tokens, g.heads};
  const int64_t strides[4] = {g.a_sb, g.a_sg, g.a_st, g.a_sh};
  for (int i = 0; i < 4; ++i) {
    if (strides[i] % 8) return false;
    if (sizes[i] > 1 && (strides[i] < 0 || strides[i] > (int64_t(1) << 30))) return false;
    if (sizes[i] > 1) extent += (sizes[i] - 1) * strides[i];
  }
  if (g.rows % (g.tokens * g.groups) || extent > (int64_t(1) << 30)) return false;
  if (g.s_row < 0 || g.w_row < 0 || wo_row < 0 || !rows_fit(g.s_row, kStageRows) || !rows_fit(g.w_row, kWideCols) ||
      !rows_fit(wo_row, kWideCols))
    return false;
  for (const void* p : {single, weight, attention, output_weight})
    if (reinterpret_cast<uintptr_t>(p) & 15) return false;
  return true;
}

namespace {
StageArgs stage_args(const oops_gate_geometry& g, const void* attention) {
  StageArgs a{};
  a.y = attention;
  a.rows = g.rows;
  a.tokens = (uint32_t)g.tokens, a.groups = (uint32_t)g.groups;
  // (a stride of a single-element axis is multiplied by zero only)
  a.a_sb = (uint32_t)g.a_sb, a.a_sg = (uint32_t)g.a_sg, a.a_st = (uint32_t)g.a_st, a.a_sh = (uint32_t)g.a_sh;
  const int64_t b = g.rows / (g.tokens * g.groups);
  int64_t extent = g.width;
  if (b > 1) extent += (b - 1) * g.a_sb;
  if (g.groups > 1) extent += (g.groups - 1) * g.a_sg;
  if (g.tokens > 1) extent += (g.tokens - 1) * g.a_st;
  if (g.heads > 1) extent += (g.heads - 1) * g.a_sh;
  a.a_bytes = (uint32_t)(extent * 2);
  a.width = g.width;
  return a;
}
}  // namespace

hipError_t launch_gate_stage_forward(const oops_gate_geometry& g, int64_t out_channels, int64_t wo_row,
                                     const void* single, const void* weight, const void* attention,
                                     const void* output_weight, void* out, void* logits, hipStream_t stream) {
  StageArgs a = stage_args(g, attention);
  a.x = single, a.w = weight, a.w_out = output_weight, a.d = out, a.e = logits;
  a.x_row = g.s_row, a.w_row = g.w_row, a.w_out_row = wo_row;
  a.kx = g.channels, a.n = g.heads * g.width, a.o = (int)out_channels;
  const int most = std::max({a.kx, a.n, a.o});
  if (most > 256 || (most > 128 && g.rows <= kStreamRows)) {
    return by_half(g.dtype, [&](auto tag) -> hipError_t {
      using T = decltype(tag);
      const dim3 grid((unsigned)((g.rows + 31) / 32));
      if (logits)
        hipLaunchKernelGGL((gate_stage_wide_kernel<T, true>), grid, dim3(kWideThreads), 0, stream, a);
      else
        hipLaunchKernelGGL((gate_stage_wide_kernel<T, false>), grid, dim3(kWideThreads), 0, stream, a);
      return hipGetLastError();
    });
  }
  const bool wide = most > 128;
  const RunPlan pl = run_plan(g.rows, wide ? 32 : 64, kStageWgs);
  a.tpw = pl.tpw, a.tiles = pl.runs;
  return by_half(g.dtype, [&](auto tag) -> hipError_t {
    using T = decltype(tag);
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)xcd_grid(a.tiles, 0)), dim3(512), 0, stream, a);
      return hipGetLastError();
    };
    if (logits) return wide ? go(gate_stage_forward_kernel<T, 256, true>) : go(gate_stage_forward_kernel<T, 128, true>);
    return wide ? go(gate_stage_forward_kernel<T, 256, false>) : go(gate_stage_forward_kernel<T, 128, false>);
  });
}

namespace {
template <bool GATE>
hipError_t launch_row_grad(int dtype, StageArgs& a, hipStream_t stream) {
  const int64_t nb = (a.n + kStageCols - 1) / kStageCols;
  const RunPlan pl = run_plan(a.rows, kStageRows, kStageWgs / nb);
  a.tpw = pl.tpw, a.tiles = pl.runs * nb;
  return by_half(dtype, [&](auto tag) -> hipError_t {
    using T = decltype(tag);
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)xcd_grid(a.tiles, 0)), dim3(512), 0, stream, a);
      return hipGetLastError();
    };
    return a.kx > 256   ? go(row_grad_kernel<T, 384, GATE>)
           : a.kx > 128 ? go(row_grad_kernel<T, 256, GATE>)
                        : go(row_grad_kernel<T, 128, GATE>);
  });
}
}  // namespace

hipError_t launch_gate_stage_backward(const oops_gate_geometry& g, int64_t out_channels, int64_t wo_row,
                                      const void* grad, const void* attention, const void* logits,
                                      const void* output_weight, void* grad_attention, void* grad_logits,
                                      float* g_parts, hipStream_t stream) {
  StageArgs a = stage_args(g, attention);
  a.x = grad, a.w = output_weight, a.logits = logits, a.d = grad_attention, a.e = grad_logits, a.parts = g_parts;
  a.x_row = out_channels, a.w_row = wo_row;
  a.kx = (int)out_channels, a.n = g.heads * g.width;
  return launch_row_grad<true>(g.dtype, a, stream);
}

bool linear_grads_ok(int dtype, int64_t rows, int64_t k, int64_t n, const void* x, int64_t x_row, const void* w,
                     int64_t w_row, const void* y, int64_t y_row, const void* d, int64_t d_row) {
  if (row_grad_parts(dtype, rows, k, n) == 0) return false;
  for (const void* p : {x, w, y, d})
    if (reinterpret_cast<uintptr_t>(p) & 15) return false;
  // (offsets within a tile's rows, and over all of the weight's: gate_stage_ok's limits)
  for (int64_t s : {x_row, y_row, d_row})
    if (s < 0 || s % 8 || !rows_fit(s, kStageRows)) return false;
  if (w_row < 0 || w_row % 8 || !rows_fit(w_row, kWideCols)) return false;
  return x_row >= k && d_row >= n;
}

hipError_t launch_linear_grads(int dtype, int64_t rows, int64_t k, int64_t n, const void* x, int64_t x_row,
                               const void* w, int64_t w_row, const void* y, int64_t y_row, void* d, int64_t d_row,
                               float* g_parts, hipStream_t stream) {
  StageArgs a{};
  a.rows = rows;
  a.x = x, a.w = w, a.y = y, a.d = d, a.parts = g_parts;
  a.x_row = x_row, a.w_row = w_row, a.y_row = y_row, a.d_row = d_row;
  a.kx = (int)k, a.n = (int)n;
  return launch_row_grad<false>(dtype, a, stream);
}

}  // namespace oops
