// float32 attention, forward and backward: head size <= 64 and a multiple of
// 4, rows of Q, K, V, O and dO 16-byte aligned, key masks; any bias layout.
//
// Bound: the exact float32 matrix instruction v_mfma_f32_32x32x2f32, 64
// cycles for 4096 flops, so a 32 x 32 score tile costs 2048 matrix cycles in
// the forward (head size 32) against some 500 of vector work.  Everything
// else is arranged to keep the matrix cores fed:
//   * 4 wavefronts per workgroup, each with 32 queries (keys in the dK/dV
//     kernel); a wave whose rows all lie past the end skips its arithmetic;
//   * K/V (Q/dO) tiles of 32 rows go straight from global memory to a
//     3-buffer LDS ring (buffer_load ... lds), issued a step and a half before
//     their use, one barrier per step;
//   * an MFMA sums any two values of k per step, so lane half g2 takes the k
//     of its half of the head dimension: both operands of Q K^T are then runs
//     of consecutive elements, four 16-byte LDS reads per row instead of 16
//     4-byte ones.  Rows are XOR-swizzled in 16-byte chunks (chunk c of row r
//     at c ^ (r % 8)), so eight lanes of such a read hit distinct banks;
//   * the bias goes from global memory to registers in accumulator order, one
//     step ahead (query rows of any alignment; no copy, no LDS);
//   * delta = rowsum(O dO) is formed by the dQ kernel from its own rows.
// The arithmetic per score is that of the generic kernels (attn_fwd.hip,
// attn_bwd.hip): x = fma(qk, scale log2 e, bias log2 e), exact running max.
// Measured against them: see attn_f32_ok.
//
// Semantics: the reference's _attend, _backward_query, _backward_key_value
// and _backward_shared_bias (oops/attention/triangle/triton/kernel.py:151-873).
#include "attn_fast_common.h"

namespace oops {

using namespace fast;

namespace {

constexpr int kRing = 3;
constexpr int kDqbTiles = 8;       // 32-key tiles of the dQ + dBias kernel: Lk <= 256
constexpr int kF32MaxTiles = 512;  // 32-key tiles: Lk <= 16384

__device__ __forceinline__ f32x16 mma2(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// Every load of this wave has landed (an asm with a memory clobber, so that neither LDS reads nor the next
// loads move across it)
__device__ __forceinline__ void vm_drain() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// float offset of (row, 16-byte chunk) in a swizzled tile of DP-float rows
template <int DP>
__device__ __forceinline__ int at4(int row, int chunk) {
  return row * DP + ((chunk ^ (row & 7)) << 2);
}

// The lane's half row (k = g2 DP/2 ..) of a tile row in LDS
template <int DP>
__device__ __forceinline__ void row_frag(const float* tile, int row, int g2, float (&f)[DP / 2]) {
#pragma unroll
  for (int i = 0; i < DP / 8; ++i) {
    const float4 v = *reinterpret_cast<const float4*>(&tile[at4<DP>(row, g2 * (DP / 8) + i)]);
    f[4 * i] = v.x, f[4 * i + 1] = v.y, f[4 * i + 2] = v.z, f[4 * i + 3] = v.w;
  }
}
// The lane's half row in global memory (zeros where !ok or past D)
template <int DP>
__device__ __forceinline__ void row_load(const float* row, bool ok, int D, int g2, float (&f)[DP / 2]) {
#pragma unroll
  for (int i = 0; i < DP / 8; ++i) {
    const int col = g2 * (DP / 2) + 4 * i;
    const float4 v = ok && col < D ? *reinterpret_cast<const float4*>(row + col) : make_float4(0.f, 0.f, 0.f, 0.f);
    f[4 * i] = v.x, f[4 * i + 1] = v.y, f[4 * i + 2] = v.z, f[4 * i + 3] = v.w;
  }
}
// Column element X[kappa(g2, j)][32 t + lq] of a swizzled tile (A operand of X^T): the lane part of the
// offset depends on j only through j % 4, the rest is an immediate.
template <int DP>
struct ColLane {
  int off[4];
  __device__ __forceinline__ ColLane(int lq, int g2) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = g2 * 4 + e;  // kappa(g2, j) % 8
      off[e] = r * DP + (((lq >> 2) ^ r) << 2) + (lq & 3);
    }
  }
  // (32 t floats are 8 t chunks, above the bits the swizzle changes)
  __device__ __forceinline__ float get(const float* tile, int j, int t) const {
    return tile[off[j & 3] + (j >> 2) * 8 * DP + 32 * t];
  }
};
// four accumulator values (head dims d0 .. d0 + 3) of one row
__device__ __forceinline__ void put4(float* row, int d0, int D, const f32x16& a, int q, float s) {
  if (d0 < D) *reinterpret_cast<float4*>(row + d0) = make_float4(a[4 * q] * s, a[4 * q + 1] * s, a[4 * q + 2] * s, a[4 * q + 3] * s);
}

// four consecutive dBias values of one row of Lk keys (rows start at any element)
__device__ __forceinline__ void put_ds(float* row, int key, int Lk, float x0, float x1, float x2, float x3) {
  typedef float F4 __attribute__((ext_vector_type(4), aligned(4)));
  if (key + 3 < Lk) {
    *reinterpret_cast<F4*>(row + key) = (F4){x0, x1, x2, x3};
  } else {
    if (key < Lk) row[key] = x0;
    if (key + 1 < Lk) row[key + 1] = x1;
    if (key + 2 < Lk) row[key + 2] = x2;
  }
}

// Direct-to-LDS loads of one tile of 32 rows of X (row stride si floats): wave
// w fills rows w IPW RPI .. of the tile, lane l slot l of its load.
template <int DP>
struct TileDma {
  static constexpr int CPR = DP / 4, RPI = 64 / CPR, IPW = 8 / RPI;
  uint32_t off[IPW], row[IPW];
  u32x4 rsrc;
  __device__ __forceinline__ void init(const float* base, int len, int si, int D, int wave, int lane) {
    rsrc = rsrc_words(base, (uint32_t)(((int64_t)(len - 1) * si + D) * 4));
#pragma unroll
    for (int i = 0; i < IPW; ++i) {
      const int r = (wave * IPW + i) * RPI + lane / CPR;
      const int col = ((lane % CPR) ^ (r & 7)) * 4;
      row[i] = (uint32_t)r;
      off[i] = col < D ? (uint32_t)((r * si + col) * 4) : kOut;
    }
  }
  // rows whose bit is clear (masked, past the end) become zeros
  __device__ __forceinline__ void issue(float* tile, int wave, uint32_t soff, uint32_t bits) const {
#pragma unroll
    for (int i = 0; i < IPW; ++i)
      dma16_asm(rsrc, tile + (wave * IPW + i) * RPI * DP, (bits >> row[i]) & 1 ? off[i] : kOut, soff);
  }
};

// bias of the lane's query and keys k0 + kappa(g2, 0..15), four at a time
struct BiasRow {
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t off;
  int Lk;
  __device__ __forceinline__ void load(int k0, float (&b)[16]) const {
    if (k0 + 32 <= Lk) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float4 v = __builtin_bit_cast(float4, buffer_load16(rsrc, off + (uint32_t)((k0 + 8 * i) * 4)));
        b[4 * i] = v.x, b[4 * i + 1] = v.y, b[4 * i + 2] = v.z, b[4 * i + 3] = v.w;
      }
    } else {  // the last tile of a length that is no multiple of 32: element by element
      const int g4 = (threadIdx.x & 32) >> 3;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int k = k0 + (j >> 2) * 8 + (j & 3);
        const uint32_t o = k + g4 < Lk ? off + (uint32_t)(k * 4) : kOut;
        b[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, o, 0, 0));
      }
    }
  }
};

__device__ __forceinline__ void load_keep(uint32_t* keep, const uint8_t* mask, int Lk, int wave, int lane) {
  for (int t = wave; t * 64 < Lk; t += 4) {
    const int key = t * 64 + lane;
    bool k = key < Lk;
    if (k && mask != nullptr) k = mask[key] != 0;
    const uint64_t bits = __ballot(k);
    if (lane == 0) {
      keep[2 * t] = (uint32_t)bits;
      keep[2 * t + 1] = (uint32_t)(bits >> 32);
    }
  }
}

// The tile of a (group, head, block) grid in the order of attn_fwd_fast.hip.
struct Where {
  int s, g, h, blk;
};
template <typename Args, typename Count>
__device__ __forceinline__ bool locate(const Args& a, Where& w, Count count) {
  int64_t tile = xcd_tile(blockIdx.x, gridDim.x, xcd_chunk(a.uniform_tiles));
  if (tile >= a.total_tiles) return false;
  const Sample* tab = reinterpret_cast<const Sample*>(a.table);
  const int s = find_sample(tile, tab, a.num_samples, a.uniform_tiles,
                            [&](const Sample& x) { return x.G * a.num_heads * count(x); });
  if (s < 0) return false;
  w.s = __builtin_amdgcn_readfirstlane(s);
  const Sample& S = tab[w.s];
  const uint32_t nb = (uint32_t)count(S), G = (uint32_t)S.G, HG = (uint32_t)a.head_group;
  w.blk = __builtin_amdgcn_readfirstlane((int)((uint32_t)tile % nb));
  uint32_t rest = (uint32_t)tile / nb;
  const uint32_t hh = rest % HG;
  rest /= HG;
  w.g = __builtin_amdgcn_readfirstlane((int)(rest % G));
  w.h = __builtin_amdgcn_readfirstlane((int)(rest / G * HG + hh));
  return true;
}

// ------------------------------------------------------------------ forward
template <int DP, bool HAS_BIAS>
__global__ __launch_bounds__(256, DP == 32 ? 4 : 2) void attn_fwd_f32_kernel(FwdArgsT<float, float> a) {
  constexpr int NS = DP / 2, NDT = DP / 32, TB = 32 * DP;
  __shared__ __attribute__((aligned(16))) float k_lds[kRing][TB];
  __shared__ __attribute__((aligned(16))) float v_lds[kRing][TB];
  __shared__ uint32_t keep_lds[kF32MaxTiles];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3, lane = threadIdx.x & 63;
  const int lq = lane & 31, g2 = lane >> 5;
  Where w;
  if (!locate(a, w, [](const Sample& s) { return cdiv(s.Lq, 128); })) return;
  const Sample& S = reinterpret_cast<const Sample*>(a.table)[w.s];
  const int g = w.g, h = w.h, H = a.num_heads, D = a.head_size;
  const int Lq = (int)S.Lq, Lk = (int)S.Lk, ntiles = (Lk + 31) >> 5;
  const int k_si = (int)S.k_si, v_si = (int)S.v_si;
  const uint8_t* mbase = a.mask != nullptr && S.m_off >= 0 ? a.mask + S.m_off + g * S.m_sg : nullptr;
  load_keep(keep_lds, mbase, Lk, wave, lane);

  // (rotated by the group: the waves that a short last block leaves idle spread over the SIMDs)
  const int q0 = w.blk * 128 + ((wave + g) & 3) * 32, q = q0 + lq;
  const bool qv = q < Lq, active = q0 < Lq;
  float qf[NS];
  row_load<DP>(a.q + S.q_off + g * S.q_sg + h * S.q_sh + (int64_t)q * S.q_si, qv, D, g2, qf);
  TileDma<DP> kd, vd;
  kd.init(a.k + S.k_off + g * S.k_sg + h * S.k_sh, Lk, k_si, D, wave, lane);
  vd.init(a.v + S.v_off + g * S.v_sg + h * S.v_sh, Lk, v_si, D, wave, lane);
  BiasRow br;
  if constexpr (HAS_BIAS) {
    br.rsrc = make_rsrc(a.bias + S.b_off + g * S.b_sg + h * S.b_sh, (uint32_t)(((int64_t)(Lq - 1) * S.b_si + Lk) * 4));
    br.off = qv ? (uint32_t)((q * (int)S.b_si + g2 * 4) * 4) : kOut;
    br.Lk = Lk;
  }
  const ColLane<DP> col(lq, g2);
  __syncthreads();  // keep bitmaps visible

  auto bits_of = [&](int t) { return t < ntiles ? __builtin_amdgcn_readfirstlane(keep_lds[t]) : 0u; };
  auto next = [&](int t) {  // fully masked tiles are skipped
    do ++t;
    while (t < ntiles && bits_of(t) == 0);
    return t < ntiles ? t : ntiles;
  };
  auto dma = [&](int t, int buf) {
    if (t >= ntiles) return;
    const uint32_t bits = bits_of(t);
    kd.issue(k_lds[buf], wave, (uint32_t)(t * 32 * k_si * 4), bits);
    vd.issue(v_lds[buf], wave, (uint32_t)(t * 32 * v_si * 4), bits);
  };

  const float c1 = a.scale * kLog2e;
  float m_run = kNegInf, l_run = 0.0f;
  f32x16 oacc[NDT];
#pragma unroll
  for (int t = 0; t < NDT; ++t) oacc[t] = f32x16{};
  float bias[16];
  int t0 = next(-1), t1 = next(t0);
  dma(t0, 0);
  dma(t1, 1);
  if constexpr (HAS_BIAS)
    if (active) br.load(t0 * 32, bias);
  vm_drain();
  __syncthreads();
  int buf = 0;
  while (t0 < ntiles) {
    const int t2 = next(t1), b2 = buf == 0 ? 2 : buf - 1;
    const uint32_t bits = bits_of(t0);
    float x[16];
    if (active) {
      f32x16 sacc = f32x16{};
      float kf[NS];
      row_frag<DP>(k_lds[buf], lq, g2, kf);
#pragma unroll
      for (int s = 0; s < NS; ++s) sacc = mma2(kf[s], qf[s], sacc);
#pragma unroll
      for (int j = 0; j < 16; ++j) x[j] = HAS_BIAS ? __builtin_fmaf(sacc[j], c1, bias[j] * kLog2e) : sacc[j] * c1;
      if (bits != 0xFFFFFFFFu) {
        const uint32_t lb = bits >> (g2 * 4);
#pragma unroll
        for (int j = 0; j < 16; ++j) x[j] = (lb >> (((j >> 2) << 3) | (j & 3))) & 1 ? x[j] : kNegInf;
      }
    }
    // this step's bias has been used and the next tile's loads, issued a step ago, are waited for; the loads
    // after that go out now (into the buffer that the last step's barrier released)
    vm_drain();
    if constexpr (HAS_BIAS)
      if (active && t1 < ntiles) br.load(t1 * 32, bias);
    dma(t2, b2);
    if (active) {
      float mx = x[0];
#pragma unroll
      for (int j = 1; j < 16; ++j) mx = fmaxf(mx, x[j]);
      mx = max_halves(mx);
      const float m_new = fmaxf(m_run, mx);
      const float m_use = m_new == kNegInf ? 0.0f : m_new;
      if (__any(m_new != m_run)) {
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
        l_run *= alpha;
#pragma unroll
        for (int t = 0; t < NDT; ++t) oacc[t] *= alpha;
        m_run = m_new;
      }
      float psum = 0.0f;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const float p = __builtin_amdgcn_exp2f(x[j] - m_use);
        psum += p;
#pragma unroll
        for (int t = 0; t < NDT; ++t) oacc[t] = mma2(col.get(v_lds[buf], j, t), p, oacc[t]);
      }
      l_run += psum;
    }
    lds_barrier();
    buf = buf == 2 ? 0 : buf + 1;
    t0 = t1;
    t1 = t2;
  }

  const float l_tot = sum_halves(l_run);
  const float inv = 1.0f / (l_tot == 0.0f ? 1.0f : l_tot);
  if (!qv) return;
  float* orow = a.out + S.o_off + g * S.o_sg + h * S.o_sh + (int64_t)q * S.o_si;
#pragma unroll
  for (int t = 0; t < NDT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) put4(orow, t * 32 + 8 * i + 4 * g2, D, oacc[t], i, inv);
  if (g2 == 0 && a.lse != nullptr) {
    const float m_use = m_run == kNegInf ? 0.0f : m_run;
    a.lse[S.l_off + ((int64_t)g * H + h) * Lq + q] = l_tot == 0.0f ? 0.0f : m_use + __log2f(l_tot);
  }
}

// ------------------------------------------------------------------ dQ (+ delta, per-group dBias)
template <int DP, bool HAS_BIAS>
__global__ __launch_bounds__(256, DP == 32 ? 3 : 2) void attn_dq_f32_kernel(BwdArgsT<float, float> a) {
  constexpr int NS = DP / 2, NDT = DP / 32, TB = 32 * DP;
  __shared__ __attribute__((aligned(16))) float k_lds[kRing][TB];
  __shared__ __attribute__((aligned(16))) float v_lds[kRing][TB];
  __shared__ uint32_t keep_lds[kF32MaxTiles];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3, lane = threadIdx.x & 63;
  const int lq = lane & 31, g2 = lane >> 5;
  Where w;
  if (!locate(a, w, [](const Sample& s) { return cdiv(s.Lq, 128); })) return;
  const Sample& S = reinterpret_cast<const Sample*>(a.table)[w.s];
  const int g = w.g, h = w.h, H = a.num_heads, D = a.head_size;
  const int Lq = (int)S.Lq, Lk = (int)S.Lk, ntiles = (Lk + 31) >> 5;
  const int k_si = (int)S.k_si, v_si = (int)S.v_si;
  const uint8_t* mbase = a.mask != nullptr && S.m_off >= 0 ? a.mask + S.m_off + g * S.m_sg : nullptr;
  load_keep(keep_lds, mbase, Lk, wave, lane);

  const int q0 = w.blk * 128 + ((wave + g) & 3) * 32, q = q0 + lq;
  const bool qv = q < Lq, active = q0 < Lq;
  const int64_t lidx = S.l_off + ((int64_t)g * H + h) * Lq + q;
  float qf[NS], df[NS], dlt = 0.0f;
  row_load<DP>(a.q + S.q_off + g * S.q_sg + h * S.q_sh + (int64_t)q * S.q_si, qv, D, g2, qf);
  row_load<DP>(a.dout + S.do_off + g * S.do_sg + h * S.do_sh + (int64_t)q * S.do_si, qv, D, g2, df);
  if (a.delta_in_dq) {
    float of[NS];
    row_load<DP>(a.out + S.o_off + g * S.o_sg + h * S.o_sh + (int64_t)q * S.o_si, qv, D, g2, of);
#pragma unroll
    for (int s = 0; s < NS; ++s) dlt = __builtin_fmaf(of[s], df[s], dlt);
    dlt = sum_halves(dlt);
    if (qv && g2 == 0) a.delta[lidx] = dlt;
  } else {
    dlt = qv ? a.delta[lidx] : 0.0f;
  }
  const float lse = qv ? a.lse[lidx] : 0.0f;
  // a per-group bias, or one shared by a single group: dBias = dS
  const bool all_tiles = a.dbias != nullptr && (S.bias_mode == OOPS_BIAS_FULL || (a.direct_dbias && S.bias_mode == OOPS_BIAS_SHARED));
  float* dbrow = all_tiles && qv ? a.dbias + S.db_off + g * S.db_sg + h * S.db_sh + (int64_t)q * S.db_si : nullptr;
  TileDma<DP> kd, vd;
  kd.init(a.k + S.k_off + g * S.k_sg + h * S.k_sh, Lk, k_si, D, wave, lane);
  vd.init(a.v + S.v_off + g * S.v_sg + h * S.v_sh, Lk, v_si, D, wave, lane);
  BiasRow br;
  if constexpr (HAS_BIAS) {
    br.rsrc = make_rsrc(a.bias + S.b_off + g * S.b_sg + h * S.b_sh, (uint32_t)(((int64_t)(Lq - 1) * S.b_si + Lk) * 4));
    br.off = qv ? (uint32_t)((q * (int)S.b_si + g2 * 4) * 4) : kOut;
    br.Lk = Lk;
  }
  const ColLane<DP> col(lq, g2);
  __syncthreads();

  auto bits_of = [&](int t) { return t < ntiles ? __builtin_amdgcn_readfirstlane(keep_lds[t]) : 0u; };
  // fully masked tiles are skipped, unless their zero dBias has to be written
  auto next = [&](int t) {
    do ++t;
    while (t < ntiles && !all_tiles && bits_of(t) == 0);
    return t < ntiles ? t : ntiles;
  };
  auto dma = [&](int t, int buf) {
    if (t >= ntiles) return;
    const uint32_t bits = bits_of(t);
    kd.issue(k_lds[buf], wave, (uint32_t)(t * 32 * k_si * 4), bits);
    vd.issue(v_lds[buf], wave, (uint32_t)(t * 32 * v_si * 4), bits);
  };

  const float c1 = a.scale * kLog2e;
  f32x16 acc[NDT];
#pragma unroll
  for (int t = 0; t < NDT; ++t) acc[t] = f32x16{};
  float bias[16];
  int t0 = next(-1), t1 = next(t0);
  dma(t0, 0);
  dma(t1, 1);
  if constexpr (HAS_BIAS)
    if (active) br.load(t0 * 32, bias);
  vm_drain();
  __syncthreads();
  int buf = 0;
  while (t0 < ntiles) {
    const int t2 = next(t1), b2 = buf == 0 ? 2 : buf - 1;
    const uint32_t bits = bits_of(t0);
    float x[16];
    f32x16 pacc = f32x16{};
    if (active) {
      f32x16 sacc = f32x16{};
      {
        float kf[NS], vf[NS];
        row_frag<DP>(k_lds[buf], lq, g2, kf);
        row_frag<DP>(v_lds[buf], lq, g2, vf);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          sacc = mma2(kf[s], qf[s], sacc);
          pacc = mma2(vf[s], df[s], pacc);
        }
      }
#pragma unroll
      for (int j = 0; j < 16; ++j) x[j] = HAS_BIAS ? __builtin_fmaf(sacc[j], c1, bias[j] * kLog2e) : sacc[j] * c1;
      if (bits != 0xFFFFFFFFu) {
        const uint32_t lb = bits >> (g2 * 4);
#pragma unroll
        for (int j = 0; j < 16; ++j) x[j] = (lb >> (((j >> 2) << 3) | (j & 3))) & 1 ? x[j] : kNegInf;
      }
    }
    vm_drain();
    if constexpr (HAS_BIAS)
      if (active && t1 < ntiles) br.load(t1 * 32, bias);
    dma(t2, b2);
    if (active) {
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        x[j] = __builtin_amdgcn_exp2f(x[j] - lse) * (pacc[j] - dlt);
#pragma unroll
        for (int t = 0; t < NDT; ++t) acc[t] = mma2(col.get(k_lds[buf], j, t), x[j], acc[t]);
      }
      if (dbrow) {
#pragma unroll
        for (int j = 0; j < 16; j += 4) put_ds(dbrow, t0 * 32 + kappa(g2, j), Lk, x[j], x[j + 1], x[j + 2], x[j + 3]);
      }
    }
    lds_barrier();
    buf = buf == 2 ? 0 : buf + 1;
    t0 = t1;
    t1 = t2;
  }
  if (!qv || a.dq == nullptr) return;
  float* row = a.dq + S.q_off + g * S.q_sg + h * S.q_sh + (int64_t)q * S.q_si;
#pragma unroll
  for (int t = 0; t < NDT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) put4(row, t * 32 + 8 * i + 4 * g2, D, acc[t], i, a.scale);
}

// ------------------------------------------------------------------ dQ + shared dBias
// dQ and the dBias of a bias shared by all groups, for at most kDqbTiles key
// tiles: a workgroup (128 queries of one head) walks the groups of one part,
// each wave summing dS of its 32 queries x all keys in registers, so the
// scores are formed once for dQ and dBias together (32 of 80 MFMAs per score
// tile saved, and the Q/dO rows are read once).  The parts' sums are added by
// attn_dbias_reduce_kernel.  NT: key tiles (the longest sample's); the sums
// take 16 NT registers, which at NT = 8 leaves two waves per SIMD.  The ring
// runs on across the group boundary: the last two tiles of a group fetch the
// first two of the next.
template <int NT>
__global__ __launch_bounds__(256, 2) void attn_dqb_f32_kernel(BwdArgsT<float, float> a) {
  constexpr int DP = 32, NS = DP / 2, TB = 32 * DP;
  __shared__ __attribute__((aligned(16))) float k_lds[kRing][TB];
  __shared__ __attribute__((aligned(16))) float v_lds[kRing][TB];
  __shared__ uint32_t keep_lds[4][kDqbTiles];  // of group g in row g % 4, stored two groups ahead

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3, lane = threadIdx.x & 63;
  const int lq = lane & 31, g2 = lane >> 5;
  int64_t tile = xcd_tile(blockIdx.x, gridDim.x, xcd_chunk(a.uniform_tiles));
  if (tile >= a.total_tiles) return;
  const Sample* tab = reinterpret_cast<const Sample*>(a.table);
  const int H = a.num_heads, P = a.parts;
  const int s_idx = find_sample(tile, tab, a.num_samples, a.uniform_tiles,
                                [&](const Sample& s) { return (int64_t)H * cdiv(s.Lq, 128) * P; });
  if (s_idx < 0) return;
  const Sample& S = tab[__builtin_amdgcn_readfirstlane(s_idx)];
  const int Lq = (int)S.Lq, Lk = (int)S.Lk, D = a.head_size;
  const uint32_t nqb = (uint32_t)cdiv(Lq, 128);
  // (head, part, query block): the query blocks of one part share their groups' K/V
  const int qb = __builtin_amdgcn_readfirstlane((int)((uint32_t)tile % nqb));
  const uint32_t rest = (uint32_t)tile / nqb;
  const int part = __builtin_amdgcn_readfirstlane((int)(rest % (uint32_t)P));
  const int h = __builtin_amdgcn_readfirstlane((int)(rest / (uint32_t)P));
  const int g_begin = (int)(S.G * part / P), g_end = (int)(S.G * (part + 1) / P);
  const int k_si = (int)S.k_si, v_si = (int)S.v_si;
  const uint8_t* mask = a.mask != nullptr && S.m_off >= 0 ? a.mask + S.m_off : nullptr;
  const int q0 = qb * 128 + ((wave + part) & 3) * 32, q = q0 + lq;
  const bool qv = q < Lq, active = q0 < Lq;
  TileDma<DP> kd, vd;
  const float* kh = a.k + S.k_off + h * S.k_sh;
  const float* vh = a.v + S.v_off + h * S.v_sh;
  kd.init(kh, Lk, k_si, D, wave, lane);
  vd.init(vh, Lk, v_si, D, wave, lane);
  const uint32_t k_bytes = kd.rsrc[2], v_bytes = vd.rsrc[2];
  BiasRow br;
  br.rsrc = make_rsrc(a.bias + S.b_off + h * S.b_sh, (uint32_t)(((int64_t)(Lq - 1) * S.b_si + Lk) * 4));
  br.off = qv ? (uint32_t)((q * (int)S.b_si + g2 * 4) * 4) : kOut;
  br.Lk = Lk;
  const ColLane<DP> col(lq, g2);
  const float c1 = a.scale * kLog2e;

  auto keep_of = [&](int g) { load_keep(keep_lds[g & 3], mask != nullptr ? mask + g * S.m_sg : nullptr, Lk, wave, lane); };
  auto bits_of = [&](int g, int t) { return t * 32 < Lk ? __builtin_amdgcn_readfirstlane(keep_lds[g & 3][t]) : 0u; };
  // tile t of group g into ring buffer buf (a tile past Lk: nothing, it is not read)
  auto dma = [&](int g, int t, int buf) {
    if (g >= g_end || t * 32 >= Lk) return;
    const uint32_t bits = bits_of(g, t);
    kd.rsrc = rsrc_words(kh + g * S.k_sg, k_bytes);
    vd.rsrc = rsrc_words(vh + g * S.v_sg, v_bytes);
    kd.issue(k_lds[buf], wave, (uint32_t)(t * 32 * k_si * 4), bits);
    vd.issue(v_lds[buf], wave, (uint32_t)(t * 32 * v_si * 4), bits);
  };

  f32x16 region[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) region[t] = f32x16{};
  float bias[16];
  static_assert(NT >= 2 && NT <= kDqbTiles, "key tiles");
  keep_of(g_begin);
  if (g_begin + 1 < g_end) keep_of(g_begin + 1);
  __syncthreads();
  dma(g_begin, 0, 0);
  dma(g_begin, 1, 1);
  if (active) br.load(0, bias);
  int buf = 0;
  for (int g = g_begin; g < g_end; ++g) {
    const int64_t lidx = S.l_off + ((int64_t)g * H + h) * Lq + q;
    float qf[NS], df[NS], dlt = 0.0f;
    row_load<DP>(a.q + S.q_off + g * S.q_sg + h * S.q_sh + (int64_t)q * S.q_si, qv, D, g2, qf);
    row_load<DP>(a.dout + S.do_off + g * S.do_sg + h * S.do_sh + (int64_t)q * S.do_si, qv, D, g2, df);
    {
      float of[NS];
      row_load<DP>(a.out + S.o_off + g * S.o_sg + h * S.o_sh + (int64_t)q * S.o_si, qv, D, g2, of);
#pragma unroll
      for (int s = 0; s < NS; ++s) dlt = __builtin_fmaf(of[s], df[s], dlt);
      dlt = sum_halves(dlt);
      if (qv && g2 == 0) a.delta[lidx] = dlt;
    }
    const float lse = qv ? a.lse[lidx] : 0.0f;
    f32x16 acc = f32x16{};
    if (g == g_begin) {
      vm_drain();
      lds_barrier();
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int b2 = buf == 0 ? 2 : buf - 1;
      const uint32_t bits = bits_of(g, t);
      const bool run = active && bits != 0;
      // (opaque, so that the offsets derived from it are not kept in registers for every tile)
      asm volatile("" : "+v"(br.off), "+s"(br.Lk));
      __builtin_amdgcn_sched_barrier(0);
      float x[16];
      f32x16 pacc = f32x16{};
      if (run) {
        f32x16 sacc = f32x16{};
        {
          float kf[NS], vf[NS];
          row_frag<DP>(k_lds[buf], lq, g2, kf);
          row_frag<DP>(v_lds[buf], lq, g2, vf);
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            sacc = mma2(kf[s], qf[s], sacc);
            pacc = mma2(vf[s], df[s], pacc);
          }
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) x[j] = __builtin_fmaf(sacc[j], c1, bias[j] * kLog2e);
        if (bits != 0xFFFFFFFFu) {
          const uint32_t lb = bits >> (g2 * 4);
#pragma unroll
          for (int j = 0; j < 16; ++j) x[j] = (lb >> (((j >> 2) << 3) | (j & 3))) & 1 ? x[j] : kNegInf;
        }
      }
      vm_drain();
      if (active) br.load((t + 1 < NT ? t + 1 : 0) * 32, bias);
      // two tiles on, in this group or the next
      dma(t + 2 < NT ? g : g + 1, (t + 2) % NT, b2);
      if (t == 0 && g + 2 < g_end) keep_of(g + 2);
      if (run) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          x[j] = __builtin_amdgcn_exp2f(x[j] - lse) * (pacc[j] - dlt);
          region[t][j] += x[j];
          acc = mma2(col.get(k_lds[buf], j, 0), x[j], acc);
        }
      }
      lds_barrier();
      buf = buf == 2 ? 0 : buf + 1;
    }
    if (qv && a.dq != nullptr) {
      float* row = a.dq + S.q_off + g * S.q_sg + h * S.q_sh + (int64_t)q * S.q_si;
#pragma unroll
      for (int i = 0; i < 4; ++i) put4(row, 8 * i + 4 * g2, D, acc, i, a.scale);
    }
  }
  if (!qv) return;
  float* dst = P == 1 ? a.dbias : a.dbias_part + (int64_t)part * a.dbias_extent;
  float* row = dst + S.db_off + h * S.db_sh + (int64_t)q * S.db_si;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int j = 0; j < 16; j += 4)
      put_ds(row, t * 32 + kappa(g2, j), Lk, region[t][j], region[t][j + 1], region[t][j + 2], region[t][j + 3]);
}

// ------------------------------------------------------------------ dK, dV
// A wave's lanes own one key each (the MFMA column); the workgroup's 128 keys
// walk the queries in tiles of 32, Q and dO through the LDS ring.
template <int DP, bool HAS_BIAS>
__global__ __launch_bounds__(256, 2) void attn_dkv_f32_kernel(BwdArgsT<float, float> a) {
  constexpr int NS = DP / 2, NDT = DP / 32, TB = 32 * DP;
  __shared__ __attribute__((aligned(16))) float q_lds[kRing][TB];
  __shared__ __attribute__((aligned(16))) float d_lds[kRing][TB];
  __shared__ __attribute__((aligned(16))) float ld_lds[kRing][64];  // LSE of the tile's queries, then delta

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3, lane = threadIdx.x & 63;
  const int lq = lane & 31, g2 = lane >> 5;
  Where w;
  if (!locate(a, w, [](const Sample& s) { return cdiv(s.Lk, 128); })) return;
  const Sample& S = reinterpret_cast<const Sample*>(a.table)[w.s];
  const int g = w.g, h = w.h, H = a.num_heads, D = a.head_size;
  const int Lq = (int)S.Lq, Lk = (int)S.Lk, ntiles = (Lq + 31) >> 5;
  const int q_si = (int)S.q_si, do_si = (int)S.do_si, b_si = (int)S.b_si;
  const int k0 = w.blk * 128 + ((wave + g) & 3) * 32, key = k0 + lq;
  const bool active = k0 < Lk;
  bool kvalid = key < Lk;
  if (kvalid && a.mask != nullptr && S.m_off >= 0) kvalid = a.mask[S.m_off + g * S.m_sg + key] != 0;
  float kf[NS], vf[NS];
  row_load<DP>(a.k + S.k_off + g * S.k_sg + h * S.k_sh + (int64_t)key * S.k_si, kvalid, D, g2, kf);
  row_load<DP>(a.v + S.v_off + g * S.v_sg + h * S.v_sh + (int64_t)key * S.v_si, kvalid, D, g2, vf);
  TileDma<DP> qd, dd;
  qd.init(a.q + S.q_off + g * S.q_sg + h * S.q_sh, Lq, q_si, D, wave, lane);
  dd.init(a.dout + S.do_off + g * S.do_sg + h * S.do_sh, Lq, do_si, D, wave, lane);
  // bias[q][key]: a row of keys per query, 128 contiguous bytes per lane half
  __amdgpu_buffer_rsrc_t b_rsrc;
  uint32_t b_off = 0;
  if constexpr (HAS_BIAS) {
    b_rsrc = make_rsrc(a.bias + S.b_off + g * S.b_sg + h * S.b_sh, (uint32_t)(((int64_t)(Lq - 1) * b_si + Lk) * 4));
    b_off = key < Lk ? (uint32_t)((g2 * 4 * b_si + key) * 4) : kOut;
  }
  auto load_bias = [&](int t, float (&b)[16]) {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const uint32_t o = b_off + (uint32_t)((t * 32 + (j >> 2) * 8 + (j & 3)) * b_si * 4);
      b[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(b_rsrc, o, 0, 0));
    }
  };
  const int64_t l_row = S.l_off + ((int64_t)g * H + h) * Lq;
  // thread t < 32: LSE of query t of the tile (queries past Lq: P = exp2(x - inf) = 0), t < 64: delta
  auto load_ld = [&](int t) {
    const int qi = t * 32 + lq;
    float v = g2 ? 0.0f : __builtin_huge_valf();
    if (wave == 0 && qi < Lq) v = g2 ? a.delta[l_row + qi] : a.lse[l_row + qi];
    return v;
  };
  auto dma = [&](int t, int buf) {
    if (t >= ntiles) return;
    const int left = Lq - t * 32;
    const uint32_t bits = left >= 32 ? 0xFFFFFFFFu : (1u << left) - 1u;
    qd.issue(q_lds[buf], wave, (uint32_t)(t * 32 * q_si * 4), bits);
    dd.issue(d_lds[buf], wave, (uint32_t)(t * 32 * do_si * 4), bits);
  };
  const ColLane<DP> col(lq, g2);
  const float c1 = a.scale * kLog2e;
  f32x16 dk[NDT], dv[NDT];
#pragma unroll
  for (int t = 0; t < NDT; ++t) dk[t] = dv[t] = f32x16{};
  float bias[16];
  dma(0, 0);
  dma(1, 1);
  if (wave == 0) {
    ld_lds[0][lane] = load_ld(0);
    ld_lds[1][lane] = load_ld(1);
  }
  float st = load_ld(2);
  if constexpr (HAS_BIAS)
    if (active) load_bias(0, bias);
  vm_drain();
  __syncthreads();
  int buf = 0;
  for (int t = 0; t < ntiles; ++t) {
    const int b2 = buf == 0 ? 2 : buf - 1;
    float p[16];
    f32x16 pacc = f32x16{};
    if (active) {
      f32x16 sacc = f32x16{};
      {
        float qa[NS], da[NS];
        row_frag<DP>(q_lds[buf], lq, g2, qa);
        row_frag<DP>(d_lds[buf], lq, g2, da);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          sacc = mma2(qa[s], kf[s], sacc);
          pacc = mma2(da[s], vf[s], pacc);
        }
      }
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        p[j] = HAS_BIAS ? __builtin_fmaf(sacc[j], c1, bias[j] * kLog2e) : sacc[j] * c1;
        p[j] = kvalid ? p[j] : kNegInf;
      }
    }
    vm_drain();
    if (wave == 0) ld_lds[b2][lane] = st;  // the tile after the next, loaded a step ago
    if constexpr (HAS_BIAS)
      if (active && t + 1 < ntiles) load_bias(t + 1, bias);
    dma(t + 2, b2);
    st = load_ld(t + 3);
    if (active) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float4 l = *reinterpret_cast<const float4*>(&ld_lds[buf][8 * i + 4 * g2]);
        const float4 d = *reinterpret_cast<const float4*>(&ld_lds[buf][32 + 8 * i + 4 * g2]);
        const float lv[4] = {l.x, l.y, l.z, l.w}, dl[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = 4 * i + e;
          p[j] = __builtin_amdgcn_exp2f(p[j] - lv[e]);
          const float ds = p[j] * (pacc[j] - dl[e]);
#pragma unroll
          for (int n = 0; n < NDT; ++n) {
            dv[n] = mma2(col.get(d_lds[buf], j, n), p[j], dv[n]);
            dk[n] = mma2(col.get(q_lds[buf], j, n), ds, dk[n]);
          }
        }
      }
    }
    lds_barrier();
    buf = buf == 2 ? 0 : buf + 1;
  }
  if (key >= Lk) return;
  float* krow = a.dk ? a.dk + S.k_off + g * S.k_sg + h * S.k_sh + (int64_t)key * S.k_si : nullptr;
  float* vrow = a.dv ? a.dv + S.v_off + g * S.v_sg + h * S.v_sh + (int64_t)key * S.v_si : nullptr;
#pragma unroll
  for (int t = 0; t < NDT; ++t) {
    if (!kvalid) dk[t] = dv[t] = f32x16{};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (krow) put4(krow, t * 32 + 8 * i + 4 * g2, D, dk[t], i, a.scale);
      if (vrow) put4(vrow, t * 32 + 8 * i + 4 * g2, D, dv[t], i, 1.0f);
    }
  }
}

// ------------------------------------------------------------------ shared dBias
// One workgroup = 128 queries (32 per wave) x 32 keys of one head, walking the
// groups of one part: the wave's bias block stays in registers, the group's
// K/V tile goes through the LDS ring, each wave's Q/dO rows straight into
// registers a group ahead.  Partial sums per part as in the generic kernel.
template <int DP>
__global__ __launch_bounds__(256, 2) void attn_dbias_f32_kernel(BwdArgsT<float, float> a) {
  constexpr int NS = DP / 2, TB = 32 * DP;
  __shared__ __attribute__((aligned(16))) float k_lds[kRing][TB];
  __shared__ __attribute__((aligned(16))) float v_lds[kRing][TB];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3, lane = threadIdx.x & 63;
  const int lq = lane & 31, g2 = lane >> 5;
  int64_t tile = xcd_tile(blockIdx.x, gridDim.x, xcd_chunk(a.uniform_tiles));
  if (tile >= a.total_tiles) return;
  const Sample* tab = reinterpret_cast<const Sample*>(a.table);
  const int H = a.num_heads, P = a.parts;
  const int s_idx = find_sample(tile, tab, a.num_samples, a.uniform_tiles, [&](const Sample& s) {
    return s.bias_mode == OOPS_BIAS_SHARED ? H * cdiv(s.Lq, 128) * cdiv(s.Lk, 32) * P : (int64_t)0;
  });
  if (s_idx < 0) return;
  const Sample& S = tab[__builtin_amdgcn_readfirstlane(s_idx)];
  const int Lq = (int)S.Lq, Lk = (int)S.Lk, D = a.head_size;
  const uint32_t nkb = (uint32_t)cdiv(Lk, 32), nqb = (uint32_t)cdiv(Lq, 128);
  // (head, part, query block, key block): neighbours share their groups' rows
  const int kb = __builtin_amdgcn_readfirstlane((int)((uint32_t)tile % nkb));
  uint32_t rest = (uint32_t)tile / nkb;
  const int qb = __builtin_amdgcn_readfirstlane((int)(rest % nqb));
  rest /= nqb;
  const int part = __builtin_amdgcn_readfirstlane((int)(rest % (uint32_t)P));
  const int h = __builtin_amdgcn_readfirstlane((int)(rest / (uint32_t)P));
  const int g_begin = (int)(S.G * part / P), g_end = (int)(S.G * (part + 1) / P);
  const int k0 = kb * 32, q0 = qb * 128 + wave * 32, q = q0 + lq;
  const bool qv = q < Lq, active = q0 < Lq;
  const uint8_t* mask = a.mask != nullptr && S.m_off >= 0 ? a.mask + S.m_off : nullptr;
  const float c1 = a.scale * kLog2e;

  float xb[16], acc[16];
  {
    const float* brow = a.bias + S.b_off + h * S.b_sh + (int64_t)q * S.b_si;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int key = k0 + kappa(g2, j);
      xb[j] = qv && key < Lk ? brow[key] * kLog2e : 0.0f;
      acc[j] = 0.0f;
    }
  }
  const float* kh = a.k + S.k_off + h * S.k_sh + (int64_t)k0 * S.k_si;
  const float* vh = a.v + S.v_off + h * S.v_sh + (int64_t)k0 * S.v_si;
  const int left = min(32, Lk - k0);
  TileDma<DP> kd, vd;
  kd.init(kh, left, (int)S.k_si, D, wave, lane);
  vd.init(vh, left, (int)S.v_si, D, wave, lane);
  const uint32_t k_bytes = kd.rsrc[2], v_bytes = vd.rsrc[2];
  const float* qrow = a.q + S.q_off + h * S.q_sh + (int64_t)q * S.q_si;
  const float* drow = a.dout + S.do_off + h * S.do_sh + (int64_t)q * S.do_si;
  const int64_t l0 = S.l_off + (int64_t)h * Lq + q, l_sg = (int64_t)H * Lq;

  // the keys of this block that group g keeps
  auto keep_of = [&](int g) {
    const int key = k0 + lq;
    bool k = g < g_end && key < Lk;
    if (k && mask != nullptr) k = mask[g * S.m_sg + key] != 0;
    return (uint32_t)__ballot(k);
  };
  auto dma = [&](int g, int buf, uint32_t bits) {
    if (g >= g_end) return;
    kd.rsrc = rsrc_words(kh + g * S.k_sg, k_bytes);
    vd.rsrc = rsrc_words(vh + g * S.v_sg, v_bytes);
    kd.issue(k_lds[buf], wave, 0, bits);
    vd.issue(v_lds[buf], wave, 0, bits);
  };
  float qf[NS], df[NS], qn[NS], dn[NS], lse, dlt, lse_n, dlt_n;
  auto load_q = [&](int g, float (&x)[NS], float (&d)[NS], float& l, float& dl) {
    const bool ok = qv && g < g_end;
    row_load<DP>(qrow + (ok ? g * S.q_sg : 0), ok, D, g2, x);
    row_load<DP>(drow + (ok ? g * S.do_sg : 0), ok, D, g2, d);
    l = ok ? a.lse[l0 + g * l_sg] : __builtin_huge_valf();
    dl = ok ? a.delta[l0 + g * l_sg] : 0.0f;
  };

  uint32_t bits0 = keep_of(g_begin), bits1 = keep_of(g_begin + 1), bits2 = keep_of(g_begin + 2);
  dma(g_begin, 0, bits0);
  dma(g_begin + 1, 1, bits1);
  load_q(g_begin, qf, df, lse, dlt);
  vm_drain();
  __syncthreads();
  int buf = 0;
  for (int g = g_begin; g < g_end; ++g) {
    const int b2 = buf == 0 ? 2 : buf - 1;
    vm_drain();  // (the next group's tile, issued a step ago)
    dma(g + 2, b2, bits2);
    const uint32_t bits3 = keep_of(g + 3);
    if (active) {
      load_q(g + 1, qn, dn, lse_n, dlt_n);
      f32x16 sacc = f32x16{}, pacc = f32x16{};
      float kf[NS], vf[NS];
      row_frag<DP>(k_lds[buf], lq, g2, kf);
      row_frag<DP>(v_lds[buf], lq, g2, vf);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        sacc = mma2(kf[s], qf[s], sacc);
        pacc = mma2(vf[s], df[s], pacc);
      }
      const uint32_t lb = bits0 >> (g2 * 4);
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        float x = __builtin_fmaf(sacc[j], c1, xb[j]);
        if (bits0 != 0xFFFFFFFFu) x = (lb >> (((j >> 2) << 3) | (j & 3))) & 1 ? x : kNegInf;
        acc[j] += __builtin_amdgcn_exp2f(x - lse) * (pacc[j] - dlt);
      }
#pragma unroll
      for (int s = 0; s < NS; ++s) qf[s] = qn[s], df[s] = dn[s];
      lse = lse_n;
      dlt = dlt_n;
    }
    lds_barrier();
    buf = buf == 2 ? 0 : buf + 1;
    bits0 = bits1;
    bits1 = bits2;
    bits2 = bits3;
  }
  if (!qv) return;
  float* dst = P == 1 ? a.dbias : a.dbias_part + (int64_t)part * a.dbias_extent;
  float* row = dst + S.db_off + h * S.db_sh + (int64_t)q * S.db_si;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int key = k0 + kappa(g2, j);
    if (key < Lk) row[key] = acc[j];
  }
}

template <typename F>
void by_dp(const Plan& plan, F&& f) {
  if (plan.dp == 32) f(std::integral_constant<int, 32>{});
  else f(std::integral_constant<int, 64>{});
}

}  // namespace

// Where these kernels do not apply (pair masks, head sizes above 64 or no
// multiple of 4, unaligned rows) the generic ones run.  Measured at 193
// residues, 4 heads of 32, shared bias, ending node (generic -> here):
// forward 112 -> 73 us, dK/dV 251 -> 126, dQ + delta + dBias 441 -> 140 (dQ
// and dBias in separate kernels: 105 + 116); forward + backward 808 -> 335 us.
// Matrix cores busy 41% (forward), 50% (dK/dV) and 34% (dQ + dBias) there, 60%
// and 70% (forward, dK/dV) at 256 residues: 193 leaves 1544 workgroups on 256
// CUs, and a CU's seventh runs alone.
bool attn_f32_ok(const oops_attn_geometry& geo, const Plan& plan) {
  return geo.force_generic != 1 && geo.dtype == OOPS_F32 && plan.dp <= 64 && geo.head_size % 4 == 0 &&
         geo.vec_ok != 0 && !plan.any_pair_mask && !plan.any_bare && plan.offsets_32bit && plan.q_offsets_32bit && plan.max_len_k <= 32 * kF32MaxTiles;
}

// The dQ + dBias kernel: its sums of all key tiles have to fit the registers
// beside the dQ kernel's (two waves per SIMD up to 256 keys of head size 32).
// Separate kernels against it: 128 residues 28 + 47 and 45 us, 256 residues
// 130 + 163 and 197 us.
bool dqb_f32_ok(const oops_attn_geometry& geo, const Plan& plan) {
  return geo.force_generic == 0 && attn_f32_ok(geo, plan) && plan.dp == 32 && plan.all_shared && !plan.f32_direct &&
         plan.max_len_k <= 32 * kDqbTiles;
}

hipError_t launch_forward_f32(const oops_attn_geometry& geo, const Plan& plan, FwdArgsT<float, float>& a,
                              hipStream_t stream) {
  a.total_tiles = plan.fwd_tiles;
  a.uniform_tiles = plan.fwd_uniform;
  a.head_group = head_group(geo);
  const dim3 grid((unsigned)xcd_grid(plan.fwd_tiles, xcd_chunk(plan.fwd_uniform)));
  by_dp(plan, [&](auto dpc) {
    constexpr int DP = decltype(dpc)::value;
    if (a.bias != nullptr) hipLaunchKernelGGL((attn_fwd_f32_kernel<DP, true>), grid, dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((attn_fwd_f32_kernel<DP, false>), grid, dim3(256), 0, stream, a);
  });
  return hipGetLastError();
}

hipError_t launch_backward_f32(const Plan& plan, BwdArgsT<float, float> a, int phase, hipStream_t stream) {
  if (phase == (OOPS_PHASE_DQ | OOPS_PHASE_DBIAS)) {
    a.parts = plan.f32_parts;
    a.total_tiles = plan.f32_tiles;
    a.uniform_tiles = plan.f32_uniform;
    const dim3 grid((unsigned)xcd_grid(a.total_tiles, xcd_chunk(a.uniform_tiles)));
    auto go = [&](auto nt) {
      hipLaunchKernelGGL((attn_dqb_f32_kernel<decltype(nt)::value>), grid, dim3(256), 0, stream, a);
    };
    const int nt = (int)((plan.max_len_k + 31) / 32);
    if (nt <= 2) go(std::integral_constant<int, 2>{});
    else if (nt == 3) go(std::integral_constant<int, 3>{});
    else if (nt == 4) go(std::integral_constant<int, 4>{});
    else if (nt == 5) go(std::integral_constant<int, 5>{});
    else if (nt == 6) go(std::integral_constant<int, 6>{});
    else if (nt == 7) go(std::integral_constant<int, 7>{});
    else go(std::integral_constant<int, 8>{});
    return hipGetLastError();
  }
  const int64_t tiles = phase == OOPS_PHASE_DQ ? plan.fwd_tiles : phase == OOPS_PHASE_DKV ? plan.dkv_tiles : plan.sbias_tiles;
  a.total_tiles = tiles;
  a.uniform_tiles = phase == OOPS_PHASE_DQ ? plan.fwd_uniform : phase == OOPS_PHASE_DKV ? plan.dkv_uniform : plan.sbias_uniform;
  const dim3 grid((unsigned)xcd_grid(tiles, xcd_chunk(a.uniform_tiles)));
  by_dp(plan, [&](auto dpc) {
    constexpr int DP = decltype(dpc)::value;
    if (phase == OOPS_PHASE_DBIAS) {
      hipLaunchKernelGGL((attn_dbias_f32_kernel<DP>), grid, dim3(256), 0, stream, a);
    } else if (phase == OOPS_PHASE_DQ) {
      if (a.bias != nullptr) hipLaunchKernelGGL((attn_dq_f32_kernel<DP, true>), grid, dim3(256), 0, stream, a);
      else hipLaunchKernelGGL((attn_dq_f32_kernel<DP, false>), grid, dim3(256), 0, stream, a);
    } else {
      if (a.bias != nullptr) hipLaunchKernelGGL((attn_dkv_f32_kernel<DP, true>), grid, dim3(256), 0, stream, a);
      else hipLaunchKernelGGL((attn_dkv_f32_kernel<DP, false>), grid, dim3(256), 0, stream, a);
    }
  });
  return hipGetLastError();
}

}  // namespace oops
