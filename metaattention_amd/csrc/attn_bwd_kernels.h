// Parallel attention backward (dq, dk, dv) for gfx950: softmax, sigmoid and relu row functions.
//
// Replaces the backward of _attention (attention_engine/core/template/tl_template/attn/attn_tl.py:
// 669-692): the delta pre-pass (:212-237), the dK/dV kernel with fp32 dQ atomics (:301-420) and the
// dQ post-pass (:239-262).  With p = rowfn(x), x = s * scale + bias, s = q.k^T:
//   softmax   p = exp(x - lse),       ds = p * (dp - delta) * scale,   delta_i = sum_d do_id * o_id
//   sigmoid   p = 1 / (1 + exp(-x)),  ds = dp * p * (1 - p) * scale
//   relu      p = max(x, 0),          ds = dp * [x > 0] * scale
//   dp = do.v^T,   dv = p^T do,   dk = ds^T q,   dq = ds k
// (p and ds are rounded to the tensor dtype before the second products, as there: :357-362; the factor
// `scale` common to dq and dk is applied once, when their accumulators are stored).
// Masks: none, causal, or an element-wise keep mask given in both orientations (the dq kernel walks a
// query row of it, the dk / dv kernel a key's column of its transpose); only tiles that a mask can
// touch evaluate it.
//
// No atomics: two kernels, each owning its outputs.
//   attn_bwd_dq_kernel   a wave owns 32 query rows and walks the kv sequence; everything transposed as in
//                        the forward kernels (S^T = K Q^T, dP^T = V dO^T: lane = query row, so lse and
//                        delta are per-lane scalars; dS^T is directly the B operand of dQ^T += K^T dS^T).
//                        It also computes delta and leaves it in the workspace for the second kernel.
//   attn_bwd_dkv_kernel  a wave owns 32 keys of one kv head (K and V fragments in registers as B
//                        operands) and walks the query rows of every query head of its group; here
//                        S = Q K^T and dP = dO V^T are NOT transposed (lane = key), so P and dS are
//                        directly the B operands of dV^T += dO^T P and dK^T += Q^T dS; lse and delta of
//                        a tile's rows come with the tile.  dk and dv in one launch or in two (then the
//                        scores are computed once more), whichever lets two waves share a SIMD.
//   attn_bwd_dkv_pair_kernel  the same work at 128 / 128, 192 / 128, 128 / 256 and 256 / 256: dk and dv in one launch, two waves
//                        per SIMD with the same 32 keys, one for dv and one for dk.
//   attn_bwd_dkv_fused_kernel  the same at 64 / 64: dk and dv in one wave, the loop pipelined inside it (see there).
// The scores are recomputed in both kernels (7 tile products instead of 5; 8 where dk and dv take two
// launches), which is what avoiding the fp32 atomics and the post-pass costs.  Tiles of 32 rows arrive by
// direct-to-LDS DMA (a wave-uniform base in scalar registers plus 32-bit lane offsets computed once),
// through a ring of stages, one barrier per tile, XOR-swizzled like the forward tiles; the column-side
// operands (K^T, dO^T, Q^T) come from the same tiles through the transposing LDS read.
#pragma once
#include "attn_bwd.h"

namespace ma {

namespace {
enum { BF_SOFTMAX = 0, BF_SIGMOID = 1, BF_RELU = 2, BF_RETENTION = 3 };   // = MA_ATTN_* of the C interface

// ds / scale (and p) of one score element: the common factor `scale` of dq and dk is applied once, when the
// accumulators are stored.  x2 = (s * scale + bias) * log2(e) for softmax / sigmoid.
// Retention (examples/retention_parallel.py:76-86 of the reference): p = s * scale * m / r with m the caller's score
// multiplier and r the row scale of the forward pass, which the backward treats as a constant (dscores = dp / r);
// `lse2` carries m / r.
template <int FAMILY>
__device__ __forceinline__ void row_fn_bwd(float s, float dp, bool masked, float c_scale, float c_bias, float scale, float bias,
                                           float lse2, float delta, float& p, float& ds) {
  if constexpr (FAMILY == BF_RETENTION) {
    p = masked ? 0.f : s * scale * lse2;
    ds = masked ? 0.f : dp * lse2;
  } else if constexpr (FAMILY == BF_SOFTMAX) {
    p = masked ? 0.f : fast_exp2(s * c_scale + lse2);   // (lse2 = c_bias - lse * log2(e), folded by the caller)
    ds = p * (dp - delta);
  } else if constexpr (FAMILY == BF_SIGMOID) {
    p = masked ? 0.f : fast_rcp(1.f + fast_exp2(-(s * c_scale + c_bias)));
    ds = dp * p * (1.f - p);
  } else {
    const float x = s * scale + bias;
    p = masked ? 0.f : fmaxf(x, 0.f);
    ds = (!masked && x > 0.f) ? dp : 0.f;
  }
}

// The same in two parts, for the pipelined kernel: p of a kept score, and ds / scale from p.
template <int FAMILY>
__device__ __forceinline__ float row_p(float s, float c_scale, float c_bias, float scale, float bias, float lse2) {
  if constexpr (FAMILY == BF_SOFTMAX) return fast_exp2(s * c_scale + lse2);
  else if constexpr (FAMILY == BF_SIGMOID) return fast_rcp(1.f + fast_exp2(-(s * c_scale + c_bias)));
  else return fmaxf(s * scale + bias, 0.f);
}
template <int FAMILY>
__device__ __forceinline__ float row_ds(float p, float dp, float delta) {
  if constexpr (FAMILY == BF_SOFTMAX) return p * (dp - delta);
  else if constexpr (FAMILY == BF_SIGMOID) return dp * p * (1.f - p);
  else return p > 0.f ? dp : 0.f;
}

// EXTRA instantiations (softmax, sigmoid, relu): the additive terms and the soft-capping of the forward pass, applied to the recomputed
// raw scores.  `extra` is (add + slope_q q + slope_kv kv) of the element; the scores stay in units of 1 / scale, so that
// everything behind sees s * scale + bias as before.  With softcap > 0, x = s * scale + bias becomes softcap * tanh(x) and
// `cap_grad` the derivative softcap * (1 - tanh^2 x), which multiplies ds; tanh(x) = 1 - 2 / (1 + e^(2x)) as in the forward.
__device__ __forceinline__ float apply_extra(float s, float extra, float scale, float inv_scale, float bias, float softcap, float& cap_grad) {
  s += extra * inv_scale;
  cap_grad = 1.f;
  if (softcap > 0.f) {
    const float x = s * scale + bias;
    const float th = 1.f - 2.f * fast_rcp(1.f + fast_exp2(x * (2.f * kLog2e)));
    s = (softcap * th - bias) * inv_scale;
    cap_grad = softcap * (1.f - th * th);
  }
  return s;
}

// DMA of a [32 x ROWB bytes] tile whose rows are `row_stride` bytes apart in memory: each instruction
// moves 1 KB; lane i fetches the 16-byte chunk that belongs at physical position i of that KB.  Rows
// beyond `limit` are clamped to the last one (whatever is computed from them is masked).
template <int ROWB, int NWAVES, int USED = ROWB / 16>
__device__ __forceinline__ void dma_tile(const char* src, int64_t row_stride, int row0, int limit, uint32_t lds_base, int wave, int lane) {
  constexpr int CPR = ROWB / 16, NI = 32 * ROWB / 1024;
  for (int ii = wave; ii < NI; ii += NWAVES) {
    const int row = ii * (1024 / ROWB) + lane / CPR, c = lane % CPR;
    const int grow = min(row0 + row, limit - 1);
    if (USED == CPR || (c ^ swz_tile<CPR>(row)) < USED)   // (chunks beyond the head size do not exist in memory)
      dma16(src + grow * row_stride + ((c ^ swz_tile<CPR>(row)) << 4), lds_base + ii * 1024);
  }
}

// Stages of the pipelined dk / dv kernel's tile ring: with eight, tiles arrive four steps ahead; beside the mask bytes of a stage (4 KB) four fit.
constexpr int fused_stages(bool masks) { return masks ? 4 : 8; }
// Workgroups of the pipelined dk / dv kernel that a CU holds.  At 64 / 64 a step is 16 MFMAs behind some 200 vector
// instructions, LDS latencies and a barrier, and one wave per SIMD waits for most of it: two workgroups (256 registers a wave,
// lse and delta requested in the step that uses them) take B4 H32 S2048 causal forward + backward from 595 to 438 us (sigmoid)
// and 557 to 421 us (softmax), B8 H32 S4096 3984 -> 3353 and 3723 -> 3130.
constexpr int FUSED_PER_CU = 2;
// Waits until at most N of this wave's vector-memory loads are outstanding (they complete in order).
template <int N>
__device__ __forceinline__ void wait_dma_but() { __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14)); }

// Retention: a wave's [32 rows x 32 columns] block of the score multiplier (64 bytes per row) by DMA into a 2 KB area of
// its own, two instructions; the 16-byte chunk c of row r sits at position c ^ ((r >> 1) & 3) of the row, so that the
// 8-byte reads of `mult_read` (lane: row r, columns 8 q4 + 4 g ..) spread over the banks.  `first` points at the wave's
// first row and the block's first column; rows from `rows_left` on are clamped to the last one.
template <typename T>
__device__ __forceinline__ void mult_dma(const T* first, int64_t row_stride, int rows_left, uint32_t lds_base, int lane) {
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int row = (lane >> 2) + 16 * j, lc = (lane & 3) ^ ((row >> 1) & 3);
    dma16(first + (int64_t)min(row, rows_left - 1) * row_stride + 8 * lc, lds_base + j * 1024);
  }
}
template <typename T>
__device__ __forceinline__ typename Elem<T>::x4 mult_read(uint32_t lds_base, int r, int g, int q4) {
  return lds_read<typename Elem<T>::x4>(lds_base + r * 64 + ((q4 ^ ((r >> 1) & 3)) << 4) + 8 * g);
}

// Element-wise keep masks: a wave's [32 rows x 32 columns] block of mask bytes by DMA into a 1 KB area of its own (one
// instruction: two lanes per row); lane (row r, half g) then reads the four bytes of columns 8 q4 + 4 g .. as one word.
__device__ __forceinline__ void keep_dma(const uint8_t* first, int64_t row_stride, int rows_left, uint32_t lds_base, int lane) {
  dma16(first + (int64_t)min(lane >> 1, rows_left - 1) * row_stride + 16 * (lane & 1), lds_base);
}
__device__ __forceinline__ uint32_t keep_read(uint32_t lds_base, int r, int g, int q4) {
  return lds_read<uint32_t>(lds_base + r * 32 + 8 * q4 + 4 * g);
}

// [32 x 32] += A B^T over DIM columns, A = the 32 rows of an LDS tile (row reads), B = fragments in registers
template <typename T, int DIM>
__device__ __forceinline__ f32x16 mm_rows(uint32_t tile, int r, int g, const typename Elem<T>::x8 (&bf)[DIM / 16]) {
  using E = Elem<T>;
  using x8 = typename E::x8;
  constexpr int ROWB = pad_width(DIM) * 2, CPR = pad_width(DIM) / 8, KS = DIM / 16, AH = 2, RING = 3;
  // (tile bases and row offsets are multiples of the row size, so the swizzled chunk index has its own address
  // bits: another k-slice is one XOR with a constant away)
  const uint32_t a0 = tile + r * ROWB + (uint32_t)((g ^ swz_tile<CPR>(r)) << 4);
  const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  f32x16 acc;
  x8 af[RING];
#pragma unroll
  for (int ks = 0; ks < AH && ks < KS; ks++) af[ks] = lds_read<x8>(a0 ^ (uint32_t)(ks * 32));
#pragma unroll
  for (int ks = 0; ks < KS; ks++) {
    if (ks + AH < KS) af[(ks + AH) % RING] = lds_read<x8>(a0 ^ (uint32_t)((ks + AH) * 32));
    __builtin_amdgcn_sched_barrier(0);
    acc = E::mfma32(af[ks % RING], bf[ks], ks == 0 ? zero16 : acc);
    __builtin_amdgcn_sched_barrier(0);
  }
  return acc;
}

// acc[DIM/32 blocks of 32 columns] += (tile columns)^T . pf, where pf holds a [32 x 32] factor in
// accumulator order rounded to T (k slot i of slice s for lane half g is tile row 16s + 8(i/4) + 4g + i%4,
// which is the row order the transposing reads below fetch)
struct NoHook { __device__ __forceinline__ void operator()(int, int) const {} };
// `between(idx, n)` runs behind MFMA idx of n: vector work that the matrix pipe covers
template <typename T, int DIM, typename Hook = NoHook>
__device__ __forceinline__ void mm_cols(uint32_t tile, int lane, const typename Elem<T>::x8 (&pf)[2], f32x16 (&acc)[DIM / 32], Hook between = Hook()) {
  using E = Elem<T>;
  using x8 = typename E::x8;
  using x4 = typename E::x4;
  constexpr int ROWB = pad_width(DIM) * 2, CPR = pad_width(DIM) / 8, NB = DIM / 32, PF = NB >= 2 ? 4 : 2;
  const int g = lane >> 5, jr = (lane & 15) >> 2;
  const int lc = (((lane >> 4) & 1) << 1) | ((lane & 3) >> 1);
  const uint32_t b0 = tile + (4 * g + jr) * ROWB + (lane & 1) * 8 + (uint32_t)((lc ^ swz_tile<CPR>(4 * g + jr)) << 4);
  x4 lo[PF], hi[PF];
  auto request = [&](int idx) {   // idx = 2 block + slice
    const int db = idx >> 1, sl = idx & 1;
    lo[idx % PF] = lds_read_tr4<T>((b0 ^ (uint32_t)((4 * db) << 4)) + 16 * sl * ROWB);
    hi[idx % PF] = lds_read_tr4<T>((b0 ^ (uint32_t)(((4 * db) ^ 2) << 4)) + (16 * sl + 8) * ROWB);
  };
#pragma unroll
  for (int i = 0; i < PF - 1; i++) request(i);
#pragma unroll
  for (int idx = 0; idx < 2 * NB; idx++) {
    if (idx + PF - 1 < 2 * NB) request(idx + PF - 1);
    __builtin_amdgcn_sched_barrier(0);
    x8 af = __builtin_shufflevector(lo[idx % PF], hi[idx % PF], 0, 1, 2, 3, 4, 5, 6, 7);
    acc[idx >> 1] = E::mfma32(af, pf[idx & 1], acc[idx >> 1]);
    between(idx, 2 * NB);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// a wave's [DIM x 32] accumulator (lane = output row, elements = columns) to global rows of DIM
// elements, through a wave-private LDS block in two halves, 16-byte coalesced stores
template <typename T, int DIM>
__device__ __forceinline__ void store_rows(const f32x16 (&acc)[DIM / 32], float mult, uint32_t stage, T* gbase, int64_t row_stride,
                                           int row0, int row_limit, int lane) {
  using x4 = typename Elem<T>::x4;
  constexpr int NB = DIM / 32, HALF = DIM / 2, OROW = HALF * 2 + 16;
  const int r = lane & 31, g = lane >> 5;
#pragma unroll
  for (int hp = 0; hp < 2; hp++) {
#pragma unroll
    for (int dbl = 0; dbl < NB / 2; dbl++)
#pragma unroll
      for (int q4 = 0; q4 < 4; q4++) {
        x4 w;
#pragma unroll
        for (int i = 0; i < 4; i++) w[i] = (T)(acc[hp * (NB / 2) + dbl][4 * q4 + i] * mult);
        lds_write<x4>(stage + r * OROW + (32 * dbl + 8 * q4 + 4 * g) * 2, w);
      }
#pragma unroll
    for (int it = 0; it < 32 * (HALF / 8) / 64; it++) {
      const int ci = lane + 64 * it, row = ci / (HALF / 8), c = ci % (HALF / 8);
      const u32x4 w = lds_read<u32x4>(stage + row * OROW + c * 16);
      if (row0 + row < row_limit) *(u32x4*)(gbase + (int64_t)(row0 + row) * row_stride + hp * HALF + c * 8) = w;
    }
  }
}
}  // namespace

// ------------------------------------------------------------------------------------------------
// dq (and delta)
// ------------------------------------------------------------------------------------------------
// LDS of a stream of the dq kernel, and of the dk / dv kernels: two stages, the row values, the retention family's multiplier
// blocks or the keep-mask blocks; at least the output staging
constexpr size_t dq_lds(int dqk, int dv, int family) {
  const size_t tiles = 2 * (size_t)32 * (pad_width(dqk) + dv) * 2 + 1024 + (family == BF_RETENTION ? 2 * 4 * 2048 : 2 * 4 * 1024);
  const size_t out = 4 * 32 * (size_t)((dqk > dv ? dqk : dv) + 16);
  return tiles > out ? tiles : out;
}

// KVS: two streams of four waves walk every other tile each, side by side with their own stages, and their sums meet in LDS.
// MASKS: with the code for element-wise and tile masks.  Without it the kernel loses registers and branches of every step, and
// 64 / 64 fits four waves on a SIMD: dq of B4 H12 S1024 64/64 sigmoid causal 29 -> 27 us; forward + backward of B2 H32 S1600 64/64 relu
// 260 -> 228, 256/256 causal 770 -> 709, B1 H16 S700 128/256 causal 142 -> 124.
template <typename T, int DQK, int DV, int FAMILY, bool CAUSAL, bool MASKS, bool EXTRA = false, int KVS = 1>
__global__ __launch_bounds__(256 * KVS, (DQK + DV >= 512 ? 1 : DQK + DV <= 128 && !MASKS ? 4 : 2)) void attn_bwd_dq_kernel(const AttnBwdArgs a) {
  using E = Elem<T>;
  using x8 = typename E::x8;
  constexpr int BM = 128, BN = 32;
  constexpr int KS = DQK / 16, VS = DV / 16, QB = DQK / 32;
  constexpr int KROW = pad_width(DQK) * 2, VROW = DV * 2;   // (LDS rows; 192-wide keys sit in 256-wide rows)
  constexpr int KTILE = BN * KROW, VTILE = BN * VROW, STAGE = KTILE + VTILE;
  constexpr int STREAM_LDS = (int)dq_lds(DQK, DV, FAMILY);   // a stream's stages and mask blocks

  extern __shared__ __align__(16) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int stream = KVS > 1 ? wave_all >> 2 : 0, wave = KVS > 1 ? wave_all & 3 : wave_all;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(MA_LDS char*)smem + (KVS > 1 ? stream * STREAM_LDS : 0);
  const int r = lane & 31, g = lane >> 5;

  // (under a causal mask the heaviest row blocks of all heads first: see attn_wide_fwd_kernel.  B8 H32 S4096, 16 rounds of
  // workgroups, would lose 20 % to the L2 in this order)
  const int nmb = a.num_blocks, BH = a.B * a.H;
  const bool heavy_first = CAUSAL && gridDim.x <= kHeavyFirstMost;
  int bh, mb;
  if ((BH & 7) == 0) {
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    bh = (heavy_first ? slot % (BH >> 3) : slot / nmb) * 8 + xcd;
    mb = heavy_first ? slot / (BH >> 3) : slot % nmb;
  } else {
    bh = heavy_first ? blockIdx.x % BH : blockIdx.x / nmb;
    mb = heavy_first ? blockIdx.x / BH : blockIdx.x % nmb;
  }
  if (CAUSAL) mb = nmb - 1 - mb;
  const int b = bh / a.H, h = bh % a.H, hk = h / a.kv_group;
  const int m_wave = mb * BM + wave * 32, m_lane = m_wave + r;
  const int m_ld = min(m_lane, a.Sq - 1);

  // B operands of this wave's 32 rows: Q (for S^T = K Q^T) and dO (for dP^T = V dO^T)
  x8 qf[KS], dof[VS];
  float delta = 0.f, lse2 = 0.f;
  {
    const T* qp = (const T*)a.q + (int64_t)b * a.qsb + (int64_t)m_ld * a.qss + (int64_t)h * a.qsh + 8 * g;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) qf[ks] = *(const x8*)(qp + 16 * ks);
    const T* dop = (const T*)a.dout + (int64_t)b * a.dosb + (int64_t)m_ld * a.doss + (int64_t)h * a.dosh + 8 * g;
#pragma unroll
    for (int sl = 0; sl < VS; sl++) dof[sl] = *(const x8*)(dop + 16 * sl);
    if constexpr (FAMILY == BF_SOFTMAX) {
      const T* op = (const T*)a.o + (int64_t)b * a.osb + (int64_t)m_ld * a.oss + (int64_t)h * a.osh + 8 * g;
      float part = 0.f;
#pragma unroll
      for (int sl = 0; sl < VS; sl++) {
        const x8 of = *(const x8*)(op + 16 * sl);
#pragma unroll
        for (int i = 0; i < 8; i++) part += (float)dof[sl][i] * (float)of[i];
      }
      delta = part + xhalf(part);
      const int64_t ri = ((int64_t)b * a.H + h) * a.Sq + m_ld;
      lse2 = a.lse[ri] * kLog2e;
      if (g == 0 && m_lane < a.Sq && stream == 0) a.delta[ri] = delta;
    }
  }
  float r_inv = 1.f;   // retention: 1 / the row scale of the forward pass
  if constexpr (FAMILY == BF_RETENTION) r_inv = 1.f / a.lse[((int64_t)b * a.H + h) * a.Sq + m_ld];
  // retention: this lane's row of the score multiplier
  const T* sm_row = FAMILY == BF_RETENTION ? (const T*)a.smask + (int64_t)b * a.sm_sb + (int64_t)h * a.sm_sh + (int64_t)m_ld * a.sm_sq : nullptr;
  const char* kb = (const char*)((const T*)a.k + (int64_t)b * a.ksb + (int64_t)hk * a.ksh);
  const char* vb = (const char*)((const T*)a.v + (int64_t)b * a.vsb + (int64_t)hk * a.vsh);
  const int64_t k_row_bytes = a.kss * 2, v_row_bytes = a.vss * 2;

  int n_tiles = (a.Skv + BN - 1) / BN;
  if (CAUSAL) n_tiles = min(n_tiles, (mb * BM + BM + BN - 1) / BN);

  // retention: whole tiles of the multiplier come with the K/V tile (a 2 KB area per wave and stage behind the stages);
  // a partial last tile, or a tensor whose rows are not 16-byte aligned, is read from global memory as it is needed
  constexpr int MULT = 2 * STAGE;
  const bool mult_ok = FAMILY == BF_RETENTION && (a.sm_sq & 7) == 0 && (a.sm_sb & 7) == 0 && (a.sm_sh & 7) == 0 && ((uintptr_t)a.smask & 15) == 0;
  const uint8_t* elem_mask = MASKS ? a.elem_mask : nullptr;
  const bool keep_ok = FAMILY != BF_RETENTION && elem_mask && ((a.em_sq | a.em_sb | a.em_sh | (int64_t)(uintptr_t)elem_mask) & 15) == 0;
  const uint8_t* bm_full = MASKS && a.kv_block_mask ? a.kv_block_mask + (int64_t)b * a.kbm_sb + (int64_t)h * a.kbm_sh + (int64_t)mb * a.kbm_sq : nullptr;
  auto tile_full = [&](int jt_) { return bm_full && bm_full[jt_] >= 2; };   // the element-wise mask keeps every score of the tile
  TileDma<KROW, 4, DQK / 8> k_dma;
  TileDma<VROW, 4> v_dma;
  k_dma.init((uint32_t)k_row_bytes, wave, lane);
  v_dma.init((uint32_t)v_row_bytes, wave, lane);
  auto issue_tile = [&](int n0, int buf) {
    if (n0 + BN <= a.Skv) {   // (wave-uniform)
      k_dma.issue(kb + (int64_t)n0 * k_row_bytes, lds0 + buf * STAGE, wave);
      v_dma.issue(vb + (int64_t)n0 * v_row_bytes, lds0 + buf * STAGE + KTILE, wave);
    } else {
      dma_tile<KROW, 4, DQK / 8>(kb, k_row_bytes, n0, a.Skv, lds0 + buf * STAGE, wave, lane);
      dma_tile<VROW, 4>(vb, v_row_bytes, n0, a.Skv, lds0 + buf * STAGE + KTILE, wave, lane);
    }
    if constexpr (FAMILY == BF_RETENTION) {
      if (mult_ok && n0 + BN <= a.Skv && m_wave < a.Sq)
        mult_dma<T>((const T*)a.smask + (int64_t)b * a.sm_sb + (int64_t)h * a.sm_sh + (int64_t)m_wave * a.sm_sq + n0, a.sm_sq, a.Sq - m_wave,
                    lds0 + MULT + (buf * 4 + wave) * 2048, lane);
    } else {
      // element-wise keep mask: whole tiles of a 16-byte aligned mask come with the K/V tile (same area, 1 KB per wave and
      // stage); a tile the block mask marks as kept in full (entry 2) needs none of it
      if (keep_ok && n0 + BN <= a.Skv && m_wave < a.Sq && !tile_full(n0 / BN))
        keep_dma(elem_mask + (int64_t)b * a.em_sb + (int64_t)h * a.em_sh + (int64_t)m_wave * a.em_sq + n0, a.em_sq, a.Sq - m_wave,
                 lds0 + MULT + (buf * 4 + wave) * 1024, lane);
    }
  };

  f32x16 dq[QB];
#pragma unroll
  for (int i = 0; i < QB; i++)
#pragma unroll
    for (int j = 0; j < 16; j++) dq[i][j] = 0.f;
  const float bias = a.bias + (a.bias_ptr ? *a.bias_ptr : 0.f);
  const float c_scale = a.scale * kLog2e, c_bias = bias * kLog2e;
  lse2 = c_bias - lse2;   // what the row function adds to s * c_scale

  // element-wise keep mask of this lane's query row
  const uint8_t* em_row = elem_mask ? elem_mask + (int64_t)b * a.em_sb + (int64_t)h * a.em_sh + (int64_t)m_ld * a.em_sq : nullptr;

  // tiles in which the mask keeps nothing for this workgroup's rows are never fetched
  const uint8_t* bm_row = MASKS && a.kv_block_mask ? a.kv_block_mask + (int64_t)b * a.kbm_sb + (int64_t)h * a.kbm_sh + (int64_t)mb * a.kbm_sq : nullptr;
  auto next_tile = [&](int jt) {
    if (bm_row)
      while (jt < n_tiles && !bm_row[jt]) jt++;
    return jt;
  };

  // (two streams: tile `jt` of the walk is stream 0's, the one behind it, `jt1`, stream 1's; both pass every barrier)
  int jt = next_tile(0), jt1 = KVS > 1 ? next_tile(jt + 1) : 0;
  auto issue_mine = [&](int buf) {
    const int t = stream == 0 ? jt : jt1;
    if (t < n_tiles) issue_tile(t * BN, buf);
  };
  issue_mine(0);
  for (int it = 0; jt < n_tiles; it++) {
    const int buf = it & 1, n0 = (stream == 0 ? jt : jt1) * BN;
    wait_dma();
    __syncthreads();
    jt = next_tile((KVS > 1 ? jt1 : jt) + 1);
    if (KVS > 1) jt1 = next_tile(jt + 1);
    issue_mine(buf ^ 1);
    if (KVS > 1 && n0 >= n_tiles * BN) continue;           // (an odd number of tiles: stream 1 has none left)
    const uint32_t kbase = lds0 + buf * STAGE, vbase = kbase + KTILE;

    // retention: the multipliers of this lane's 16 scores, requested before the products that hide their latency
    typename E::x4 mk[4];
    if constexpr (FAMILY == BF_RETENTION) {
      if (mult_ok && n0 + BN <= a.Skv && m_wave < a.Sq) {
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) mk[q4] = mult_read<T>(lds0 + MULT + (buf * 4 + wave) * 2048, r, g, q4);
      } else {
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) {
          const int n = n0 + 8 * q4 + 4 * g;
          if (n + 3 < a.Skv) {
            mk[q4] = *(const typename E::x4*)(sm_row + n);
          } else {
#pragma unroll
            for (int i = 0; i < 4; i++) mk[q4][i] = n + i < a.Skv ? sm_row[n + i] : (T)0.f;
          }
        }
      }
    }
    f32x16 s = mm_rows<T, DQK>(kbase, r, g, qf);           // S^T: lane = row m_lane, element jj = key n0 + 8(jj/4) + 4g + jj%4
    const f32x16 dp = mm_rows<T, DV>(vbase, r, g, dof);   // dP^T, same layout
    x8 dsf[2];
    float cap_grad[16];
    if constexpr (EXTRA) {
      const float inv_scale = 1.f / a.scale;
      const float sl_q = a.slope_q ? a.slope_q[h] * (float)m_ld : 0.f, sl_kv = a.slope_kv ? a.slope_kv[h] : 0.f;
      const int64_t add_row = (int64_t)b * a.add_sb + (int64_t)h * a.add_sh + (int64_t)m_ld * a.add_sq;
#pragma unroll
      for (int jj = 0; jj < 16; jj++) {
        const int n = min(n0 + 8 * (jj >> 2) + 4 * g + (jj & 3), a.Skv - 1);
        float e = sl_q + sl_kv * (float)n;
        if (a.add) e += a.add_f32 ? ((const float*)a.add)[add_row + (int64_t)n * a.add_sk] : (float)((const T*)a.add)[add_row + (int64_t)n * a.add_sk];
        s[jj] = apply_extra(s[jj], e, a.scale, inv_scale, bias, a.softcap, cap_grad[jj]);
      }
    }
    float mr[16];   // retention: multiplier / r per element
    if constexpr (FAMILY == BF_RETENTION) {
#pragma unroll
      for (int jj = 0; jj < 16; jj++) mr[jj] = (float)mk[jj >> 2][jj & 3] * r_inv;
    }
    // only tiles that touch the diagonal or the end of the keys pay for the mask (the test is wave-uniform);
    // with an element-wise mask every tile does
    const bool full = tile_full(n0 / BN);
    if ((CAUSAL && n0 + BN - 1 > m_wave) || n0 + BN > a.Skv || (em_row && !full)) {
      uint32_t keep[4] = {0x01010101u, 0x01010101u, 0x01010101u, 0x01010101u};   // the bytes of this lane's four keys per group
      if (full) {
      } else if (keep_ok && n0 + BN <= a.Skv && m_wave < a.Sq) {
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) keep[q4] = keep_read(lds0 + MULT + (buf * 4 + wave) * 1024, r, g, q4);
      } else if (em_row) {
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) {
          const int n = n0 + 8 * q4 + 4 * g;
          if (n + 3 < a.Skv) {
            keep[q4] = *(const uint32_t*)(em_row + n);
          } else {
            keep[q4] = 0;
#pragma unroll
            for (int i = 0; i < 4; i++)
              if (n + i < a.Skv) keep[q4] |= (uint32_t)em_row[n + i] << (8 * i);
          }
        }
      }
#pragma unroll
      for (int jj = 0; jj < 16; jj++) {
        const int n = n0 + 8 * (jj >> 2) + 4 * g + (jj & 3);
        const bool masked = (CAUSAL && n > m_lane) || n >= a.Skv || ((keep[jj >> 2] >> (8 * (jj & 3))) & 0xffu) == 0;
        float p, ds;
        row_fn_bwd<FAMILY>(s[jj], dp[jj], masked, c_scale, c_bias, a.scale, bias, FAMILY == BF_RETENTION ? mr[jj] : lse2, delta, p, ds);
        if constexpr (EXTRA) ds *= cap_grad[jj];
        dsf[jj >> 3][jj & 7] = (T)ds;
      }
    } else {
#pragma unroll
      for (int jj = 0; jj < 16; jj++) {
        float p, ds;
        row_fn_bwd<FAMILY>(s[jj], dp[jj], false, c_scale, c_bias, a.scale, bias, FAMILY == BF_RETENTION ? mr[jj] : lse2, delta, p, ds);
        if constexpr (EXTRA) ds *= cap_grad[jj];
        dsf[jj >> 3][jj & 7] = (T)ds;
      }
    }
    mm_cols<T, DQK>(kbase, lane, dsf, dq);                 // dQ^T += K^T dS^T
  }
  __syncthreads();   // every wave is done with the tiles: they become output staging

  if constexpr (KVS > 1) {
    // stream 1 hands its sums to stream 0: 16 bytes a lane, lane-major
    const uint32_t at = (uint32_t)(uintptr_t)(MA_LDS char*)smem + wave * (QB * 4096) + lane * 16;
    if (stream == 1) {
#pragma unroll
      for (int i = 0; i < QB; i++)
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++)
          lds_write<f32x4>(at + (i * 4 + q4) * 1024, f32x4{dq[i][4 * q4], dq[i][4 * q4 + 1], dq[i][4 * q4 + 2], dq[i][4 * q4 + 3]});
    }
    __syncthreads();
    if (stream == 1) return;
#pragma unroll
    for (int i = 0; i < QB; i++)
#pragma unroll
      for (int q4 = 0; q4 < 4; q4++) {
        const f32x4 x = lds_read<f32x4>(at + (i * 4 + q4) * 1024);
#pragma unroll
        for (int j = 0; j < 4; j++) dq[i][4 * q4 + j] += x[j];
      }
  }
  // (two streams: a wave stages its output where the sums that only it has read were)
  constexpr int OROW = DQK + 16, OUT = KVS > 1 ? QB * 4096 : 32 * OROW;
  static_assert(KVS == 1 || (OUT >= 32 * OROW && 4 * OUT <= KVS * STREAM_LDS), "LDS of the merged sums and the output staging");
  T* dqb = (T*)a.dq + (int64_t)b * a.dqsb + (int64_t)h * a.dqsh;
  store_rows<T, DQK>(dq, a.scale, lds0 + wave * OUT, dqb, a.dqss, m_wave, a.Sq, lane);
}

// ------------------------------------------------------------------------------------------------
// dk, dv
// ------------------------------------------------------------------------------------------------
// WHAT: 3 = dk and dv in one launch, 1 = dv only, 2 = dk only.  Both [D x 32] accumulators plus the K and V
// fragments take 192 registers at 128/128, which leaves one wave per SIMD (forcing two makes the compiler
// spill the fragments and is slower); computing dv and dk in two launches (the scores are then computed once
// more) lets each run two waves per SIMD.
template <typename T, int DQK, int DV, int FAMILY, bool CAUSAL, int WHAT, bool EXTRA = false>
__global__ __launch_bounds__(256, (WHAT == 3 ? (DQK + DV >= 256 ? 1 : 2) : (DQK + DV >= 512 ? 1 : 2))) void attn_bwd_dkv_kernel(const AttnBwdArgs a) {
  constexpr bool DO_DV = (WHAT & 1) != 0, DO_DK = (WHAT & 2) != 0;
  using E = Elem<T>;
  using x8 = typename E::x8;
  constexpr int BNW = 128, BMT = 32;   // keys per workgroup, query rows per tile
  constexpr int KS = DQK / 16, VS = DV / 16, QB = DQK / 32, VB = DV / 32;
  constexpr int QROW = pad_width(DQK) * 2, DOROW = DV * 2;   // (LDS rows; 192-wide queries sit in 256-wide rows)
  // a stage: the Q tile and the dO tile; behind both stages, lse and delta of each stage's 32 rows (softmax; 2 x 128
  // bytes per stage -- not inside the stages: the swizzled reads address a tile as base XOR offset, which needs the
  // tile bases aligned to the row size)
  constexpr int QTILE = BMT * QROW, DOTILE = BMT * DOROW, STAGE = QTILE + DOTILE, ROWVALS = 2 * STAGE;
  // retention: behind those, a 2 KB block of the transposed multiplier per wave and stage (see the dq kernel)
  constexpr int MULT = ROWVALS + 1024;

  extern __shared__ __align__(16) char smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(MA_LDS char*)smem;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, g = lane >> 5;

  const bool heavy_first = CAUSAL && gridDim.x <= kHeavyFirstMost;   // (as in the dq kernel)
  const int nnb = a.num_blocks, BHK = a.B * a.Hkv;
  int bhk, nb;
  if ((BHK & 7) == 0) {
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    bhk = (heavy_first ? slot % (BHK >> 3) : slot / nnb) * 8 + xcd;
    nb = heavy_first ? slot / (BHK >> 3) : slot % nnb;
  } else {
    bhk = heavy_first ? blockIdx.x % BHK : blockIdx.x / nnb;
    nb = heavy_first ? blockIdx.x / BHK : blockIdx.x % nnb;
  }
  const int b = bhk / a.Hkv, hk = bhk % a.Hkv;
  const int n_wave = nb * BNW + wave * 32, n_lane = n_wave + r;
  const int n_ld = min(n_lane, a.Skv - 1);

  // B operands of this wave's 32 keys: K (for S = Q K^T) and V (for dP = dO V^T)
  x8 kf[KS], vf[VS];
  {
    const T* kp = (const T*)a.k + (int64_t)b * a.ksb + (int64_t)n_ld * a.kss + (int64_t)hk * a.ksh + 8 * g;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) kf[ks] = *(const x8*)(kp + 16 * ks);
    const T* vp = (const T*)a.v + (int64_t)b * a.vsb + (int64_t)n_ld * a.vss + (int64_t)hk * a.vsh + 8 * g;
#pragma unroll
    for (int sl = 0; sl < VS; sl++) vf[sl] = *(const x8*)(vp + 16 * sl);
  }
  f32x16 dk[QB], dv[VB];
#pragma unroll
  for (int i = 0; i < QB; i++)
#pragma unroll
    for (int j = 0; j < 16; j++) dk[i][j] = 0.f;
#pragma unroll
  for (int i = 0; i < VB; i++)
#pragma unroll
    for (int j = 0; j < 16; j++) dv[i][j] = 0.f;
  const float bias = a.bias + (a.bias_ptr ? *a.bias_ptr : 0.f);
  const float c_scale = a.scale * kLog2e, c_bias = bias * kLog2e;

  // query tiles that can see this workgroup's keys, for every query head of the kv head's group
  const int t_first = CAUSAL ? (nb * BNW) / BMT : 0;
  const int t_count = (a.Sq + BMT - 1) / BMT - t_first;
  const int n_steps = t_count > 0 ? t_count * a.kv_group : 0;
  const int64_t q_row_bytes = a.qss * 2, do_row_bytes = a.doss * 2;
  // tiles in which the mask keeps nothing for this workgroup's keys are never fetched
  const uint8_t* qbm = a.q_block_mask ? a.q_block_mask + (int64_t)b * a.qbm_sb + (int64_t)nb * a.qbm_sk : nullptr;
  // (entry 2: the element-wise mask keeps every score of the tile)
  // a step = (query head of the group, tile of that head's rows), counted without divisions
  struct Pos { int step, hg, t; };
  auto advance = [&](Pos& p) {
    p.step++;
    if (++p.t == t_count) { p.t = 0; p.hg++; }
  };
  auto qbm_at = [&](const Pos& p) { return qbm[(int64_t)(hk * a.kv_group + p.hg) * a.qbm_sh + t_first + p.t]; };
  auto step_full = [&](const Pos& p) { return qbm && qbm_at(p) >= 2; };
  auto skip_empty = [&](Pos& p) {
    if (qbm)
      while (p.step < n_steps && !qbm_at(p)) advance(p);
  };
  const bool keep_ok = FAMILY != BF_RETENTION && a.elem_mask_t && ((a.emt_sk | a.emt_sb | a.emt_sh | (int64_t)(uintptr_t)a.elem_mask_t) & 15) == 0;
  const bool mult_ok = FAMILY == BF_RETENTION && (a.smt_sk & 7) == 0 && (a.smt_sb & 7) == 0 && (a.smt_sh & 7) == 0 && ((uintptr_t)a.smask_t & 15) == 0;
  TileDma<QROW, 4, DQK / 8> q_dma;
  TileDma<DOROW, 4> do_dma;
  q_dma.init((uint32_t)q_row_bytes, wave, lane);
  do_dma.init((uint32_t)do_row_bytes, wave, lane);
  auto issue_step = [&](const Pos& step, int buf) {
    const int h = hk * a.kv_group + step.hg, m0 = (t_first + step.t) * BMT;
    const char* qb = (const char*)((const T*)a.q + (int64_t)b * a.qsb + (int64_t)h * a.qsh);
    const char* dob = (const char*)((const T*)a.dout + (int64_t)b * a.dosb + (int64_t)h * a.dosh);
    if (m0 + BMT <= a.Sq) {   // (wave-uniform)
      q_dma.issue(qb + (int64_t)m0 * q_row_bytes, lds0 + buf * STAGE, wave);
      do_dma.issue(dob + (int64_t)m0 * do_row_bytes, lds0 + buf * STAGE + QTILE, wave);
    } else {
      dma_tile<QROW, 4, DQK / 8>(qb, q_row_bytes, m0, a.Sq, lds0 + buf * STAGE, wave, lane);
      dma_tile<DOROW, 4>(dob, do_row_bytes, m0, a.Sq, lds0 + buf * STAGE + QTILE, wave, lane);
    }
    if constexpr (FAMILY == BF_SOFTMAX) {
      // lse (lanes 0..31) and delta (lanes 32..63) of the tile's rows come with it: read from global memory inside
      // the loop, their latency is not covered by the little work a tile is
      // (wave 0 fetches lse, wave 1 delta: a scalar base and the lane's row; the upper lanes repeat the lower ones into
      // the other half of the wave's 256 bytes)
      if (wave < 2) {
        const float* src = (wave == 0 ? a.lse : (const float*)a.delta) + ((int64_t)b * a.H + h) * a.Sq + m0;
        dma4_so(src, (uint32_t)(min(m0 + (lane & 31), a.Sq - 1) - m0) * 4u, lds0 + ROWVALS + buf * 512 + wave * 256);
      }
    }
    if constexpr (FAMILY == BF_RETENTION) {
      // the row scales r of the tile's rows (twice: both halves of the wave fetch them) and, for whole tiles of an
      // aligned tensor, each wave's block of the transposed multiplier
      if (wave == 0)
        dma4_so(a.lse + ((int64_t)b * a.H + h) * a.Sq + m0, (uint32_t)(min(m0 + (lane & 31), a.Sq - 1) - m0) * 4u, lds0 + ROWVALS + buf * 512);
      if (mult_ok && m0 + BMT <= a.Sq && n_wave < a.Skv)
        mult_dma<T>((const T*)a.smask_t + (int64_t)b * a.smt_sb + (int64_t)h * a.smt_sh + (int64_t)n_wave * a.smt_sk + m0, a.smt_sk, a.Skv - n_wave,
                    lds0 + MULT + (buf * 4 + wave) * 2048, lane);
    } else {
      // the transposed element-wise keep mask: whole tiles of a 16-byte aligned mask come with the Q/dO tile
      if (keep_ok && m0 + BMT <= a.Sq && n_wave < a.Skv && !step_full(step))
        keep_dma(a.elem_mask_t + (int64_t)b * a.emt_sb + (int64_t)h * a.emt_sh + (int64_t)n_wave * a.emt_sk + m0, a.emt_sk, a.Skv - n_wave,
                 lds0 + MULT + (buf * 4 + wave) * 1024, lane);
    }
  };

  Pos step_next = {0, 0, 0};
  skip_empty(step_next);
  if (step_next.step < n_steps) issue_step(step_next, 0);
  for (int it = 0; step_next.step < n_steps; it++) {
    const int buf = it & 1;
    const Pos step = step_next;
    const int h = hk * a.kv_group + step.hg, m0 = (t_first + step.t) * BMT;
    wait_dma();
    __syncthreads();
    advance(step_next);
    skip_empty(step_next);
    if (step_next.step < n_steps) issue_step(step_next, buf ^ 1);
    // (a wave whose keys all lie behind this tile's rows has nothing to add; it still takes part in the barriers.  With
    // the large accumulators of the 256 / 512 head size the second way round the loop costs register copies that spill,
    // and the few such tiles are computed instead: every element of them is masked)
    if (CAUSAL && DQK + DV < 768 && m0 + BMT - 1 < n_wave) continue;
    const uint32_t qbase = lds0 + buf * STAGE, dobase = qbase + QTILE;

    // retention: 1 / r of the rows this lane holds and the multipliers of its 16 scores (from the transposed
    // multiplier tensor: this key's row, indexed by query position)
    float lse2[16], dl[16];
    if constexpr (FAMILY == BF_RETENTION) {
      const uint32_t rv = lds0 + ROWVALS + buf * 512;
      const T* smt_row = (const T*)a.smask_t + (int64_t)b * a.smt_sb + (int64_t)h * a.smt_sh + (int64_t)n_ld * a.smt_sk;
      const bool staged = mult_ok && m0 + BMT <= a.Sq && n_wave < a.Skv;
#pragma unroll
      for (int q4 = 0; q4 < 4; q4++) {
        const int m = m0 + 8 * q4 + 4 * g;
        const f32x4 tr = lds_read<f32x4>(rv + (8 * q4 + 4 * g) * 4);
        typename E::x4 tm;
        if (staged) {
          tm = mult_read<T>(lds0 + MULT + (buf * 4 + wave) * 2048, r, g, q4);
        } else {
#pragma unroll
          for (int i = 0; i < 4; i++) tm[i] = smt_row[min(m + i, a.Sq - 1)];
        }
#pragma unroll
        for (int i = 0; i < 4; i++) lse2[4 * q4 + i] = (float)tm[i] * fast_rcp(tr[i]);
      }
    }
    // lse and delta of the rows this lane holds: m0 + 8q4 + 4g + {0..3}
    if constexpr (FAMILY == BF_SOFTMAX) {
      const uint32_t rv = lds0 + ROWVALS + buf * 512;
#pragma unroll
      for (int q4 = 0; q4 < 4; q4++) {
        const f32x4 tl = lds_read<f32x4>(rv + (8 * q4 + 4 * g) * 4);
        const f32x4 td = lds_read<f32x4>(rv + 256 + (8 * q4 + 4 * g) * 4);
#pragma unroll
        for (int i = 0; i < 4; i++) {
          lse2[4 * q4 + i] = c_bias - tl[i] * kLog2e;   // what the row function adds to s * c_scale
          dl[4 * q4 + i] = td[i];
        }
      }
    }
    f32x16 s = mm_rows<T, DQK>(qbase, r, g, kf);           // S: lane = key n_lane, element jj = row m0 + 8(jj/4) + 4g + jj%4
    float cap_grad[16];
    if constexpr (EXTRA) {
      const float inv_scale = 1.f / a.scale;
      const float sl_q = a.slope_q ? a.slope_q[h] : 0.f, sl_kv = a.slope_kv ? a.slope_kv[h] * (float)n_ld : 0.f;
      const int64_t add_col = (int64_t)b * a.add_sb + (int64_t)h * a.add_sh + (int64_t)n_ld * a.add_sk;
#pragma unroll
      for (int jj = 0; jj < 16; jj++) {
        const int m = min(m0 + 8 * (jj >> 2) + 4 * g + (jj & 3), a.Sq - 1);
        float e = sl_q * (float)m + sl_kv;
        if (a.add) e += a.add_f32 ? ((const float*)a.add)[add_col + (int64_t)m * a.add_sq] : (float)((const T*)a.add)[add_col + (int64_t)m * a.add_sq];
        s[jj] = apply_extra(s[jj], e, a.scale, inv_scale, bias, a.softcap, cap_grad[jj]);
      }
    }
    f32x16 dp;
    if constexpr (DO_DK) dp = mm_rows<T, DV>(dobase, r, g, vf);   // dP, same layout
    else
#pragma unroll
      for (int j = 0; j < 16; j++) dp[j] = 0.f;
    x8 pf[2], dsf[2];
    // only tiles that touch the diagonal or an end of the sequences pay for the mask (the test is wave-uniform);
    // with an element-wise mask every tile does
    const bool full = step_full(step);
    if ((CAUSAL && n_wave + 31 > m0) || m0 + BMT > a.Sq || n_wave + 32 > a.Skv || (a.elem_mask_t && !full)) {
      uint32_t keep[4] = {0x01010101u, 0x01010101u, 0x01010101u, 0x01010101u};   // the bytes of this lane's four rows per group
      if (full) {
      } else if (keep_ok && m0 + BMT <= a.Sq && n_wave < a.Skv) {
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) keep[q4] = keep_read(lds0 + MULT + (buf * 4 + wave) * 1024, r, g, q4);
      } else if (a.elem_mask_t) {
        // the transposed mask: this key's row, indexed by query position
        const uint8_t* emt_row = a.elem_mask_t + (int64_t)b * a.emt_sb + (int64_t)h * a.emt_sh + (int64_t)n_ld * a.emt_sk;
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) {
          const int m = m0 + 8 * q4 + 4 * g;
          if (m + 3 < a.Sq) {
            keep[q4] = *(const uint32_t*)(emt_row + m);
          } else {
            keep[q4] = 0;
#pragma unroll
            for (int i = 0; i < 4; i++)
              if (m + i < a.Sq) keep[q4] |= (uint32_t)emt_row[m + i] << (8 * i);
          }
        }
      }
#pragma unroll
      for (int jj = 0; jj < 16; jj++) {
        const int m = m0 + 8 * (jj >> 2) + 4 * g + (jj & 3);
        const bool masked = (CAUSAL && n_lane > m) || m >= a.Sq || n_lane >= a.Skv || ((keep[jj >> 2] >> (8 * (jj & 3))) & 0xffu) == 0;
        float p, ds;
        row_fn_bwd<FAMILY>(s[jj], dp[jj], masked, c_scale, c_bias, a.scale, bias, FAMILY == BF_SOFTMAX || FAMILY == BF_RETENTION ? lse2[jj] : 0.f,
                           FAMILY == BF_SOFTMAX ? dl[jj] : 0.f, p, ds);
        if (masked) ds = 0.f;
        if constexpr (EXTRA) ds *= cap_grad[jj];
        pf[jj >> 3][jj & 7] = (T)p;
        dsf[jj >> 3][jj & 7] = (T)ds;
      }
    } else {
#pragma unroll
      for (int jj = 0; jj < 16; jj++) {
        float p, ds;
        row_fn_bwd<FAMILY>(s[jj], dp[jj], false, c_scale, c_bias, a.scale, bias, FAMILY == BF_SOFTMAX || FAMILY == BF_RETENTION ? lse2[jj] : 0.f,
                           FAMILY == BF_SOFTMAX ? dl[jj] : 0.f, p, ds);
        if constexpr (EXTRA) ds *= cap_grad[jj];
        pf[jj >> 3][jj & 7] = (T)p;
        dsf[jj >> 3][jj & 7] = (T)ds;
      }
    }
    if constexpr (DO_DV) mm_cols<T, DV>(dobase, lane, pf, dv);     // dV^T += dO^T P
    if constexpr (DO_DK) mm_cols<T, DQK>(qbase, lane, dsf, dk);    // dK^T += Q^T dS
  }
  __syncthreads();   // every wave is done with the tiles: they become output staging

  constexpr int DMAX = DQK > DV ? DQK : DV, OROW = DMAX + 16;
  const uint32_t stage = lds0 + wave * 32 * OROW;
  T* dkb = (T*)a.dk + (int64_t)b * a.dksb + (int64_t)hk * a.dksh;
  T* dvb = (T*)a.dv + (int64_t)b * a.dvsb + (int64_t)hk * a.dvsh;
  if constexpr (DO_DK) store_rows<T, DQK>(dk, a.scale, stage, dkb, a.dkss, n_wave, a.Skv, lane);
  if constexpr (DO_DV) store_rows<T, DV>(dv, 1.f, stage, dvb, a.dvss, n_wave, a.Skv, lane);
}


// ------------------------------------------------------------------------------------------------
// dk and dv in one launch at 64 / 64, software pipelined inside the wave
// ------------------------------------------------------------------------------------------------
// Few key blocks (short sequences, one or two sequences with grouped-query heads) leave CUs idle: the steps of every key block
// are then dealt to n_parts runs, taken by workgroups side by side (attn_bwd_parts chooses): tile t of the group's head hg
// goes to run (t + hg) % n_parts.  (By the tile's place in the sequence, so that a mask's runs hold what a causal call's hold
// and the sums come out the same, whatever tiles a mask leaves in the list.)
// The tiles of a run in order: tile t (from the first that sees the key block) of head hg; skip: the head's first tile of the run.
struct DkvWalk {
  int hg, t, skip;
  template <bool PARTS>
  __device__ __forceinline__ void next(int n_parts, int t_count, int kv_group) {
    if constexpr (PARTS) to_tile(t + n_parts, n_parts, t_count, kv_group);
    else if (++t == t_count) { t = 0; hg++; }
  }
  __device__ __forceinline__ void to_tile(int tile, int n_parts, int t_count, int kv_group) {
    t = tile;
    while (t >= t_count && hg < kv_group) {
      hg++;
      skip = skip == 0 ? n_parts - 1 : skip - 1;
      t = skip;
    }
  }
};
// the fp32 partial sums of (run, batch and kv head, key block): [wave][column block of dk, then of dv][q4][lane] x 4 elements
template <int DQK, int DV>
__device__ __forceinline__ float* dkv_partial(const AttnBwdArgs& a, int run, int bhk, int nb) {
  return a.dkv_part + (((int64_t)run * a.B * a.Hkv + bhk) * a.num_blocks + nb) * (128 * (DQK + DV));
}
template <int N>
__device__ __forceinline__ void partial_store(float* to, const f32x16 (&acc)[N]) {
#pragma unroll
  for (int i = 0; i < N; i++)
#pragma unroll
    for (int q4 = 0; q4 < 4; q4++)
      *(f32x4*)(to + (i * 4 + q4) * 256) = f32x4{acc[i][4 * q4], acc[i][4 * q4 + 1], acc[i][4 * q4 + 2], acc[i][4 * q4 + 3]};
}

// At 64 / 64 the K and V fragments and both [D x 32] accumulators of a wave's 32 keys fit the registers of one wave of two on a
// SIMD, and dk and dv share the recomputed scores (7 tile products in all instead of 8).  The loop is pipelined inside the wave.  A
// step is ONE sequence of MFMAs:
//   phase F  S(u+1) = Q(u+1) K^T and dP(u+1) = dO(u+1) V^T of the NEXT tile, with p of the current step's 16 score elements
//            spread behind them,
//   phase V  dV^T += dO(u)^T P(u), with ds of the 16 elements behind them,
//   phase K  dK^T += Q(u)^T dS(u),
// whose LDS operand fragments travel through one ring of registers, requested AH MFMAs ahead across the phases and across
// steps (the last MFMAs of phase K request the first fragments of the next step).  Tiles come through a ring of stages, LA
// steps ahead; the step's single barrier sits between phases V and K: behind it tile u+2 is visible to every wave, and
// every wave is done with tile u-1, whose stage takes tile u+LA.  lse and delta of a tile's rows come with it.  The loop
// body is written for two steps (the registers of "this" and "the next" step swap roles) so that nothing is copied; an odd
// number of steps is padded with a step in which everything is masked.  Masked scores are set to -inf and their dp to
// 0 before the row function, in the few tiles that touch the diagonal or an end of the sequences: p = 0 and so ds = 0 follow.
// Larger head sizes take the pair kernel below; the retention family, 256 / 512, additive score terms and
// masks with more steps than the list holds the kernels above.
template <int I>
struct IntC { static constexpr int value = I; };
template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {   // f(IntC<I>()), ..., f(IntC<N - 1>()): indices that are constants by construction
  if constexpr (I < N) {
    f(IntC<I>());
    static_for<I + 1, N>(f);
  }
}

template <typename T>
struct FusedStepRegs {
  f32x16 s, dp;        // S and dP of the step's tile (lane = key, element jj = row 8(jj/4) + 4g + jj%4 of the tile)
  f32x4 tl[4], td[4];  // lse and delta of those rows (softmax)
};

// MASKS: with an element-wise keep mask (its transpose: a lane walks a key's column) and / or a tile mask.  The steps of a
// key block are then a list in LDS, built by wave 0 before the loop: the (query head, tile) pairs whose tile-mask entry is
// not 0, each with the flag "kept in full" (entry 2: the element mask is not consulted).  A wave's [32 x 32] block of mask
// bytes comes with the tile (whole tiles of a 16-byte aligned mask; others are read from global memory), and the
// masked scores are set to -inf in the same place as for the structural masks.
constexpr int FUSED_LIST_MAX = 2048;   // steps of a key block that the list holds (the launcher checks)
// STREAMS 2 (64 / 64, see dkv_two_streams): two streams of four waves walk every other tile of the workgroup's steps each, with
// stages of their own, as two runs would; at the end one keeps dk and the other dv, and each hands the other one over through LDS.
// PARTS: n_parts > 1 (an instantiation of its own: the walk over a run's tiles costs the one-run loop 3 % at 64 / 64).
template <typename T, int DQK, int DV, int FAMILY, bool CAUSAL, bool MASKS, bool PARTS, int STREAMS = 1>
__global__ __launch_bounds__(256 * STREAMS, FUSED_PER_CU) void attn_bwd_dkv_fused_kernel(const AttnBwdArgs a) {
  using E = Elem<T>;
  using x8 = typename E::x8;
  using x4 = typename E::x4;
  constexpr int BNW = 128, BMT = 32;
  constexpr int KS = DQK / 16, VS = DV / 16, QB = DQK / 32, VB = DV / 32;
  constexpr int QROW = DQK * 2, DOROW = DV * 2;
  // a stage: the Q tile and the dO tile; behind the stages, 512 bytes per stage: lse (first 128) and delta (at 256) of its rows
  constexpr int QTILE = BMT * QROW, DOTILE = BMT * DOROW, STAGE = QTILE + DOTILE;
  constexpr int NST = fused_stages(MASKS), LA = NST == 8 ? 4 : 3, ROWVALS = NST * STAGE;
  // (MASKS) behind the row values: 1 KB of mask bytes per stage and wave, then the step list and its length
  constexpr int KEEP = ROWVALS + NST * 512, LIST = KEEP + NST * 4 * 1024, LIST_N = LIST + FUSED_LIST_MAX * 4;
  constexpr int STREAM_LDS = (MASKS ? LIST_N + 4 : ROWVALS + NST * 512) + 1023 & ~1023;
  // the MFMAs of a step and the fragment ring
  constexpr int NF = KS + VS, NV = 2 * VB, NK = 2 * QB, NTOT = NF + NV + NK;
  constexpr int RING = 8, AH = FAMILY == BF_SOFTMAX ? 2 : (NK < 6 ? NK : 6);
  static_assert(NTOT % RING == 0 && AH < RING && AH <= NK && AH <= NF, "fragment ring");
  // phase F alternates the k slices of S and dP: MFMA j is slice j / 2 of S (j even) or of dP
  static_assert(DQK == DV, "phase F");

  extern __shared__ __align__(16) char smem[];
  constexpr bool WALK = PARTS || STREAMS > 1;
  static_assert(STREAMS == 2 || (STREAMS == 1 && !PARTS), "two streams share a SIMD; runs are theirs");
  const int tid = threadIdx.x, lane = tid & 63, wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int stream = STREAMS > 1 ? wave_all >> 2 : 0, wave = STREAMS > 1 ? wave_all & 3 : wave_all;   // wave: within its stream
  const uint32_t lds_all = (uint32_t)(uintptr_t)(MA_LDS char*)smem, lds0 = lds_all + (STREAMS > 1 ? stream * (uint32_t)STREAM_LDS : 0u);
  const int r = lane & 31, g = lane >> 5;

  // STREAMS 2: an item, a workgroup of its own, is one key block (or a run of it).
  // STREAMS 1 is persistent: the grid is one workgroup per CU, and every workgroup walks items  item = blockIdx.x, + gridDim.x, ...  An
  // item is a (batch, kv head) and, under a causal mask, the PAIR of key blocks (k, n - 1 - k), which together see the
  // same number of query tiles whatever k is: every item weighs the same.  Items that follow each other on an XCD
  // (item % 8) belong to the same (batch, kv head) pairs, whose Q and dO tiles then come from that XCD's L2.
  const int nnb = a.num_blocks, BHK = a.B * a.Hkv, n_parts = PARTS ? a.n_parts : 1;
  // With n_parts > 1 (two streams) an item is one of the n_parts runs of each block's steps, whose fp32 sums go to the workspace
  // (attn_bwd_dkv_reduce_kernel adds the runs up).
  const int per_bh = (CAUSAL && STREAMS == 1 ? (nnb + 1) / 2 : nnb) * n_parts, n_items = BHK * per_bh;
  for (int item = blockIdx.x; item < n_items; item += gridDim.x) {
  int bhk, ki, run;
  if (STREAMS > 1) {
    // the heaviest blocks of all heads first
    const int xcds = (BHK & 7) == 0 ? 8 : 1, slot = item / xcds, heads = BHK / xcds;
    run = slot % n_parts;
    bhk = (slot / n_parts) % heads * xcds + item % xcds;
    ki = slot / (n_parts * heads);
  } else if ((BHK & 7) == 0) {
    const int slot = item >> 3;
    bhk = (slot / per_bh) * 8 + (item & 7);
    ki = slot % per_bh;
    run = ki % n_parts;
    ki /= n_parts;
    // (without the causal pairing a key block's work depends on the mask: a workgroup, whose items are a whole number of
    // (batch, kv head) pairs apart, takes another key block each time round instead of the same one)
    if (!CAUSAL) ki = (ki + slot / per_bh) % nnb;
  } else {
    bhk = item / per_bh;
    ki = item % per_bh;
    run = ki % n_parts;
    ki /= n_parts;
    if (!CAUSAL) ki = (ki + bhk) % nnb;
  }
  const int b = bhk / a.Hkv, hk = bhk % a.Hkv;
  for (int part = 0; part < (STREAMS == 1 && CAUSAL && ki != nnb - 1 - ki ? 2 : 1); part++) {
  const int nb = part == 0 ? ki : nnb - 1 - ki;
  const int n_wave = nb * BNW + wave * 32, n_lane = n_wave + r;
  const int n_ld = min(n_lane, a.Skv - 1);

  x8 kf[KS], vf[VS];
  {
    const T* kp = (const T*)a.k + (int64_t)b * a.ksb + (int64_t)n_ld * a.kss + (int64_t)hk * a.ksh + 8 * g;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) kf[ks] = *(const x8*)(kp + 16 * ks);
    const T* vp = (const T*)a.v + (int64_t)b * a.vsb + (int64_t)n_ld * a.vss + (int64_t)hk * a.vsh + 8 * g;
#pragma unroll
    for (int sl = 0; sl < VS; sl++) vf[sl] = *(const x8*)(vp + 16 * sl);
  }
  f32x16 dk[QB], dv[VB];
#pragma unroll
  for (int i = 0; i < QB; i++)
#pragma unroll
    for (int j = 0; j < 16; j++) dk[i][j] = 0.f;
#pragma unroll
  for (int i = 0; i < VB; i++)
#pragma unroll
    for (int j = 0; j < 16; j++) dv[i][j] = 0.f;
  const float bias = a.bias + (a.bias_ptr ? *a.bias_ptr : 0.f);
  const float c_scale = a.scale * kLog2e, c_bias = bias * kLog2e;
  const float s_masked = -__builtin_inff();   // a score whose p is 0 (scale > 0)

  // steps: for every query head of the kv head's group, the 32-row tiles that can see this workgroup's keys
  const int t_first = CAUSAL ? (nb * BNW) / BMT : 0;
  const int t_count = (a.Sq + BMT - 1) / BMT - t_first;
  int n_steps = t_count > 0 ? t_count * a.kv_group : 0;
  DkvWalk first{0, 0, 0};
  // (the streams of a workgroup are runs side by side, whose sums meet in LDS)
  const int n_runs = n_parts * STREAMS;
  int n_bodies = 0;      // (STREAMS > 1) steps of the longer stream: the barriers are everybody's
  if (WALK && !MASKS && n_steps > 0) {
    const int each = t_count / n_runs, more = t_count % n_runs;
    auto steps_of = [&](int skip) {
      int n = 0;
      for (int hg = 0; hg < a.kv_group; hg++, skip = skip == 0 ? n_runs - 1 : skip - 1) n += each + (skip < more ? 1 : 0);
      return n;
    };
    const int mine = run * STREAMS + stream;
    auto skip_of = [&](int any_run) { return ((any_run - t_first) % n_runs + n_runs) % n_runs; };
    first.skip = skip_of(mine);
    n_steps = steps_of(first.skip);
    if (STREAMS > 1) n_bodies = max(n_steps, steps_of(skip_of(mine ^ 1)));
    first.to_tile(first.skip, n_runs, t_count, a.kv_group);
  }
  if (STREAMS == 1) n_bodies = n_steps;
  const bool keep_ok = MASKS && a.elem_mask_t && ((a.emt_sk | a.emt_sb | a.emt_sh | (int64_t)(uintptr_t)a.elem_mask_t) & 15) == 0;
  if constexpr (MASKS) {
    // the step list: entry = tile | head of the group << 16 | kept in full << 31
    const uint8_t* qbm = a.q_block_mask ? a.q_block_mask + (int64_t)b * a.qbm_sb + (int64_t)nb * a.qbm_sk : nullptr;
    if (wave == 0) {
      int count = 0;
      for (int i0 = 0; i0 < n_steps; i0 += 64) {
        const int i = i0 + lane;
        bool keep = false;
        uint32_t entry = 0;
        if (i < n_steps) {
          const int hg = i / t_count, t = i - hg * t_count;
          const uint8_t e = qbm ? qbm[(int64_t)(hk * a.kv_group + hg) * a.qbm_sh + t_first + t] : (uint8_t)1;
          keep = e != 0 && (!WALK || (t_first + t + hg) % n_runs == run * STREAMS + stream);
          entry = (uint32_t)t | ((uint32_t)hg << 16) | (e >= 2 || !a.elem_mask_t ? 0x80000000u : 0u);
        }
        const uint64_t votes = __ballot(keep);
        if (keep) lds_write<uint32_t>(lds0 + LIST + 4 * (count + __popcll(votes & ((1ull << lane) - 1ull))), entry);
        count += __popcll(votes);
      }
      if (lane == 0) lds_write<uint32_t>(lds0 + LIST_N, (uint32_t)count);
    }
    __syncthreads();
    n_steps = __builtin_amdgcn_readfirstlane((int)lds_read<uint32_t>(lds0 + LIST_N));
    n_bodies = n_steps;
    if (STREAMS > 1) n_bodies = max(n_steps, __builtin_amdgcn_readfirstlane((int)lds_read<uint32_t>(lds_all + (stream ^ 1) * (uint32_t)STREAM_LDS + LIST_N)));
  }
  // (list entries are requested a step before they are used and made wave-uniform only then: a read that is waited for
  // at once would drain the ring of operand fragments)
  auto list_request = [&](int i) { return lds_read<uint32_t>(lds0 + LIST + 4 * (i < n_steps ? i : 0)); };
  auto uniform = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
  const int64_t q_row_bytes = a.qss * 2, do_row_bytes = a.doss * 2;
  TileDma<QROW, 4> q_dma;
  TileDma<DOROW, 4> do_dma;
  q_dma.init((uint32_t)q_row_bytes, wave, lane);
  do_dma.init((uint32_t)do_row_bytes, wave, lane);
  // what a wave issues per tile at least
  constexpr int TILE_DMAS = TileDma<QROW, 4>::NJ + TileDma<DOROW, 4>::NJ;
  auto issue_tile = [&](int hg, int t, int st, bool full = true) {
    const int h = hk * a.kv_group + hg, m0 = (t_first + t) * BMT;
    if constexpr (MASKS) {
      // the transposed element-wise keep mask: whole tiles of a 16-byte aligned mask come with the Q / dO tile
      if (keep_ok && !full && m0 + BMT <= a.Sq && n_wave < a.Skv)
        keep_dma(a.elem_mask_t + (int64_t)b * a.emt_sb + (int64_t)h * a.emt_sh + (int64_t)n_wave * a.emt_sk + m0, a.emt_sk, a.Skv - n_wave,
                 lds0 + KEEP + (st * 4 + wave) * 1024, lane);
    }
    const char* qb = (const char*)((const T*)a.q + (int64_t)b * a.qsb + (int64_t)h * a.qsh);
    const char* dob = (const char*)((const T*)a.dout + (int64_t)b * a.dosb + (int64_t)h * a.dosh);
    if (m0 + BMT <= a.Sq) {   // (wave-uniform)
      q_dma.issue(qb + (int64_t)m0 * q_row_bytes, lds0 + st * STAGE, wave);
      do_dma.issue(dob + (int64_t)m0 * do_row_bytes, lds0 + st * STAGE + QTILE, wave);
    } else {
      dma_tile<QROW, 4>(qb, q_row_bytes, m0, a.Sq, lds0 + st * STAGE, wave, lane);
      dma_tile<DOROW, 4>(dob, do_row_bytes, m0, a.Sq, lds0 + st * STAGE + QTILE, wave, lane);
    }
    if constexpr (FAMILY == BF_SOFTMAX) {
      if (wave < 2) {   // wave 0 fetches lse, wave 1 delta (the upper lanes repeat the lower ones)
        const float* src = (wave == 0 ? a.lse : (const float*)a.delta) + ((int64_t)b * a.H + h) * a.Sq + m0;
        dma4_so(src, (uint32_t)(min(m0 + (lane & 31), a.Sq - 1) - m0) * 4u, lds0 + ROWVALS + st * 512 + wave * 256);
      }
    }
  };
  auto row_lse = [&](int st, FusedStepRegs<T>& x) {
    if constexpr (FAMILY == BF_SOFTMAX)
#pragma unroll
      for (int q4 = 0; q4 < 4; q4++) x.tl[q4] = lds_read<f32x4>(lds0 + ROWVALS + st * 512 + (8 * q4 + 4 * g) * 4);
  };
  auto row_delta = [&](int st, FusedStepRegs<T>& x) {
    if constexpr (FAMILY == BF_SOFTMAX)
#pragma unroll
      for (int q4 = 0; q4 < 4; q4++) x.td[q4] = lds_read<f32x4>(lds0 + ROWVALS + st * 512 + 256 + (8 * q4 + 4 * g) * 4);
  };
  // the lane's part of the fragment addresses, relative to a tile: row reads (A operands of S and dP) and
  // transposing reads (A operands of dV^T and dK^T: the tile's columns)
  const uint32_t aq_l = (uint32_t)(r * QROW) + (uint32_t)((g ^ swz_tile<QROW / 16>(r)) << 4);
  const uint32_t ad_l = (uint32_t)(r * DOROW) + (uint32_t)((g ^ swz_tile<DV / 8>(r)) << 4);
  const int jr = (lane & 15) >> 2, lc = (((lane >> 4) & 1) << 1) | ((lane & 3) >> 1);
  const uint32_t bq_l = (uint32_t)((4 * g + jr) * QROW + (lane & 1) * 8) + (uint32_t)((lc ^ swz_tile<QROW / 16>(4 * g + jr)) << 4);
  const uint32_t bd_l = (uint32_t)((4 * g + jr) * DOROW + (lane & 1) * 8) + (uint32_t)((lc ^ swz_tile<DV / 8>(4 * g + jr)) << 4);
  // the fragment of MFMA j of a step whose current tile sits at `cur` and whose next tile at `nxt` (LDS addresses)
  auto fragment = [&](auto jc, uint32_t cur, uint32_t nxt) __attribute__((always_inline)) -> x8 {
    constexpr int j = decltype(jc)::value;
    // (consecutive MFMAs go to different accumulators: with one wave on the SIMD a dependent MFMA waits for the result
    // of the one before it.  Phase F alternates S and dP; phases V and K walk the column blocks before the k slices)
    if constexpr (j < NF && j % 2 == 0) {
      return lds_read<x8>((nxt + aq_l) ^ (uint32_t)(j / 2 * 32));
    } else if constexpr (j < NF) {
      return lds_read<x8>((nxt + QTILE + ad_l) ^ (uint32_t)(j / 2 * 32));
    } else {
      constexpr bool is_v = j < NF + NV;
      constexpr int idx = is_v ? j - NF : j - NF - NV, db = idx % (is_v ? VB : QB), sl = idx / (is_v ? VB : QB);
      constexpr int rowb = is_v ? DOROW : QROW;
      const uint32_t b0 = is_v ? cur + QTILE + bd_l : cur + bq_l;
      const x4 lo = lds_read_tr4<T>((b0 ^ (uint32_t)((4 * db) << 4)) + 16 * sl * rowb);
      const x4 hi = lds_read_tr4<T>((b0 ^ (uint32_t)(((4 * db) ^ 2) << 4)) + (16 * sl + 8) * rowb);
      return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
  };

  if (n_bodies > 0) {
    // the next tile to fetch
    DkvWalk fetch = first, at = first;   // (without MASKS) the next tile to fetch, the current step's
    int i_n = 0;
    uint32_t i_next = MASKS ? list_request(0) : 0u;   // (MASKS) the list entry of the next tile to fetch
    auto issue_next = [&]() {
      if constexpr (MASKS) {
        const uint32_t e = uniform(i_next);
        issue_tile((int)((e >> 16) & 0x7fffu), (int)(e & 0xffffu), i_n & (NST - 1), (e >> 31) != 0);
        i_n++;
        i_next = list_request(i_n);
      } else {
        issue_tile(fetch.hg, fetch.t, i_n & (NST - 1));
        i_n++;
        fetch.template next<WALK>(n_runs, t_count, a.kv_group);
      }
    };
#pragma unroll
    for (int i = 0; i < LA; i++)
      if (i_n < n_steps) issue_next();
    // (the padding step of an odd number of steps evaluates S, dP, lse and delta of the stage behind the last tile's:
    // where no earlier tile has been there, the first one goes there, so that what it computes is 0 unless a tile that this key block
    // sees is not finite)
    if ((n_steps & 1) && n_steps < NST) {
      if constexpr (MASKS) {
        const uint32_t e = uniform(list_request(0));
        issue_tile((int)((e >> 16) & 0x7fffu), (int)(e & 0xffffu), n_steps);
      } else {
        issue_tile(first.hg, first.t, n_steps);
      }
    }
    wait_dma();
    __syncthreads();
    FusedStepRegs<T> ra, rb;
    ra.s = mm_rows<T, DQK>(lds0, r, g, kf);
    ra.dp = mm_rows<T, DV>(lds0 + QTILE, r, g, vf);
    x8 fr[RING];
    static_for<0, AH>([&](auto jc) __attribute__((always_inline)) { fr[decltype(jc)::value] = fragment(jc, lds0, lds0 + STAGE); });   // (of step 0)
    const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

    uint32_t c_next = MASKS ? list_request(0) : 0u;   // (MASKS) the list entry of the step about to begin, requested a step ahead
    auto body = [&](int u, FusedStepRegs<T>& cur, FusedStepRegs<T>& nxt) __attribute__((always_inline)) {
      const bool real = u < n_steps;                 // (the padding step: the last tile once more, everything masked)
      const uint32_t c_entry = MASKS ? uniform(c_next) : 0u;
      if constexpr (MASKS) c_next = list_request(u + 1);
      const uint32_t cur_tile = lds0 + (uint32_t)(((real ? u : n_steps - 1) & (NST - 1)) * STAGE);
      const uint32_t nxt_tile = lds0 + (uint32_t)(((u + 1) & (NST - 1)) * STAGE);
      const uint32_t nn_tile = lds0 + (uint32_t)(((u + 2) & (NST - 1)) * STAGE);
      const int m0 = real ? (t_first + (MASKS ? (int)(c_entry & 0xffffu) : at.t)) * BMT : a.Sq;
      if (!MASKS) at.template next<WALK>(n_runs, t_count, a.kv_group);
      row_lse(u & (NST - 1), cur);      // (row values are requested in the step that uses them: 32 registers less, with a second wave on the SIMD)
      // the tiles that touch the diagonal, an end of the sequences or an element-wise mask (the test is wave-uniform)
      const bool by_elem = MASKS && real && a.elem_mask_t && (c_entry >> 31) == 0;
      if ((CAUSAL && n_wave + 31 > m0) || m0 + BMT > a.Sq || n_wave + 32 > a.Skv || by_elem) {
        // (m0 through an empty asm statement: the compiler would otherwise evaluate the 32 compares in every step, ahead
        // of the branch, and turn the assignments into selects)
        int m0e = m0;
        asm volatile("; a tile that touches a mask" : "+s"(m0e));
        uint32_t keep[4] = {0x01010101u, 0x01010101u, 0x01010101u, 0x01010101u};   // the bytes of this lane's four rows per group
        if constexpr (MASKS) {
          if (by_elem) {
            if (keep_ok && m0e + BMT <= a.Sq && n_wave < a.Skv) {
#pragma unroll
              for (int q4 = 0; q4 < 4; q4++) keep[q4] = keep_read(lds0 + KEEP + ((u & (NST - 1)) * 4 + wave) * 1024, r, g, q4);
            } else {
              // this key's row of the transposed mask, indexed by query position
              const int h = hk * a.kv_group + (int)((c_entry >> 16) & 0x7fffu);
              const uint8_t* emt_row = a.elem_mask_t + (int64_t)b * a.emt_sb + (int64_t)h * a.emt_sh + (int64_t)n_ld * a.emt_sk;
#pragma unroll
              for (int q4 = 0; q4 < 4; q4++) {
                const int m = m0e + 8 * q4 + 4 * g;
                keep[q4] = 0;
#pragma unroll
                for (int i = 0; i < 4; i++)
                  if (m + i < a.Sq) keep[q4] |= (uint32_t)emt_row[m + i] << (8 * i);
              }
            }
          }
        }
#pragma unroll
        for (int jj = 0; jj < 16; jj++) {
          const int m = m0e + 8 * (jj >> 2) + 4 * g + (jj & 3);
          if ((CAUSAL && n_lane > m) || m >= a.Sq || n_lane >= a.Skv || (MASKS && ((keep[jj >> 2] >> (8 * (jj & 3))) & 0xffu) == 0)) {
            cur.s[jj] = s_masked;
            cur.dp[jj] = 0.f;      // (p = 0 times a hidden key's row of V that is not finite is not 0)
            // (a row without any kept key has lse = -inf: its masked scores must still give p = 0)
            if constexpr (FAMILY == BF_SOFTMAX) cur.tl[jj >> 2][jj & 3] = 0.f;
          }
        }
      }
      x8 pf[2], dsf[2];
      float p32[16];
      static_for<0, NTOT>([&](auto jc) __attribute__((always_inline)) {
        constexpr int j = decltype(jc)::value;
        if constexpr (j == NF + NV) {
          // tile u + 2 has landed (what may still be in flight: the tiles behind it) and every wave is done with
          // tile u - 1, whose stage takes tile u + LA
          if (LA > 3 && u + LA - 1 < n_steps) wait_dma_but<(LA - 3) * TILE_DMAS>();
          else wait_dma();
          asm volatile("" ::: "memory");
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
          if (i_n < n_steps) issue_next();
        }
        if constexpr (j == NF - 2) row_delta(u & (NST - 1), cur);
        // the fragment of the MFMA AH places on (the last ones of the step: of the next step's first MFMAs)
        if constexpr (j + AH < NTOT) fr[(j + AH) % RING] = fragment(IntC<j + AH>(), cur_tile, nxt_tile);
        else fr[(j + AH) % RING] = fragment(IntC<j + AH - NTOT>(), nxt_tile, nn_tile);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (j < NF && j % 2 == 0) nxt.s = E::mfma32(fr[j % RING], kf[j / 2], j == 0 ? zero16 : nxt.s);
        else if constexpr (j < NF) nxt.dp = E::mfma32(fr[j % RING], vf[j / 2], j == 1 ? zero16 : nxt.dp);
        else if constexpr (j < NF + NV) dv[(j - NF) % VB] = E::mfma32(fr[j % RING], pf[(j - NF) / VB], dv[(j - NF) % VB]);
        else dk[(j - NF - NV) % QB] = E::mfma32(fr[j % RING], dsf[(j - NF - NV) / QB], dk[(j - NF - NV) % QB]);
        // vector work behind the MFMA: p of the step's 16 elements in phase F, ds in phase V
        if constexpr (j < NF) {
#pragma unroll
          for (int jj = j * 16 / NF; jj < (j + 1) * 16 / NF; jj++) {
            p32[jj] = row_p<FAMILY>(cur.s[jj], c_scale, c_bias, a.scale, bias, FAMILY == BF_SOFTMAX ? fmaf(cur.tl[jj >> 2][jj & 3], -kLog2e, c_bias) : 0.f);
            pf[jj >> 3][jj & 7] = (T)p32[jj];
          }
        } else if constexpr (j < NF + NV) {
#pragma unroll
          for (int jj = (j - NF) * 16 / NV; jj < (j - NF + 1) * 16 / NV; jj++)
            dsf[jj >> 3][jj & 7] = (T)row_ds<FAMILY>(p32[jj], cur.dp[jj], FAMILY == BF_SOFTMAX ? cur.td[jj >> 2][jj & 3] : 0.f);
          // (evaluated here, behind this MFMA: left alone the compiler moves it down to its use behind the barrier)
          asm volatile("" : "+v"(dsf[((j - NF) * 16 / NV) >> 3]));
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    for (int u = 0; u < n_steps; u += 2) {
      body(u, ra, rb);
      body(u + 1, rb, ra);
    }
    // (the steps that only the other stream has: their barriers and nothing else.  No tile stands in for them, as this stream may have
    // none that its key block sees, and zeros times a tile that is not finite are not 0)
    if (STREAMS > 1)
      for (int u = (n_steps + 1) & ~1; u < ((n_bodies + 1) & ~1); u++) __builtin_amdgcn_s_barrier();
  }
  wait_dma();
  __syncthreads();   // every wave is done with the tiles: they become output staging

  if constexpr (STREAMS > 1) {
    // stream 0 keeps dk and stream 1 dv: each hands the other one over, 16 bytes a lane, lane-major
    static_assert(QB == VB && 8 * QB * 4096 <= STREAMS * STREAM_LDS, "LDS of the sums");
    const uint32_t out = lds_all + wave_all * (QB * 4096) + lane * 16, in = lds_all + (wave_all ^ 4) * (QB * 4096);
#pragma unroll
    for (int i = 0; i < QB; i++)
#pragma unroll
      for (int q4 = 0; q4 < 4; q4++) {
        const f32x16& x = stream == 0 ? dv[i] : dk[i];
        lds_write<f32x4>(out + (i * 4 + q4) * 1024, f32x4{x[4 * q4], x[4 * q4 + 1], x[4 * q4 + 2], x[4 * q4 + 3]});
      }
    __syncthreads();
    if (stream == 1) {
#pragma unroll
      for (int i = 0; i < QB; i++) dk[i] = dv[i];
    }
#pragma unroll
    for (int i = 0; i < QB; i++)
#pragma unroll
      for (int q4 = 0; q4 < 4; q4++) {
        const f32x4 x = lds_read<f32x4>(in + lane * 16 + (i * 4 + q4) * 1024);
#pragma unroll
        for (int j = 0; j < 4; j++) dk[i][4 * q4 + j] += x[j];      // (from here on a stream's own output)
      }
    if constexpr (PARTS) {
      partial_store<QB>(dkv_partial<DQK, DV>(a, run, bhk, nb) + wave * (32 * (DQK + DV)) + lane * 4 + (stream == 0 ? 0 : 32 * DQK), dk);
    } else {
      // (staged where only this wave has read)
      T* base = stream == 0 ? (T*)a.dk + (int64_t)b * a.dksb + (int64_t)hk * a.dksh : (T*)a.dv + (int64_t)b * a.dvsb + (int64_t)hk * a.dvsh;
      store_rows<T, DQK>(dk, stream == 0 ? a.scale : 1.f, in, base, stream == 0 ? a.dkss : a.dvss, n_wave, a.Skv, lane);
    }
    __syncthreads();   // the sums have left the stages: the next key block's tiles may arrive
    continue;
  }
  constexpr int DMAX = DQK > DV ? DQK : DV, OROW = DMAX + 16;
  const uint32_t stage = lds0 + wave * 32 * OROW;
  T* dkb = (T*)a.dk + (int64_t)b * a.dksb + (int64_t)hk * a.dksh;
  T* dvb = (T*)a.dv + (int64_t)b * a.dvsb + (int64_t)hk * a.dvsh;
  store_rows<T, DQK>(dk, a.scale, stage, dkb, a.dkss, n_wave, a.Skv, lane);
  store_rows<T, DV>(dv, 1.f, stage, dvb, a.dvss, n_wave, a.Skv, lane);
  __syncthreads();   // the staged output has left the stages: the next key block's tiles may arrive
  }   // the item's key blocks
  }   // items
}

// ------------------------------------------------------------------------------------------------
// dk and dv in one launch: two waves per SIMD, one for dv and one for dk
// ------------------------------------------------------------------------------------------------
// The work of the kernel above where the accumulators of one product and the fragments of one operand fit half a
// SIMD's registers: eight waves take 128 keys, two waves the same 32 of them, on one SIMD.  For every tile u of 32 query rows
//   wave A   S(u+1) = Q(u+1) K^T with p(u) behind its MFMAs, p(u) to the partner through LDS (fp32);  dV^T += dO(u)^T P(u)
//   wave B   dP(u+1) = dO(u+1) V^T with ds(u) behind its MFMAs;                                       dK^T += Q(u)^T dS(u)
// as many MFMAs each whatever the head sizes.  One barrier a tile, between the two halves of A's step and in front of B's: between
// two barriers A runs its pure MFMA half beside B's row function and then its own row function beside B's pure MFMA half.
// What bounded the one-wave kernel was issue: 250 k of 412 k clocks a wave, one instruction at a time, the matrix pipe idle for the rest.
// B2 H32 Hkv8 S2047 128/128 causal 198 -> 170 us = 0.865 PFLOP/s of MFMAs (147 GFLOP; 40 % of the cycles at 2.07 GHz; the LDS is busy for 32 %, without
// conflicts).  From there on longer and shorter rings (4, 5 or 7 MFMAs ahead), p written earlier and fewer scalar instructions change
// 1 % or nothing: the forward kernel's 1.1 PFLOP/s at the clock that random operands leave is near.  Forward + backward B8 H32 S4096
// 5740 -> 5120 us, B2 H16 S1600 159 -> 144, B2 H32 Hkv8 S1500 sigmoid without a mask 443 -> 389, B4 H16 S1024 192/128 179 -> 163; at
// 128 / 256, which took a launch for dk and one for dv before, B2 H16 S2048 causal 371 -> 286, B4 H32 S2500 1825 -> 1610; 256 / 256
// likewise, B4 H16 S1024 286 -> 263, B4 H12 S1024 sigmoid without a mask 388 -> 318.
// Ring of NST stages: behind barrier u the tiles u, u + 1 and u + 2 are read, and the stage of tile u - 1 takes tile u + NST - 1.
// The same products in the same order as the kernel above: the same bits where everything is finite.
// MASKS: as in the kernel above, from a list of the steps in LDS.  Both waves know what a mask hides: A makes p = 0 of it, and B, where dp or
// delta is not finite, ds = 0; tiles that a wave's keys do not see under a causal mask stay out of its sums.  (With B's part forward + backward
// of B2 H32 Hkv8 S2047 128/128 causal 355 -> 360 us, B2 H16 S1600 141.6 -> 142.8; the mask evaluated by B in every tile that it touches
// cost 6 % under a window.)
// At 256 / 256 fragments, accumulators and one set of scores fill the registers: there a wave's step is its scores, the row function, its
// accumulators, one after the other, beside the partner's (pair_serial; a tile is then read in two steps, not three).  There a softmax step
// reads its operand fragments two MFMAs ahead instead of three, and the lane's part of every address but the fragments' is made where it is
// used: held in registers they were spilled, and a reload waits for all loads under way, the next tiles' among them (causal: 8 of them a
// step; now none).  Forward + backward, B8 H12 S829 causal 366 -> 304 us, B8 H16 S600 302 -> 253, B4 H16 S4096 3020 -> 2725, without a mask
// 5345 -> 4912; with three fragments ahead, one reload left, 318, 262, 2740 and 5003.
constexpr bool pair_serial(int dqk, int dv) { return dqk + dv >= 512; }
constexpr int pair_stages(int dqk, int dv, bool masks) { return pair_serial(dqk, dv) ? 3 : (pad_width(dqk) + dv <= 256 ? 6 : 5) - masks; }
constexpr size_t pair_lds(int dqk, int dv, bool masks) {
  return pair_stages(dqk, dv, masks) * (32 * (size_t)(pad_width(dqk) + dv) * 2 + 512 + (masks ? 4 * 1024 : 0)) + 2 * 4 * 4096 + (masks ? FUSED_LIST_MAX * 4 + 16 : 0);
}

template <typename T, int DQK, int DV, int FAMILY, bool CAUSAL, bool MASKS, bool PARTS>
__global__ __launch_bounds__(512, 2) void attn_bwd_dkv_pair_kernel(const AttnBwdArgs a) {
  using E = Elem<T>;
  using x8 = typename E::x8;
  using x4 = typename E::x4;
  constexpr int BNW = 128, BMT = 32;
  constexpr int QROW = pad_width(DQK) * 2, DOROW = DV * 2;   // (LDS rows; 192-wide queries sit in 256-wide rows)
  // a stage: the Q tile, the dO tile, lse (first 128 bytes) and delta (at 256) of its rows
  constexpr int QTILE = BMT * QROW, DOTILE = BMT * DOROW, ROWVALS = QTILE + DOTILE, STAGE = ROWVALS + 512;
  constexpr int NST = pair_stages(DQK, DV, MASKS), XCHG = NST * STAGE;
  // (MASKS) behind the exchanged p: 1 KB of mask bytes per stage and wave, then the step list and its length
  constexpr int KEEP = XCHG + 2 * 4 * 4096, LIST = KEEP + NST * 4 * 1024, LIST_N = LIST + FUSED_LIST_MAX * 4;
  constexpr bool SERIAL = pair_serial(DQK, DV);
  constexpr int READ = SERIAL ? 3 : 4;      // tiles that are read or must have landed
  static_assert(NST >= READ && pair_lds(DQK, DV, MASKS) <= 160 * 1024 && STAGE % QROW == 0 && STAGE % DOROW == 0 && 8 * 32 * ((DQK > DV ? DQK : DV) + 16) <= NST * STAGE, "LDS");

  extern __shared__ __align__(16) char smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(MA_LDS char*)smem;
  const int tid = threadIdx.x, lane = tid & 63, wave_all = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave_all & 3;
  // (where registers are short what is rarely needed is made from the lane's number anew: derived from the one above, the compiler
  // carries it through the loop in spilled registers.  128 / 128 has the registers: 201 us for 203, B2 H16 S1500)
  auto lane_here = [&]() { return DQK + DV > 256 ? lane_anew() : lane; };
  const int r = lane & 31, g = lane >> 5, jr = (lane & 15) >> 2, lc = (((lane >> 4) & 1) << 1) | ((lane & 3) >> 1);

  // persistent, items as in the kernel above
  const int nnb = a.num_blocks, BHK = a.B * a.Hkv, n_parts = PARTS ? a.n_parts : 1;
  const int per_bh = (CAUSAL ? (nnb + 1) / 2 : nnb) * n_parts, n_items = BHK * per_bh;
  const float bias = a.bias + (a.bias_ptr ? *a.bias_ptr : 0.f);
  const float c_scale = a.scale * kLog2e, c_bias = bias * kLog2e;
  const float s_masked = -__builtin_inff();   // a score whose p is 0 (scale > 0)
  const int64_t q_row_bytes = a.qss * 2, do_row_bytes = a.doss * 2;
  TileDma<QROW, 8, DQK / 8> q_dma;
  TileDma<DOROW, 8> do_dma;
  q_dma.init((uint32_t)q_row_bytes, wave_all, lane);
  do_dma.init((uint32_t)do_row_bytes, wave_all, lane);
  constexpr int TILE_DMAS = TileDma<QROW, 8>::NJ + TileDma<DOROW, 8>::NJ;   // what a wave issues per tile at least (a lane may sit out instructions at 192, a whole wave never does)

  for (int item = blockIdx.x; item < n_items; item += gridDim.x) {
  int bhk, ki, run;
  if ((BHK & 7) == 0) {
    const int slot = item >> 3;
    bhk = (slot / per_bh) * 8 + (item & 7);
    ki = slot % per_bh;
    run = ki % n_parts;
    ki /= n_parts;
    if (MASKS) ki = (ki + slot / per_bh) % nnb;      // (another key block each time round, see above)
  } else {
    bhk = item / per_bh;
    ki = item % per_bh;
    run = ki % n_parts;
    ki /= n_parts;
    if (MASKS) ki = (ki + bhk) % nnb;
  }
  const int b = bhk / a.Hkv, hk = bhk % a.Hkv;
  for (int part = 0; part < (CAUSAL && ki != nnb - 1 - ki ? 2 : 1); part++) {
  const int nb = part == 0 ? ki : nnb - 1 - ki;
  const int n_wave = nb * BNW + wave * 32, n_lane = n_wave + r;
  const int n_ld = min(n_lane, a.Skv - 1);

  const int t_first = CAUSAL ? (nb * BNW) / BMT : 0;
  const int t_count = (a.Sq + BMT - 1) / BMT - t_first;
  int n_steps = t_count > 0 ? t_count * a.kv_group : 0;
  DkvWalk first{0, 0, 0};
  int each = 0, more = 0;      // a run's tiles of a head: one more than `each` where its first one comes before `more`
  if (PARTS && !MASKS && n_steps > 0) {
    each = t_count / n_parts;
    more = t_count % n_parts;
    first.skip = ((run - t_first) % n_parts + n_parts) % n_parts;
    n_steps = 0;
    for (int hg = 0, skip = first.skip; hg < a.kv_group; hg++, skip = skip == 0 ? n_parts - 1 : skip - 1) n_steps += each + (skip < more ? 1 : 0);
    first.to_tile(first.skip, n_parts, t_count, a.kv_group);
  }
  const bool keep_ok = MASKS && a.elem_mask_t && ((a.emt_sk | a.emt_sb | a.emt_sh | (int64_t)(uintptr_t)a.elem_mask_t) & 15) == 0;
  if constexpr (MASKS) {
    // the step list: entry = tile | head of the group << 16 | kept in full << 31
    const uint8_t* qbm = a.q_block_mask ? a.q_block_mask + (int64_t)b * a.qbm_sb + (int64_t)nb * a.qbm_sk : nullptr;
    if (wave_all == 0) {
      int count = 0;
      for (int i0 = 0; i0 < n_steps; i0 += 64) {
        const int i = i0 + lane;
        bool keep = false;
        uint32_t entry = 0;
        if (i < n_steps) {
          const int hg = i / t_count, t = i - hg * t_count;
          const uint8_t e = qbm ? qbm[(int64_t)(hk * a.kv_group + hg) * a.qbm_sh + t] : (uint8_t)1;
          keep = e != 0 && (!PARTS || (t + hg) % n_parts == run);
          entry = (uint32_t)t | ((uint32_t)hg << 16) | (e >= 2 || !a.elem_mask_t ? 0x80000000u : 0u);
        }
        const uint64_t votes = __ballot(keep);
        if (keep) lds_write<uint32_t>(lds0 + LIST + 4 * (count + __popcll(votes & ((1ull << lane) - 1ull))), entry);
        count += __popcll(votes);
      }
      if (lane == 0) lds_write<uint32_t>(lds0 + LIST_N, (uint32_t)count);
    }
    __syncthreads();
    n_steps = __builtin_amdgcn_readfirstlane((int)lds_read<uint32_t>(lds0 + LIST_N));
  }
  // (list entries are requested a step before they are used and made wave-uniform only then)
  auto list_request = [&](int i) { return lds_read<uint32_t>(lds0 + LIST + 4 * (i < n_steps ? i : 0)); };
  auto uniform = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
  auto entry_walk = [&](uint32_t e) { return DkvWalk{(int)((e >> 16) & 0x7fffu), (int)(e & 0xffffu), 0}; };
  // The next tile to fetch: a run's tiles of a head follow each other at fixed distances, so that its rows' addresses are sums.
  // (Made anew for every tile they are 48 scalar instructions behind the barrier, where no MFMA is under way.)
  struct Fetch {
    DkvWalk w;
    const char *q, *d;
    const float *lse, *delta;
  } fetch;
  const int64_t q_step = (int64_t)(BMT * n_parts) * q_row_bytes, do_step = (int64_t)(BMT * n_parts) * do_row_bytes;
  const int t_whole = a.Sq / BMT - t_first;      // (tiles of a head that lie inside the sequence)
  auto fetch_at = [&](DkvWalk w) {
    const int h = hk * a.kv_group + w.hg;
    const int64_t m0 = (int64_t)(t_first + w.t) * BMT, row = ((int64_t)b * a.H + h) * a.Sq + m0;
    fetch.w = w;
    fetch.q = (const char*)((const T*)a.q + (int64_t)b * a.qsb + (int64_t)h * a.qsh) + m0 * q_row_bytes;
    fetch.d = (const char*)((const T*)a.dout + (int64_t)b * a.dosb + (int64_t)h * a.dosh) + m0 * do_row_bytes;
    fetch.lse = a.lse + row;
    fetch.delta = (const float*)a.delta + row;
  };
  auto issue_tile = [&](uint32_t to, bool full) {
    if constexpr (MASKS) {
      // the transposed element-wise keep mask of A's keys: whole tiles of a 16-byte aligned mask come with the Q / dO tile
      const int m0 = (t_first + fetch.w.t) * BMT, h = hk * a.kv_group + fetch.w.hg;
      if (wave_all < 4 && keep_ok && !full && m0 + BMT <= a.Sq && n_wave < a.Skv)
        keep_dma(a.elem_mask_t + (int64_t)b * a.emt_sb + (int64_t)h * a.emt_sh + (int64_t)n_wave * a.emt_sk + m0, a.emt_sk, a.Skv - n_wave,
                 lds0 + KEEP + ((to - lds0) / STAGE * 4 + wave) * 1024, lane_here());
    }
    const int rows = fetch.w.t < t_whole ? BMT : a.Sq % BMT;   // (wave-uniform)
    if (rows == BMT) {
      if constexpr (SERIAL) {
        const int ln = lane_anew();
        q_dma.init((uint32_t)q_row_bytes, wave_all, ln);
        do_dma.init((uint32_t)do_row_bytes, wave_all, ln);
      }
      q_dma.issue(fetch.q, to, wave_all);
      do_dma.issue(fetch.d, to + QTILE, wave_all);
    } else {
      const int ln = lane_here();
      dma_tile<QROW, 8, DQK / 8>(fetch.q, q_row_bytes, 0, rows, to, wave_all, ln);
      dma_tile<DOROW, 8>(fetch.d, do_row_bytes, 0, rows, to + QTILE, wave_all, ln);
    }
    if constexpr (FAMILY == BF_SOFTMAX) {
      // wave 0 fetches lse, wave 1 delta (the upper lanes repeat the lower ones)
      if (wave_all < 2) dma4_so(wave_all == 0 ? fetch.lse : fetch.delta, (uint32_t)min(lane & 31, rows - 1) * 4u, to + ROWVALS + wave_all * 256);
    }
    if constexpr (MASKS) return;
    DkvWalk w = fetch.w;
    w.next<PARTS>(n_parts, t_count, a.kv_group);
    if (w.hg == fetch.w.hg) {
      fetch.w = w;
      fetch.q += q_step;
      fetch.d += do_step;
      if constexpr (FAMILY == BF_SOFTMAX) {
        fetch.lse += BMT * n_parts;
        fetch.delta += BMT * n_parts;
      }
    } else if (w.hg < a.kv_group) {
      fetch_at(w);
    }
  };

  auto work = [&](auto role) __attribute__((always_inline)) {
    constexpr bool ROLE_B = decltype(role)::value != 0;
    // rows of one tile against the wave's fragments make the scores, the columns of the other the accumulators
    constexpr int DR = ROLE_B ? DV : DQK, DC = ROLE_B ? DQK : DV;
    constexpr int RROW = ROLE_B ? DOROW : QROW, CROW = ROLE_B ? QROW : DOROW, ROFF = ROLE_B ? QTILE : 0, COFF = ROLE_B ? 0 : QTILE;
    // (128 / 256: with the longer ring 40 registers spill, B2 H16 S2048 causal 302 us, 286 with four)
    constexpr int NR = DR / 16, CB = DC / 32, NTOT = NR + 2 * CB, RING = NTOT % 8 == 0 && DQK + DV <= 256 ? 8 : 4, AH = RING == 8 ? 5 : SERIAL && FAMILY == BF_SOFTMAX ? 2 : 3;
    static_assert(NTOT % RING == 0 && AH <= NR && AH <= 2 * CB, "fragment ring");
    x8 wf[NR];
    {
      const T* p = ROLE_B ? (const T*)a.v + (int64_t)b * a.vsb + (int64_t)n_ld * a.vss + (int64_t)hk * a.vsh + 8 * g
                          : (const T*)a.k + (int64_t)b * a.ksb + (int64_t)n_ld * a.kss + (int64_t)hk * a.ksh + 8 * g;
#pragma unroll
      for (int i = 0; i < NR; i++) wf[i] = *(const x8*)(p + 16 * i);
    }
    f32x16 acc[CB];
#pragma unroll
    for (int i = 0; i < CB; i++)
#pragma unroll
      for (int j = 0; j < 16; j++) acc[i][j] = 0.f;

    if (n_steps > 0) {
      const uint32_t row_l = ROFF + (uint32_t)(r * RROW) + (uint32_t)((g ^ swz_tile<RROW / 16>(r)) << 4);
      const uint32_t col_l = COFF + (uint32_t)((4 * g + jr) * CROW + (lane & 1) * 8) + (uint32_t)((lc ^ swz_tile<CROW / 16>(4 * g + jr)) << 4);
      // the fragment of MFMA j of a step: the row reads from `rows`, the transposing reads from `cols` (stages)
      auto fragment = [&](auto jc, uint32_t rows, uint32_t cols) __attribute__((always_inline)) -> x8 {
        constexpr int j = decltype(jc)::value;
        if constexpr (j < NR) {
          return lds_read<x8>((rows + row_l) ^ (uint32_t)(j * 32));
        } else {
          constexpr int db = (j - NR) % CB, sl = (j - NR) / CB;
          const x4 lo = lds_read_tr4<T>(((cols + col_l) ^ (uint32_t)((4 * db) << 4)) + 16 * sl * CROW);
          const x4 hi = lds_read_tr4<T>(((cols + col_l) ^ (uint32_t)(((4 * db) ^ 2) << 4)) + (16 * sl + 8) * CROW);
          return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
      };
      const uint32_t x_l = lds0 + XCHG + wave * 4096 + lane * 16;      // p of the even tiles, 16 KB on of the odd ones
      f32x4 rv[4];      // lse (A) or delta (B) of the rows 8 q4 + 4 g + {0..3} of the step's tile
      auto row_values = [&](uint32_t tile) {
        if constexpr (FAMILY == BF_SOFTMAX) {
          uint32_t at = tile + ROWVALS + (ROLE_B ? 256 : 0);
          if constexpr (SERIAL) {
            at += lane_anew() >> 5 << 4;
            asm volatile("" : "+v"(at));      // (one address and four offsets, not four addresses)
          }
#pragma unroll
          for (int q4 = 0; q4 < 4; q4++) rv[q4] = lds_read<f32x4>(at + (SERIAL ? 8 * q4 : 8 * q4 + 4 * g) * 4);
        }
      };

      DkvWalk at = first;      // the current step's tile
      if (!MASKS) fetch_at(first);
      uint32_t i_next = MASKS ? list_request(0) : 0u, c_next = i_next;      // (MASKS) the entries of the next tile to fetch and of the next step
      int i_n = 0;
      uint32_t to = lds0;
      auto after = [&](uint32_t stage) { return stage == lds0 + (NST - 1) * STAGE ? lds0 : stage + STAGE; };
      auto issue_next = [&]() {
        bool full = true;
        if constexpr (MASKS) {
          const uint32_t e = uniform(i_next);
          fetch_at(entry_walk(e));
          full = (e >> 31) != 0;
        }
        issue_tile(to, full);
        to = after(to);
        i_n++;
        if constexpr (MASKS) i_next = list_request(i_n);
      };
#pragma unroll
      for (int i = 0; i < NST - 1; i++)
        if (i_n < n_steps) issue_next();
      wait_dma();
      __syncthreads();
      uint32_t t0 = lds0, t1 = lds0 + STAGE, t2 = lds0 + 2 * STAGE;      // the stages of tiles u, u + 1, u + 2
      f32x16 sa, sb;
      x8 fr[RING];
      if constexpr (!SERIAL) sa = mm_rows<T, DR>(t0 + ROFF, r, g, wf);
      // what a step finds ready beside its scores
      auto fill = [&]() __attribute__((always_inline)) {
        static_for<0, AH>([&](auto jc) __attribute__((always_inline)) { fr[decltype(jc)::value] = fragment(jc, SERIAL ? t0 : t1, t0); });
        if constexpr (!SERIAL) row_values(t0);
      };
      const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

      // None of the wave's keys sees the tile at hand: the accumulators are to be left alone (p = 0 times a row of dO that is not finite
      // is not 0).
      auto unseen = [&](const DkvWalk& w) { return n_wave >= (t_first + w.t + 1) * BMT; };
      // The elements that a mask hides: p = 0 (A) and ds = 0 (B, from dp = delta = 0) whatever the rows and keys hold.  B leaves out what
      // does not matter: relu's ds is 0 where p is, and without a mask all that is hidden is the last row again and keys that do not exist.
      constexpr bool HIDES = !ROLE_B || ((CAUSAL || MASKS) && FAMILY != BF_RELU);
      auto hide = [&](int u, f32x16& cur) __attribute__((always_inline)) {
        if constexpr (!HIDES && !CAUSAL) return;
        const uint32_t c_entry = MASKS ? uniform(c_next) : 0u;
        if constexpr (MASKS) {
          c_next = list_request(u + 1);
          at = entry_walk(c_entry);
        }
        const int m0 = (t_first + at.t) * BMT;
        if (!MASKS) at.template next<PARTS>(n_parts, t_count, a.kv_group);
        if constexpr (!HIDES) return;
        const bool by_elem = MASKS && a.elem_mask_t && (c_entry >> 31) == 0;
        if ((CAUSAL && n_wave + 31 > m0) || m0 + BMT > a.Sq || n_wave + 32 > a.Skv || by_elem) {
          if constexpr (ROLE_B) {
            // (as a rule nothing here is not finite, and 0 times it is 0: one look at all of it instead of the mask)
            f32x4 any = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int jj = 0; jj < 16; jj++) any[jj & 3] = FAMILY == BF_SOFTMAX ? fmaf(cur[jj], rv[jj >> 2][jj & 3], any[jj & 3]) : any[jj & 3] + cur[jj];
            if (__all(__builtin_isfinite((any[0] + any[1]) + (any[2] + any[3])))) return;
          }
          int m0e = m0;
          asm volatile("; a tile that touches a mask" : "+s"(m0e));      // (see the kernel above)
          const int ln = lane_here(), r = ln & 31, g = ln >> 5, n_lane = n_wave + r, n_ld = min(n_lane, a.Skv - 1);
          uint32_t keep[4] = {0x01010101u, 0x01010101u, 0x01010101u, 0x01010101u};   // the bytes of this lane's four rows per group
          if constexpr (MASKS) {
            if (by_elem) {
              if (keep_ok && m0e + BMT <= a.Sq && n_wave < a.Skv) {
#pragma unroll
                for (int q4 = 0; q4 < 4; q4++) keep[q4] = keep_read(lds0 + KEEP + ((t0 - lds0) / STAGE * 4 + wave) * 1024, r, g, q4);
              } else {
                // this key's row of the transposed mask, indexed by query position
                const uint8_t* emt_row = a.elem_mask_t + (int64_t)b * a.emt_sb + (int64_t)(hk * a.kv_group + at.hg) * a.emt_sh + (int64_t)n_ld * a.emt_sk;
#pragma unroll
                for (int q4 = 0; q4 < 4; q4++) {
                  const int m = m0e + 8 * q4 + 4 * g;
                  keep[q4] = 0;
#pragma unroll
                  for (int i = 0; i < 4; i++)
                    if (m + i < a.Sq) keep[q4] |= (uint32_t)emt_row[m + i] << (8 * i);
                }
              }
            }
          }
#pragma unroll
          for (int jj = 0; jj < 16; jj++) {
            const int m = m0e + 8 * (jj >> 2) + 4 * g + (jj & 3);
            if ((CAUSAL && n_lane > m) || m >= a.Sq || n_lane >= a.Skv || (MASKS && ((keep[jj >> 2] >> (8 * (jj & 3))) & 0xffu) == 0)) {
              cur[jj] = ROLE_B ? 0.f : s_masked;
              // (a row without any kept key has lse = -inf: its masked scores must still give p = 0)
              if constexpr (FAMILY == BF_SOFTMAX) rv[jj >> 2][jj & 3] = 0.f;
            }
          }
        }
      };
      // tile u + 2 (SERIAL: u + 1) has landed (what may still be in flight: the tiles behind it), p(u) is in LDS, and every wave is done
      // with tile u - 1, whose stage takes tile u + NST - 1
      auto meet = [&](int u) __attribute__((always_inline)) {
        if (u + NST - 2 < n_steps) wait_dma_but<(NST - READ) * TILE_DMAS>();
        else wait_dma();
        if constexpr (!ROLE_B) __builtin_amdgcn_s_waitcnt(0xC07F);      // lgkmcnt(0)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      };
      auto ahead = [&]() {
        t0 = t1;
        t1 = SERIAL ? after(t1) : t2;
        if constexpr (!SERIAL) t2 = after(t2);
      };
      auto body = [&](int u, f32x16& cur, f32x16& nxt) __attribute__((always_inline)) {
        if constexpr (!ROLE_B) hide(u, cur);
        const uint32_t x = x_l + (u & 1) * 16384;
        x8 f[2];
        f32x4 p4[4];
        static_for<0, NTOT>([&](auto jc) __attribute__((always_inline)) {
          constexpr int j = decltype(jc)::value;
          if constexpr (j == (ROLE_B ? 0 : NR)) {
            meet(u);
            if constexpr (ROLE_B) {
#pragma unroll
              for (int q4 = 0; q4 < 4; q4++) p4[q4] = lds_read<f32x4>(x + q4 * 1024);
            }
          }
          if constexpr (ROLE_B && j == 2) hide(u, cur);
          if constexpr (j == (ROLE_B ? 2 : NR + 2))      // (two MFMAs on: behind the barrier itself, B2 H16 S1600 148 us for 144)
            if (i_n < n_steps) issue_next();
          if constexpr (j == NTOT - 4) row_values(t1);
          // the fragment of the MFMA AH places on (the last ones of the step: of the next step's first MFMAs)
          if constexpr (j + AH < NTOT) fr[(j + AH) % RING] = fragment(IntC<j + AH>(), t1, t0);
          else fr[(j + AH) % RING] = fragment(IntC<j + AH - NTOT>(), t2, t1);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (j < NR) nxt = E::mfma32(fr[j % RING], wf[j], j == 0 ? zero16 : nxt);
          else acc[(j - NR) % CB] = E::mfma32(fr[j % RING], f[(j - NR) / CB], acc[(j - NR) % CB]);
          // vector work behind the MFMA: p, or ds, of the step's 16 elements (ds from the second MFMA on: its p come from LDS)
          if constexpr (j < NR) {
            constexpr int J0 = ROLE_B ? 2 : 0;
            constexpr int from = j < J0 ? 0 : (j - J0) * 16 / (NR - J0), upto = j < J0 ? 0 : (j + 1 - J0) * 16 / (NR - J0);
#pragma unroll
            for (int jj = from; jj < upto; jj++) {
              if constexpr (!ROLE_B) {
                p4[jj >> 2][jj & 3] = row_p<FAMILY>(cur[jj], c_scale, c_bias, a.scale, bias, FAMILY == BF_SOFTMAX ? fmaf(rv[jj >> 2][jj & 3], -kLog2e, c_bias) : 0.f);
                f[jj >> 3][jj & 7] = (T)p4[jj >> 2][jj & 3];
                if ((jj & 3) == 3) lds_write<f32x4>(x + (jj >> 2) * 1024, p4[jj >> 2]);
              } else {
                f[jj >> 3][jj & 7] = (T)row_ds<FAMILY>(p4[jj >> 2][jj & 3], cur[jj], FAMILY == BF_SOFTMAX ? rv[jj >> 2][jj & 3] : 0.f);
              }
            }
            // (evaluated here, behind this MFMA)
            if constexpr (upto > from) asm volatile("" : "+v"(f[(upto - 1) >> 3]));
          }
          __builtin_amdgcn_sched_barrier(0);
        });
        ahead();
      };
      auto serial_body = [&](int u) __attribute__((always_inline)) {
        x8 f[2];
        static_for<0, NTOT>([&](auto jc) __attribute__((always_inline)) {
          constexpr int j = decltype(jc)::value;
          if constexpr (ROLE_B && j == 0) meet(u);
          if constexpr (j == NR - 1) row_values(t0);
          if constexpr (j == NR) {
            hide(u, sa);
            const uint32_t x = lds0 + XCHG + wave * 4096 + (u & 1) * 16384 + lane_anew() * 16;
#pragma unroll
            for (int q4 = 0; q4 < 4; q4++) {
              f32x4 p;
              if constexpr (ROLE_B) p = lds_read<f32x4>(x + q4 * 1024);
#pragma unroll
              for (int i = 0; i < 4; i++) {
                const float row = FAMILY == BF_SOFTMAX ? rv[q4][i] : 0.f;
                if constexpr (!ROLE_B) p[i] = row_p<FAMILY>(sa[4 * q4 + i], c_scale, c_bias, a.scale, bias, FAMILY == BF_SOFTMAX ? fmaf(row, -kLog2e, c_bias) : 0.f);
                f[q4 >> 1][4 * (q4 & 1) + i] = (T)(ROLE_B ? row_ds<FAMILY>(p[i], sa[4 * q4 + i], row) : p[i]);
              }
              if constexpr (!ROLE_B) lds_write<f32x4>(x + q4 * 1024, p);
            }
            if constexpr (!ROLE_B) meet(u);
          }
          if constexpr (j == (ROLE_B ? 2 : NR + 2))
            if (i_n < n_steps) issue_next();
          if constexpr (j + AH < NTOT) fr[(j + AH) % RING] = fragment(IntC<j + AH>(), t0, t0);
          else fr[(j + AH) % RING] = fragment(IntC<j + AH - NTOT>(), t1, t0);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (j < NR) sa = E::mfma32(fr[j % RING], wf[j], j == 0 ? zero16 : sa);
          else acc[(j - NR) % CB] = E::mfma32(fr[j % RING], f[(j - NR) / CB], acc[(j - NR) % CB]);
          __builtin_amdgcn_sched_barrier(0);
        });
        ahead();
      };
      for (int u = 0, upto; u < n_steps; u = upto) {
        // The tiles in front of the diagonal come first of every head, for the waves of the later keys: those take part in the barriers
        // and have the next step's scores ready.  (A way round the products inside the step instead makes the compiler spill 60 to 900
        // registers.)
        upto = n_steps;
        if constexpr (CAUSAL) {
          int passed = 0;      // of the head at hand
          for (; u < n_steps && unseen(at); u++) {
            const int hg = at.hg;
            at.template next<PARTS>(n_parts, t_count, a.kv_group);
            passed = at.hg == hg ? passed + 1 : 0;
            if constexpr (!SERIAL)
              if (!unseen(at)) sa = mm_rows<T, DR>(t1 + ROFF, r, g, wf);
            meet(u);
            if (i_n < n_steps) issue_next();
            ahead();
          }
          if (n_wave > t_first * BMT) {
            upto = u - passed;
            DkvWalk w = at;
            do {
              upto += PARTS ? each + (w.skip < more ? 1 : 0) : t_count;
              w.to_tile(t_count, n_parts, t_count, a.kv_group);
            } while (upto < n_steps && !unseen(w));
            upto = min(upto, n_steps);      // (a run may end in front of the diagonal)
          }
        }
        fill();
        if constexpr (SERIAL) {
          for (; u < upto; u++) serial_body(u);
        } else {
          for (; u + 1 < upto; u += 2) {
            body(u, sa, sb);
            body(u + 1, sb, sa);
          }
          if (u < upto) body(u, sa, sb);
        }
      }
    }
    wait_dma();
    __syncthreads();   // every wave is done with the tiles: they become output staging

    if constexpr (PARTS) {
      partial_store<CB>(dkv_partial<DQK, DV>(a, run, bhk, nb) + wave * (32 * (DQK + DV)) + lane_here() * 4 + (ROLE_B ? 0 : 32 * DQK), acc);
    } else {
      T* base = ROLE_B ? (T*)a.dk + (int64_t)b * a.dksb + (int64_t)hk * a.dksh : (T*)a.dv + (int64_t)b * a.dvsb + (int64_t)hk * a.dvsh;
      store_rows<T, DC>(acc, ROLE_B ? a.scale : 1.f, lds0 + wave_all * (32 * ((DQK > DV ? DQK : DV) + 16)), base, ROLE_B ? a.dkss : a.dvss, n_wave, a.Skv, lane_here());
      __syncthreads();   // the staged output has left the stages: the next key block's tiles may arrive
    }
  };
  if (wave_all < 4) work(IntC<0>());
  else work(IntC<1>());
  }   // the item's key blocks
  }   // items
}

// dk, dv = the sum of the runs' fp32 partial sums (in the order of the runs), rounded once.  A workgroup of 4 waves takes
// dk (blockIdx.y 0) or dv (1) of a key block, a wave the 32 keys that it has in the kernel above, in the same registers.
template <typename T, int DQK, int DV>
__global__ __launch_bounds__(256) void attn_bwd_dkv_reduce_kernel(const AttnBwdArgs a) {
  constexpr int DMAX = DQK > DV ? DQK : DV;
  __shared__ __align__(16) char smem[4 * 32 * (DMAX + 16)];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nnb = a.num_blocks, bhk = blockIdx.x / nnb, nb = blockIdx.x % nnb;
  const int b = bhk / a.Hkv, hk = bhk % a.Hkv, n_wave = nb * 128 + wave * 32;
  const uint32_t stage = (uint32_t)(uintptr_t)(MA_LDS char*)smem + wave * 32 * (DMAX + 16);
  auto sum = [&](auto& acc, int offset) __attribute__((always_inline)) {
    constexpr int N = sizeof(acc) / sizeof(f32x16);
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
      for (int j = 0; j < 16; j++) acc[i][j] = 0.f;
    for (int run = 0; run < a.n_parts; run++) {
      const float* from = dkv_partial<DQK, DV>(a, run, bhk, nb) + wave * (32 * (DQK + DV)) + offset + lane * 4;
#pragma unroll
      for (int i = 0; i < N; i++)
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) {
          const f32x4 x = *(const f32x4*)(from + (i * 4 + q4) * 256);
#pragma unroll
          for (int j = 0; j < 4; j++) acc[i][4 * q4 + j] += x[j];
        }
    }
  };
  if (blockIdx.y == 0) {
    f32x16 dk[DQK / 32];
    sum(dk, 0);
    store_rows<T, DQK>(dk, a.scale, stage, (T*)a.dk + (int64_t)b * a.dksb + (int64_t)hk * a.dksh, a.dkss, n_wave, a.Skv, lane);
  } else {
    f32x16 dv[DV / 32];
    sum(dv, 32 * DQK);
    store_rows<T, DV>(dv, 1.f, stage, (T*)a.dv + (int64_t)b * a.dvsb + (int64_t)hk * a.dvsh, a.dvss, n_wave, a.Skv, lane);
  }
}

// ------------------------------------------------------------------------------------------------
// Two streams of key tiles in the dq kernel where row blocks are few: a tile is a serial chain of about a microsecond, and with
// at most one workgroup of four waves per CU half of the wave slots are empty.  Under a causal mask (heaviest blocks first)
// the chains of the longest blocks still bind at 1.5 row blocks per CU, and about there the sizes cross.  Forward + backward,
// two streams against one at 320, 384, 416 and 448 row blocks: 128/128 S1024 0.96, 0.99, 1.01, 1.03, 192/128 S1024 0.97, 0.99, 1.02,
// 1.02, 64/64 S600 0.93, 1.01, 1.04, .. (480) 1.02; longer chains cross later (64/64 S1024 0.91, 0.93, 0.96, 0.98; 128/128 S2048 0.93,
// 0.94, 0.97, 0.98).  Without a mask, at 192, 256 and 288: 128/128 0.97, 0.99, 1.08, 64/64 0.92, 0.91, 1.06.
inline bool dq_two_streams(int64_t blocks, bool causal) { return 2 * blocks <= (causal ? 3 : 2) * (int64_t)device_cus(); }

// Masked calls at 128 / 256 in one run, where key blocks have few steps: the pair kernel holds one workgroup a CU, so that its list of steps, first
// tiles and outputs stand alone and a last round that is nearly empty costs a whole one; the two-launch kernels hold two.  Forward + backward,
// two launches and pairs, windows of 147 and 600, S1115 (35 steps, 9 key blocks a head), by key blocks a CU: 1.1 156, 172 and 221, 240 us; 1.4
// 159, 174 and 234, 242; 2.0 168, 181 and 243, 248; 2.25 232, 258 and 314, 345; 2.5 267, 272; 2.8 283, 281; 3.1 295, 329.  Full rounds: 3.0, S679
// 249, 246; 4.0, S400 226, 204; 5.0, S1200 598, 492.  More steps: 1.1, S2300 (72) 192, 197; 1.5, S3000 (94) 229, 222; 2.0, S2000 in groups of
// four heads (252) 538, 425.
inline bool masked_two_launches(int64_t key_blocks, int64_t steps) {
  const int64_t cus = device_cus(), rounds = cus > 0 ? (key_blocks + cus - 1) / cus : 1;
  return steps <= 72 && rounds > 1 && (rounds == 2 || 10 * key_blocks < 8 * rounds * cus);
}

template <typename T, int DQK, int DV, int FAMILY, bool CAUSAL>
static int launch_bwd(const AttnBwdArgs& a, hipStream_t stream) {
  constexpr int DMAX = DQK > DV ? DQK : DV;
  constexpr size_t ostage = 4 * 32 * (size_t)(DMAX + 16);
  constexpr size_t lds = dq_lds(DQK, DV, FAMILY);
  constexpr bool NOT_RETENTION = FAMILY != BF_RETENTION;      // (which takes no masks)
  const bool masked = a.elem_mask || a.kv_block_mask;
  auto k1 = attn_bwd_dq_kernel<T, DQK, DV, FAMILY, CAUSAL, false>;
  auto k1m = attn_bwd_dq_kernel<T, DQK, DV, FAMILY, CAUSAL, NOT_RETENTION>;
  // one dk/dv launch where both accumulators fit beside a second wave, else one launch each (at 256 / 256 the single launch
  // held both 128-register accumulators in a 512-register wave and spilled 170 registers: the whole backward at B4 H16 S4096
  // took 9.7 ms under the causal mask and 6.2 ms without; with one launch each 3.3 ms and 4.8 ms)
  constexpr bool SPLIT = DQK + DV >= 256;
  auto k2 = attn_bwd_dkv_kernel<T, DQK, DV, FAMILY, CAUSAL, SPLIT ? 1 : 3>;
  auto k3 = attn_bwd_dkv_kernel<T, DQK, DV, FAMILY, CAUSAL, 2>;
  static std::atomic<uint64_t> lds_ok{0};
  if (allow_lds(lds_ok, lds, k1, k1m, k2, k3) != 0) return -1;
  AttnBwdArgs args = a;
  if (a.add || a.slope_q || a.slope_kv || a.softcap != 0.f) {
    // additive score terms / soft-capping: instantiations of their own (not for the retention family, whose score function
    // is the multiplier tensor; soft-capping goes with softmax only, as in the forward), dk and dv by the two-launch kernels
    if constexpr (FAMILY != BF_RETENTION) {
      if (a.softcap != 0.f && FAMILY != BF_SOFTMAX) return -2;
      auto e1 = attn_bwd_dq_kernel<T, DQK, DV, FAMILY, CAUSAL, true, true>;
      auto e2 = attn_bwd_dkv_kernel<T, DQK, DV, FAMILY, CAUSAL, SPLIT ? 1 : 3, true>;
      auto e3 = attn_bwd_dkv_kernel<T, DQK, DV, FAMILY, CAUSAL, 2, true>;
      static std::atomic<uint64_t> elds_ok{0};
      if (allow_lds(elds_ok, lds, e1, e2, e3) != 0) return -1;
      args.num_blocks = (a.Sq + 127) / 128;
      hipLaunchKernelGGL(e1, dim3((unsigned)(args.num_blocks * a.B * a.H)), dim3(256), lds, stream, args);
      args.num_blocks = (a.Skv + 127) / 128;
      hipLaunchKernelGGL(e2, dim3((unsigned)(args.num_blocks * a.B * a.Hkv)), dim3(256), lds, stream, args);
      if (SPLIT) hipLaunchKernelGGL(e3, dim3((unsigned)(args.num_blocks * a.B * a.Hkv)), dim3(256), lds, stream, args);
      return launch_status();
    } else {
      return -2;
    }
  }
  args.num_blocks = (a.Sq + 127) / 128;
  bool dq_done = false;
  if constexpr (FAMILY != BF_RETENTION && DQK + DV <= 320) {   // (128 / 256: measured no faster)
    if (dq_two_streams(args.num_blocks * (int64_t)a.B * a.H, CAUSAL)) {
      auto k1s = attn_bwd_dq_kernel<T, DQK, DV, FAMILY, CAUSAL, false, false, 2>;
      auto k1sm = attn_bwd_dq_kernel<T, DQK, DV, FAMILY, CAUSAL, true, false, 2>;
      static std::atomic<uint64_t> slds_ok{0};
      if (allow_lds(slds_ok, 2 * lds, k1s, k1sm) != 0) return -1;
      hipLaunchKernelGGL(masked ? k1sm : k1s, dim3((unsigned)(args.num_blocks * a.B * a.H)), dim3(512), 2 * lds, stream, args);
      dq_done = true;
    }
  }
  if (!dq_done) hipLaunchKernelGGL(masked ? k1m : k1, dim3((unsigned)(args.num_blocks * a.B * a.H)), dim3(256), lds, stream, args);
  args.num_blocks = (a.Skv + 127) / 128;
  if constexpr (FAMILY != BF_RETENTION && DQK <= 256 && DV <= 256) {
    // dk and dv by the pipelined single launch (with masks: as long as a key block's steps fit its list)
    const bool masks = a.elem_mask_t || a.q_block_mask;
    // (256 / 256 with masks in one run: the list's loop has no registers to spare, and its two launches were the faster ones, B2 H16 S1500 with
    // a window of 300 forward + backward 352 and 357 us)
    const int64_t steps = (int64_t)((a.Sq + 31) / 32) * a.kv_group;
    const bool one_run = !a.dkv_part || a.n_parts <= 1;
    const bool two_launches = masks && one_run && (pair_serial(DQK, DV) || (DQK + DV == 384 && masked_two_launches((int64_t)args.num_blocks * a.B * a.Hkv, steps)));
    if (!two_launches && (!masks || steps <= FUSED_LIST_MAX)) {
      if (!a.dkv_part) args.n_parts = 1;
      const bool parts = args.n_parts > 1;
      if (CAUSAL && masks) return -2;   // (masks go with MA_MASK_NONE)
      const int cus = device_cus();
      if (cus <= 0) return -1;
      const int items = (CAUSAL ? (args.num_blocks + 1) / 2 : args.num_blocks) * a.B * a.Hkv * args.n_parts;
      if constexpr (DQK + DV <= 128) {
        constexpr size_t stage = (size_t)32 * (DQK + DV) * 2 + 512;
        constexpr size_t ftiles = fused_stages(false) * stage, mtiles = fused_stages(true) * (stage + 4 * 1024) + FUSED_LIST_MAX * 4 + 16;
        constexpr size_t fmax = ftiles > mtiles ? ftiles : mtiles, flds = fmax > ostage ? fmax : ostage;
        const int64_t workgroups = (int64_t)args.num_blocks * a.B * a.Hkv * args.n_parts;
        if (parts || dkv_two_streams(workgroups, CAUSAL)) {
          auto kf = attn_bwd_dkv_fused_kernel<T, DQK, DV, FAMILY, CAUSAL, false, false, 2>;
          auto kfp = attn_bwd_dkv_fused_kernel<T, DQK, DV, FAMILY, CAUSAL, false, true, 2>;
          auto km = attn_bwd_dkv_fused_kernel<T, DQK, DV, FAMILY, false, true, false, 2>;
          auto kmp = attn_bwd_dkv_fused_kernel<T, DQK, DV, FAMILY, false, true, true, 2>;
          constexpr size_t slds = 2 * ((flds + 1023) & ~(size_t)1023);
          static std::atomic<uint64_t> slds_ok{0};
          if (allow_lds(slds_ok, slds, kf, kfp, km, kmp) != 0) return -1;
          hipLaunchKernelGGL(masks ? (parts ? kmp : km) : (parts ? kfp : kf), dim3((unsigned)workgroups), dim3(512), slds, stream, args);
        } else {
          auto kf = attn_bwd_dkv_fused_kernel<T, DQK, DV, FAMILY, CAUSAL, false, false>;
          auto km = attn_bwd_dkv_fused_kernel<T, DQK, DV, FAMILY, false, true, false>;
          static std::atomic<uint64_t> flds_ok{0};
          if (allow_lds(flds_ok, flds, kf, km) != 0) return -1;
          const int slots = cus * FUSED_PER_CU;
          hipLaunchKernelGGL(masks ? km : kf, dim3((unsigned)(items < slots ? items : slots)), dim3(256), flds, stream, args);
        }
      } else {
        auto kf = attn_bwd_dkv_pair_kernel<T, DQK, DV, FAMILY, CAUSAL, false, false>;
        auto kfp = attn_bwd_dkv_pair_kernel<T, DQK, DV, FAMILY, CAUSAL, false, true>;
        auto km = attn_bwd_dkv_pair_kernel<T, DQK, DV, FAMILY, false, true, pair_serial(DQK, DV)>;      // (pair_serial: never in one run)
        auto kmp = attn_bwd_dkv_pair_kernel<T, DQK, DV, FAMILY, false, true, true>;
        constexpr size_t plain = pair_lds(DQK, DV, false), with_masks = pair_lds(DQK, DV, true);
        static std::atomic<uint64_t> plds_ok{0};
        if (allow_lds(plds_ok, plain > with_masks ? plain : with_masks, kf, kfp, km, kmp) != 0) return -1;
        hipLaunchKernelGGL(masks ? (parts ? kmp : km) : (parts ? kfp : kf), dim3((unsigned)(items < cus ? items : cus)), dim3(512), masks ? with_masks : plain, stream, args);
      }
      if (parts) {
        const dim3 grid((unsigned)(args.num_blocks * a.B * a.Hkv), 2);
        hipLaunchKernelGGL((attn_bwd_dkv_reduce_kernel<T, DQK, DV>), grid, dim3(256), 0, stream, args);
      }
      return launch_status();
    }
  }
  hipLaunchKernelGGL(k2, dim3((unsigned)(args.num_blocks * a.B * a.Hkv)), dim3(256), lds, stream, args);
  if (SPLIT) hipLaunchKernelGGL(k3, dim3((unsigned)(args.num_blocks * a.B * a.Hkv)), dim3(256), lds, stream, args);
  return launch_status();
}

template <typename T, int DQK, int DV>
static int bwd_family(const AttnBwdArgs& a, int family, bool causal, hipStream_t stream) {
  switch (family) {
    case BF_SOFTMAX:
      return causal ? launch_bwd<T, DQK, DV, BF_SOFTMAX, true>(a, stream) : launch_bwd<T, DQK, DV, BF_SOFTMAX, false>(a, stream);
    case BF_SIGMOID:
      return causal ? launch_bwd<T, DQK, DV, BF_SIGMOID, true>(a, stream) : launch_bwd<T, DQK, DV, BF_SIGMOID, false>(a, stream);
    case BF_RELU:
      return causal ? launch_bwd<T, DQK, DV, BF_RELU, true>(a, stream) : launch_bwd<T, DQK, DV, BF_RELU, false>(a, stream);
  }
  return -2;
}

// One head size: the retention family (where it is built at this size) or softmax / sigmoid / relu.
template <typename T, int DQK, int DV, bool RETENTION_TOO>
static int bwd_size(const AttnBwdArgs& a, int family, bool causal, hipStream_t stream) {
  if (family == BF_RETENTION) {
    if constexpr (RETENTION_TOO)
      return causal ? launch_bwd<T, DQK, DV, BF_RETENTION, true>(a, stream) : launch_bwd<T, DQK, DV, BF_RETENTION, false>(a, stream);
    else
      return -2;
  }
  return bwd_family<T, DQK, DV>(a, family, causal, stream);
}

}  // namespace ma
