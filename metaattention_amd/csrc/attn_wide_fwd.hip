// Parallel attention forward: which kernel and cut a call takes, split-kv decode and its merge, and the general kernel
// (attn_wide_fwd_kernel.h) in its form with one stream per row block.
#include "attn_wide_fwd_kernel.h"

#include <cmath>
#include <type_traits>

namespace ma {

// Merge of the kv splits: o = sum_s exp(lse_s - lse) o_s with lse = log sum_s exp(lse_s) (examples/mha_decode.py:72-80).
// One wave per (batch, head, row).  Latency is all there is to it (two trips to memory: the log-sum-exps, a lane each, and the
// partial results, requested before the first have come), so DV / 8 lanes take a row of 16 bytes each and the wave reads
// 512 / DV splits at a time, four times over.  B9 H32 Hkv8 KV3672 64/64, 26 splits: 12.6 us with a load of every split behind
// the one before it, DV / 64 columns a lane.
// P: the partial results' type.
template <typename T, typename P, int DV>
__global__ __launch_bounds__(256) void attn_split_combine_kernel(const AttnArgs a) {
  using x8 = typename Elem<T>::x8;
  typedef P p8 __attribute__((ext_vector_type(8), aligned(16)));
  constexpr int LPR = DV / 8, AT_ONCE = 64 / LPR, FLY = 4;
  const int lane = threadIdx.x & 63, part = lane / LPR, col = (lane % LPR) * 8;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);   // (b * H + h) * Sq + m
  const int64_t rows = (int64_t)a.B * a.H * a.Sq;
  if (row >= rows) return;
  const int m = (int)(row % a.Sq), h = (int)((row / a.Sq) % a.H), b = (int)(row / ((int64_t)a.Sq * a.H));
  const int64_t part_row = ((int64_t)b * a.n_split * a.H + h) * a.Sq + m, split_stride = (int64_t)a.H * a.Sq;
  const P* src = (const P*)a.o_part + part_row * DV + col;
  p8 v[FLY];
  auto fetch = [&](int s0) {
#pragma unroll
    for (int k = 0; k < FLY; k++) {
      const int s = s0 + k * AT_ONCE + part;
      if (s < a.n_split) v[k] = *(const p8*)(src + s * split_stride * DV);
    }
  };
  fetch(0);
  const float my = lane < a.n_split ? a.lse_part[part_row + lane * split_stride] : -INFINITY;   // (at most 64 splits)
  float mx = my;
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) mx = fmaxf(mx, __shfl_xor(mx, d, 64));
  const float e = my == -INFINITY ? 0.f : __expf(my - mx);   // (a split without keys, or a row without any: zeros)
  float tot = e;
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) tot += __shfl_xor(tot, d, 64);
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < a.n_split; s0 += FLY * AT_ONCE) {
    if (s0 > 0) fetch(s0);
#pragma unroll
    for (int k = 0; k < FLY; k++) {
      const int s = s0 + k * AT_ONCE + part;
      const float w = __shfl(e, s & 63, 64);
      if (s < a.n_split) {   // (a weight of 0 too: every split has written its rows, and 0 x NaN is to stay NaN)
#pragma unroll
        for (int i = 0; i < 8; i++) acc[i] += w * (float)v[k][i];
      }
    }
  }
#pragma unroll
  for (int d = LPR; d < 64; d *= 2)
#pragma unroll
    for (int i = 0; i < 8; i++) acc[i] += __shfl_xor(acc[i], d, 64);
  // (only a row without any key has a sum of exactly 0; one that is NaN makes the row and its scale NaN, as the unsplit kernel does)
  const float inv = tot == 0.f ? 0.f : 1.f / tot;
  if (part == 0) {
    x8 w;
#pragma unroll
    for (int i = 0; i < 8; i++) w[i] = (T)(acc[i] * inv);
    *(x8*)((T*)a.o + (int64_t)b * a.osb + (int64_t)m * a.oss + (int64_t)h * a.osh + col) = w;
  }
  if (a.row_scale && lane == 0) a.row_scale[row] = tot == 0.f ? -INFINITY : mx + __logf(tot);
}

// the one-wave workgroups that run side by side on 256 CUs
static int64_t decode_slots(int dqk, int dv) {
  const int per_cu = (160 * 1024) / (2 * 32 * (pad_width(dqk) + dv) * 2);
  return (int64_t)(per_cu > 4 ? 4 : per_cu) * 256;
}

// Rounding the partial results to the tensor dtype in front of the merge adds a fifth to the error of the output (300 keys, bf16:
// 2.3e-3 of it unsplit, 2.2e-3 split with fp32 partial results, 2.8e-3 with bf16).  They are fp32 where the call could as well
// run unsplit: a cache of at most 15 tiles, or (batch, head) pairs that take more than half of the slots by themselves.  Between
// the few pairs of a long cache they are 16-bit, as the reference's Output_partial is (mla_decode_tl.py:160).
bool attn_decode_partials_f32(int B, int H, int Skv, int dqk, int dv) {
  return Skv <= 15 * 32 || 2 * (int64_t)B * H > decode_slots(dqk, dv);
}

// Decode shapes: at most 32 query rows per (batch, head), softmax, no structural mask.  A one-wave workgroup takes one
// (batch, head, kv split); a CU holds four of them, or as many as their two tile stages fit into its 160 KB of LDS.  The
// split count is the one with the shortest schedule, in microseconds: rounds of resident workgroups x (3 for a workgroup's
// beginning and end + its tiles of 32 keys at 2.3 each, what a tile takes on a stream from HBM; unsplit, with four waves
// to begin and end it, 1), put together with the time that the whole cache takes to stream in (as the root of their squares:
// the closer the two, the longer they are in each other's way), plus the merge: 3.5 and the partial results' way through memory.  Every split gets at least two tiles.
// B1 H32 Hkv8 KV1000: 16 splits, 10.2 us the call; with 4 (at least 8 tiles a split) 15.9.
int attn_decode_splits(int family, bool causal, int B, int H, int Sq, int Skv, int dqk, int dv) {
  if (family != WF_SOFTMAX || causal || Sq > 32) return 1;
  if (!((dqk == 128 && dv == 128) || (dqk == 64 && dv == 64) || (dqk == 128 && dv == 256) || (dqk == 256 && dv == 256) || (dqk == 192 && dv == 128))) return 1;
  const int64_t tiles = ((int64_t)Skv + 31) / 32, groups = (int64_t)B * H, slots = decode_slots(dqk, dv);
  const int part_bytes = attn_decode_partials_f32(B, H, Skv, dqk, dv) ? 4 : 2;
  const double stream_us = (double)groups * (double)Skv * (dqk + dv) * 2 / 5.5e6, part_us = (double)groups * Sq * dv * part_bytes * 1.5 / 5.5e6;
  int best = 1;
  double best_us = 0;
  for (int n = 1; n <= 64 && (n == 1 || 2 * n <= tiles); n++) {
    const int64_t per = (tiles + n - 1) / n;
    if (n > 1 && (tiles + per - 1) / per != n) continue;   // (some of the splits would be empty)
    const double run = (double)((groups * n + slots - 1) / slots) * ((n > 1 ? 3 : 1) + (double)per * 2.3);
    const double us = std::sqrt(run * run + stream_us * stream_us) + (n > 1 ? 3.5 + n * part_us : 0);
    if (n == 1 || us < best_us) {
      best_us = us;
      best = n;
    }
  }
  return best;
}

// The tile DMA of attn_wide_fwd_kernel addresses a tile's 32 rows with 32-bit byte offsets from its first row.
static constexpr int64_t kWideRowStride = (int64_t)1 << 26;

// Prefill calls whose workgroups of 128 (or 256: attn_fwd.hip) query rows are too few to keep the chip busy: a row block's tiles
// are then walked by several streams side by side (KVS of attn_wide_fwd_kernel), or the row blocks are smaller.  A step of a
// stream is a serial chain of about 0.78 us at 128 / 128 whatever else the CU does, 1.0 with a second wave on the SIMD, so the
// cut is the one with the shortest schedule in microseconds: the longest workgroup, or all of them over the slots where that is
// more.  The constants are fitted to all cuts' times at 354 shapes (64/64, 128/128, 192/128; 4 to 128 heads of 64 to 4096 rows,
// causal and not): the choice costs 0.9 % over the best of the cuts that it may take on average, 14 % at the worst.  (The streams may be
// taken only below the line drawn in the code; at the line, B1 H16 S4096 128/128 causal, that costs 19 %: 99 us, 83 with streams.)
// 128 / 256 is always row blocks of 128: the persistent kernel, which takes the value columns in two halves, lost at every size
// once the general kernel had its registers to itself (B1 H16 S300 28 us and 14.5, B2 H32 S1653 causal 139 and 84, B8 H32 S4096 2087
// and 1736, without a mask 3710 and 2988); it is left with the rows that are too far apart for the general kernel.
AttnCut attn_prefill_cut(const AttnArgs& a, int family, bool causal, int dqk, int dv) {
  if (family == WF_RETENTION || a.kv_lens || a.o_part || (a.kv_block_mask && !a.kbm_by_query_head)) return AttnCut::kRows128;
  const bool plain = !a.kv_block_mask && !a.elem_mask && !a.add && !a.slope_q && !a.slope_kv && !(a.softcap > 0.f);
  const bool persistent = plain && dqk == 128 && (dv == 128 || (dv == 256 && a.Sq >= 256));
  if (persistent && (a.kss >= kWideRowStride || a.vss >= kWideRowStride)) return AttnCut::kPersistent;   // (the other cuts would refuse them)
  const bool small = dqk + dv <= 128;
  const double step_alone = small ? 0.65 : dqk == 192 ? 1.15 : 0.78, step_two = small ? 0.81 : dqk == 192 ? 1.35 : 1.0;
  const int64_t bh = (int64_t)a.B * a.H, tiles = ((int64_t)a.Skv + 31) / 32;
  const bool half = causal || a.kv_block_mask || a.elem_mask;   // (what a mask keeps is not known here: taken as a causal one)
  AttnCut best = AttnCut::kRows128;
  double best_us = 1e30;
  auto consider = [&](AttnCut cut, int nw, int kvs, double fixed) {
    const int64_t blocks = ((int64_t)a.Sq + 32 * nw - 1) / (32 * nw), n = bh * blocks;
    // (64 / 64: the LDS of six streams; 192 / 128: of two)
    const int64_t slots = dqk == 192 && kvs > 1 ? 256 : (small ? 768 : 512) * 4 / (nw * kvs);
    const double step = nw * kvs == 4 && n <= 256 ? step_alone : step_two, longest = (double)((tiles + kvs - 1) / kvs);
    const double mean = half ? longest * (double)(blocks + 1) / (double)(2 * blocks) : longest;
    // (one workgroup to a CU, all of a weight: whole rounds)
    const double rounds = dqk == 192 && kvs > 1 && !causal ? (double)((n + slots - 1) / slots) : 0, part = 1.15 * (double)n / (double)slots;
    const double one = fixed + longest * step, all = (fixed + mean * step) * (rounds > part ? rounds : part), us = one > all ? one : all;
    if (us < best_us) {
      best_us = us;
      best = cut;
    }
  };
  const bool sizes = (dqk == 64 && dv == 64) || (dqk == 128 && dv == 128) || (dqk == 192 && dv == 128);
  consider(AttnCut::kRows128, 4, 1, 4.9);
  // (only where row blocks of 128 leave slots empty.  With batch x heads in the rule, a row's sums, and so its last bits, may be formed
  // in another order in a batch than in a call of its own: at one block a slot too, an entry of 32 heads and 2048 rows would be, and the
  // calls beyond 4 GiB are compared to the bit with those of their entries)
  if (sizes && bh * (((int64_t)a.Sq + 127) / 128) < (small ? 768 : 512)) {
    consider(AttnCut::kStreams4x2, 4, 2, 8.9);
    if (dqk <= 128) consider(AttnCut::kStreams2x4, 2, 4, 7.3);
    consider(AttnCut::kStreams2x2, 2, 2, 5.5);
  }
  if (persistent && dv == 128) {
    // the persistent kernel: rounds of row blocks of 256 (under a causal mask, pairs of them), 32 keys in 0.64 us, 0.92 once all
    // CUs take part
    const int64_t blocks = ((int64_t)a.Sq + 255) / 256, units = bh * (causal ? (blocks + 1) / 2 : blocks);
    const double steps = causal && blocks > 1 ? (double)(8 * blocks + 8) : (double)tiles;
    const double busy = units <= 128 ? 0.0 : units >= 256 ? 1.0 : (double)(units - 128) / 128.0;
    const double us = 5.3 + (double)((units + 255) / 256) * (3.1 + (steps < 2 * tiles ? steps : 2 * tiles) * (0.64 + 0.28 * busy));
    if (us < best_us) best = AttnCut::kPersistent;
  }
  return best;
}

template <typename T, int DQK, int DV>
static int wide_family(const AttnArgs& a, int family, bool causal, hipStream_t stream) {
  switch (family) {
    case WF_SOFTMAX:
      if constexpr (DV <= 256) {
        if (!causal && a.Sq <= 32 && a.o_part) {   // decode
          if (const int rc = launch_wide<T, DQK, DV, WF_SOFTMAX, false, 1>(a, stream)) return rc;
          if (a.n_split > 1) {
            const int64_t rows = (int64_t)a.B * a.H * a.Sq;
            const dim3 grid((unsigned)((rows + 3) / 4));
            if (a.part_f32) hipLaunchKernelGGL((attn_split_combine_kernel<T, float, DV>), grid, dim3(256), 0, stream, a);
            else hipLaunchKernelGGL((attn_split_combine_kernel<T, T, DV>), grid, dim3(256), 0, stream, a);
          }
          return launch_status();
        }
      }
      return causal ? launch_wide<T, DQK, DV, WF_SOFTMAX, true>(a, stream) : launch_wide<T, DQK, DV, WF_SOFTMAX, false>(a, stream);
    case WF_SIGMOID:
      return causal ? launch_wide<T, DQK, DV, WF_SIGMOID, true>(a, stream) : launch_wide<T, DQK, DV, WF_SIGMOID, false>(a, stream);
    case WF_RELU:
      return causal ? launch_wide<T, DQK, DV, WF_RELU, true>(a, stream) : launch_wide<T, DQK, DV, WF_RELU, false>(a, stream);
  }
  return -2;
}

template <typename T>
static int wide_dims(const AttnArgs& a, int family, bool causal, int dqk, int dv, hipStream_t stream) {
  if (family == WF_RETENTION) {
    if (dqk == 256 && dv == 512) return retention_pair_fwd_dispatch(a, causal, std::is_same<T, __bf16>::value, stream);   // retention_fwd.hip
#define MA_RET_FWD(DQ, DVV) \
  if (dqk == DQ && dv == DVV) return causal ? launch_wide<T, DQ, DVV, WF_RETENTION, true>(a, stream) : launch_wide<T, DQ, DVV, WF_RETENTION, false>(a, stream);
    MA_RET_FWD(128, 128)
    MA_RET_FWD(64, 64)
    MA_RET_FWD(128, 256)
    MA_RET_FWD(256, 256)
#undef MA_RET_FWD
    return -2;
  }
  if (dqk == 128 && dv == 128) return wide_family<T, 128, 128>(a, family, causal, stream);   // (only with kv selection: see attn_fwd_dispatch)
  if (dqk == 64 && dv == 64) return wide_family<T, 64, 64>(a, family, causal, stream);
  if (dqk == 128 && dv == 256) return wide_family<T, 128, 256>(a, family, causal, stream);
  if (dqk == 256 && dv == 256) return wide_family<T, 256, 256>(a, family, causal, stream);
  if (dqk == 192 && dv == 128) return wide_family<T, 192, 128>(a, family, causal, stream);   // (the reference's DeepSeek-V2-Lite benchmark shape)
  if (dqk == 256 && dv == 512 && (family != WF_SOFTMAX || !(a.Sq <= 32 && a.o_part))) return wide_family<T, 256, 512>(a, family, causal, stream);
  // Softmax decode (split kv, one wave per workgroup) at 256/512: a workgroup's two tile stages would take 96 KB of LDS,
  // one wave per CU.  Given the probabilities the value columns are independent, so the two halves of V and of the
  // output go through the 256/256 decode kernel one after the other (the scores are computed twice; both launches write
  // the same row scales).
  if (dqk == 256 && dv == 512) {
    AttnArgs half = a;
    const int rc = wide_family<T, 256, 256>(half, family, causal, stream);
    if (rc != 0) return rc;
    half.v = (const T*)a.v + 256;
    half.o = (T*)a.o + 256;
    return wide_family<T, 256, 256>(half, family, causal, stream);
  }
  return -2;
}

// returns 0 ok, -1 launch failure, -2 unsupported
int attn_wide_fwd_dispatch(const AttnArgs& a, int family, bool causal, bool is_bf16, int dqk, int dv, hipStream_t stream) {
  for (int64_t row_stride : {a.kss, a.vss})
    if (row_stride < 0 || row_stride >= kWideRowStride) return -2;
  const AttnCut cut = attn_prefill_cut(a, family, causal, dqk, dv);
  if (cut == AttnCut::kStreams4x2 || cut == AttnCut::kStreams2x4 || cut == AttnCut::kStreams2x2)
    return (is_bf16 ? attn_streams_bf16 : attn_streams_fp16)(a, cut, family, causal, dqk, dv, stream);
  return is_bf16 ? wide_dims<__bf16>(a, family, causal, dqk, dv, stream) : wide_dims<_Float16>(a, family, causal, dqk, dv, stream);
}

}  // namespace ma
