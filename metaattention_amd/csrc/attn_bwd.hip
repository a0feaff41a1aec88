// Parallel attention backward: dispatch by head size to the translation units that hold the kernels (attn_bwd_kernels.h,
// instantiated per group of head sizes in attn_bwd_128.hip, attn_bwd_64.hip, attn_bwd_192.hip, attn_bwd_256.hip).
#include "attn_bwd.h"

namespace ma {

int attn_bwd_128_128(const AttnBwdArgs& a, int family, bool causal, bool is_bf16, hipStream_t stream);
int attn_bwd_64_64(const AttnBwdArgs& a, int family, bool causal, bool is_bf16, hipStream_t stream);
int attn_bwd_128_256(const AttnBwdArgs& a, int family, bool causal, bool is_bf16, hipStream_t stream);
int attn_bwd_256_256(const AttnBwdArgs& a, int family, bool causal, bool is_bf16, hipStream_t stream);
int attn_bwd_192_128(const AttnBwdArgs& a, int family, bool causal, bool is_bf16, hipStream_t stream);   // (the reference's DeepSeek-V2-Lite benchmark shape; not the retention family)
int attn_bwd_256_512(const AttnBwdArgs& a, int family, bool causal, bool is_bf16, hipStream_t stream);   // (256 / 512 is the head size of the retention operator itself, examples/retention_parallel.py)

// The kernels that make dk and dv in one launch run one workgroup per CU on items of a key block (a pair of them under a causal mask).  The number
// of runs per item is the one with the shortest schedule: rounds of workgroups x (steps of a run + a workgroup's fixed cost of
// about six steps), a step taking 1.2 us at 128 / 128, plus the partial sums' way through memory (written and read at about
// 4 TB/s) and their launch.  B2 H32 Hkv8 S2047 128/128 causal: 128 pairs of 272 steps on 256 CUs; B1 H16 Hkv4 S700
// 128/256 causal, 12 pairs: forward + backward 187 us in one run, 106 in those that this chooses.  (Steps of 0.7 and 0.9 us: within 3 % either way.)  What element-wise and tile
// masks keep is not known here: they count as half the pairs, as a causal mask does (and so get as many runs: a triangular mask
// gives a causal call's bits).
int attn_bwd_parts(const AttnBwdArgs& a, bool half, int dqk, int dv) {
  const bool fused = (dqk == 128 && dv == 128) || (dqk == 64 && dv == 64) || (dqk == 192 && dv == 128) || (dqk == 128 && dv == 256) || (dqk == 256 && dv == 256);
  if (!fused || a.add || a.slope_q || a.slope_kv || a.softcap != 0.f) return 1;
  const int cus = device_cus();
  if (cus <= 0) return 1;
  const int64_t blocks = (a.Skv + 127) / 128, tiles = (a.Sq + 31) / 32;
  const int64_t items = (half ? (blocks + 1) / 2 : blocks) * a.B * a.Hkv;
  if (items >= 4 * (int64_t)cus) return 1;
  const int64_t steps = (half && blocks > 1 ? (2 * tiles > 4 * (blocks - 1) ? 2 * tiles - 4 * (blocks - 1) : 1) : tiles) * a.kv_group;
  const double step_us = 1.2 * (dqk + dv) / 256, sum_us = 2.0 * (double)attn_bwd_part_bytes(a, 1, dqk, dv) / 4e6;
  int best = 1;
  double best_us = 0;
  if (dqk + dv <= 128) {
    // two streams a workgroup and a key block each (dkv_two_streams; beyond that rule one run): 0.64 us a tile, about 4.5 a
    // workgroup; the longest block or all of them over the CUs, in whole rounds where they weigh the same.  Backward of B1 H16 S700
    // causal, 96 blocks: 35.5 us in one run, 38 in two, 42 in three; B1 H4 S2000 causal, 64 blocks: 71.5, 62, 58, 56.5 in four, 59 in
    // six; H16 Hkv4: 180, 117, 95, 83, 78 in six.
    const bool causal = half && !a.elem_mask_t && !a.q_block_mask;
    const int64_t blocks_all = blocks * a.B * a.Hkv, most = tiles * a.kv_group;
    if (!dkv_two_streams(blocks_all, causal)) return 1;
    for (int n = 1; n <= 16 && (n == 1 || (most >= 4 * n && blocks_all * n <= 4 * (int64_t)cus)); n++) {
      const double longest = 6.5 + 0.64 * (double)((most + n - 1) / n), mean = (half ? 0.5 : 1.0) * 0.64 * (double)most / n + 4.5;
      const double rounds = causal ? (double)(blocks_all * n) / cus : (double)((blocks_all * n + cus - 1) / cus), all = 2 + mean * rounds;
      const double us = (longest > all ? longest : all) + (n > 1 ? 4 + n * sum_us : 0);
      if (n == 1 || us < best_us) {
        best_us = us;
        best = n;
      }
    }
    return best;
  }
  for (int n = 1; n <= 16 && (n == 1 || steps >= 4 * n); n++) {
    const double us = (double)((items * n + cus - 1) / cus) * ((double)((steps + n - 1) / n) + 6) * step_us + (n > 1 ? 4 + n * sum_us : 0);
    if (n == 1 || us < best_us) {
      best_us = us;
      best = n;
    }
  }
  return best;
}
size_t attn_bwd_part_bytes(const AttnBwdArgs& a, int n_parts, int dqk, int dv) {
  return (size_t)n_parts * a.B * a.Hkv * ((a.Skv + 127) / 128) * 128 * (dqk + dv) * sizeof(float);
}

// returns 0 ok, -1 launch failure, -2 unsupported
int attn_bwd_dispatch(const AttnBwdArgs& a, int family, bool causal, bool is_bf16, int dqk, int dv, hipStream_t stream) {
  // (the tile DMA addresses a tile's 32 rows with 32-bit byte offsets from its first row)
  for (int64_t row_stride : {a.qss, a.kss, a.vss, a.doss})
    if (row_stride < 0 || row_stride >= ((int64_t)1 << 26)) return -2;
  if (dqk == 128 && dv == 128) return attn_bwd_128_128(a, family, causal, is_bf16, stream);
  if (dqk == 64 && dv == 64) return attn_bwd_64_64(a, family, causal, is_bf16, stream);
  if (dqk == 128 && dv == 256) return attn_bwd_128_256(a, family, causal, is_bf16, stream);
  if (dqk == 256 && dv == 256) return attn_bwd_256_256(a, family, causal, is_bf16, stream);
  if (dqk == 192 && dv == 128) return attn_bwd_192_128(a, family, causal, is_bf16, stream);
  if (dqk == 256 && dv == 512) return attn_bwd_256_512(a, family, causal, is_bf16, stream);
  return -2;
}

}  // namespace ma
