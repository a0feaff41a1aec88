// Chunked linear / stateful attention forward (RetNet retention, Mamba2 SSD,
// gated retention) for gfx950.
//
// Replaces the three launches of LinearAttention.forward in
// attention_engine/core/template/tl_template/linear/linear_tl.py:1240-1269
// (chunk_local_cumsum :36-60, chunk_fwd_h :146-221, chunk_o :322-399) with ONE
// kernel that keeps the inter-chunk state on chip:
//
//   o_t = q_scale * q_t . sum_{s<=t} exp(G_t - G_s) k_s^T (v_s * vs_s),   G = cumsum(log_decay)
//
// Work split.  A workgroup owns one (batch, head) and a slice of 32*NW value
// columns; wave w owns 32 of them and the matching DK x 32 block of the fp32
// state, which lives in its accumulator registers for the whole sequence (the
// reference writes the state to HBM as bf16 every chunk and reads it back).  The
// sequence is walked in chunks of 32 tokens; per chunk and wave, with
// g = chunk-local cumsum of the log decay, everything is computed TRANSPOSED so
// each lane owns one token column:
//   A^T = K Q^T                      [32 x 32]
//   P^T = A^T * q_scale * exp(g_i - g_j) * vs_j * [j <= i]
//   O^T = h^T (Q^T) * exp(g_i) q_scale + V^T P^T          [32 dv x 32 tokens]
//   h   = exp(g_last) h + K^T (V * vs * exp(g_last - g))  [DK x 32 dv]
// The state accumulator of K^T V (lane = value column, rows = key dims) is,
// register for register, the A operand of h^T Q^T, so the state never moves.
// Q/K/V chunk tiles arrive by direct-to-LDS DMA with a single workgroup barrier per chunk.
//
// Where a workgroup has four waves or more and produces outputs the chunk loop is pipelined (see PIPE): P^T, which is the
// same for every wave of a head, is made once, by three waves and a chunk ahead, the chunk's scalars two chunks ahead by a
// fourth, tiles arrive two or three chunks ahead.  Vector issue bounds this loop (61 % of the cycles of a chunk at 256 / 512
// with P^T formed by every wave, the matrix pipe 23 %), so what pays is fewer vector instructions per wave: 650 -> 450 a chunk.
// 8 x 16 heads, 2048 tokens, 256 / 512: 290 -> 222 us a pass.  At that rate the clock gives way (2.1 -> 1.65 GHz with random
// operands): 9500 -> 6000 clocks a chunk.
//
// Heads that share their q and k head (Mamba2: one B/C group for all heads) can be
// grouped HG to a workgroup, which then shares the Q/K tiles in LDS.
//
// Segments.  One (batch, head) is a serial chain of T/32 chunks; when batch x heads
// is too small to give every SIMD several waves, the sequence is cut into segments
// that run side by side: a first launch (MODE 1) computes, for every segment but the
// last, the state it ends in when entered with a zero state and its total log decay;
// the second launch (MODE 2) enters segment s with
//   sum_{s' < s} exp(sum_{s' < s'' < s} D[s'']) h_local[s']
// (states are exchanged in accumulator-register order, fp32, through the workspace; with many
// segments a launch between the two, linear_states_kernel, forms the entering states once)
// and produces the outputs.  MODE 0 is the single pass.
#include "linear_fwd.h"

#include <type_traits>

namespace ma {

namespace {
constexpr int L = 32;  // tokens per chunk
// What the waves of a head share in the pipelined loop.  P^T of two chunks, as the B operand of V^T P^T: slice 0 64 lanes x 16 bytes,
// slice 1 its 32 lanes of tokens 16..31.  Scalars of three chunks: running log2 decay and value scale x q_scale of the tokens, factors
// of the state update's rows and of the tokens' inter-chunk term, decay of the chunk.
constexpr int kPipeP1 = 1024, kPipeP = 1536, kScalG = 0, kScalV = 4 * L, kScalW = 8 * L, kScalE = 12 * L, kScalD = 16 * L, kPipeScal = kScalD + 16;
constexpr int pipe_shared(int heads) { return heads * (2 * kPipeP + 3 * kPipeScal) + 16; }     // (the last 16 bytes: zeros)

template <int CTRL>
__device__ __forceinline__ float dpp_f32(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}

__device__ __forceinline__ const LinArgs& one_scan(const LinArgs& a, int) { return a; }
__device__ __forceinline__ const LinArgs& one_scan(const LinScans& a, int i) { return a.s[i]; }

template <typename X8>
__device__ __forceinline__ X8 scale_bf16x8(X8 v, const float (&w)[8]) {
  X8 r;
#pragma unroll
  for (int i = 0; i < 8; i++) r[i] = (__bf16)((float)v[i] * w[i]);
  return r;
}

// The natural logarithm as exactly as the operators that take it in front of the kernel have it.  (-ffast-math makes logf the
// hardware's log2 times ln 2, one rounded product; here ln 2 is hi + lo and the product's rounding error comes from a fused
// multiply-add, so that what is left is the error of log2 and one rounding.  The asm statements keep the compiler from reordering
// the sums as if they were exact.)
__device__ __forceinline__ float log_f32(float x) {
  constexpr double kLn2 = 0.693147180559945309417;
  constexpr float hi = (float)kLn2, lo = (float)(kLn2 - (double)hi);
  const bool subnormal = x < 0x1p-126f;      // (log2 would take it for 0)
  const float y = fast_log2(subnormal ? x * 0x1p32f : x);
  float p = y * hi;
  asm("" : "+v"(p));
  float r = p + __builtin_fmaf(y, lo, __builtin_fmaf(y, hi, -p));
  asm("" : "+v"(r));
  r = __builtin_fabsf(y) < __builtin_inff() ? r : y;      // (of 0 and infinity; NaN)
  asm("" : "+v"(r));
  float shifted = subnormal ? r - (float)(32 * kLn2) : r;
  asm("" : "+v"(shifted));
  return shifted;
}
}  // namespace

// The pipelined chunk loop (P^T shared by the waves of a head and made one chunk ahead): workgroups of four waves or more that
// produce outputs.
template <int NWH, int HG, int MODE>
constexpr bool pipelined() { return NWH * HG >= 4 && MODE != 1; }
// ... and where a workgroup has four state waves of at most 128 key dims by four waves of their own (`helpers`), one beside each state
// wave of a SIMD, which write the outputs too.  A chunk of a state wave alone takes 1900 clocks, that of its helper 2300; without them
// P^T, scalars and outputs stand in the state waves' chain (4700 clocks) and only further workgroups on the CU, with sequence
// segments to supply them, hide it.  8 x 64 heads sharing q and k, 2048 tokens, 128 / 64: three workgroups a CU in three segments
// 127 us, one with helpers in a single pass 87 us; 8 x 16 heads, 128 / 128, forward and backward 386 -> 363 us.
template <int DK, int NWH, int HG, int MODE>
constexpr int helpers() { return pipelined<NWH, HG, MODE>() && NWH * HG == 4 && DK <= 128 ? 4 : 0; }
// waves of a workgroup
template <int DK, int NWH, int HG, int MODE>
constexpr int workgroup_waves() { return NWH * HG + helpers<DK, NWH, HG, MODE>(); }
// minimum waves per SIMD asked of the register allocator: the eight waves of a workgroup need two
template <int DK, int NWH, int HG, int MODE>
constexpr int min_waves_per_simd() { return HG > 1 && MODE == 1 ? 3 : NWH == 4 && DK > 128 ? 1 : 2; }

// GEN: the operands' general addressing (reversed time, row strides, v head broadcast) of LinArgs; without it the
// addressing is the plain one, with compile-time row sizes.
// GEN 1: one scan, 2: the scans of a LinScans, one blockIdx.y each (with the arguments behind an index the single scan takes 1 %
// longer: B8 H16 T2048 256 / 512 forward + backward 1516, 1530 us).
// GEN 3, 4: like 1 and 2, of scans that leave or take in partial results (o_part, o_add): instantiations of their own, because the code for
// them (and their earlier tile loads) cost the others 1 - 2 %: 8 x 8 heads, 256 / 512, forward + backward, 129 tokens 93.6 -> 92.2 us, 300
// tokens 140.2 -> 137.4.
constexpr bool gen_scans(int gen) { return gen == 2 || gen == 4; }
template <int DK, int NWH, int HG, int MODE, int GEN = 0>
__global__ __launch_bounds__((64 * workgroup_waves<DK, NWH, HG, MODE>()), (min_waves_per_simd<DK, NWH, HG, MODE>())) void linear_fwd_kernel(const std::conditional_t<gen_scans(GEN), LinScans, LinArgs> all) {
  const LinArgs& a = one_scan(all, gen_scans(GEN) ? (int)blockIdx.y : 0);
  constexpr int NW = NWH * HG;
  constexpr bool PIPE = pipelined<NWH, HG, MODE>();
  constexpr bool HELP = helpers<DK, NWH, HG, MODE>() > 0;
  constexpr int NT = 64 * workgroup_waves<DK, NWH, HG, MODE>();
  static_assert(!HELP || NWH * HG == 4, "helper w serves state wave w");
  constexpr bool ALIAS_OST = HG > 1 || PIPE;     // output staging block inside the wave's own (already consumed) V columns
  using T = __bf16;
  using E = Elem<T>;
  using x8 = typename E::x8;
  using x4 = typename E::x4;
  constexpr int DVS = 32 * NW;
  constexpr int RBQ = DK * 2, RBV = DVS * 2;       // row bytes
  constexpr int CPRQ = DK / 8, CPRV = DVS / 8;     // 16-byte chunks per row
  constexpr int QT = L * RBQ, VT = L * RBV;
  constexpr int STAGE = 2 * QT + VT;
  constexpr int KB = DK / 32;                      // 32-row blocks of the state
  constexpr int OROW = 64 + 16;                    // padded row of the per-wave output staging block
  constexpr int SCAL_BYTES = 3 * L * 4;            // per-wave g / pv*q_scale / w
  constexpr int NIQ = QT / 1024, NIV = VT / 1024;  // DMA instructions per tile
  static_assert(CPRQ >= 16, "DK < 128 needs its own Q/K swizzle");
  extern __shared__ __align__(16) char smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(MA_LDS char*)smem;
  const int tid = threadIdx.x, lane = tid & 63, wave_id = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool helper = HELP && wave_id >= NW;
  const int wave = helper ? wave_id - NW : wave_id;       // (a helper's: the state wave whose outputs it writes)
  const int r0 = lane & 31;
  constexpr int NST = HELP ? 4 : PIPE ? 3 : 2;             // stages of chunk tiles
  const uint32_t lds_scal = lds0 + NST * STAGE + wave * SCAL_BYTES;                                     // (unused with PIPE)
  const uint32_t lds_ost = lds0 + NST * STAGE + NW * SCAL_BYTES + wave * (L * OROW);   // (unused with ALIAS_OST)
  const uint32_t lds_p = lds0 + NST * STAGE, lds_scalars = lds_p + HG * 2 * kPipeP, lds_zero = lds_scalars + HG * 3 * kPipeScal;   // PIPE: [slot][head] (see kPipeP)

  // workgroup -> (head group, value slice, segment); the workgroups of one head group share
  // id % 8 (one XCD, shared L2)
  const int n_seg = MODE == 0 ? 1 : (MODE == 1 ? a.nseg - 1 : a.nseg);
  const int BG = a.bg_n > 0 ? a.bg_n : a.B * a.H / HG;     // head groups of this launch
  int bg, dvb, seg, piece = 0;      // (pieces of a contraction side by side: see LinArgs)
  {
    int slot = blockIdx.x;
    if (GEN) {
      const int of_piece = BG * a.dv_blocks * n_seg;
      piece = slot / of_piece;
      slot -= piece * of_piece;
      if (piece >= (a.n_pieces > 1 ? a.n_pieces : 1)) return;    // (the launch is as wide as its largest scan)
    }
    if ((BG & 7) == 0) {
      const int xcd = slot & 7;
      slot >>= 3;
      seg = slot % n_seg;
      slot /= n_seg;
      dvb = slot % a.dv_blocks;
      bg = (slot / a.dv_blocks) * 8 + xcd;
    } else {
      seg = slot % n_seg;
      slot /= n_seg;
      dvb = slot % a.dv_blocks;
      bg = slot / a.dv_blocks;
    }
  }
  const int bg_local = bg;      // (indexes the launch's workspace)
  bg += a.bg0;
  const int hl = wave / NWH;                      // head of the group this wave works for
  const int bh0 = bg * HG, bh = bh0 + hl;
  const int b = bh0 / a.H, h0 = bh0 % a.H;        // (HG divides H, and the heads of a group share hq and hk)
  const int hq = h0 / (a.H / a.Hq), hk = h0 / (a.H / a.Hk);
  const int Tn = a.T;
  const bool rev = GEN && a.rev != 0, rev_o = GEN && a.rev_o != 0;
  const int64_t q_rb = GEN ? a.q_row * 2 : (int64_t)RBQ, k_rb = GEN ? a.k_row * 2 : (int64_t)RBQ;   // bytes between an operand's rows in memory
  const int64_t v_row_bytes = (GEN ? a.v_row : (int64_t)a.Dv) * 2;
  const int64_t bh0_v = GEN ? (int64_t)b * a.Hv + h0 / (a.H / a.Hv) : (int64_t)bh0;
  const char* qb = (const char*)a.q + ((int64_t)(b * a.Hq + hq) * Tn) * q_rb + (int64_t)piece * a.piece_qk * 2;
  const char* kb = (const char*)a.k + ((int64_t)(b * a.Hk + hk) * Tn) * k_rb + (int64_t)piece * a.piece_qk * 2;
  const char* vb = (const char*)a.v + bh0_v * Tn * v_row_bytes + (int64_t)dvb * (32 * NWH) * 2;
  const int64_t v_head_bytes = (int64_t)Tn * v_row_bytes;
  T* ob = (T*)a.o + (int64_t)bh * Tn * a.Dv + dvb * (32 * NWH) + 32 * (wave % NWH);
  const float* ldp = a.log_decay + (int64_t)bh * Tn;
  const int64_t tok0 = (int64_t)bh * Tn;
  // A token's value scale, and its log decay from what log_decay holds.  As passes of their own in front of this kernel the
  // conversion of a bf16 scale and the product with a head's factor were 9.8 of 99 us at 8 x 64 heads, 2048 tokens, 128 / 64.
  // (Not with general addressing: the code alone cost the two-head kernels of a 64-wide key 2 %, 42.9 -> 44.1 us at 8 x 16 heads,
  // 1024 tokens.)
  // (The scale is loaded as it is and converted where it is used: a conversion behind the load, in a branch, waits for it there,
  // 12 us of that pass.)
  auto v_scale_at = [&](int64_t i) {
    return GEN == 0 && a.v_scale_bf16 ? __builtin_bit_cast(float, (uint32_t)((const uint16_t*)a.v_scale)[i]) : a.v_scale[i];
  };
  auto v_scale_of = [&](float x) { return GEN == 0 && a.v_scale_bf16 ? __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) << 16) : x; };
  auto log_decay_of = [&](float x, float head_factor) {
    if (GEN == 0 && a.decay_log) x = log_f32(x);
    return GEN == 0 && a.decay_head ? x * head_factor : x;
  };
  const int n_chunks_all = (Tn + L - 1) / L;
  const int c_begin = MODE == 0 ? 0 : seg * a.seg_chunks;
  const int c_end = MODE == 0 ? n_chunks_all : min(c_begin + a.seg_chunks, n_chunks_all);
  // this wave's block of the exchanged states: [segment][wave][KB*16 registers][64 lanes]
  float* ws_mine = nullptr;
  if (MODE != 0)
    ws_mine = a.ws_state + (((((int64_t)piece * BG + bg_local) * a.dv_blocks + dvb) * (a.nseg - 1)) * NW + wave) * (int64_t)(KB * 16 * 64) + lane;
  constexpr int64_t WS_SEG = (int64_t)NW * KB * 16 * 64;

  // ---- DMA of one chunk: each instruction moves 1 KB (1024/row_bytes tile rows); lane i fetches
  //      the 16-byte chunk that belongs at physical position i of that KB.
  //      (Spreading a chunk's instructions over the chunk's phases instead of issuing them together behind the
  //      barrier was measured: no gain at the RetNet shape, 5 % slower at the Mamba2 shape.)
  const uint32_t qk_chunks = GEN && a.qk_cols > 0 ? (uint32_t)a.qk_cols / 8 : (uint32_t)CPRQ;   // 16-byte chunks of a q / k row that exist
  // (columns beyond the operand's are zeros: the 16- and 32-wide slices of the contraction that hold nothing else are skipped)
  const int qk_used = GEN && a.qk_cols > 0 ? a.qk_cols : DK;
  if (GEN && qk_chunks < (uint32_t)CPRQ) {
    // the Q and K tiles of all stages start as zeros: the missing columns are never written
    for (uint32_t off = (uint32_t)tid * 16; off < (uint32_t)(2 * QT); off += NT * 16)
#pragma unroll
      for (int st = 0; st < NST; st++) lds_write<u32x4>(lds0 + st * STAGE + off, u32x4{0u, 0u, 0u, 0u});
    __syncthreads();
  }
  // a partial chunk: rows beyond the sequence are clamped to its last row
  auto issue_rows = [&](int t0, uint32_t base) {
    constexpr int NQK = MODE == 1 ? NIQ : 2 * NIQ;      // (the state-only pass needs no Q)
#pragma unroll 1
    for (int ii = wave; ii < NQK + NIV; ii += NW) {
      if (ii < NQK) {
        const int which = MODE == 1 ? 1 : ii >= NIQ, i2 = (MODE != 1 && which) ? ii - NIQ : ii;
        const int row = i2 * (1024 / RBQ) + lane / CPRQ, c = lane % CPRQ;
        const int tpos = min(t0 + row, Tn - 1), trow = rev ? Tn - 1 - tpos : tpos;
        const uint32_t lc = (uint32_t)(c ^ swz_tile<CPRQ>(row));
        const char* src = (which ? kb + (int64_t)trow * k_rb : qb + (int64_t)trow * q_rb) + (lc << 4);
        if (!GEN || lc < qk_chunks) dma16(src, base + which * QT + i2 * 1024);
      } else {
        const int i2 = ii - NQK;
        const int row = i2 * (1024 / RBV) + lane / CPRV, c = lane % CPRV;
        const int tpos = min(t0 + row, Tn - 1), trow = rev ? Tn - 1 - tpos : tpos;
        const int lc = c ^ swz_tile<CPRV>(row);          // logical 16-byte chunk: head lc / (4 NWH), then its columns
        const char* src = vb + (int64_t)trow * v_row_bytes + ((lc % (4 * NWH)) << 4);
        if (HG > 1) src += (lc / (4 * NWH)) * v_head_bytes;
        dma16(src, base + 2 * QT + i2 * 1024);
      }
    }
  };
  auto issue_chunk = [&](int t0, int buf) {
    const uint32_t base = lds0 + buf * STAGE;
    constexpr int NQK = MODE == 1 ? NIQ : 2 * NIQ;      // (the state-only pass needs no Q)
    constexpr int RQ = 1024 / RBQ, RV = 1024 / RBV;     // tile rows per instruction
    static_assert(HG == 1 || RV % 4 == 0, "the V swizzle of an instruction's first row must stay inside a head's columns");
    if (t0 + L <= Tn && v_head_bytes < ((int64_t)1 << 31)) {
      // Whole chunk: no row clamping, so an instruction's source is a wave-uniform base (SGPRs) plus a
      // 32-bit lane offset.  The swizzle is a bit permutation of the row index, so it splits into the
      // lane's part (row within the instruction) and the instruction's part (its first row), and since row
      // offsets are multiples of the row size the instruction's part is one XOR on the finished lane offset.
      int ln2 = lane;
      asm volatile("" : "+v"(ln2));   // rebuilt per chunk: kept live across the chunk these would cost registers
      const int lrq = ln2 / CPRQ, lrv = ln2 / CPRV;
      // (reversed time: an instruction's rows lie behind each other in memory the other way round; its base is then
      // its LAST row's address, the lowest, and the lane's row offset counts from there)
      // With the general addressing a row distance need not be a multiple of the tile's row size, so the instruction's
      // part of the swizzle goes onto the chunk index before the row offset is added; chunks beyond the operand's columns
      // are not loaded (their LDS stays zero).
      const uint32_t cq = (uint32_t)((ln2 % CPRQ) ^ swz_tile<CPRQ>(lrq));
      const uint32_t aq = (uint32_t)(rev ? RQ - 1 - lrq : lrq) * (uint32_t)q_rb + (GEN ? 0u : cq << 4);
      const uint32_t ak = GEN ? (uint32_t)(rev ? RQ - 1 - lrq : lrq) * (uint32_t)k_rb : aq;
      const uint32_t lc0 = (ln2 % CPRV) ^ swz_tile<CPRV>(lrv);       // logical chunk: head lc / (4 NWH), then its columns
      uint32_t av = (uint32_t)(rev ? RV - 1 - lrv : lrv) * (uint32_t)v_row_bytes + ((lc0 % (4 * NWH)) << 4);
      if (HG > 1) av += (lc0 / (4 * NWH)) * (uint32_t)v_head_bytes;
#pragma unroll (DK <= 128 ? 16 : 1)   // (with a 256-wide key the state leaves no registers for an unrolled burst)
      for (int it = 0; it < (NQK + NIV + NW - 1) / NW; it++) {
        const int ii = wave + NW * it;
        if ((NQK + NIV) % NW != 0 && ii >= NQK + NIV) break;
        if (ii < NQK) {
          const int which = MODE == 1 ? 1 : ii >= NIQ, i2 = (MODE != 1 && which) ? ii - NIQ : ii;
          const int64_t row0 = rev ? Tn - t0 - (i2 + 1) * RQ : t0 + i2 * RQ;
          const char* sb = (which ? kb + row0 * k_rb : qb + row0 * q_rb);
          if constexpr (GEN) {
            const uint32_t lc = cq ^ (uint32_t)swz_tile<CPRQ>(i2 * RQ);
            if (lc < qk_chunks) dma16_so(sb, (which ? ak : aq) + (lc << 4), base + which * QT + i2 * 1024);
          } else {
            dma16_so(sb, aq ^ (uint32_t)(swz_tile<CPRQ>(i2 * RQ) << 4), base + which * QT + i2 * 1024);
          }
        } else {
          const int i2 = ii - NQK;
          const int64_t row0 = rev ? Tn - t0 - (i2 + 1) * RV : t0 + i2 * RV;
          const char* sb = vb + row0 * v_row_bytes;
          dma16_so(sb, av ^ (uint32_t)(swz_tile<CPRV>(i2 * RV) << 4), base + 2 * QT + i2 * 1024);
        }
      }
      return;
    }
    issue_rows(t0, base);
  };

  f32x16 hst[KB];
#pragma unroll
  for (int i = 0; i < KB; i++)
#pragma unroll
    for (int j = 0; j < 16; j++) hst[i][j] = 0.f;

  // scalars of the chunk about to be processed (loaded one chunk ahead)
  const int ti = r0;
  float ld_next = 0.f, vs_next = 1.f;
  if (!PIPE && c_begin * L + ti < Tn) {
    ld_next = ldp[c_begin * L + ti];
    if (a.v_scale) vs_next = v_scale_at(tok0 + c_begin * L + ti);
  }
  if (!helper) {
    if (c_begin < c_end) issue_chunk(c_begin * L, 0);
    if (PIPE && c_begin + 1 < c_end) issue_chunk((c_begin + 1) * L, 1);
    if (HELP && c_begin + 2 < c_end) issue_chunk((c_begin + 2) * L, 2);
  }

  if (MODE == 2 && !helper && seg > 0 && a.ws_entering) {
    // entering state, formed by linear_states_kernel
    const float* src = ws_mine + (seg - 1) * WS_SEG;
#pragma unroll
    for (int i = 0; i < KB; i++)
#pragma unroll
      for (int j = 0; j < 16; j++) hst[i][j] = src[(i * 16 + j) * 64];
  } else if (MODE == 2 && !helper && seg > 0) {
    // entering state: the local end states of the earlier segments, each decayed by the segments between
    const float* dec = a.ws_decay + (int64_t)(bh - a.bg0 * HG) * (a.nseg - 1);
    float acc_log = 0.f;
    for (int sp = seg - 1; sp >= 0; sp--) {
      const float coef = fast_exp2(acc_log * kLog2e), d = dec[sp];   // (d: requested with the state, not behind it)
      const float* src = ws_mine + sp * WS_SEG;
      // 64 loads in flight at a time, held apart from the sums: left alone the compiler may wait for each load before it asks
      // for the next (five segments at 256 / 512: 22 -> 132 us)
      constexpr int NB = KB < 4 ? KB : 4;
#pragma unroll
      for (int i0 = 0; i0 < KB; i0 += NB) {
        float x[NB][16];
#pragma unroll
        for (int i = 0; i < NB; i++)
#pragma unroll
          for (int j = 0; j < 16; j++) x[i][j] = src[((i0 + i) * 16 + j) * 64];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NB; i++)
#pragma unroll
          for (int j = 0; j < 16; j++) hst[i0 + i][j] += coef * x[i][j];
      }
      acc_log += d;
    }
  }
  float seg_log = 0.f;   // MODE 1: total log decay of the segment

  auto write_out = [&](const f32x16& o, int t0, uint32_t vbase) {
    // ---- write this wave's [32 tokens x 32 columns] block: stage (wave private), then 16-byte row pieces.
    //      With ALIAS_OST the staging block is the wave's own 4 chunks per row of the V tile just consumed
    //      (only this wave reads them, and the next DMA into this buffer is issued behind the next barrier).
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int r = ln & 31, g = ln >> 5;
    if (MODE != 1 && a.out_f32) {
      // fp32 outputs (used by the backward pass, whose decay gradient is a difference of sums over these
      // values): the same staging block, 16 columns at a time
      const int sw_r = swz_tile<CPRV>(r);
      float* ob32 = (float*)a.o + (int64_t)piece * a.piece_o + (int64_t)bh * Tn * a.Dv + dvb * (32 * NWH) + 32 * (wave % NWH);
#pragma unroll
      for (int half = 0; half < 2; half++) {
#pragma unroll
        for (int q2 = 0; q2 < 2; q2++) {
          const int q4 = 2 * half + q2;
          f32x4 w;
#pragma unroll
          for (int i = 0; i < 4; i++)
            w[i] = o[4 * q4 + i];
          if (ALIAS_OST) lds_write<f32x4>(vbase + r * RBV + (uint32_t)(((4 * wave + 2 * q2 + g) ^ sw_r) << 4), w);
          else lds_write<f32x4>(lds_ost + r * OROW + (8 * q2 + 4 * g) * 4, w);
        }
#pragma unroll
        for (int it = 0; it < 2; it++) {
          const int ci = ln + 64 * it, row = ci >> 2, cc = ci & 3;
          const u32x4 w = ALIAS_OST ? lds_read<u32x4>(vbase + row * RBV + (uint32_t)(((4 * wave + cc) ^ swz_tile<CPRV>(row)) << 4))
                                    : lds_read<u32x4>(lds_ost + row * OROW + cc * 16);
          if (t0 + row < Tn) {
            f32x4* dst = (f32x4*)(ob32 + (int64_t)(rev_o ? Tn - 1 - (t0 + row) : t0 + row) * a.Dv + 16 * half + cc * 4);
            f32x4 val = __builtin_bit_cast(f32x4, w);
            if (a.out_f32 == 2) val += *dst;   // (a contraction cut into pieces: the pieces' outputs add up)
            *dst = val;
          }
        }
      }
    } else if constexpr (MODE != 1) {
      const int sw_r = swz_tile<CPRV>(r);
#pragma unroll
      for (int q4 = 0; q4 < 4; q4++) {
        x4 w;
#pragma unroll
        for (int i = 0; i < 4; i++)
          w[i] = (T)o[4 * q4 + i];
        if (ALIAS_OST) lds_write<x4>((vbase + r * RBV + (uint32_t)(((4 * wave) ^ sw_r) << 4) + g * 8) ^ (uint32_t)(q4 << 4), w);
        else lds_write<x4>(lds_ost + r * OROW + (8 * q4 + 4 * g) * 2, w);
      }
      // (rows 16 apart share their swizzle)
      const uint32_t ra = vbase + (ln >> 2) * RBV + (uint32_t)(((4 * wave + (ln & 3)) ^ swz_tile<CPRV>(ln >> 2)) << 4);
#pragma unroll
      for (int it = 0; it < 2; it++) {
        const int ci = ln + 64 * it, row = ci >> 2, cc = ci & 3;
        const u32x4 w = ALIAS_OST ? lds_read<u32x4>(ra + 16 * it * RBV) : lds_read<u32x4>(lds_ost + row * OROW + cc * 16);
        if (t0 + row < Tn) *(u32x4*)(ob + (int64_t)(rev_o ? Tn - 1 - (t0 + row) : t0 + row) * a.Dv + cc * 8) = w;
      }
    }
  };
  if constexpr (PIPE) {
    constexpr int RQ = 1024 / RBQ, RV = 1024 / RBV, NLQ = NIQ / NW, NLV = NIV / NW, NL = 2 * NLQ + NLV;
    static_assert(NIQ % NW == 0 && NIV % NW == 0, "every wave moves the same number of instructions");
    constexpr int JOBS = 4;        // waves 0..2: a quadrant of P^T each, wave 3: scalars
    auto scalars_of = [&](int cn) { return lds_scalars + (uint32_t)((cn - c_begin) % 3) * (HG * kPipeScal); };

    // ---- Scalars of chunk cn, lane: token lane % 32, head lane / 32 of the group (one head: both halves alike).  ld, vs: its log
    //      decay and value scale.  Inclusive scan over the tokens (DPP: shifts within rows of 16 lanes, then lane 15 of rows 0
    //      and 2 carried into rows 1 and 3), in the log2 domain.
    const int64_t lane_head = (int64_t)(bh0 + (HG > 1 ? lane >> 5 : 0)) * Tn;
    const float head_factor = GEN == 0 && a.decay_head ? a.decay_head[h0 + (HG > 1 ? lane >> 5 : 0)] : 1.f;
    auto load_scalars = [&](int cn, float& ld, float& vs) {
      const int t = cn * L + r0;
      ld = 0.f;
      vs = 1.f;
      if (cn < c_end && t < Tn) {
        ld = a.log_decay[lane_head + t];
        if (a.v_scale) vs = v_scale_at(lane_head + t);
      }
    };
    auto publish = [&](int cn, float ld, float vs_loaded) {
      const float vs = v_scale_of(vs_loaded);
      const bool valid = cn * L + r0 < Tn;
      float x = valid ? log_decay_of(ld, head_factor) : 0.f;
      x += dpp_f32<0x111>(x);   // row_shr:1, lanes shifted in from outside the row read 0
      x += dpp_f32<0x112>(x);
      x += dpp_f32<0x114>(x);
      x += dpp_f32<0x118>(x);
      x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x142, 0xa, 0xf, false));   // row_bcast:15
      const float gi2 = x * kLog2e;
      const float last0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, gi2), 31));
      const float last1 = HG > 1 ? __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, gi2), 63)) : last0;
      const float g_last2 = HG > 1 && lane >= 32 ? last1 : last0;
      if (HG > 1 || lane < 32) {
        const uint32_t at = scalars_of(cn) + (HG > 1 ? (uint32_t)(lane >> 5) * kPipeScal : 0u) + (uint32_t)r0 * 4;
        lds_write<float>(at + kScalG, gi2);
        lds_write<float>(at + kScalV, valid ? vs * a.q_scale : 0.f);
        lds_write<float>(at + kScalW, valid ? vs * fast_exp2(g_last2 - gi2) : 0.f);
        lds_write<float>(at + kScalE, fast_exp2(gi2) * a.q_scale);
        if (r0 == 0) lds_write<float>(at + kScalD, fast_exp2(g_last2));
      }
    };

    // ---- A 16 x 16 quadrant of
    //        P^T = (K Q^T) * q_scale * exp(g_i - g_j) * vs_j * [j <= i]
    //      of chunk cn (wave 0: keys 0..15 x queries 0..15, 1: keys 0..15 x queries 16..31, 2: keys 16..31 x queries 16..31; the
    //      fourth lies above the diagonal), for every head of the group, straight into the B operand layout of V^T P^T.  A / B
    //      operand of the 16 x 16 MFMA: lane holds row (column) lane % 16, k = 8 (lane / 16) .. +7 of a 32-wide slice; C: lane holds
    //      column lane % 16, rows 4 (lane / 16) + {0..3}.
    //      Every wave of a head used to take A^T and form all of P^T for itself: 200 of its 650 vector instructions a
    //      chunk, in a loop that vector issue bounds.
    auto make_p = [&](int cn, int stage) {
      int la = lane;
      asm volatile("" : "+v"(la));
      const int kq = wave >> 1, qq = wave > 0;        // key and query half of the quadrant
      const int rr = la & 15, kg = la >> 4;
      const uint32_t qbase = lds0 + stage * STAGE, kbase = qbase + QT;
      // (tile bases and row offsets are multiples of the row size, so the swizzled chunk index occupies its own
      // address bits: one XOR with a constant per read moves to another slice)
      const uint32_t c0 = (uint32_t)((kg ^ swz16(rr)) << 4);
      const uint32_t ka = kbase + (16 * kq + rr) * RBQ + c0, qa = qbase + (16 * qq + rr) * RBQ + c0;
      f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      // (operands are requested three slices ahead: read as they are needed they cost an LDS latency each)
      constexpr int NS = DK / 32, AH = 3;
      x8 kf[AH + 1], qf[AH + 1];
      auto request = [&](int s2) {
        kf[s2 % (AH + 1)] = lds_read<x8>(ka ^ (uint32_t)(s2 * 64));
        qf[s2 % (AH + 1)] = lds_read<x8>(qa ^ (uint32_t)(s2 * 64));
      };
#pragma unroll
      for (int s2 = 0; s2 < AH; s2++) request(s2);
      const uint32_t sc = scalars_of(cn);
      float gq[HG];
      f32x4 gk[HG], pk[HG];
#pragma unroll
      for (int h = 0; h < HG; h++) {
        gq[h] = lds_read<float>(sc + h * kPipeScal + kScalG + (uint32_t)(16 * qq + rr) * 4);
        gk[h] = lds_read<f32x4>(sc + h * kPipeScal + kScalG + (uint32_t)(16 * kq + 4 * kg) * 4);
        pk[h] = lds_read<f32x4>(sc + h * kPipeScal + kScalV + (uint32_t)(16 * kq + 4 * kg) * 4);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s2 = 0; s2 < NS; s2++) {
        if (GEN && s2 * 32 >= qk_used) break;
        if (s2 + AH < NS) request(s2 + AH);
        __builtin_amdgcn_sched_barrier(0);
        acc[s2 & 1] = E::mfma16(kf[s2 % (AH + 1)], qf[s2 % (AH + 1)], acc[s2 & 1]);
        __builtin_amdgcn_sched_barrier(0);
      }
      const bool low[4] = {wave == 1 || 4 * kg <= rr, wave == 1 || 4 * kg + 1 <= rr, wave == 1 || 4 * kg + 2 <= rr, wave == 1 || 4 * kg + 3 <= rr};
#pragma unroll
      for (int h = 0; h < HG; h++) {
        float p[4];
        x4 w;
        // (above the diagonal the exponent is positive and the product may be inf or NaN: the select drops it)
#pragma unroll
        for (int t = 0; t < 4; t++) p[t] = (acc[0][t] + acc[1][t]) * fast_exp2(gq[h] - gk[h][t]) * pk[h][t];
        asm volatile("" : "+v"(p[0]), "+v"(p[1]), "+v"(p[2]), "+v"(p[3]));   // computed for every lane, then selected: no branch per element
#pragma unroll
        for (int t = 0; t < 4; t++) w[t] = (T)(low[t] ? p[t] : 0.f);
        // keys 16 kq + 4 kg + {0..3} of token i: slice kq, lane half kg % 2, elements 4 (kg / 2) ..
        const uint32_t at = lds_p + (uint32_t)(((cn - c_begin) & 1) * HG + h) * kPipeP + (uint32_t)(kg >> 1) * 8 +
                            (kq ? kPipeP1 + (uint32_t)(rr + 16 * (kg & 1)) * 16 : (uint32_t)(16 * qq + rr + 32 * (kg & 1)) * 16);
        lds_write<x4>(at, w);
      }
    };
    // what waves 0..3 (or the helpers) prepare while chunk c is under way: P^T of c + 1, scalars of c + 2
    auto prepare = [&](int c, int buf, float ld, float vs) {
      if (wave < 3) {
        if (c + 1 < c_end) make_p(c + 1, buf == NST - 1 ? 0 : buf + 1);
      } else if (c + 2 < c_end) {
        publish(c + 2, ld, vs);
      }
    };

    // ---- Loads of a chunk inside the loop: each wave moves instructions wave, wave + NW .. of each tile.  Bases are the tile's
    //      first row (reversed time: its last, the lowest address) plus the instruction's rows, lane offsets do not change; what is
    //      not to be loaded is switched off in the execution mask, without a branch.
    const int ln_q = wave * RQ + lane / CPRQ, ln_v = wave * RV + lane / CPRV;        // the lane's row in instruction 0
    const uint32_t lcq = (uint32_t)((lane % CPRQ) ^ swz_tile<CPRQ>(ln_q)), lcv = (uint32_t)((lane % CPRV) ^ swz_tile<CPRV>(ln_v));
    const uint32_t row_q = (uint32_t)(rev ? L - 1 - ln_q : ln_q) * (uint32_t)q_rb, row_k = GEN ? (uint32_t)(rev ? L - 1 - ln_q : ln_q) * (uint32_t)k_rb : row_q;
    const uint32_t row_v = (uint32_t)(rev ? L - 1 - ln_v : ln_v) * (uint32_t)v_row_bytes + (HG > 1 ? (lcv / (4 * NWH)) * (uint32_t)v_head_bytes : 0u);
    const uint64_t qk_lanes = GEN ? (uint64_t)__ballot(lcq < qk_chunks) : ~(uint64_t)0;      // (qk_chunks is a multiple of 4: the same lanes in every load)
    auto load_one = [&](int x, int t2, uint32_t base2, uint64_t on) {
      const int64_t first = rev ? Tn - t2 - L : t2;
      if (x < 2 * NLQ) {
        const int j = x % NLQ;
        const bool is_k = x >= NLQ;
        const int64_t rows = first + (rev ? -1 : 1) * j * NW * RQ;
        const uint32_t ch = (lcq ^ (uint32_t)swz_tile<CPRQ>(j * NW * RQ)) << 4;
        dma16_masked(is_k ? kb + rows * k_rb : qb + rows * q_rb, (is_k ? row_k : row_q) + ch, base2 + (is_k ? QT : 0) + (wave + NW * j) * 1024, on & qk_lanes);
      } else {
        const int j = x - 2 * NLQ;
        const int64_t rows = first + (rev ? -1 : 1) * j * NW * RV;
        const uint32_t ch = ((lcv ^ (uint32_t)swz_tile<CPRV>(j * NW * RV)) % (4 * NWH)) << 4;
        dma16_masked(vb + rows * v_row_bytes, row_v + ch, base2 + 2 * QT + (wave + NW * j) * 1024, on);
      }
    };

    float ld_next = 0.f, vs_next = 1.f;      // of the next chunk to be published
    const bool jobs = HELP ? helper : wave < JOBS;
    if (tid == 0) lds_write<u32x4>(lds_zero, u32x4{0u, 0u, 0u, 0u});
    if (jobs && wave == 3) {
      load_scalars(c_begin, ld_next, vs_next);
      publish(c_begin, ld_next, vs_next);
      load_scalars(c_begin + 1, ld_next, vs_next);
      publish(c_begin + 1, ld_next, vs_next);
      load_scalars(c_begin + 2, ld_next, vs_next);
    }
    wait_dma();
    __syncthreads();
    if (jobs && wave < 3 && c_begin < c_end) make_p(c_begin, 0);
    __syncthreads();

    // HELP: [chunk parity][wave] blocks of 32 tokens x 32 columns fp32 on their way out, rows padded by 16 bytes
    constexpr uint32_t OSTR = 128 + 16;
    auto out_block = [&](int c) { return lds_zero + 16 + (uint32_t)(((c - c_begin) & 1) * NW + wave) * (L * OSTR); };
    auto write_block = [&](int c) {
      int ln = lane;
      asm volatile("" : "+v"(ln));
      const int t0 = c * L;
      const uint32_t from = out_block(c);
      if (a.out_f32) {
        float* ob32 = (float*)a.o + (int64_t)piece * a.piece_o + (int64_t)bh * Tn * a.Dv + dvb * (32 * NWH) + 32 * (wave % NWH);
#pragma unroll
        for (int it = 0; it < 4; it++) {
          const int row = 8 * it + (ln >> 3), cc = ln & 7;
          f32x4 val = lds_read<f32x4>(from + row * OSTR + cc * 16);
          if (t0 + row < Tn) {
            f32x4* dst = (f32x4*)(ob32 + (int64_t)(rev_o ? Tn - 1 - (t0 + row) : t0 + row) * a.Dv + cc * 4);
            if (a.out_f32 == 2) val += *dst;   // (a contraction cut into pieces: the pieces' outputs add up)
            *dst = val;
          }
        }
      } else {
#pragma unroll
        for (int it = 0; it < 2; it++) {
          const int row = 16 * it + (ln >> 2), cc = ln & 3;
          const f32x4 lo = lds_read<f32x4>(from + row * OSTR + cc * 32), hi = lds_read<f32x4>(from + row * OSTR + cc * 32 + 16);
          x8 w;
#pragma unroll
          for (int i = 0; i < 4; i++) { w[i] = (T)lo[i]; w[4 + i] = (T)hi[i]; }
          if (t0 + row < Tn) *(x8*)(ob + (int64_t)(rev_o ? Tn - 1 - (t0 + row) : t0 + row) * a.Dv + cc * 8) = w;
        }
      }
    };

    f32x16 o_out;         // outputs of chunk c - 1, written while chunk c is under way: nobody waits for the stores
    // What is added to a chunk's outputs (o_add) is asked for when they are there and the state loop's operand registers are free
    // again, and waited for where they are written, behind the next chunk's first reads.  (Asked for in the middle of the state loop,
    // with V^T P^T behind it, it is no faster: what these passes wait for is memory, 4.5 - 4.9 TB/s.)
    f32x4 add[4];
    constexpr bool PARTIAL = GEN >= 3, EARLY = !HELP && (PARTIAL || (GEN == 0 && MODE == 0));
    static_assert(!PARTIAL || !HELP, "partial results");
    const bool adds = PARTIAL && a.o_add != nullptr;
    // the wave's 32 x 32 block of chunk c in the order of its accumulators: four rows of 64 lanes x 16 bytes
    auto part_at = [&](const float* part, int c) {
      return (f32x4*)(part + ((((int64_t)bh * a.dv_blocks + dvb) * n_chunks_all + c) * NW + wave) * (16 * 64));
    };
    auto load_add = [&](int c) {
      const f32x4* src = part_at(a.o_add, c);
#pragma unroll
      for (int q4 = 0; q4 < 4; q4++) add[q4] = src[64 * q4 + lane];
    };
    auto finish = [&](int c, uint32_t vbase) {
      if (adds) {
#pragma unroll
        for (int j = 0; j < 16; j++) o_out[j] += add[j >> 2][j & 3];
      }
      if (PARTIAL && a.o_part) {
        f32x4* dst = part_at(a.o_part, c);
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) dst[64 * q4 + lane] = f32x4{o_out[4 * q4], o_out[4 * q4 + 1], o_out[4 * q4 + 2], o_out[4 * q4 + 3]};
      } else {
        write_out(o_out, c * L, vbase);
      }
    };
    // a state wave's work of chunk c
    auto run_chunk = [&](int c, int buf) {
      const int t0 = c * L;
      const uint32_t base = lds0 + buf * STAGE, qbase = base, kbase = base + QT, vbase = base + 2 * QT;
      // the loads of this chunk: chunk c + NST - 1, into the stage that chunk c - 1 has left
      const int t2 = t0 + (NST - 1) * L;
      const uint32_t base2 = lds0 + (uint32_t)(buf == 0 ? NST - 1 : buf - 1) * STAGE;
      const bool loads = c + NST - 1 < c_end, whole = t2 + L <= Tn && v_head_bytes < ((int64_t)1 << 31);
      const uint64_t on = loads && whole ? ~(uint64_t)0 : 0;
      int ln = lane;
      asm volatile("" : "+v"(ln));
      const int r = ln & 31, g = ln >> 5;
      const int jr = (ln & 15) >> 2, lc = (((ln >> 4) & 1) << 1) | ((ln & 3) >> 1);
      constexpr int X8 = 2;          // swz(row + 8) ^ swz(row); rows 16 apart share their swizzle
      // ---- V^T fragments (rows = this wave's 32 value columns; k-slot i of slice s is token
      //      16s + 8(i/4) + 4g + i%4, the order P^T comes in)
      x8 vf[2];
      {
        const uint32_t va = vbase + (4 * g + jr) * RBV + (ln & 1) * 8 + (uint32_t)(((4 * wave + lc) ^ swz_tile<CPRV>(4 * g + jr)) << 4);
#pragma unroll
        for (int s = 0; s < 2; s++) {
          const x4 lo = lds_read_tr4<T>(va + 16 * s * RBV), hi = lds_read_tr4<T>((va ^ (uint32_t)(X8 << 4)) + (16 * s + 8) * RBV);
          vf[s] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
      }
      const uint32_t ph = lds_p + (uint32_t)(((c - c_begin) & 1) * HG + hl) * kPipeP, sh = scalars_of(c) + hl * kPipeScal;
      const x8 pf0 = lds_read<x8>(ph + ln * 16);
      const x8 pf1 = lds_read<x8>(r >= 16 ? ph + kPipeP1 + (r - 16 + 16 * g) * 16 : lds_zero);
      const float eg = lds_read<float>(sh + kScalE + r * 4);
      float decay_all = lds_read<float>(sh + kScalD);
      f32x4 w4[4];
#pragma unroll
      for (int i = 0; i < 4; i++) w4[i] = lds_read<f32x4>(sh + kScalW + 16 * g + 32 * i);
      if (!HELP && c > c_begin) finish(c - 1, vbase);

      const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      f32x16 o_intra = E::mfma32(vf[0], pf0, zero16);
      o_intra = E::mfma32(vf[1], pf1, o_intra);
      // value-scaled V^T for the state update
      x8 vsf[2];
#pragma unroll
      for (int s = 0; s < 2; s++) {
        const float w8[8] = {w4[2 * s][0], w4[2 * s][1], w4[2 * s][2], w4[2 * s][3], w4[2 * s + 1][0], w4[2 * s + 1][1], w4[2 * s + 1][2], w4[2 * s + 1][3]};
        vsf[s] = scale_bf16x8(vf[s], w8);
      }
      if (!HELP && wave < JOBS) {
        prepare(c, buf, ld_next, vs_next);
        if (wave == 3) load_scalars(c + 3, ld_next, vs_next);
      }

      // ---- per 32-row state block: inter-chunk product with the OLD state (as bf16 operand), decay, state update.  The
      //      conversion and the decay of the next block are dealt into the gaps behind the four MFMAs of this block, operands
      //      are requested one block ahead.  The chunk's loads go out behind all blocks, but with the first half of them in a plain scan
      //      of one pass and with partial results, which fill the device and wait for memory (EARLY; the last
      //      loads of a chunk are waited for at its end).  Forward + backward, 256 / 512, all early and all late: 8 x 16 heads, 2048 tokens
      //      1031 and 1042 us; 8 x 8 heads, 300 tokens, whose scans run side by side, 142.7 and 140.6.  A choice made in the kernel, by a
      //      branch at every load: 1017 and 143 where the early ones alone took 1001 and 140.6, on one box.  Not with helpers, which have
      //      a stage more to land in: Mamba2's scan 86 us late and 87 early.
      if (loads && !whole) issue_rows(t2, base2);
      const uint32_t qpa = qbase + r * RBQ + (uint32_t)(((2 * g) ^ swz16(r)) << 4);
      const uint32_t kta = kbase + (4 * g + jr) * RBQ + ((ln >> 1) & 1) * 8 + (uint32_t)(((((ln & 1) << 1) | ((ln >> 4) & 1)) ^ swz16(4 * g + jr)) << 4);
      f32x16 o_inter;
      {
        x8 qf[2][2];
        x4 klo[2][2], khi[2][2];
        u32x4 hf[2];       // (slice s of the next block's operand is written behind the MFMA that reads this block's)
        auto request = [&](int bb) {
#pragma unroll
          for (int s = 0; s < 2; s++) {
            qf[bb % 2][s] = lds_read<x8>(qpa ^ (uint32_t)((4 * bb + s) << 4));
            klo[bb % 2][s] = lds_read_tr4<T>((kta ^ (uint32_t)((4 * bb) << 4)) + 16 * s * RBQ);
            khi[bb % 2][s] = lds_read_tr4<T>((kta ^ (uint32_t)(((4 * bb) ^ X8) << 4)) + (16 * s + 8) * RBQ);
          }
        };
        auto convert = [&](int bb, int part) {      // a quarter of block bb: operand in bf16, then decayed in place
          typename E::x2 x, y;
#pragma unroll
          for (int i = 0; i < 2; i++) { x[i] = (T)hst[bb][4 * part + i]; y[i] = (T)hst[bb][4 * part + 2 + i]; }
          uint32_t lo = __builtin_bit_cast(uint32_t, x), hi = __builtin_bit_cast(uint32_t, y);
          // (pinned here, the products through their factor: the compiler otherwise gathers the vector work of a block in
          // front of its MFMAs)
          asm volatile("" : "+v"(lo), "+v"(hi), "+v"(decay_all));
#pragma unroll
          for (int i = 0; i < 4; i++) hst[bb][4 * part + i] *= decay_all;
          hf[part >> 1][2 * (part & 1)] = lo;
          hf[part >> 1][2 * (part & 1) + 1] = hi;
        };
        request(0);
#pragma unroll
        for (int part = 0; part < 4; part++) convert(0, part);
#pragma unroll
        for (int bb = 0; bb < KB; bb++) {
          const bool used = !GEN || bb * 32 < qk_used, more = bb + 1 < KB;
          if (used) {
            if (more) request(bb + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 2; s++) {
              o_inter = E::mfma32(__builtin_bit_cast(x8, hf[s]), qf[bb % 2][s], bb == 0 && s == 0 ? zero16 : o_inter);
              __builtin_amdgcn_sched_barrier(0);
              if (more) convert(bb + 1, s);
              __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int s = 0; s < 2; s++) {
              const x8 kf = __builtin_shufflevector(klo[bb % 2][s], khi[bb % 2][s], 0, 1, 2, 3, 4, 5, 6, 7);
              hst[bb] = E::mfma32(kf, vsf[s], hst[bb]);
              __builtin_amdgcn_sched_barrier(0);
              if (more) convert(bb + 1, 2 + s);
              __builtin_amdgcn_sched_barrier(0);
            }
          }
#pragma unroll
          for (int x = 0; x < NL; x++)
            if (x * (EARLY ? KB / 2 : KB) / NL == bb) load_one(x, t2, base2, on);
        }
      }
#pragma unroll
      for (int j = 0; j < 16; j++) o_out[j] = o_inter[j] * eg + o_intra[j];
      if constexpr (HELP) {
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) {
          const f32x4 w = {o_out[4 * q4], o_out[4 * q4 + 1], o_out[4 * q4 + 2], o_out[4 * q4 + 3]};
          lds_write<f32x4>(out_block(c) + r * OSTR + (8 * q4 + 4 * g) * 4, w);
        }
      }
      // chunk c + 2 must be there for P^T of c + 2, made in c + 1: with four stages it was asked for a chunk ago and the loads of this
      // chunk may go on; with three, its V, not read before c + 2, may
      if (adds) {
        load_add(c);
      } else {
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) add[q4] = f32x4{0.f, 0.f, 0.f, 0.f};     // (not carried through the chunk)
      }
      if (loads && !whole) wait_dma();
      else if (adds) wait_vm<NLV + 4>();
      else wait_vm<HELP ? NL : NLV>();
    };
    // a helper's: scalars' loads of chunk c + 3, outputs of c - 1, P^T of c + 1 or scalars of c + 2
    auto help_chunk = [&](int c, int buf) {
      const float ld_now = ld_next, vs_now = vs_next;
      if (wave == 3) load_scalars(c + 3, ld_next, vs_next);
      if (c > c_begin) write_block(c - 1);
      prepare(c, buf, ld_now, vs_now);
    };
    int buf = 0;          // stage of chunk c
    if (HELP && helper) {
      for (int c = c_begin; c < c_end; c++) {
        help_chunk(c, buf);
        __syncthreads();
        buf = buf == NST - 1 ? 0 : buf + 1;
      }
      if (c_begin < c_end) write_block(c_end - 1);
    } else {
      for (int c = c_begin; c < c_end; c++) {
        run_chunk(c, buf);
        __syncthreads();
        buf = buf == NST - 1 ? 0 : buf + 1;
      }
      if (!HELP && c_begin < c_end) finish(c_end - 1, lds0 + (uint32_t)(buf == 0 ? NST - 1 : buf - 1) * STAGE + 2 * QT);
    }
  }
  if constexpr (!PIPE) {
  const float head_factor = GEN == 0 && a.decay_head ? a.decay_head[h0 + hl] : 1.f;
  for (int c = c_begin; c < c_end; c++) {
    const int buf = (c - c_begin) & 1, t0 = c * L;
    wait_dma();
    __syncthreads();
    const float ld = ld_next, vs = v_scale_of(vs_next);
    const bool has_next = c + 1 < c_end;
    if (has_next) {
      const int tn = t0 + L + ti;
      ld_next = 0.f;
      vs_next = 1.f;
      if (tn < Tn) {
        ld_next = ldp[tn];
        if (a.v_scale) vs_next = v_scale_at(tok0 + tn);
      }
    }
    if (has_next) issue_chunk(t0 + L, buf ^ 1);
    const uint32_t base = lds0 + buf * STAGE;
    const uint32_t qbase = base, kbase = base + QT, vbase = base + 2 * QT;

    // ---- per-lane LDS read offsets.  They are loop invariant; left outside the loop, they (and every
    //      swizzled address derived from them, dozens) stay in registers across chunks, which the state
    //      accumulator leaves no room for.  The lane id is laundered so that they are rebuilt per chunk.
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int r = ln & 31, g = ln >> 5;
    // K rows / Q rows as MFMA operands of A^T = K Q^T: row r, logical chunk 2ks + g
    const uint32_t qk_row = r * RBQ;
    const int qk_c0 = g ^ swz16(r);
    // A 32-row block of the state holds its key dims in an order that makes the Q^T operand of h^T Q^T one 128-bit read per
    // slice: accumulator rows 8q + 4g + {0..3} of lane half g are key dims 16g + 4q + {0..3}, so slice s (q = 2s, 2s + 1) of
    // lane half g is the eight dims of chunk 4b + 2g + s.  (In the rows' own order it was two 64-bit reads that left half of the
    // banks idle and met twice in the other half: SQ_LDS_BANK_CONFLICT 15.7 M -> 7.3 M a pass at 8 x 16 heads, 2048 tokens,
    // 256 / 512, 290 -> 280 us before anything else changed.)
    const uint32_t qp_row = r * RBQ;
    const int qp_c0 = (2 * g) ^ swz16(r);
    // transposing reads (K^T and V^T): lane block lane/16 -> (row group g, column half), rows 16s + 4g + jr (+8)
    const int jr = (ln & 15) >> 2;
    const int lc = (((ln >> 4) & 1) << 1) | ((ln & 3) >> 1);
    // (K^T: the four columns that become rows 4m .. 4m + 3 of a state block, m = 4 ((ln >> 4) & 1) + ln % 4, are its dims
    // 16 (m % 2) + 4 (m / 2) ..: chunk 2 (m % 2) + m / 4, half (m / 2) % 2)
    const uint32_t kt_row = (4 * g + jr) * RBQ + ((ln >> 1) & 1) * 8;
    const int kt_c0 = (((ln & 1) << 1) | ((ln >> 4) & 1)) ^ swz16(4 * g + jr);                      // rows +8 / +16: see Q_X8 below
    const uint32_t vt_row = (4 * g + jr) * RBV + (ln & 1) * 8;
    const int vt_c0 = (4 * wave + lc) ^ swz_tile<CPRV>(4 * g + jr);
    // swz(row + 8) ^ swz(row) and swz(row + 16) ^ swz(row) for rows < 8
    constexpr int Q_X8 = 2, Q_X16 = 0;
    constexpr int V_X8 = CPRV >= 16 ? 2 : 2, V_X16 = CPRV >= 16 ? 0 : 0;


    // ---- chunk scalars: inclusive scan of the log decay over the 32 tokens (both lane halves hold a copy)
    const bool valid = t0 + ti < Tn;
    // (DPP: shifts within rows of 16 lanes, then lane 15 of rows 0 and 2 carried into rows 1 and 3; the
    // two halves of the wave scan the same 32 values)
    float gi = valid ? log_decay_of(ld, head_factor) : 0.f;
    gi += dpp_f32<0x111>(gi);   // row_shr:1, lanes shifted in from outside the row read 0
    gi += dpp_f32<0x112>(gi);
    gi += dpp_f32<0x114>(gi);
    gi += dpp_f32<0x118>(gi);
    gi += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, gi), 0x142, 0xa, 0xf, false));   // row_bcast:15
    const float g_last = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, gi), 31));
    const float gi2 = gi * kLog2e, g_last2 = g_last * kLog2e;    // (exponents in the log2 domain from here on)
    const float pvq = valid ? vs * a.q_scale : 0.f;               // factor of column j in P
    const float wl = valid ? vs * fast_exp2(g_last2 - gi2) : 0.f;   // factor of row l in the state update
    const float eg = fast_exp2(gi2) * a.q_scale;                  // factor of token i in the inter-chunk term
    const float decay_all = fast_exp2(g_last2);
    if (MODE == 1) seg_log += g_last;
    if (g == 0) {
      lds_write<float>(lds_scal + ti * 4, gi2);
      lds_write<float>(lds_scal + (L + ti) * 4, pvq);
      lds_write<float>(lds_scal + (2 * L + ti) * 4, wl);
    }
    // ---- A^T = K Q^T (lane: token i = r, rows j = 8(jj/4) + 4g + jj%4)
    // two accumulation chains, so that consecutive MFMAs do not wait for each other, where registers allow
    constexpr bool TWO_CHAINS = HG == 1;
    // (a chain's first MFMA takes the constant zero as its accumulator input: no registers to clear)
    const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    f32x16 sacc, sacc2;
#pragma unroll
    for (int j = 0; j < 16; j++) { sacc[j] = 0.f; sacc2[j] = 0.f; }
    if constexpr (MODE != 1) {
      constexpr int NS = DK / 16, AH = 2, RING = 3;
      x8 kf[RING], qf[RING];
      const uint32_t kq_a = kbase + qk_row + (uint32_t)(qk_c0 << 4), qq_a = qbase + qk_row + (uint32_t)(qk_c0 << 4);
      auto request = [&](int ks) {
        kf[ks % RING] = lds_read<x8>(kq_a ^ (uint32_t)(ks * 32));
        qf[ks % RING] = lds_read<x8>(qq_a ^ (uint32_t)(ks * 32));
      };
#pragma unroll
      for (int ks = 0; ks < AH; ks++) request(ks);
#pragma unroll
      for (int ks = 0; ks < NS; ks++) {
        if (GEN && ks * 16 >= qk_used) break;
        if (ks + AH < NS) request(ks + AH);
        __builtin_amdgcn_sched_barrier(0);
        if (TWO_CHAINS && (ks & 1)) sacc2 = E::mfma32(kf[ks % RING], qf[ks % RING], ks == 1 ? zero16 : sacc2);
        else sacc = E::mfma32(kf[ks % RING], qf[ks % RING], ks == 0 ? zero16 : sacc);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // rows held by this lane in a 32 x 32 accumulator block: 8q4 + 4g + {0..3}
    float gj[16], pj[16];
    uint32_t scal_g = lds_scal + 16 * g;   // one lane register; every read below is this plus an immediate
    asm volatile("" : "+v"(scal_g));
    if constexpr (MODE != 1) {
#pragma unroll
    for (int q4 = 0; q4 < 4; q4++) {
      const f32x4 tg = lds_read<f32x4>(scal_g + 32 * q4);
      const f32x4 tp = lds_read<f32x4>(scal_g + (L + 8 * q4) * 4);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        gj[4 * q4 + i] = tg[i];
        pj[4 * q4 + i] = tp[i];
      }
    }
    }
    // ---- P^T: decay, per-token value scale, causal mask (exact zeros above the diagonal)
    x8 pf[2];
    if constexpr (MODE != 1) {
#pragma unroll
    for (int jj = 0; jj < 16; jj++) {
      const int j = 8 * (jj >> 2) + 4 * g + (jj & 3);
      // (above the diagonal the exponent is positive and the product may be inf or NaN: the select drops it)
      const float e = fast_exp2(gi2 - gj[jj]);
      float p = (TWO_CHAINS ? sacc[jj] + sacc2[jj] : sacc[jj]) * e * pj[jj];
      asm volatile("" : "+v"(p));   // computed for every lane, then selected: no branch per element
      pf[jj >> 3][jj & 7] = (T)(j <= ti ? p : 0.f);
    }
    }

    // ---- V^T fragments (rows = this wave's 32 value columns; k-slot i of slice s is token
    //      16s + 8(i/4) + 4g + i%4, the order P^T comes in)
    x8 vf[2];
    {
      const uint32_t va = vbase + vt_row + (uint32_t)(vt_c0 << 4);
#pragma unroll
      for (int s = 0; s < 2; s++) {
        const int cx = s ? V_X16 : 0;
        x4 lo = lds_read_tr4<T>((va ^ (uint32_t)(cx << 4)) + 16 * s * RBV);
        x4 hi = lds_read_tr4<T>((va ^ (uint32_t)((cx ^ V_X8) << 4)) + (16 * s + 8) * RBV);
        vf[s] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      }
    }

    // ---- O^T = (h^T Q^T) * eg + V^T P^T
    f32x16 o_inter, o_inter2, o_intra;
#pragma unroll
    for (int j = 0; j < 16; j++) { o_inter[j] = 0.f; o_inter2[j] = 0.f; o_intra[j] = 0.f; }
    if constexpr (MODE != 1) {
      o_intra = E::mfma32(vf[0], pf[0], zero16);
      o_intra = E::mfma32(vf[1], pf[1], o_intra);
    }
    // value-scaled V^T for the state update (k-slot i of slice s is token 16s + 8(i/4) + 4g + i%4 -> wj[8s + i])
    x8 vsf[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
      float w8[8];
#pragma unroll
      for (int h2 = 0; h2 < 2; h2++) {
        const f32x4 tw = lds_read<f32x4>(scal_g + (2 * L + 16 * s + 8 * h2) * 4);
#pragma unroll
        for (int i = 0; i < 4; i++) w8[4 * h2 + i] = tw[i];
      }
      vsf[s] = scale_bf16x8(vf[s], w8);
    }

    {
      // per 32-row state block b: inter-chunk product with the OLD state, then the state update
      constexpr int RING = 2;
      x8 qf[RING][2];
      x4 klo[RING][2], khi[RING][2];
      const uint32_t qpa = qbase + qp_row + (uint32_t)(qp_c0 << 4), kta = kbase + kt_row + (uint32_t)(kt_c0 << 4);
      auto request = [&](int bb) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
          if constexpr (MODE != 1) qf[bb % RING][s] = lds_read<x8>(qpa ^ (uint32_t)((4 * bb + s) << 4));
          const int cx = s ? Q_X16 : 0;
          klo[bb % RING][s] = lds_read_tr4<T>((kta ^ (uint32_t)(((4 * bb) ^ cx) << 4)) + 16 * s * RBQ);
          khi[bb % RING][s] = lds_read_tr4<T>((kta ^ (uint32_t)(((4 * bb) ^ cx ^ Q_X8) << 4)) + (16 * s + 8) * RBQ);
        }
      };
      // operands are requested one block ahead, except where three waves per SIMD (two heads a workgroup, states alone) hide the LDS
      // latency and the registers are needed elsewhere
      constexpr bool AHEAD = HG == 1;
      if (AHEAD) request(0);
#pragma unroll
      for (int bb = 0; bb < KB; bb++) {
        if (GEN && bb * 32 >= qk_used) break;
        if (!AHEAD) request(bb);
        else if (bb + 1 < KB) request(bb + 1);
        __builtin_amdgcn_sched_barrier(0);
        // the old state as bf16 operands first, then the decay in place (left to itself the compiler decays into a
        // second register block while the old values are still waiting to be converted, and copies it back)
        x8 hf[2];
        if constexpr (MODE != 1) {
#pragma unroll
          for (int s = 0; s < 2; s++)
#pragma unroll
            for (int i = 0; i < 8; i++) hf[s][i] = (T)hst[bb][8 * s + i];
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int j = 0; j < 16; j++) hst[bb][j] *= decay_all;
        if constexpr (MODE != 1) {
#pragma unroll
          for (int s = 0; s < 2; s++) {
            if (DK < 256 && HG == 1 && s) o_inter2 = E::mfma32(hf[s], qf[bb % RING][s], bb == 0 ? zero16 : o_inter2);   // (a second chain where registers allow)
            else o_inter = E::mfma32(hf[s], qf[bb % RING][s], (bb == 0 && (s == 0 || (DK < 256 && HG == 1))) ? zero16 : o_inter);
          }
        }
#pragma unroll
        for (int s = 0; s < 2; s++) {
          x8 kf = __builtin_shufflevector(klo[bb % RING][s], khi[bb % RING][s], 0, 1, 2, 3, 4, 5, 6, 7);
          hst[bb] = E::mfma32(kf, vsf[s], hst[bb]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }

    if constexpr (MODE != 1) {
      f32x16 o;
#pragma unroll
      for (int j = 0; j < 16; j++) o[j] = (DK < 256 && HG == 1 ? o_inter[j] + o_inter2[j] : o_inter[j]) * eg + o_intra[j];
      write_out(o, t0, vbase);
    }
  }
  }
  if (MODE == 1) {
    // the state this segment ends in when entered with zeros, and its total log decay
    float* dst = ws_mine + seg * WS_SEG;
#pragma unroll
    for (int i = 0; i < KB; i++)
#pragma unroll
      for (int j = 0; j < 16; j++) dst[(i * 16 + j) * 64] = hst[i][j];
    if (piece == 0 && dvb == 0 && wave % NWH == 0 && lane == 0) a.ws_decay[(int64_t)(bh - a.bg0 * HG) * (a.nseg - 1) + seg] = seg_log;
  }
}

// Entering states of segments 1 .. nseg-1 from the local end states, in place: slot s (the state segment s ends in when entered
// with zeros) becomes the state that segment s + 1 is entered with, E_{s+1} = exp(D_s) E_s + h_s.  One thread per four floats
// of a group's state, walking the segments; head_floats of a group's group_floats belong to one head.  Bound by memory latency
// (each state once in and once out); the loads of four segments are in flight together.
// (blockIdx.z: the scan, blockIdx.y: piece, head group, value slice)
__global__ __launch_bounds__(256) void linear_states_kernel(const LinScans all, int group_floats, int head_floats, int HG) {
  const LinArgs& a = all.s[blockIdx.z];
  const int off = (blockIdx.x * 256 + threadIdx.x) * 4;       // (group_floats is a multiple of 1024: whole workgroups)
  const int grp = blockIdx.y, BG = a.B * a.H / HG, slots = a.nseg - 1;
  if (grp >= BG * a.dv_blocks * (a.n_pieces > 1 ? a.n_pieces : 1)) return;
  const int bg = (grp / a.dv_blocks) % BG, hl = off / head_floats;
  const float* dec = a.ws_decay + ((int64_t)bg * HG + hl) * slots;
  float* p = a.ws_state + (int64_t)grp * slots * group_floats + off;
  f32x4 e = *(const f32x4*)p;
  int s = 1;
  for (; s + 3 < slots; s += 4) {
    f32x4 h[4];
    float d[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      h[i] = *(const f32x4*)(p + (int64_t)(s + i) * group_floats);
      d[i] = dec[s + i];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      e = e * fast_exp2(d[i] * kLog2e) + h[i];
      *(f32x4*)(p + (int64_t)(s + i) * group_floats) = e;
    }
  }
  for (; s < slots; s++) {
    e = e * fast_exp2(dec[s] * kLog2e) + *(const f32x4*)(p + (int64_t)s * group_floats);
    *(f32x4*)(p + (int64_t)s * group_floats) = e;
  }
}

namespace {
// Resident workgroups per CU and the CU count, asked of the runtime once per configuration.
template <int DK, int NWH, int HG>
struct Config {
  static constexpr int NW = NWH * HG;
  static constexpr size_t stage = (size_t)L * (4 * DK + 2 * 32 * NW);
  static constexpr int waves = workgroup_waves<DK, NWH, HG, 0>();      // of a workgroup that produces outputs
  static constexpr size_t lds_states = 2 * stage + NW * (3 * L * 4);
  static constexpr size_t lds = pipelined<NWH, HG, 0>() ? (waves > NW ? 4 : 3) * stage + pipe_shared(HG) + (waves > NW ? 2 * NW * L * 144 : 0) : lds_states + NW * (L * 80);
  static_assert(lds <= 160 * 1024, "a workgroup's LDS");
  static constexpr int64_t ws_wave_floats = (int64_t)(DK / 32) * 16 * 64;

  // partial results (o_part, o_add): by the pipelined chunk loop without helpers
  static constexpr bool can_leave_parts = pipelined<NWH, HG, 0>() && helpers<DK, NWH, HG, 0>() == 0;
  static bool prepare(int& resident, int& cus) {
    // (threads that meet in a first call compute the same numbers; a device other than the first one asked is assumed to
    // be of the same kind)
    static std::atomic<uint64_t> lds_ok{0};
    static std::atomic<int> s_resident{-1};
    if (allow_lds(lds_ok, lds, linear_fwd_kernel<DK, NWH, HG, 0>, linear_fwd_kernel<DK, NWH, HG, 1>, linear_fwd_kernel<DK, NWH, HG, 2>,
                  linear_fwd_kernel<DK, NWH, HG, 0, 1>, linear_fwd_kernel<DK, NWH, HG, 1, 1>, linear_fwd_kernel<DK, NWH, HG, 2, 1>,
                  linear_fwd_kernel<DK, NWH, HG, 0, 2>, linear_fwd_kernel<DK, NWH, HG, 1, 2>, linear_fwd_kernel<DK, NWH, HG, 2, 2>) != 0)
      return false;
    if constexpr (can_leave_parts) {
      static std::atomic<uint64_t> parts_ok{0};
      if (allow_lds(parts_ok, lds, linear_fwd_kernel<DK, NWH, HG, 0, 3>, linear_fwd_kernel<DK, NWH, HG, 2, 3>,
                    linear_fwd_kernel<DK, NWH, HG, 0, 4>, linear_fwd_kernel<DK, NWH, HG, 2, 4>) != 0)
        return false;
    }
    cus = device_cus();
    if (cus <= 0) return false;
    int r = s_resident.load(std::memory_order_relaxed);
    if (r < 0) {
      if (hip_check(hipOccupancyMaxActiveBlocksPerMultiprocessor(&r, linear_fwd_kernel<DK, NWH, HG, 2>, 64 * waves, lds)) != 0) return false;
      r = r < 1 ? 1 : r;
      s_resident.store(r, std::memory_order_relaxed);
    }
    resident = r;
    return true;
  }

  // workgroups of a single pass
  static int64_t groups(const LinArgs& a) { return (a.bg_n > 0 ? a.bg_n : (int64_t)a.B * a.H / HG) * (a.Dv / (32 * NWH)) * (a.n_pieces > 1 ? a.n_pieces : 1); }

  // Number of segments and chunks per segment for this problem.  want: 0 = choose, n >= 1 = at most n.
  // Chosen: as many segments as keep every CU's resident workgroup slots busy.  A chunk is a chain of 2 - 4 us however few
  // workgroups there are, and both launches walk a segment's chunks, so that short sequences go down to 2 chunks a segment
  // (1 x 16 heads, 300 tokens, 256 / 512: 2 segments 42.6 us, 5 segments 35.0); more than 8 segments pay for
  // linear_states_kernel and are at least 4 chunks long (1 x 4 heads, 2048 tokens, 256 / 512: 8 segments 68.5 us, 16 of 4
  // chunks 53.1, 32 of 2 chunks 58.4; 8 heads, 4096 tokens, 128 / 128: 8 segments 60.3, 32 segments 31.1).
  static void plan(const LinArgs& a, int64_t all_groups, int want, int resident, int cus, int& nseg, int& seg_chunks) {
    const int n_chunks = (a.T + L - 1) / L;
    int n;
    if (want >= 1) n = want;
    else {
      n = (int)((int64_t)resident * cus / all_groups);
      const int direct = n_chunks / 2 < 8 ? n_chunks / 2 : 8, scanned = n_chunks / 4 < 32 ? n_chunks / 4 : 32;
      if (n > (direct > scanned ? direct : scanned)) n = direct > scanned ? direct : scanned;
    }
    if (n > n_chunks) n = n_chunks;
    if (n < 1) n = 1;
    seg_chunks = (n_chunks + n - 1) / n;
    nseg = (n_chunks + seg_chunks - 1) / seg_chunks;
  }

  static size_t ws_bytes(const LinArgs& a, int nseg) {
    if (nseg <= 1) return 0;
    return (size_t)((groups(a) * (nseg - 1) * NW * ws_wave_floats + (int64_t)a.B * a.H * (nseg - 1)) * 4);
  }

  // A single pass over more head groups than the device holds at once ends in a round that is mostly empty (320 workgroups
  // on 256 CUs take as long as 512).  When the last round would be at most half full, the head groups of the full rounds run
  // the single pass and the rest is cut into sequence segments, as many as fill the device once: tail_bg head groups from
  // full_bg on, in nseg segments (tail_bg = 0: no such split).
  struct Tail { int full_bg, tail_bg, nseg, seg_chunks; };
  static Tail tail_plan(const LinArgs& a, int want, int resident, int cus) {
    Tail t{0, 0, 1, 0};
    const int dvb = a.Dv / (32 * NWH), n_chunks = (a.T + L - 1) / L;
    const int64_t BG = (int64_t)a.B * a.H / HG, per_round = (int64_t)resident * cus / dvb;     // head groups
    if (want != 0 || a.n_pieces > 1 || per_round < 1 || BG <= per_round) return t;
    const int64_t tail = BG % per_round;
    int n = tail > 0 ? (int)(per_round / tail) : 1;
    if (n > 8) n = 8;
    if (n > n_chunks / 4) n = n_chunks / 4;
    if (tail == 0 || tail * 2 > per_round || n < 2) return t;
    t.full_bg = (int)(BG - tail);
    t.tail_bg = (int)tail;
    t.seg_chunks = (n_chunks + n - 1) / n;
    t.nseg = (n_chunks + t.seg_chunks - 1) / t.seg_chunks;
    if (t.nseg < 2) t.tail_bg = 0;
    return t;
  }
  static size_t tail_ws_bytes(const Tail& t, int dvb) {
    if (t.tail_bg <= 0) return 0;
    return (size_t)(((int64_t)t.tail_bg * dvb * (t.nseg - 1) * NW * ws_wave_floats + (int64_t)t.tail_bg * HG * (t.nseg - 1)) * 4);
  }

  // general operand addressing: defaults for what is left at zero; the row distances must be multiples of the tile
  // rows (the kernel XORs the swizzle of an instruction's first row onto the finished lane offset)
  static bool general(const LinArgs& a) {
    return a.rev != 0 || a.q_row != 0 || a.k_row != 0 || a.v_row != 0 || (a.Hv != 0 && a.Hv != a.H) || a.qk_cols != 0 || a.n_pieces > 1 || a.rev_o != 0 || a.o_add != nullptr || a.o_part != nullptr;
  }
  static int fill(LinArgs& a) {
    a.dv_blocks = a.Dv / (32 * NWH);
    if (a.q_row == 0) a.q_row = DK;
    if (a.k_row == 0) a.k_row = DK;
    if (a.v_row == 0) a.v_row = a.Dv;
    if (a.Hv == 0) a.Hv = a.H;
    if (a.q_row % 8 != 0 || a.k_row % 8 != 0 || a.v_row % (32 * NWH) != 0 || a.Hv <= 0 || a.H % a.Hv != 0) return -2;
    if (a.qk_cols < 0 || a.qk_cols > DK || a.qk_cols % 32 != 0) return -2;
    if (HG > 1 && a.Hv != a.H) return -2;
    if (a.n_pieces > 1 && !a.out_f32) return -2;
    if ((a.o_add || a.o_part) && (!can_leave_parts || a.out_f32)) return -2;
    return 0;
  }

  // MODE 0, 1 or 2 of n scans; the grid is as wide as the widest
  template <int MODE>
  static void launch(const LinScans& all, int n, bool gen, hipStream_t stream) {
    unsigned width = 0;
    for (int i = 0; i < n; i++) {
      const LinArgs& a = all.s[i];
      const int64_t heads = a.bg_n > 0 ? a.bg_n : (int64_t)a.B * a.H / HG;
      const unsigned w = (unsigned)(heads * a.dv_blocks * (a.n_pieces > 1 ? a.n_pieces : 1) * (MODE == 0 ? 1 : MODE == 1 ? a.nseg - 1 : a.nseg));
      width = w > width ? w : width;
    }
    const dim3 grid(width, (unsigned)n), block(64 * (MODE == 1 ? NW : waves));
    const size_t l = MODE == 1 ? lds_states : lds;
    if constexpr (can_leave_parts && MODE != 1) {
      bool parts = false;
      for (int i = 0; i < n; i++) parts = parts || all.s[i].o_add || all.s[i].o_part;
      if (parts) {
        if (n > 1) hipLaunchKernelGGL((linear_fwd_kernel<DK, NWH, HG, MODE, 4>), grid, block, l, stream, all);
        else hipLaunchKernelGGL((linear_fwd_kernel<DK, NWH, HG, MODE, 3>), grid, block, l, stream, all.s[0]);
        return;
      }
    }
    if (n > 1) hipLaunchKernelGGL((linear_fwd_kernel<DK, NWH, HG, MODE, 2>), grid, block, l, stream, all);
    else if (gen) hipLaunchKernelGGL((linear_fwd_kernel<DK, NWH, HG, MODE, 1>), grid, block, l, stream, all.s[0]);
    else hipLaunchKernelGGL((linear_fwd_kernel<DK, NWH, HG, MODE>), grid, block, l, stream, all.s[0]);
  }

  // n scans side by side (see linear_scans_dispatch; more than one: all with the general addressing).
  // query != null: only report the workspace the launch would use
  static int run(const LinArgs* scans, int n, int want_segments, void* ws, size_t ws_size, hipStream_t stream, size_t* query) {
    int resident = 1, cus = 256;
    if (!prepare(resident, cus)) {
      if (query) { *query = 0; return 0; }
      return -1;
    }
    LinScans all{};
    bool gen = n > 1;
    int64_t all_groups = 0;
    for (int i = 0; i < n; i++) {
      all.s[i] = scans[i];
      gen = gen || general(scans[i]);
      all_groups += groups(scans[i]);
    }
    for (int i = 0; i < n; i++) {
      if (gen) {
        if (const int rc = fill(all.s[i])) return rc;
      } else {
        all.s[i].dv_blocks = scans[i].Dv / (32 * NWH);
      }
    }
    const LinArgs& a = all.s[0];
    int nseg = 1, seg_chunks = 0;
    plan(a, all_groups, want_segments, resident, cus, nseg, seg_chunks);
    const Tail tail = nseg <= 1 && n == 1 ? tail_plan(a, want_segments, resident, cus) : Tail{0, 0, 1, 0};
    size_t need = 0;
    for (int i = 0; i < n; i++) need += ws_bytes(all.s[i], nseg);
    if (query) {
      *query = tail.tail_bg > 0 ? tail_ws_bytes(tail, a.dv_blocks) : need;
      return 0;
    }
    if (nseg > 1 && (!ws || ws_size < need || ((uintptr_t)ws & 3) != 0)) nseg = 1;   // no workspace: single pass
    if (nseg <= 1 && tail.tail_bg > 0 && ws && ws_size >= tail_ws_bytes(tail, a.dv_blocks) && ((uintptr_t)ws & 3) == 0) {
      // the full rounds in a single pass, then the tail in segments (see tail_plan)
      LinScans full = all;
      full.s[0].nseg = 1;
      full.s[0].bg0 = 0;
      full.s[0].bg_n = tail.full_bg;
      launch<0>(full, 1, gen, stream);
      LinScans rest = all;
      LinArgs& r = rest.s[0];
      r.nseg = tail.nseg;
      r.seg_chunks = tail.seg_chunks;
      r.bg0 = tail.full_bg;
      r.bg_n = tail.tail_bg;
      r.ws_state = (float*)ws;
      r.ws_decay = r.ws_state + (int64_t)tail.tail_bg * a.dv_blocks * (tail.nseg - 1) * NW * ws_wave_floats;
      launch<1>(rest, 1, gen, stream);
      launch<2>(rest, 1, gen, stream);
    } else if (nseg <= 1) {
      // scans that each fill whole rounds of the device gain nothing side by side and lose some of the L2 (B8 H16 T2048 256 / 512,
      // forward + backward: 1520 us one after the other, 1536 side by side)
      bool whole_rounds = true;
      for (int i = 0; i < n; i++) {
        all.s[i].nseg = 1;
        whole_rounds = whole_rounds && groups(all.s[i]) % ((int64_t)resident * cus) == 0;
      }
      if (!whole_rounds) {
        launch<0>(all, n, gen, stream);
      } else {
        for (int i = 0; i < n; i++) {
          LinScans one{};
          one.s[0] = all.s[i];
          launch<0>(one, 1, gen, stream);
        }
      }
    } else {
      // the scans' states behind each other, then their decays
      float* at = (float*)ws;
      int64_t widest = 0;
      for (int i = 0; i < n; i++) {
        all.s[i].nseg = nseg;
        all.s[i].seg_chunks = seg_chunks;
        all.s[i].ws_state = at;
        at += groups(all.s[i]) * (nseg - 1) * NW * ws_wave_floats;
        widest = groups(all.s[i]) > widest ? groups(all.s[i]) : widest;
      }
      // With direct sums the last segment reads nseg - 1 states, one behind the other; the scan reads and writes each once but
      // is a launch.  Measured (direct, scan): 256 / 512 with 8 segments 78.2, 68.5 us, 256 / 256 with 4 segments 75.1, 81.1,
      // 128 / 128 with 8 segments 26.7, 29.1 us.
      const bool scan = nseg >= (DK > 128 ? 8 : 9) && ((uintptr_t)ws & 15) == 0 && widest <= 65535;
      for (int i = 0; i < n; i++) {
        all.s[i].ws_decay = at;
        at += (int64_t)a.B * a.H * (nseg - 1);
        all.s[i].ws_entering = scan;
      }
      launch<1>(all, n, gen, stream);
      if (scan)
        hipLaunchKernelGGL(linear_states_kernel, dim3((unsigned)(NW * ws_wave_floats / 1024), (unsigned)widest, (unsigned)n), dim3(256), 0, stream, all,
                           (int)(NW * ws_wave_floats), (int)(NWH * ws_wave_floats), HG);
      launch<2>(all, n, gen, stream);
    }
    return launch_status();
  }
};
}  // namespace

// the instantiation for a problem: key width x waves of 32 value columns (x heads of a workgroup)
namespace {
enum LinConfig { kNone, kC256x8, kC256x4, kC256x2, kC128x8, kC128x4, kC128x2x2, kC128x2 };
LinConfig linear_config(const LinArgs& a, int dk) {
  // two heads per workgroup when they share their q and k heads (Mamba2: all heads of a batch entry do)
  const bool pairable = a.H % 2 == 0 && (a.H / a.Hq) % 2 == 0 && (a.H / a.Hk) % 2 == 0 && (a.Hv == 0 || a.Hv == a.H);
  const int dv = a.Dv;
  if (dk == 256) return dv % 256 == 0 ? kC256x8 : dv % 128 == 0 ? kC256x4 : dv % 64 == 0 ? kC256x2 : kNone;
  if (dk == 128) return dv % 256 == 0 ? kC128x8 : dv % 128 == 0 ? kC128x4 : dv % 64 != 0 ? kNone : pairable ? kC128x2x2 : kC128x2;
  return kNone;
}
}  // namespace

// returns 0 ok, -1 launch failure, -2 unsupported.  With query != null nothing is launched and *query
// receives the workspace size the same call would use.
static int run_scans(const LinArgs* scans, int n, int dk, int want_segments, void* ws, size_t ws_size, hipStream_t stream, size_t* query) {
  switch (linear_config(scans[0], dk)) {
    case kC256x8: return Config<256, 8, 1>::run(scans, n, want_segments, ws, ws_size, stream, query);
    case kC256x4: return Config<256, 4, 1>::run(scans, n, want_segments, ws, ws_size, stream, query);
    case kC256x2: return Config<256, 2, 1>::run(scans, n, want_segments, ws, ws_size, stream, query);
    case kC128x8: return Config<128, 8, 1>::run(scans, n, want_segments, ws, ws_size, stream, query);
    case kC128x4: return Config<128, 4, 1>::run(scans, n, want_segments, ws, ws_size, stream, query);
    case kC128x2x2: return Config<128, 2, 2>::run(scans, n, want_segments, ws, ws_size, stream, query);
    case kC128x2: return Config<128, 2, 1>::run(scans, n, want_segments, ws, ws_size, stream, query);
    default: return -2;
  }
}

int linear_fwd_dispatch(const LinArgs& a, int dk, int want_segments, void* ws, size_t ws_size, hipStream_t stream, size_t* query) {
  return run_scans(&a, 1, dk, want_segments, ws, ws_size, stream, query);
}

bool linear_scans_together(const LinArgs* scans, int n, int dk) {
  for (int i = 1; i < n; i++)
    if (linear_config(scans[i], dk) != linear_config(scans[0], dk)) return false;
  return n <= kLinScans;
}

int linear_scans_dispatch(const LinArgs* scans, int n, int dk, void* ws, size_t ws_size, hipStream_t stream, size_t* query) {
  return run_scans(scans, n, dk, 0, ws, ws_size, stream, query);
}

}  // namespace ma
