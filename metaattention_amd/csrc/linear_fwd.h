// Kernel-side argument block of the chunked linear attention forward kernel.
#pragma once
#include "common.h"

namespace ma {

struct LinArgs {
  const void* q; const void* k; const void* v; void* o;
  const float* log_decay;  // [B,H,T]
  const float* v_scale;    // [B,H,T] or null (v_scale_bf16, set only with a scale: bf16)
  float q_scale;
  int B, H, Hq, Hk, T, Dv, dv_blocks;
  // sequence segments (see linear_fwd.hip): nseg segments of seg_chunks 32-token chunks; local end
  // states [group][segment][wave][registers][lane] fp32 and per-(batch*head, segment) log decays
  int nseg, seg_chunks;
  int out_f32;   // 1: o is fp32 [B,H,T,Dv] instead of bf16; 2: fp32, and the result is added to what o holds
  // General operand addressing (the backward's scans; all zero: q [B,Hq,T,Dk], k [B,Hk,T,Dk], v [B,H,T,Dv] as they
  // are): rev = the operands are read in reversed time order (token T-1-t at position t); q_row / k_row / v_row = elements
  // between consecutive tokens of an operand (a column slice of a wider tensor: the pointer carries the column offset);
  // Hv = heads of v (dividing H: head h reads v head h / (H / Hv)).
  int rev, Hv;
  int64_t q_row, k_row, v_row;
  // qk_cols (general addressing only; 0: all Dk): the q and k operands hold only this many columns (a multiple of 32); the
  // rest of the Dk-wide contraction is zeros that are never loaded (the tiles' LDS is cleared once, the loads of the missing
  // columns are switched off).
  int qk_cols;
  // rev_o (general addressing only): the outputs are written in reversed time order (row T-1-t holds the scan's token t), so
  // that a scan over reversed operands leaves its result in the operands' own order.
  int rev_o;
  // pieces (general addressing only; 0 or 1: none): the launch runs n_pieces independent scans side by side, piece p with
  // its q and k pointers moved on by p * piece_qk elements (the next slice of the contraction's columns) and its output
  // (fp32) by p * piece_o elements; the caller adds the pieces' outputs up.
  int n_pieces;
  int64_t piece_qk, piece_o;
  // o_part, o_add (general addressing and the pipelined chunk loop only; null: none): the pieces of a contraction in turn.  o_part: the
  // outputs go there, fp32, instead of to o; o_add: what an earlier piece left is added to the outputs (before they are rounded).  Both
  // in the order of the accumulators, [batch * head][value slice][chunk of 32 tokens][wave][4][64 lanes] x 16 bytes (the last chunk's
  // missing tokens included): a wave writes and reads whole lines, without a trip through LDS.
  float* o_part;
  const float* o_add;
  float* ws_state;
  float* ws_decay;
  int ws_entering;   // ws_state holds, in slot s, the state that segment s + 1 is entered with (linear_states_kernel), not the one segment s ends in
  // head-group range of this launch (a workgroup handles head group bg0 + its own index; bg_n groups in all; bg_n = 0: every
  // group, from 0).  The workspace of a launch with sequence segments is indexed by the launch's own group index.
  int bg0, bg_n;
  // (not with general addressing) what log_decay holds where it is not the log decay itself: its exponential (decay_log), or the log decay over a head's factor
  // (decay_head [H] or null)
  int v_scale_bf16, decay_log;
  const float* decay_head;
};

// Scans that go out in one launch (general addressing): scan i is blockIdx.y = i.
constexpr int kLinScans = 3;
struct LinScans {
  LinArgs s[kLinScans];
};

// n scans of the same B, H, T, kernel width dk and value-slice configuration, independent of each other; ws holds
// linear_scans_ws_bytes of them (n = 1: what linear_fwd_dispatch asks for).  Returns as linear_fwd_dispatch.
bool linear_scans_together(const LinArgs* scans, int n, int dk);
int linear_scans_dispatch(const LinArgs* scans, int n, int dk, void* ws, size_t ws_size, hipStream_t stream, size_t* query);

int linear_fwd_dispatch(const LinArgs& a, int dk, int want_segments, void* ws, size_t ws_size, hipStream_t stream, size_t* query);

}  // namespace ma
