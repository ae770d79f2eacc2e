// fp32 matrix form of the recurrence over 16-token pieces (piece32.hip): the
// route of long calls whose contract is fp32 arithmetic (the fp32-state
// recurrence on fp16 tokens or at head sizes 128 and 256, and training at head
// size 256), given scratch memory.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "../../include/flashrwkv_amd.h"

namespace frwkv {

struct Piece32Params {
  int32_t num_heads;
  int32_t num_sequences;
  int32_t total_tokens;
  // Token layout, one of: cu_seqlens (packed sequences); seg_offsets, starts
  // and ends (caller chunks); dense_t (sequence s holds tokens s * dense_t ..).
  const int32_t* cu_seqlens;
  const int32_t* seg_offsets;
  const int32_t* seg_starts;
  const int32_t* seg_ends;
  int32_t num_segments;
  int32_t dense_t;
  // State: [slots, H, D, D] fp32, in place at slots[s] (null: s); null: zero
  // start and no final state.
  float* state;
  const int32_t* slots;
  int32_t state_slots;
  const int32_t* status;  // metadata status word, or null
  const void* r;
  const void* decay;  // logits
  const void* bias;
  const void* k;
  const void* v;
  const void* a;
  const void* b;
  void* out;
  int64_t out_elems;
  float scale;
  // Training: the state at each caller chunk start ([num_segments, H, D, D]),
  // or every 16 tokens of the dense layout ([B, H, T / 16, D, D]); at further
  // piece starts inside a caller chunk, at slot (piece start) / 16 of
  // interior; and a^T S_{t-1} ([N, H, D]). Written by the forward, read by the
  // backward. Null: not wanted.
  float* boundary;
  float* interior;
  float* state_dot_a;
  // Backward.
  const void* dy;             // or null (zero)
  const float* dstate_final;  // or null (zero)
  void* dr;
  void* ddecay;
  void* dk;
  void* dv;
  void* da;
  void* db;
  float* dstate0;  // or null
  // Scratch areas (piece32_forward_bytes / piece32_backward_bytes).
  int4* table;      // caller chunks: {first token, tokens, chunk, piece of chunk} per piece
  int32_t* base;    // caller chunks: first piece of each chunk, [num_segments + 1], then
                    // 1 if the chunks have more pieces than there are slots
  // [H, piece slots]: 1 where the piece holds a value that is not finite (or
  // products of its tokens overflow). Such a unit runs token by token.
  uint32_t* flags;
  int32_t slots_total;
  float* tiles;     // operand tiles per (piece, head)
  float* adjoints;  // backward: dS at the piece end per (piece, head), [D, D]
  float* dz;        // backward: dZ per (piece, head), [16, D]
};

// Piece slots of a call: packed or dense sequences of `tokens` tokens in all
// in `lists` sequences, or caller chunks of `tokens` tokens in `lists` chunks.
inline int64_t piece32_slots(int64_t tokens, int64_t lists) { return tokens / 16 + lists; }

// The recurrent operator's calls on this route: decay logits, 16-bit tokens
// that the chunk kernel of bf16 tokens at head size 64 does not take, at least
// 32 tokens in the longest sequence, and less time than the per-token kernel by
// the estimates below (us), which tell batches with long prompts from decoding
// batches with a short one. Both follow measured calls of 1 to 256 sequences
// within 30%, and within 10% where the two are close (us per token / pieces;
// "+": single tokens beside one prompt):
//                            16 tokens    32 tokens    64 tokens
//   D = 64,  1 x 32 heads    10.0 / 12.2  15.4 / 14.1  26.1 / 17.8
//   D = 64,  9 x 32 heads    18.6 / 18.5  30.5 / 23.5  54.3 / 35.9
//   D = 64,  64 x 32 heads   58.2 / 59.9  99.0 / 76.9   184 / 151
//   D = 128, 64 x 16 heads   94.5 / 94.1   165 / 125    312 / 218
//   D = 256, 64 x 8 heads     218 / 179    377 / 286    697 / 458
//                            32 tokens    128 tokens   512 tokens
//   D = 64,  63 + 1, 32 h.   33.4 / 53.5  75.8 / 63.9   251 / 107
//   D = 64,  255 + 1, 32 h.  78.2 / 191    121 / 207    295 / 256
//   D = 128, 63 + 1, 16 h.   55.4 / 87.3   120 / 106    380 / 186
//   D = 256, 63 + 1, 8 h.     111 / 175    223 / 205    674 / 358
// Calls whose tiles would take more than 2 GiB stay on the per-token kernel.
constexpr int32_t kPiece32MinSeqlen = 32;
constexpr size_t kPiece32RecurrentBytes = size_t{2} << 30;

// Per token: every unit's state once (0.0073 us per 16 KiB), and the longest
// sequence's chain, whose step is longer where several waves share a SIMD. The
// tokens in all make up `full` units of the longest length.
inline double per_token_time(int head_size, double units, double full, double longest) {
  const double wide = head_size / 64.0;
  const double waves = __builtin_ceil(full * (head_size / 16) / 1024);
  double step = head_size == 64    ? 0.14 + 0.307 * waves
                : head_size == 128 ? 0.115 + 0.56 * waves
                                   : 1.22 * waves;
  if (head_size == 64 && units * 8 <= 1024) step = 0.343;  // 8-column slabs
  return 4.5 + 0.0073 * wide * wide * units + longest * step;
}
// Pieces: every unit's state and workgroups, every piece's tiles, and the chain,
// in as many rounds as its workgroups (two per CU) need. Sequences other than
// the longest have at least one piece each, and end in half a one.
inline double piece32_time(int head_size, double sequences, double heads, double total,
                           double longest) {
  const double wide = head_size / 64.0;
  const double chain = __builtin_ceil(longest / 16);
  double rest = (total - longest) / 16 + 0.5 * (sequences - 1);
  if (rest < sequences - 1) rest = sequences - 1;
  const double pieces = (chain + rest) * heads;
  double rounds = pieces / chain * wide * wide / 512;
  if (rounds < 1) rounds = 1;
  const double step = head_size == 64 ? 1.86 : head_size == 128 ? 2.31 : 2.38;
  const double unit = head_size == 64 ? 0.012 : head_size == 128 ? 0.048 : 0.30;
  const double tile = head_size == 64 ? 0.0075 : head_size == 128 ? 0.0135 : 0.025;
  return 10 + step * chain * rounds + unit * sequences * heads + tile * pieces;
}

inline bool piece32_recurrent(int io_dtype, int decay_mode, int head_size, int32_t sequences,
                              int32_t heads, int32_t total, int32_t longest) {
  const bool head = head_size == 64 || head_size == 128 || head_size == 256;
  if (decay_mode != FRWKV_DECAY_LOGITS || !head || longest < kPiece32MinSeqlen ||
      !(io_dtype == FRWKV_DTYPE_F16 || (io_dtype == FRWKV_DTYPE_BF16 && head_size != 64))) {
    return false;
  }
  if (longest > total) longest = total;
  const double units = static_cast<double>(sequences) * heads;
  return piece32_time(head_size, sequences, heads, total, longest) <
         per_token_time(head_size, units, static_cast<double>(total) * heads / longest, longest);
}

size_t piece32_forward_bytes(int head_size, int64_t heads, int64_t tokens, int64_t lists);

// Lays out p's scratch areas and launches. head_size 64, 128 or 256; 16-bit io.
int piece32_forward(Piece32Params p, int head_size, int io_dtype, void* scratch,
                    hipStream_t stream);

// Backward at head size 256, from the forward's boundary, interior (chunks
// longer than 16 tokens) and state_dot_a.
size_t piece32_backward_bytes(int64_t heads, int64_t tokens, int64_t lists);
int piece32_backward(Piece32Params p, int io_dtype, void* scratch, hipStream_t stream);

}  // namespace frwkv
