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
// that the chunk kernel of bf16 tokens at head size 64 does not take, and at
// least 32 tokens in the longest sequence. Measured (us per token / pieces):
//                            16 tokens    24 tokens    32 tokens    64 tokens
//   D = 64,  1 x 32 heads    10.0 / 12.2  12.7 / 14.4  15.4 / 14.1  26.1 / 17.8
//   D = 64,  9 x 32 heads    18.6 / 18.5  24.7 / 22.9  30.5 / 23.5  54.3 / 35.9
//   D = 64,  64 x 32 heads   58.2 / 59.9  79.3 / 74.2  99.0 / 76.9   184 / 151
//   D = 128, 64 x 16 heads   94.5 / 94.1   130 / 122    165 / 125    312 / 218
//   D = 256, 64 x 8 heads     218 / 179    298 / 279    377 / 286    697 / 458
// Calls whose tiles would take more than 2 GiB stay on the per-token kernel.
constexpr int32_t kPiece32MinSeqlen = 32;
constexpr size_t kPiece32RecurrentBytes = size_t{2} << 30;
inline bool piece32_recurrent(int io_dtype, int decay_mode, int head_size, int32_t max_seqlen) {
  const bool head = head_size == 64 || head_size == 128 || head_size == 256;
  return decay_mode == FRWKV_DECAY_LOGITS && head && max_seqlen >= kPiece32MinSeqlen &&
         (io_dtype == FRWKV_DTYPE_F16 || (io_dtype == FRWKV_DTYPE_BF16 && head_size != 64));
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
