// Sequence parts: the chunked kernels on few, long sequences.
//
// A chunked kernel walks one (sequence, head) with one workgroup, so a launch
// of few sequences leaves most CUs idle for the whole serial chain of chunks.
// The recurrence is affine in the state, so a run of chunks ("part") maps its
// start state to its end state as S -> M S + N, with a 64 x 64 map M over the
// keys that does not depend on the value columns. A split call is two
// launches:
//   1. chunk_transfer_kernel, one workgroup per part but the last of its
//      sequence: M and N of the part, both by walking its chunks as the main
//      kernel does (N from a zero state, M from the identity with V = 0,
//      without outputs). The first part starts from the real state, so it
//      gives its end state directly and needs no map;
//   2. the main kernel, one workgroup per part: part j composes its start
//      state from the first part's end state and the maps of parts
//      1 .. j - 1 in fp32 (compose_start), then walks its chunks.
// The work is about twice that of the unsplit kernel, over `parts` times the
// workgroups.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "chunk_common.h"

namespace frwkv {

struct ChunkFwdParams {
  int32_t num_heads;
  // Packed varlen batches of at most 64 sequences (cu_seqlens mode) run
  // their sequences longest first: workgroup b takes the sequence of length
  // rank b / H. 0 keeps the natural order.
  int32_t longest_first_sequences;
  int32_t total_tokens;
  int32_t state_slots;
  const int32_t* cu_seqlens;    // sequence token ranges when seg_offsets == null
  const int32_t* seg_offsets;   // [B+1] segment lists (StateTune chunks) or null
  const int32_t* seg_starts;
  const int32_t* seg_ends;
  int32_t num_segments;         // length of seg_starts / seg_ends / boundary
  const int32_t* slots;         // [B] state slot per sequence, or null (identity)
  const int32_t* status;        // metadata status word, or null
  void* state;
  const void* r;
  const void* decay;
  const void* bias;
  const void* k;
  const void* v;
  const void* a;
  const void* b;
  void* out;
  float* boundary;              // state at each segment start, or null
  float* state_dot_a;           // per-token a^T S_{t-1}, or null
  float scale;
  int64_t out_elems;
  // Dense layout: > 0 means every sequence has dense_t tokens (sequence s
  // covers tokens s * dense_t ..), with no cu_seqlens or segment arrays.
  int32_t dense_t;
  // 1: boundary is [B, H, dense_t / 16, D, D], the state every 16 tokens.
  int32_t boundary16;
  // 1: the initial states are read and never written back (replay from
  // stored boundaries).
  int32_t read_only_state;
  // [ceil(total_tokens / 64), H, D, D] or null: the state at every 64-token
  // piece start inside a segment (not at the segment start), at slot
  // (piece start) / 64. Interior starts of different segments lie more than
  // 64 tokens apart, so the slots are distinct.
  float* interior;
  // 1 (replay layout, one segment per unit): only the interior states are
  // wanted; segments of at most 64 tokens have none and are skipped, and a
  // segment's last piece is not computed.
  int32_t fill_only;
  // Sequence parts (chunk_parts.h): every sequence's chunks are cut into runs
  // of part_len chunks (longer ones where a sequence would need more than
  // `parts` runs), one workgroup each; part_states holds the runs' transfer
  // states. parts is 1 and part_states null otherwise.
  int32_t parts;
  int32_t part_len;
  float* part_states;
};

constexpr int kMinParts = 3;
constexpr int kMaxParts = 16;

constexpr int kStateElems = kHead * kHead;

// States of part `part` of unit (sequence, head) `unit`: [M][N], 64 x 64 fp32
// each, row-major over keys. Part 0 keeps the sequence's start state in place
// of M (the pool is overwritten by the last part while the first one still
// needs it) and its end state in place of N. The last part has none.
__device__ __forceinline__ float* part_state(const ChunkFwdParams& p, int unit, int part,
                                             int which) {
  return p.part_states +
         ((static_cast<int64_t>(unit) * (p.parts - 1) + part) * 2 + which) * kStateElems;
}

// Part `part` of a sequence's `count` items (64-token chunks, or caller
// chunks): items [begin, end), the same split in both launches. Part 0 exists
// always, the others when they have an item.
struct PartRange {
  int begin, end;
  bool exists, last;
};
__device__ __forceinline__ PartRange part_range(const ChunkFwdParams& p, int count, int part) {
  const int per = max((count + p.parts - 1) / p.parts, p.part_len);
  PartRange r;
  r.begin = min(part * per, count);
  r.end = min(r.begin + per, count);
  r.exists = part == 0 || r.begin < count;
  r.last = r.end >= count;
  return r;
}

// How a call is split: at most `parts` parts of `len` chunks each.
struct PartPlan {
  int32_t parts, len;
};

// Measured time of one chunk step of a kernel (us): with at most one workgroup
// per CU (256 CUs), and with two on each, in proportion between. Further
// workgroups wait for a place, and the last round of them fills the GPU only
// in part (768 workgroups of equal length took 1.8 times as long as 512, 1024
// 2.6 times). A kernel whose LDS admits one per CU starts a second round
// beyond 256 (`rounds`).
struct ChunkTime {
  double alone, shared;
  bool rounds;
  double of(double workgroups) const {
    if (workgroups <= 256) return alone;
    if (workgroups > 512) return shared * (1.0 + 1.6 * (workgroups / 512 - 1.0));
    return rounds ? shared : alone + (shared - alone) * (workgroups - 256) / 256;
  }
};
constexpr ChunkTime kForwardTime{5.2, 7.2, false};
constexpr ChunkTime kPreciseTime{6.4, 12.8, true};
constexpr ChunkTime kTransferTime{5.2, 8.3, false};

// The split of a call of `heads` heads whose sequences have `chunks` chunks in
// all and at most `longest` each: the part length with the least estimated
// time of both launches (every chunk is walked by each, and composing a part's
// start state costs about a fifth of a chunk per part), if that beats the
// unsplit kernel. Measured, one sequence of 32 heads (unsplit / split): 4
// chunks 29 / 22 us (split-precision), 16 chunks 89 / 39, 64 chunks 331 / 88;
// two parts never paid (170 / 162), four paid up to 128 units (64 chunks
// 337 / 237), and at 256 units no split did (32 chunks 177 / 204).
inline PartPlan plan_parts(int64_t sequences, int64_t heads, int64_t chunks, int64_t longest,
                           const ChunkTime& main, const ChunkTime& transfer) {
  PartPlan best{1, 0};
  if (sequences <= 0 || heads <= 0 || chunks <= 0 || longest <= 2) return best;
  const double units = static_cast<double>(sequences) * heads;
  double least = longest * (units <= 512 ? main.of(units) : main.alone);
  const double full = static_cast<double>(chunks) * heads * main.shared / 512;
  if (least < full) least = full;
  least *= 0.95;
  for (int32_t parts = kMinParts; parts <= kMaxParts; ++parts) {
    const int64_t len = (longest + parts - 1) / parts;
    if ((longest + len - 1) / len != parts) continue;
    // The last part of a sequence of a ragged batch is half full on average.
    const bool ragged = len > 1 && chunks < longest * sequences;
    const double groups = heads * (static_cast<double>(chunks) / len +
                                   (ragged ? 0.5 * (sequences - 1) : 0.0));
    const double time =
        5.0 + (len + 0.2 * parts) * main.of(groups) + len * transfer.of(groups - units);
    if (time < least) {
      least = time;
      best = PartPlan{parts, static_cast<int32_t>(len)};
    }
  }
  return best;
}

// Bytes of part states of a split call (0 when it does not split).
inline size_t part_bytes(int64_t units, const PartPlan& plan) {
  return plan.parts > 1 ? static_cast<size_t>(units) * (plan.parts - 1) * 2 * kStateElems *
                              sizeof(float)
                        : 0;
}

// Splits the call when the caller's scratch holds its part states.
inline void use_parts(ChunkFwdParams& p, int64_t units, const PartPlan& plan, void* scratch,
                      size_t scratch_bytes) {
  const bool split = plan.parts > 1 && scratch != nullptr &&
                     scratch_bytes >= part_bytes(units, plan);
  p.parts = split ? plan.parts : 1;
  p.part_len = split ? plan.len : 0;
  p.part_states = split ? static_cast<float*>(scratch) : nullptr;
}

inline int64_t chunks_of(int64_t tokens) {
  return tokens > 0 ? (tokens + kChunk - 1) / kChunk : 0;
}

// The plan of a call with caller chunks, whose lengths are on the device: by
// the mean chunk count (a longer sequence gets as many, longer parts).
inline PartPlan plan_caller_chunks(int64_t sequences, int64_t heads, int64_t chunks) {
  if (sequences <= 0) return PartPlan{1, 0};
  return plan_parts(sequences, heads, chunks, (chunks + sequences - 1) / sequences, kForwardTime,
                    kTransferTime);
}

// Launches chunk_transfer_kernel (chunk_transfer.hip) for p.parts > 1.
template <typename T, DecayMode M, typename PoolT, bool kPrecise>
int launch_chunk_transfer(const ChunkFwdParams& p, int units, hipStream_t stream);

}  // namespace frwkv
