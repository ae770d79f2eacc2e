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
// workgroups. A sequence of one part takes no transfer and no part states.
//
// The backward's state adjoint is affine in the adjoint behind it, so it is
// split the same way from the end: part 0 is a sequence's last run of chunks,
// chunk_adjoint_kernel gives dS_start = M dS_end + N of each part, and the
// backward kernel composes the adjoint at its part's end.
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
  // Packed sequences: their number, and the slots of a head (0: states by unit).
  int32_t packed_sequences;
  int32_t part_slots;
};

struct ChunkBwdParams {
  int32_t num_heads;
  int32_t total_tokens;
  int32_t num_segments;
  const int32_t* seg_offsets;
  const int32_t* seg_starts;
  const int32_t* seg_ends;
  const float* checkpoint;      // [num_segments, H, 64, 64]: state at each segment start
  const float* interior;        // [ceil(N/64), H, 64, 64] piece-start states, or null
  const void* r;
  const void* decay;
  const void* bias;
  const void* k;
  const void* v;
  const void* a;
  const void* b;
  const void* dy;               // or null (zero)
  const float* dstate_final;    // or null (zero)
  void* dr;
  void* ddecay;
  void* dk;
  void* dv;
  void* da;
  void* db;
  float* dstate0;               // or null (not needed)
  float scale;
  // Dense layout: > 0 means every sequence has dense_t tokens (one segment)
  // and checkpoint is [B, H, dense_t / 16, D, D], the state every 16 tokens.
  int32_t dense_t;
  // Sequence parts (see above): part 0 is a sequence's last run of chunks.
  int32_t parts;
  int32_t part_len;
  float* part_states;
};

constexpr int kMinParts = 3;
constexpr int kMaxParts = 16;

constexpr int kStateElems = kHead * kHead;
// A part's states are [M][N], 64 x 64 each, row-major over keys: M as three bf16
// planes, M = hi + mid + lo exactly (split3_bf16x2), as compose_start multiplies
// it (every later part reads it, so it is split once here), N in fp32. Sizes in
// floats.
constexpr int kMapElems = 3 * kStateElems / 2;
constexpr int kPartElems = kMapElems + kStateElems;

// Where a part's workgroup is: its (sequence, head), its part, and the states
// of the unit's parts. Part 0 keeps the sequence's start state in place of M
// (the pool is overwritten by the last part while the first one still needs it)
// and its end state in place of N, both fp32. The last part has none.
struct PartPlace {
  int seq, head, part;
  float* states;
  int64_t step;  // from one part's states to the next
  __device__ __forceinline__ float* state(int i, int which) const {
    return states + i * step + which * kMapElems;
  }
};

// Packed sequences: sequence s has its states at slots part_slot(s) .. of each
// head. It needs at most ceil(chunks / len) - 1 = floor((tokens - 1) / (64 len))
// of them, so the slots of disjoint, ascending sequences are disjoint and below
// floor(total_tokens / (64 len)), and short sequences have none.
__device__ __forceinline__ int part_slot(const ChunkFwdParams& p, int seq) {
  return max(p.cu_seqlens[seq], 0) / (kChunk * p.part_len);
}
// The sequence that owns a slot (or the last one that starts at or before it).
// Every lane tries one of 64 equal steps, so 64 sequences take one round.
__device__ __forceinline__ int sequence_of_part_slot(const ChunkFwdParams& p, int slot,
                                                     int lane) {
  int lo = 0, hi = p.packed_sequences;
  while (hi - lo > 1) {
    const int stride = (hi - lo + 63) / 64;
    const int s = lo + lane * stride;
    const bool before = s < hi && part_slot(p, s) <= slot;
    const int count = max(__builtin_popcountll(__builtin_amdgcn_ballot_w64(before)), 1);
    lo = uniform(lo + (count - 1) * stride);
    hi = min(lo + stride, hi);
  }
  return lo;
}
// Blocks (slot, head): the parts with a successor (kTransfer) or, in the main
// launch, those with a predecessor, followed by every sequence's first part.
template <bool kTransfer>
__device__ __forceinline__ PartPlace packed_place(const ChunkFwdParams& p, int lane) {
  PartPlace at;
  const int blocks = p.part_slots * p.num_heads;
  const int block = static_cast<int>(blockIdx.x);
  int first;
  if (kTransfer || block < blocks) {
    const int slot = block / p.num_heads;
    at.head = block % p.num_heads;
    at.seq = sequence_of_part_slot(p, slot, lane);
    first = uniform(part_slot(p, at.seq));
    at.part = slot - first + (kTransfer ? 0 : 1);
  } else {
    at.seq = (block - blocks) / p.num_heads;
    at.head = (block - blocks) % p.num_heads;
    at.part = 0;
    first = uniform(part_slot(p, at.seq));
  }
  at.step = static_cast<int64_t>(p.num_heads) * kPartElems;
  at.states = p.part_states + first * at.step + at.head * kPartElems;
  return at;
}
// Dense sequences and caller chunks: block part * units + unit, so that (for a
// unit count divisible by the 8 XCDs) a unit's parts share an XCD, and its L2,
// in both launches.
template <bool kTransfer, typename P>
__device__ __forceinline__ PartPlace unit_place(const P& p) {
  PartPlace at;
  const uint32_t units = gridDim.x / (kTransfer ? p.parts - 1 : p.parts);
  const uint32_t unit = blockIdx.x % units;
  at.part = blockIdx.x / units;
  at.seq = unit / p.num_heads;
  at.head = unit % p.num_heads;
  at.step = kPartElems;
  at.states = p.part_states + static_cast<int64_t>(unit) * (p.parts - 1) * at.step;
  return at;
}

// Part `part` of a sequence's `count` items (64-token chunks, or caller
// chunks): items [begin, end), the same split in both launches. Part 0 exists
// always, the others when they have an item.
struct PartRange {
  int begin, end;
  bool exists, last;
};
template <typename P>
__device__ __forceinline__ PartRange part_range(const P& p, int count, int part) {
  const int per = max((count + p.parts - 1) / p.parts, p.part_len);
  PartRange r;
  r.begin = min(part * per, count);
  r.end = min(r.begin + per, count);
  r.exists = part == 0 || r.begin < count;
  r.last = r.end >= count;
  return r;
}

// Start state of part `part`, columns 16w .. of the wave (w = wave % 4) in C
// layout (S[kb][j]: row 16kb + 4g + j, column 16w + n): part 0 takes the kept
// start state, part j the first part's end state through the maps of parts
// 1 .. j - 1, S <- M_i S + N_i. All waves need all of each map, so maps go
// through LDS (tiles: kComposeBytes, not yet in use), two at a time, and the
// state is split into three bf16 as they are: M S is the six products of at
// least 2^-16 times the whole, so the state is carried at fp32's precision, as
// it is from chunk to chunk. The next two maps are loaded while these are
// applied.
constexpr int kComposeMaps = 2;
constexpr size_t kComposeBytes = kComposeMaps * 3 * kOpTile * sizeof(uint16_t);
template <int kThreads>
__device__ __forceinline__ void compose_start(void* space, const PartPlace& where,
                                              f32x4 (&S)[4]) {
  const int part = where.part;
  constexpr int kShare = kStateElems / kThreads;  // a thread's elements of a map
  constexpr int kPerRow = kHead / kShare;
  const int tid = threadIdx.x;
  const int w = uniform(tid >> 6) & 3;
  const int lane = tid & 63;
  const int g = lane >> 4, n = lane & 15;
  uint16_t* const tiles = static_cast<uint16_t*>(space);  // [map][hi, mid, lo][row][col]
  const int col = (4 * g) * kHead + 16 * w + n;
  auto load_slab = [&](int i, int which, f32x4 (&x)[4]) {
    const float* src = where.state(i, which) + col;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
      for (int j = 0; j < 4; ++j) x[kb][j] = src[(16 * kb + j) * kHead];
    }
  };
  load_slab(0, part > 0 ? 1 : 0, S);
  if (part < 2) return;
  const int share = kShare * tid;
  const int place = (tid / kPerRow) * kOpStride + kShare * (tid % kPerRow);
  uint4 m[kComposeMaps][3][kShare / 8];
  f32x4 off[kComposeMaps][4];
  auto load_maps = [&](int first) {
#pragma unroll
    for (int u = 0; u < kComposeMaps; ++u) {
      if (first + u < part) {
        const uint16_t* src =
            reinterpret_cast<const uint16_t*>(where.state(first + u, 0)) + share;
#pragma unroll
        for (int x = 0; x < 3; ++x) {
#pragma unroll
          for (int c = 0; c < kShare / 8; ++c) {
            m[u][x][c] = *reinterpret_cast<const uint4*>(src + x * kStateElems + 8 * c);
          }
        }
      }
    }
  };
  load_maps(1);
  for (int first = 1; first < part; first += kComposeMaps) {
#pragma unroll
    for (int u = 0; u < kComposeMaps; ++u) {
      if (first + u < part) load_slab(first + u, 1, off[u]);
    }
    if (first > 1) __syncthreads();  // the maps before these are applied
#pragma unroll
    for (int u = 0; u < kComposeMaps; ++u) {
      if (first + u < part) {
        uint16_t* dst = tiles + 3 * u * kOpTile + place;
#pragma unroll
        for (int x = 0; x < 3; ++x) {
#pragma unroll
          for (int c = 0; c < kShare / 8; ++c) {
            const uint4 q = m[u][x][c];
            uint2* to = reinterpret_cast<uint2*>(dst + x * kOpTile + 8 * c);
            to[0] = make_uint2(q.x, q.y);
            to[1] = make_uint2(q.z, q.w);
          }
        }
      }
    }
    __syncthreads();
    load_maps(first + kComposeMaps);
#pragma unroll
    for (int u = 0; u < kComposeMaps; ++u) {
      if (first + u < part) {
        const uint16_t* map = tiles + 3 * u * kOpTile;
        i16x4 s[3][4];
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
          to_operand_split3(S[kb], s[0][kb], s[1][kb], s[2][kb]);
          S[kb] = off[u][kb];
        }
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          const i16x8 bh = cat(s[0][2 * kk], s[0][2 * kk + 1]);
          const i16x8 bm = cat(s[1][2 * kk], s[1][2 * kk + 1]);
          const i16x8 bl = cat(s[2][2 * kk], s[2][2 * kk + 1]);
#pragma unroll
          for (int rb = 0; rb < 4; ++rb) {
            const int row = 16 * rb + n;
            const i16x8 ah = lds_operand32<kOpStride>(map, row, 32 * kk, g);
            const i16x8 am = lds_operand32<kOpStride>(map + kOpTile, row, 32 * kk, g);
            const i16x8 al = lds_operand32<kOpStride>(map + 2 * kOpTile, row, 32 * kk, g);
            S[rb] = mfma32(al, bh, S[rb]);
            S[rb] = mfma32(ah, bl, S[rb]);
            S[rb] = mfma32(am, bm, S[rb]);
            S[rb] = mfma32(am, bh, S[rb]);
            S[rb] = mfma32(ah, bm, S[rb]);
            S[rb] = mfma32(ah, bh, S[rb]);
          }
        }
      }
    }
  }
  __syncthreads();  // before the chunk tiles are written
}

// Stores a wave's columns of a map or an offset (C layout, element (4g, column)
// at `offset` of it): a map of parts 1 .. as planes, all else as fp32.
__device__ __forceinline__ void store_part_state(const PartPlace& where, int part, bool map,
                                                 uint32_t offset, const f32x4 (&S)[4]) {
  float* dst = where.state(part, map ? 0 : 1);
  if (!map || part == 0) {
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
      for (int j = 0; j < 4; ++j) dst[offset + (16 * kb + j) * kHead] = S[kb][j];
    }
    return;
  }
  uint16_t* planes = reinterpret_cast<uint16_t*>(dst) + offset;
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
    for (int j = 0; j < 4; j += 2) {
      const uint3 x = split3_bf16x2(S[kb][j], S[kb][j + 1]);
      uint16_t* row = planes + (16 * kb + j) * kHead;
      row[0] = static_cast<uint16_t>(x.x);
      row[kHead] = static_cast<uint16_t>(x.x >> 16);
      row[kStateElems] = static_cast<uint16_t>(x.y);
      row[kStateElems + kHead] = static_cast<uint16_t>(x.y >> 16);
      row[2 * kStateElems] = static_cast<uint16_t>(x.z);
      row[2 * kStateElems + kHead] = static_cast<uint16_t>(x.z >> 16);
    }
  }
}

// How a call is split: at most `parts` parts of `len` chunks each.
struct PartPlan {
  int32_t parts, len;
};

// Measured time of one chunk step of a kernel (us; the adjoint transfer kernel
// takes 5.9 + 4.9 per chunk): with at most one workgroup per CU (256 CUs), and
// with two on each, in proportion between. Further workgroups wait for a place,
// and the last round of them fills the GPU only in part (768 workgroups of
// equal length took 1.8 times as long as 512, 1024 2.6 times). A kernel whose
// LDS admits one per CU runs in rounds of 256 (`rounds`; 576 workgroups of the
// backward, 2 chunks each, took 82 us, 256 of 5 chunks 64).
// Packed batches add, per sequence or part of one, the start of its workgroup
// (`unit`; with the rank search of at most 64 sequences, `sorted`; with the
// search for its part, `part`) and each map that a part composes (`map`), all
// in the time that a workgroup takes when its CU is shared.
struct ChunkTime {
  double alone, shared;
  bool rounds;
  double unit, sorted, part, map;
  double of(double workgroups) const {
    if (workgroups <= 256) return alone;
    if (rounds) return alone * __builtin_ceil(workgroups / 256);
    if (workgroups > 512) return shared * (1.0 + 1.6 * (workgroups / 512 - 1.0));
    return alone + (shared - alone) * (workgroups - 256) / 256;
  }
};
constexpr ChunkTime kForwardTime{5.2, 7.2, false, 1.0, 6.4, 1.5, 1.5};
constexpr ChunkTime kPreciseTime{5.9, 11.8, true, 4.5, 13.2, 6.6, 2.2};
constexpr ChunkTime kTransferTime{5.2, 8.3, false};
constexpr ChunkTime kBackwardTime{11.5, 23.0, true};
constexpr ChunkTime kAdjointTime{5.2, 8.3, false};

// The split of a call of `heads` heads whose sequences have `chunks` chunks in
// all and at most `longest` each: the part length with the least estimated
// time of both launches (every chunk is walked by each, and composing a part's
// start state costs about a fifth of a forward chunk per part), if that beats
// the unsplit kernel. Measured, one sequence of 32 heads (unsplit / split): 4
// chunks 29 / 22 us (split-precision), 16 chunks 89 / 39, 64 chunks 331 / 88;
// two parts never paid (170 / 162), four paid up to 128 units (64 chunks
// 337 / 237), and at 256 units no split did (32 chunks 177 / 204). Backward
// (unsplit / split): 32 units of 4 chunks 46 / 26, of 16 chunks 170 / 51, of
// 64 chunks 702 / 160; 96 units of 16 chunks 174 / 120, 128 units 182 / 134;
// from 192 units on the estimate keeps it whole.
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
    const bool ragged = chunks < longest * sequences;
    const double groups =
        ragged ? heads * (static_cast<double>(chunks) / len + (len > 1 ? 0.5 * (sequences - 1) : 0))
               : units * parts;
    const double time = 5.0 + len * main.of(groups) + 0.2 * parts * kForwardTime.of(groups) +
                        len * transfer.of(groups - units);
    if (time < least) {
      least = time;
      best = PartPlan{parts, static_cast<int32_t>(len)};
    }
  }
  return best;
}

// The same for packed or dense sequences of `tokens` tokens in all, `longest` in
// the longest. The other lengths are not known: sequences that share the other
// tokens evenly end in half a chunk, and have one chunk at least. A call takes
// the longer of its longest chain and of all its workgroups' work, and a split
// adds work: beside short sequences enough to fill the GPU it pays only where
// the prompt's chain is the longer one by far: the estimate must promise 22%, or
// 5% where every workgroup has a CU at once.
//
// Against every part count, forced, on 142 batches (one to 300 sequences, equal,
// similar, mixed, and prompts beside short ones or single tokens; 12 to 40
// heads): 2.0% (bf16) and 3.0% (split-precision) above the fastest in the mean
// and at most 5% slower than unsplit (at 18% three of 190 others were 6 to 13%
// slower); counting the chunks from the tokens alone, as for caller chunks, 4.2
// and 4.4%, and up to 1.26 and 1.44 times unsplit. 32 heads: 15 sequences of 100
// tokens and one of 320 in split precision took 1.41 times as long split, 255
// single tokens and a prompt of 512 1.20 times and in bf16 1.23 times, and stay
// whole; 63 single tokens and a prompt of 2048 in bf16 take 171 us unsplit and
// 86 split.
inline PartPlan plan_packed_parts(int64_t sequences, int64_t heads, int64_t tokens,
                                  int64_t longest_tokens, const ChunkTime& main,
                                  const ChunkTime& transfer) {
  PartPlan best{1, 0};
  if (longest_tokens > tokens) longest_tokens = tokens;
  const int64_t longest = (longest_tokens + kChunk - 1) / kChunk;
  if (sequences <= 0 || heads <= 0 || longest <= 2) return best;
  const double units = static_cast<double>(sequences) * heads;
  const double others = static_cast<double>(sequences - 1);
  const bool equal = sequences * longest_tokens <= tokens;
  double rest = others * longest;
  if (!equal) {
    rest = static_cast<double>(tokens - longest_tokens) / kChunk + 0.5 * others;
    if (rest < others) rest = others;
  }
  const double chunks = longest + rest;

  // Unsplit: the longest chain, on CUs shared by as many workgroups of its
  // length as the work amounts to, or the work.
  const double alike = equal ? units : heads * chunks / longest;
  double chain = main.shared;
  if (main.rounds && !equal) chain = main.alone;
  else if (alike <= 512) chain = main.of(alike);
  const double start = equal ? 0.0 : sequences <= 64 ? main.sorted : main.unit;
  double least = longest * chain;
  const double full = heads * (chunks * main.shared + sequences * start) / 512;
  if (least < full) least = full;
  const double unsplit = least;

  for (int32_t parts = kMinParts; parts <= kMaxParts; ++parts) {
    const int64_t len = (longest + parts - 1) / parts;
    if ((longest + len - 1) / len != parts) continue;
    double each = static_cast<double>(sequences) * parts;  // workgroups of a head
    if (!equal) {
      each = chunks / len + (len > 1 ? 0.5 * others : 0.0);
      if (each < sequences + parts - 1) each = static_cast<double>(sequences) + parts - 1;
    }
    const double groups = heads * each;
    const bool alone = equal || groups <= (main.rounds ? 256 : 512);
    double walk = 0.0;
    // Parts of one length, where the other sequences are as long as a part too.
    if (alone || (!main.rounds && rest > len * others)) {
      walk = len * main.of(groups) + 0.2 * parts * kForwardTime.of(groups);
    }
    if (!alone) {
      const double maps = (each - sequences) * parts / 2;
      const double work = (chunks * main.shared + maps * main.map) / each + main.part;
      const double all =
          main.rounds ? __builtin_ceil(groups / 256) * work / 2 : groups / 512 * work;
      // The longest sequence's own parts, at least, run at the same time.
      const double own = main.rounds ? 256 : __builtin_fmin(heads * (parts - 1.0), 512);
      const double last = len * main.of(own) + 0.2 * parts * kForwardTime.of(own);
      if (walk < all) walk = all;
      if (walk < last) walk = last;
    }
    const double time = 4.0 + len * transfer.of(groups - units) + walk;
    if (time < least && time < unsplit * (alone ? 0.95 : 0.78)) {
      least = time;
      best = PartPlan{parts, static_cast<int32_t>(len)};
    }
  }
  return best;
}

// Bytes of part states of a split call (0 when it does not split): parts - 1 per
// unit for equal sequences, caller chunks (planned by their mean) and packed
// sequences of similar lengths, else as many as the packed tokens can need (see
// part_slot). Either way it is proportional to the call's tokens, whatever the
// sequences' lengths. Three sequences of 817 to 1654 tokens take 109.5 us by
// units and 111.9 by slots (the search for a slot's sequence); 63 single tokens
// and a prompt of 2048 173.6 by units (most workgroups without a part) and 94.1.
inline size_t part_bytes(int64_t states) {
  return static_cast<size_t>(states) * kPartElems * sizeof(float);
}
inline size_t unit_part_bytes(int64_t units, const PartPlan& plan) {
  return part_bytes(units * (plan.parts - 1));
}
// Slots per head of packed sequences, or 0 for states by unit.
inline int64_t packed_part_slots(int64_t tokens, int64_t sequences, const PartPlan& plan) {
  const int64_t slots = plan.parts > 1 ? tokens / (kChunk * plan.len) : 0;
  return sequences * (plan.parts - 1) <= 2 * slots ? 0 : slots;
}
inline size_t packed_part_bytes(int64_t tokens, int64_t sequences, int64_t heads,
                                const PartPlan& plan) {
  const int64_t slots = packed_part_slots(tokens, sequences, plan);
  return slots > 0 ? part_bytes(slots * heads) : unit_part_bytes(sequences * heads, plan);
}

// Splits the call when the caller's scratch holds its `bytes` of part states.
template <typename P>
inline void use_parts(P& p, const PartPlan& plan, size_t bytes, void* scratch,
                      size_t scratch_bytes) {
  const bool split = bytes > 0 && scratch != nullptr && scratch_bytes >= bytes;
  p.parts = split ? plan.parts : 1;
  p.part_len = split ? plan.len : 0;
  p.part_states = split ? static_cast<float*>(scratch) : nullptr;
}
inline void use_packed_parts(ChunkFwdParams& p, int32_t sequences, const PartPlan& plan,
                             void* scratch, size_t scratch_bytes) {
  use_parts(p, plan, packed_part_bytes(p.total_tokens, sequences, p.num_heads, plan), scratch,
            scratch_bytes);
  p.packed_sequences = sequences;
  p.part_slots =
      p.parts > 1 ? static_cast<int32_t>(packed_part_slots(p.total_tokens, sequences, plan)) : 0;
}
template <typename P>
inline void use_unit_parts(P& p, int64_t units, const PartPlan& plan, void* scratch,
                           size_t scratch_bytes) {
  use_parts(p, plan, unit_part_bytes(units, plan), scratch, scratch_bytes);
}

inline int64_t chunks_of(int64_t tokens) {
  return tokens > 0 ? (tokens + kChunk - 1) / kChunk : 0;
}

// The plan of a call with caller chunks, whose lengths are on the device: by
// the mean chunk count (a longer sequence gets as many, longer parts).
inline PartPlan plan_caller_chunks(int64_t sequences, int64_t heads, int64_t chunks,
                                   const ChunkTime& main = kForwardTime,
                                   const ChunkTime& transfer = kTransferTime) {
  if (sequences <= 0) return PartPlan{1, 0};
  return plan_parts(sequences, heads, chunks, (chunks + sequences - 1) / sequences, main,
                    transfer);
}

// Launches chunk_transfer_kernel (chunk_transfer.hip) for p.parts > 1.
template <typename T, DecayMode M, typename PoolT, bool kPrecise>
int launch_chunk_transfer(const ChunkFwdParams& p, int units, hipStream_t stream);
// Launches chunk_adjoint_kernel for p.parts > 1.
template <typename T, DecayMode M>
int launch_chunk_adjoint(const ChunkBwdParams& p, int units, hipStream_t stream);

}  // namespace frwkv
