// fp32 matrix form of the recurrence over 16-token pieces.
//
// The per-token kernels (recurrent.hip, train_recurrent.hip) do one dependent
// step per token: about five VALU instructions per state element and a
// reduction over the keys on the critical path. This file takes the chunk form
// of chunk_fwd_kernel.h with 16-token pieces and fp32 operands throughout, on the
// fp32 matrix instruction (v_mfma_f32_16x16x4_f32, twice the rate of unpacked
// fp32 VALU): per piece, with cumulative decays G (inclusive) and Gp
// (exclusive), At = a 2^Gp, Rt = r 2^G, Bh = b 2^-G, Kh = k 2^-G,
//   SA = T (At S0 + Lak V),  T = (I - Lab)^{-1},
//   Y  = scale (Rt S0 + Arb SA + Ark V),
//   S' = g (S0 + Bh^T SA + Kh^T V),  g = 2^G(last token).
// Operands, sums and states are fp32, as in the per-token kernels; results
// differ by the order of the sums. Decay logits only: their retention is at
// least exp(-e^{-1/2}), so a piece's decay stays above 2^-15 and one reference
// point serves a piece (raw retentions stay on the per-token kernels).
//
// The matrix products spread a NaN or an infinity over a whole piece (a masked
// zero times NaN is NaN), and to earlier tokens of it. A (sequence, head) with
// one anywhere in its tokens therefore runs token by token, as the per-token
// kernels do, so that it reaches later tokens only: the preparation flags its
// pieces, the forward walks the unit's tokens (token_form) and the backward
// leaves it to train_recurrent.hip.
//
// Several kernels, so that the serial chain over pieces holds nothing but the
// state products:
//   piece32_prepare   every piece at once: decodes the rows, scans the decay
//                     and writes the scaled tiles and the four triangles in
//                     the operand layouts of the chain;
//   piece32_forward   one wave per 64 keys x 16 value columns of a state,
//                     walking the pieces; operands are read from the tiles
//                     straight into registers, one piece ahead. Waves sharing
//                     columns (D / 64 of them) add their key sums through LDS,
//                     one barrier per piece; at D = 64 there is none;
// and for the backward at D = 256, the same preparation, the adjoint chain
// (piece32_adjoint_kernel) and every piece's gradients at once from its start
// state and its adjoint (piece32_gradient_kernel).
//
// Operand layouts (16x16x4: A[m = n][k = g], B[k = g][n], C[m = 4g + j][n] for
// lane (g, n)): step j of a 16-wide contraction takes k = 4g + j, so a 16 x 16
// block as B operand is its C layout, and as A operand four consecutive
// elements of one row.
#include "capi_internal.h"
#include "chunk_common.h"
#include "piece32.h"
#include "train_common.h"

namespace frwkv {
namespace {

constexpr int kTriElems = kPiece * kPiece;

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// C += A B for 16 x 16 blocks in operand layouts.
__device__ __forceinline__ f32x4 mm16(f32x4 a, f32x4 b, f32x4 c) {
#pragma unroll
  for (int j = 0; j < 4; ++j) c = mfma4(a[j], b[j], c);
  return c;
}

// Sum over a wave's 64 keys (A operands x, B operands s): four chains, so that
// consecutive matrix instructions do not depend on each other.
__device__ __forceinline__ f32x4 over_keys(const f32x4 (&x)[4], const f32x4 (&s)[4]) {
  f32x4 c[4] = {zero4(), zero4(), zero4(), zero4()};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) c[kb] = mfma4(x[kb][j], s[kb][j], c[kb]);
  }
  return (c[0] + c[1]) + (c[2] + c[3]);
}
// s[kb] += x[kb] b: 64 keys (rows of the A operands) by one 16-token block.
__device__ __forceinline__ void add_columns(const f32x4 (&x)[4], f32x4 b, f32x4 (&s)[4]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) s[kb] = mfma4(x[kb][j], b[j], s[kb]);
  }
}

// Schedule of a chain step: one load of the next piece after every two matrix
// instructions. Issued as one burst at the top of the step, the loads of a
// CU's waves fill the address unit, and no wave reaches its first product
// before its last load is accepted.
__device__ __forceinline__ void spread_loads() {
#pragma unroll
  for (int i = 0; i < 28; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);  // MFMA
    __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // vector memory read
  }
}

// Tiles of one (piece, head), in floats.
template <int D>
struct Tiles {
  static constexpr int kTile = kPiece * D;
  // Forward: At, Rt [t][k]; Bh^T, Kh^T [k][t]; g [k]; T, Lak, Arb, Ark [t][i].
  static constexpr int kAt = 0, kRt = kTile, kBhT = 2 * kTile, kKhT = 3 * kTile;
  static constexpr int kG = 4 * kTile;
  static constexpr int kTri = kG + D;
  static constexpr int kForward = kTri + 4 * kTriElems;
  // Backward: Bh, Kh [t][k]; At^T, Rt^T, Bh^T, Kh^T [k][t]; g [k]; T^T, Lak^T,
  // Arb^T, Ark^T [i][t].
  static constexpr int kBh = 0, kKh = kTile, kAtT = 2 * kTile, kRtT = 3 * kTile;
  static constexpr int kBackBhT = 4 * kTile, kBackKhT = 5 * kTile;
  static constexpr int kBackG = 6 * kTile;
  static constexpr int kBackTri = kBackG + D;
  static constexpr int kBackward = kBackTri + 4 * kTriElems;
};

// A pointer known to be the same in every lane, in scalar registers.
template <typename P>
__device__ __forceinline__ P* uniform_pointer(P* x) {
  const uint64_t bits = reinterpret_cast<uint64_t>(x);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(bits));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(bits >> 32));
  return reinterpret_cast<P*>(static_cast<uint64_t>(hi) << 32 | lo);
}

// x[q] for a wave-uniform q by selects (a branch would end the scheduling
// region).
__device__ __forceinline__ float pick4(f32x4 x, int q) {
  const float a = q & 1 ? x[1] : x[0], b = q & 1 ? x[3] : x[2];
  return q & 2 ? b : a;
}

// Pieces of sequence `seq`: slots first .. first + count - 1; with the packed
// and dense layouts, piece i holds tokens begin + 16 i .. of [begin, end).
struct Walk {
  int first, count, begin, end;
};
__device__ __forceinline__ Walk walk_of(const Piece32Params& p, int seq) {
  Walk w{0, 0, 0, 0};
  if (p.seg_offsets != nullptr) {
    const int lo = min(max(meta_at(p.seg_offsets, seq), 0), p.num_segments);
    const int hi = min(max(meta_at(p.seg_offsets, seq + 1), lo), p.num_segments);
    w.first = meta_at(p.base, lo);
    w.count = meta_at(p.base, hi) - w.first;
  } else if (p.dense_t > 0) {
    w.begin = seq * p.dense_t;
    w.end = w.begin + p.dense_t;
    w.first = seq * (p.dense_t / kPiece);
    w.count = p.dense_t / kPiece;
  } else {
    // floor(begin / 16) + seq: sequences of ascending, disjoint ranges then
    // have disjoint slots.
    w.begin = max(meta_at(p.cu_seqlens, seq), 0);
    w.end = min(meta_at(p.cu_seqlens, seq + 1), p.total_tokens);
    w.first = w.begin / kPiece + seq;
    w.count = (max(w.end - w.begin, 0) + kPiece - 1) / kPiece;
  }
  w.first = uniform(w.first);
  w.count = uniform(w.count);
  w.begin = uniform(w.begin);
  w.end = uniform(w.end);
  return w;
}
// Piece i of a walk: {first token, tokens, caller chunk, piece of the chunk}.
__device__ __forceinline__ int4 piece_at(const Piece32Params& p, const Walk& w, int i) {
  if (p.seg_offsets != nullptr) {
    const int32_t* e = reinterpret_cast<const int32_t*>(p.table + w.first + i);
    return make_int4(meta_at(e, 0), meta_at(e, 1), meta_at(e, 2), meta_at(e, 3));
  }
  const int start = w.begin + kPiece * i;
  return make_int4(start, min(kPiece, w.end - start), 0, i);
}

// True when the unit runs token by token (uniform over its workgroups).
__device__ __forceinline__ bool unit_flagged(const Piece32Params& p, const Walk& w, int head,
                                             int lane) {
  bool bad = p.seg_offsets != nullptr && meta_at(p.base, p.num_segments + 1) != 0;
  const uint32_t* flags = p.flags + static_cast<int64_t>(head) * p.slots_total + w.first;
  for (int i = lane; i < w.count; i += 64) bad |= flags[i] != 0;
  return __builtin_amdgcn_ballot_w64(bad) != 0;
}

// The packed sequence that owns a slot (or the last one that starts at or
// before it): the first slots ascend, and every lane tries one of 64 equal
// steps, so a batch of 64 sequences takes one round.
__device__ __forceinline__ int sequence_of_slot(const Piece32Params& p, int slot, int lane) {
  int lo = 0, hi = p.num_sequences;
  while (hi - lo > 1) {
    const int stride = (hi - lo + 63) / 64;
    const int s = lo + lane * stride;
    const bool before = s < hi && max(p.cu_seqlens[s], 0) / kPiece + s <= slot;
    const int count = max(__builtin_popcountll(__builtin_amdgcn_ballot_w64(before)), 1);
    lo = uniform(lo + (count - 1) * stride);
    hi = min(lo + stride, hi);
  }
  return lo;
}

// Slots of the caller chunks' pieces in chunk order, one workgroup. Token
// ranges are clamped to the call's; an empty chunk has one piece of no tokens
// (its start state is an output too). Overlapping chunks can have more pieces
// than there are slots; every unit then runs token by token.
constexpr int kTableThreads = 1024;
__global__ __launch_bounds__(kTableThreads) void piece32_table(Piece32Params p, int slots) {
  __shared__ int sums[kTableThreads];
  const int tid = threadIdx.x;
  int before = 0;
  for (int c0 = 0; c0 < p.num_segments; c0 += kTableThreads) {
    const int c = c0 + tid;
    int start = 0, len = 0;
    if (c < p.num_segments) {
      start = min(max(p.seg_starts[c], 0), p.total_tokens);
      len = max(min(p.seg_ends[c], p.total_tokens) - start, 0);
    }
    const int count = c < p.num_segments ? max((len + kPiece - 1) / kPiece, 1) : 0;
    sums[tid] = count;
    __syncthreads();
    for (int step = 1; step < kTableThreads; step *= 2) {
      const int add = tid >= step ? sums[tid - step] : 0;
      __syncthreads();
      sums[tid] += add;
      __syncthreads();
    }
    const int first = before + sums[tid] - count;
    if (c < p.num_segments) {
      p.base[c] = min(first, slots);
      for (int i = 0; i < count && first + i < slots; ++i) {
        p.table[first + i] = make_int4(start + kPiece * i, min(kPiece, len - kPiece * i), c, i);
      }
    }
    before += sums[kTableThreads - 1];
    __syncthreads();
  }
  if (tid == 0) {
    p.base[p.num_segments] = min(before, slots);
    p.base[p.num_segments + 1] = before > slots;
  }
  for (int i = before + tid; i < slots; i += kTableThreads) p.table[i] = make_int4(0, 0, -1, 0);
}

// Four consecutive 16-bit values at a buffer offset, as loaded.
__device__ __forceinline__ u32x2 load4(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0);
}
template <typename T>
__device__ __forceinline__ f32x4 widen4(u32x2 q) {
  return f32x4{to_f32<T>(static_cast<uint16_t>(q.x)), to_f32<T>(static_cast<uint16_t>(q.x >> 16)),
               to_f32<T>(static_cast<uint16_t>(q.y)), to_f32<T>(static_cast<uint16_t>(q.y >> 16))};
}

// Whether one of two packed 16-bit values is an infinity or NaN (its exponent
// bits, five or eight, are all set).
template <typename T>
__device__ __forceinline__ bool not_finite(uint32_t x) {
  constexpr uint32_t kExponent = __is_same(T, Bf16) ? 0x7f80u : 0x7c00u;
  return (x & kExponent) == kExponent || ((x >> 16) & kExponent) == kExponent;
}

// Cumulative decay of a piece at token n of the lane's 16-lane row, from the
// logits' log2 retentions: 2^G, 2^Gp and 2^-G of sums of logs. A sum of small
// logs keeps the slow channels (the largest states) more exact than a product
// of retentions near 1 (states 4.9e-7 off fp64 with the per-token product,
// 5.7e-7 with a scanned one).
struct Decay {
  float sig;              // sigmoid of the logit
  float incl, excl, inv;  // 2^G, 2^Gp, 2^-G
};
__device__ __forceinline__ Decay piece_decay(float logit, bool on) {
  Decay d;
  d.sig = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-kLog2E * logit));
  const float sum = prefix16(on ? -(kExpNegHalf * kLog2E) * d.sig : 0.0f);
  const float before = __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(sum), 0x111, 0xf, 0xf, true));
  d.incl = __builtin_amdgcn_exp2f(sum);
  d.excl = __builtin_amdgcn_exp2f(before);
  d.inv = __builtin_amdgcn_exp2f(-sum);
  return d;
}

// One workgroup of D / 64 waves per (piece, head); lane (g, n) of wave q holds
// token n, keys 64q + 16kb + 4g .. +3, which is the A and the B operand layout
// of the triangles' products over the keys. Bound by its writes (21 KB per
// (piece, head) at D = 64, 69 KB at 256, beside 10 and 40 KB of rows read):
// 3600 of them at D = 64 take 27 us (4.3 TB/s), 512 at D = 256 17 us.
template <typename T, int D, bool kBackward>
__global__ __launch_bounds__(D) void piece32_prepare(Piece32Params p) {
  constexpr int kWaves = D / 64;
  using L = Tiles<D>;
  __shared__ f32x4 part[kWaves > 1 ? kWaves : 1][5][64];
  __shared__ bool wave_bad[kWaves];
  if (p.status != nullptr && p.status[0] != 0) return;
  const int heads = p.num_heads;
  const int head = static_cast<int>(blockIdx.x) % heads;
  const int index = static_cast<int>(blockIdx.x) / heads;
  int slot, start, ntok;
  if (p.seg_offsets != nullptr) {
    slot = index;
    const int4 e = p.table[slot];
    start = uniform(e.x);
    ntok = uniform(e.y);
    if (e.z < 0) return;
  } else {
    slot = index;
    const Walk w = walk_of(p, p.dense_t > 0 ? slot / (p.dense_t / kPiece)
                                            : sequence_of_slot(p, slot, threadIdx.x & 63));
    const int i = slot - w.first;
    if (i >= w.count) return;
    start = w.begin + kPiece * i;
    ntok = min(kPiece, w.end - start);
  }
  const int wave = uniform(static_cast<int>(threadIdx.x) >> 6);
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4, n = lane & 15;
  const bool on = n < ntok;

  using S16 = typename IoTraits<T>::storage;
  const uint32_t row_bytes = static_cast<uint32_t>(heads) * D * 2;
  const int64_t row0 = (static_cast<int64_t>(start) * heads + head) * D;
  auto rows = [&](const void* x) {
    return buffer_rsrc(static_cast<const S16*>(x) + row0, static_cast<uint32_t>(ntok) * row_bytes);
  };
  const auto rw = rows(p.decay), ra = rows(p.a), rr = rows(p.r), rb = rows(p.b), rk = rows(p.k);
  const uint32_t off = static_cast<uint32_t>(n) * row_bytes + 2 * (64 * wave + 4 * g);
  u32x2 qw[4], qa[4], qr[4], qb[4], qk[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) qw[kb] = load4(rw, off + 32 * kb);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    qa[kb] = load4(ra, off + 32 * kb);
    qr[kb] = load4(rr, off + 32 * kb);
    qb[kb] = load4(rb, off + 32 * kb);
    qk[kb] = load4(rk, off + 32 * kb);
  }
  // Values that the tiles do not hold: V, and dY in the backward.
  const auto rv = rows(p.v);
  const bool with_dy = kBackward && p.dy != nullptr;
  const auto rdy = with_dy ? rows(p.dy) : buffer_rsrc(static_cast<const S16*>(nullptr), 0u);
  bool bad = false;
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const u32x2 x = load4(rv, off + 32 * kb);
    bad |= not_finite<T>(x.x) || not_finite<T>(x.y);
    if constexpr (kBackward) {
      const u32x2 y = load4(rdy, off + 32 * kb);
      bad |= not_finite<T>(y.x) || not_finite<T>(y.y);
    }
  }
  float* const tiles = p.tiles + (static_cast<int64_t>(slot) * heads + head) *
                                     (kBackward ? L::kBackward : L::kForward);
  const int key0 = 64 * wave + 4 * g;  // + 16 kb + j
  auto store_rows = [&](int tile, int key, f32x4 x) {  // [t][k]
    *reinterpret_cast<f32x4*>(tiles + tile + n * D + key) = x;
  };
  auto store_cols = [&](int tile, int key, f32x4 x) {  // [k][t]
#pragma unroll
    for (int j = 0; j < 4; ++j) tiles[tile + (key + j) * kPiece + n] = x[j];
  };
  f32x4 at[4], rt[4], bh[4], kh[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    f32x4 x = widen4<T>(qw[kb]);
    if (p.bias != nullptr) {
      const S16* bias = static_cast<const S16*>(p.bias) + static_cast<int64_t>(head) * D + key0 + 16 * kb;
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] += to_f32<T>(bias[j]);
    }
    const f32x4 av = widen4<T>(qa[kb]), rv = widen4<T>(qr[kb]), bv = widen4<T>(qb[kb]),
                kv = widen4<T>(qk[kb]);
    f32x4 total;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const Decay dec = piece_decay(x[j], on);
      total[j] = dec.incl;
      at[kb][j] = on ? av[j] * dec.excl : 0.0f;
      rt[kb][j] = on ? rv[j] * dec.incl : 0.0f;
      bh[kb][j] = on ? bv[j] * dec.inv : 0.0f;
      kh[kb][j] = on ? kv[j] * dec.inv : 0.0f;
    }
    const int key = key0 + 16 * kb;
    if (n == 15) {
      *reinterpret_cast<f32x4*>(tiles + (kBackward ? L::kBackG : L::kG) + key) = total;
    }
    if constexpr (kBackward) {
      store_rows(L::kBh, key, bh[kb]);
      store_rows(L::kKh, key, kh[kb]);
      store_cols(L::kAtT, key, at[kb]);
      store_cols(L::kRtT, key, rt[kb]);
      store_cols(L::kBackBhT, key, bh[kb]);
      store_cols(L::kBackKhT, key, kh[kb]);
    } else {
      store_rows(L::kAt, key, at[kb]);
      store_rows(L::kRt, key, rt[kb]);
      store_cols(L::kBhT, key, bh[kb]);
      store_cols(L::kKhT, key, kh[kb]);
    }
  }

  // Triangles X[t][i] = sum_k X_t Y_i, as X^T in C layout (lane (g, n): row
  // t = n, i = 4g + j), and Lab in C layout too for the inverse. The backward
  // takes the transposed matrices: the same products with the operands
  // exchanged (lane (g, n): i = n, t = 4g + j).
  auto tri_product = [](f32x4 x, f32x4 y, f32x4 c) {
    return kBackward ? mm16(x, y, c) : mm16(y, x, c);
  };
  f32x4 tri[5] = {zero4(), zero4(), zero4(), zero4(), zero4()};
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    tri[0] = mm16(bh[kb], at[kb], tri[0]);
    tri[1] = mm16(at[kb], bh[kb], tri[1]);
    tri[2] = tri_product(at[kb], kh[kb], tri[2]);
    tri[3] = tri_product(rt[kb], bh[kb], tri[3]);
    tri[4] = tri_product(rt[kb], kh[kb], tri[4]);
  }
  if constexpr (kWaves > 1) {
#pragma unroll
    for (int m = 0; m < 5; ++m) part[wave][m][lane] = tri[m];
    wave_bad[wave] = __builtin_amdgcn_ballot_w64(bad) != 0;
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int q = 1; q < kWaves; ++q) {
#pragma unroll
      for (int m = 0; m < 5; ++m) tri[m] += part[q][m][lane];
      bad |= wave_bad[q];
    }
  }
  // A value of r, w, k, a or b that is not finite makes a sum of Lab or Ark so
  // (before the masks, every row meets every other).
  float probe = 0.0f;
#pragma unroll
  for (int m = 0; m < 5; ++m) {
#pragma unroll
    for (int j = 0; j < 4; ++j) probe = fmaf(tri[m][j], 0.0f, probe);
  }
  const f32x4 lab_r = tri[0], lab_c = tri[1];
  f32x4 lak = tri[2], arb = tri[3], ark = tri[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int i = 4 * g + j;
    const bool strict = kBackward ? n < i : i < n;  // source before target
    lak[j] = strict ? lak[j] : 0.0f;
    arb[j] = strict || i == n ? arb[j] : 0.0f;
    ark[j] = strict || i == n ? ark[j] : 0.0f;
  }
  // (I - L)^{-1} by block substitution (wkv7_mfma.h): in fp32 too, products of
  // powers of L lose up to four digits to cancellation where the keys are
  // similar (states 1e-5 off fp64 against 2e-7). The backward takes T^T, T_C.
  f32x4 t_r, t_c;
  invert_diagonal4(lab_r, lab_c, t_r, t_c);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float one = 4 * g + j == n ? 1.0f : 0.0f;
    t_r[j] += one;
    t_c[j] += one;
  }
  const f32x4 x = mm16(in_lanes(kJoins8) ? lab_c : zero4(), t_r, zero4());
  const f32x4 t8_r = mm16(t_c, x, t_r), t8_c = mm16(x, t_c, t_c);
  const f32x4 y = mm16(in_lanes(kJoins16) ? lab_c : zero4(), t8_r, zero4());
  const f32x4 t = kBackward ? mm16(y, t8_c, t8_c) : mm16(t8_c, y, t8_r);
#pragma unroll
  for (int j = 0; j < 4; ++j) probe = fmaf(t[j], 0.0f, probe);
  bad |= !(probe == 0.0f);
  const uint32_t flag = __builtin_amdgcn_ballot_w64(bad) != 0;
  if (lane == 0) p.flags[static_cast<int64_t>(head) * p.slots_total + slot] = flag;
  float* const out = tiles + (kBackward ? L::kBackTri : L::kTri) + n * kPiece + 4 * g;
  *reinterpret_cast<f32x4*>(out) = t;
  *reinterpret_cast<f32x4*>(out + kTriElems) = lak;
  *reinterpret_cast<f32x4*>(out + 2 * kTriElems) = arb;
  *reinterpret_cast<f32x4*>(out + 3 * kTriElems) = ark;
}

// A flagged unit's tokens one by one, on the state slab of the forward kernel
// (wave: keys 64q .. +63, lane: keys 64q + 16kb + 4g + j of column col), with
// the outputs of the chain:
//   sa = a^T S,  S <- diag(w) S + b sa^T + k v^T,  y = scale r^T S.
// red: 8 x 64 floats of LDS for the sums over the waves that share columns.
template <typename T, int D, bool kTrain, typename Store>
__device__ __forceinline__ void token_form(const Piece32Params& p, const Walk& walk, int seq,
                                           int head, int col, f32x4 (&S)[4], f32x4* red,
                                           Store&& store_state) {
  constexpr int kKeyWaves = D / 64;
  using S16 = typename IoTraits<T>::storage;
  const int wave = uniform(static_cast<int>(threadIdx.x) >> 6);
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4, n = lane & 15;
  const int kq = wave % kKeyWaves;
  const int key0 = 64 * kq + 4 * g;
  constexpr int64_t kState = static_cast<int64_t>(D) * D;
  // Sum over the keys. Two areas in turn: a wave writes one again only after
  // the barrier that follows its reads.
  auto over_waves = [&](float x, int area) {
    x = add_xor32(add_xor16(x));
    if constexpr (kKeyWaves > 1) {
      float* const at = reinterpret_cast<float*>(red) + 64 * area;
      if (g == 0) at[16 * wave + n] = x;
      __syncthreads();
      x = 0.0f;
#pragma unroll
      for (int q = 0; q < kKeyWaves; ++q) x += at[16 * (wave - kq + q) + n];
    }
    return x;
  };
  f32x4 bias[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    bias[kb] = zero4();
    if (p.bias != nullptr) {
      const S16* src = static_cast<const S16*>(p.bias) + static_cast<int64_t>(head) * D + key0;
#pragma unroll
      for (int j = 0; j < 4; ++j) bias[kb][j] = to_f32<T>(src[16 * kb + j]);
    }
  }
  auto tokens = [&](int begin, int end) {
    for (int t = begin; t < end; ++t) {
      const int64_t row = (static_cast<int64_t>(t) * p.num_heads + head) * D;
      auto row4 = [&](const void* x, int kb) {
        return widen4<T>(*reinterpret_cast<const u32x2*>(static_cast<const S16*>(x) + row + key0 +
                                                         16 * kb));
      };
      const float v = to_f32<T>(static_cast<const S16*>(p.v)[row + col]);
      f32x4 w[4], a[4], b[4], k[4], r[4];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        w[kb] = row4(p.decay, kb) + bias[kb];
        a[kb] = row4(p.a, kb);
        b[kb] = row4(p.b, kb);
        k[kb] = row4(p.k, kb);
        r[kb] = row4(p.r, kb);
      }
      float sa = 0.0f, y = 0.0f;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
        for (int j = 0; j < 4; ++j) sa = fmaf(a[kb][j], S[kb][j], sa);
      }
      sa = over_waves(sa, 0);
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float x = decay_retention<DecayMode::kLogits>(w[kb][j]);
          S[kb][j] = fmaf(x, S[kb][j], fmaf(b[kb][j], sa, k[kb][j] * v));
          y = fmaf(r[kb][j], S[kb][j], y);
        }
      }
      y = over_waves(y, 1);
      if (g == 0 && kq == 0) {
        static_cast<S16*>(p.out)[row + col] = from_f32<T>(p.scale * y);
        if constexpr (kTrain) p.state_dot_a[row + col] = sa;
      }
    }
  };
  if constexpr (kTrain) {
    // The state at every chunk start, and every 16 tokens inside a chunk.
    auto chunk = [&](int start, int end, float* at_start, bool interior) {
      store_state(at_start);
      for (int t = start; t < end; t += kPiece) {
        if (interior && t > start) {
          store_state(p.interior +
                      (static_cast<int64_t>(t / kPiece) * p.num_heads + head) * kState);
        }
        tokens(t, min(t + kPiece, end));
      }
    };
    if (p.seg_offsets != nullptr) {
      const int hi = min(meta_at(p.seg_offsets, seq + 1), p.num_segments);
      for (int c = max(meta_at(p.seg_offsets, seq), 0); c < hi; ++c) {
        const int start = min(max(meta_at(p.seg_starts, c), 0), p.total_tokens);
        const int end = min(meta_at(p.seg_ends, c), p.total_tokens);
        chunk(start, end, p.boundary + (static_cast<int64_t>(c) * p.num_heads + head) * kState,
              p.interior != nullptr);
      }
      return;
    }
    float* at = p.boundary + (static_cast<int64_t>(seq) * p.num_heads + head) *
                                 (p.dense_t / kPiece) * kState;
    for (int t = walk.begin; t < walk.end; t += kPiece, at += kState) {
      chunk(t, t + kPiece, at, false);
    }
  } else {
    tokens(walk.begin, walk.end);
  }
}

// The chain over a sequence's pieces. Wave: keys 64q .. +63 (q = wave % (D /
// 64)), value columns col0 .. +15; S[kb][j] is key 64q + 16kb + 4g + j, column
// col0 + n. kTrain: boundary, interior and a^T S outputs. Bound by the serial
// chain of its matrix products (a sequence and head occupy D / 16 waves at
// D = 64, 4 D / 16 at 256). Measured: 24 pieces in 288 units at D = 64 46 us;
// 32 pieces in 16 units at D = 256 98 us, where the per-token kernel takes 567.
template <typename T, int D, bool kTrain>
__global__ __launch_bounds__(256, 2) void piece32_forward_kernel(Piece32Params p) {
  using L = Tiles<D>;
  constexpr int kKeyWaves = D / 64;
  constexpr int kSlabs = 4 / kKeyWaves;  // column slabs per workgroup
  using S16 = typename IoTraits<T>::storage;
  __shared__ f32x4 part[2][kKeyWaves > 1 ? 4 : 1][2][64];
  if (p.status != nullptr && p.status[0] != 0) {
    fill_nan<T>(static_cast<S16*>(p.out), p.out_elems);
    return;
  }
  const int heads = p.num_heads;
  const int units = p.num_sequences * heads;
  // Blocks of one unit are `units` apart: on one XCD where that is a multiple
  // of 8, so that they share its tiles' L2 lines.
  const int unit = static_cast<int>(blockIdx.x) % units;
  const int seq = unit / heads, head = unit % heads;
  const int slot = uniform(p.slots != nullptr ? p.slots[seq] : seq);
  if (p.state != nullptr && (slot < 0 || slot >= p.state_slots)) return;
  const int wave = uniform(static_cast<int>(threadIdx.x) >> 6);
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4, n = lane & 15;
  const int kq = wave % kKeyWaves;
  const int col =
      16 * (static_cast<int>(blockIdx.x) / units * kSlabs + wave / kKeyWaves) + n;
  const int key0 = 64 * kq + 4 * g;  // + 16 kb + j
  const Walk walk = walk_of(p, seq);

  constexpr int64_t kState = static_cast<int64_t>(D) * D;
  // Element (16 kb + j) * D floats after s_off; a null state reads as zero.
  const uint32_t s_off = static_cast<uint32_t>(key0 * D + col) * 4;
  float* const state =
      p.state != nullptr ? p.state + (static_cast<int64_t>(slot) * heads + head) * kState : nullptr;
  const auto state_rs = buffer_rsrc(state, state != nullptr ? static_cast<uint32_t>(kState) * 4 : 0u);
  f32x4 S[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      S[kb][j] = __uint_as_float(
          __builtin_amdgcn_raw_buffer_load_b32(state_rs, s_off, (16 * kb + j) * D * 4, 0));
    }
  }
  auto store_state = [&](float* dst) {
    const auto rs = buffer_rsrc(dst, dst != nullptr ? static_cast<uint32_t>(kState) * 4 : 0u);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(S[kb][j]), rs, s_off,
                                              (16 * kb + j) * D * 4, 0);
      }
    }
  };

  // A piece's operands: registers in operand layout. The triangles' products
  // with V and SA (four steps of four tokens) are shared out over the waves
  // that add up a sum anyway: wave q takes steps kSteps q .. of each.
  constexpr int kSteps = 4 / kKeyWaves;
  const int step0 = kSteps * kq;
  const int lane_step0 = kSteps * ((static_cast<int>(threadIdx.x) >> 6) % kKeyWaves);
  struct Ops {
    f32x4 at[4], rt[4], bt[4], kt[4], t;
    float lak[kSteps], arb[kSteps], ark[kSteps];
    uint16_t v[4];  // V[4g + j][col]
    int start, ntok, chunk, index;
  };
  const uint32_t row_bytes = static_cast<uint32_t>(heads) * D * 2;
  auto load = [&](Ops& o, int i, const int4& e) {
    o.start = e.x;
    o.ntok = e.y;
    o.chunk = e.z;
    o.index = e.w;
    const float* tiles =
        p.tiles + (static_cast<int64_t>(walk.first + i) * heads + head) * L::kForward;
    auto at4 = [&](int offset) { return *reinterpret_cast<const f32x4*>(tiles + offset); };
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      o.at[kb] = at4(L::kAt + n * D + key0 + 16 * kb);
      o.rt[kb] = at4(L::kRt + n * D + key0 + 16 * kb);
    }
    const auto vs = buffer_rsrc(static_cast<const S16*>(p.v) +
                                    (static_cast<int64_t>(e.x) * heads + head) * D,
                                static_cast<uint32_t>(e.y) * row_bytes);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      o.v[j] = __builtin_amdgcn_raw_buffer_load_b16(
          vs, static_cast<uint32_t>(4 * g + j) * row_bytes + 2 * col, 0, 0);
    }
    const int tri = L::kTri + n * kPiece + 4 * g;
#pragma unroll
    for (int j = 0; j < kSteps; ++j) {
      o.lak[j] = tiles[tri + kTriElems + step0 + j];
      o.arb[j] = tiles[tri + 2 * kTriElems + step0 + j];
      o.ark[j] = tiles[tri + 3 * kTriElems + step0 + j];
    }
    o.t = at4(tri);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const int key = 64 * kq + 16 * kb + n;
      o.kt[kb] = at4(L::kKhT + key * kPiece + 4 * g);
      o.bt[kb] = at4(L::kBhT + key * kPiece + 4 * g);
    }
  };

  // Rows 4g + step0 .. of a token block of the column, from its C layout.
  auto store_y = [&](int start, int ntok, const float (&y)[kSteps]) {
    const auto ys = buffer_rsrc(
        static_cast<S16*>(p.out) + (static_cast<int64_t>(start) * heads + head) * D,
        static_cast<uint32_t>(ntok) * row_bytes);
#pragma unroll
    for (int j = 0; j < kSteps; ++j) {
      __builtin_amdgcn_raw_buffer_store_b16(
          from_f32<T>(p.scale * y[j]), ys,
          static_cast<uint32_t>(4 * g + step0 + j) * row_bytes + 2 * col, 0, 0);
    }
  };
  // The wave's rows of the output of piece i from the key waves' sums, after
  // the barrier that follows them.
  auto finish_y = [&](int i, int start, int ntok) {
    const int first = wave - kq;
    float y[kSteps];
#pragma unroll
    for (int j = 0; j < kSteps; ++j) {
      y[j] = 0.0f;
#pragma unroll
      for (int q = 0; q < kKeyWaves; ++q) {
        y[j] += reinterpret_cast<const float*>(&part[i & 1][first + q][1][lane])[step0 + j];
      }
    }
    store_y(start, ntok, y);
  };
  int done_start = 0, done_ntok = 0;  // the piece whose output is still in LDS
  auto step = [&](const Ops& o, Ops& next, int i) {
    // Everything with a branch first: one scheduling region follows.
    const int following = min(i + 1, walk.count - 1);
    const int4 e = piece_at(p, walk, following);
    float* boundary = nullptr;
    if constexpr (kTrain) {
      int64_t at = (static_cast<int64_t>(seq) * heads + head) * (p.dense_t / kPiece) + i;
      float* base = p.boundary;
      if (p.dense_t == 0) {
        const bool first = o.index == 0;
        at = static_cast<int64_t>(first ? o.chunk : o.start / kPiece) * heads + head;
        base = first ? p.boundary : p.interior;
      }
      boundary = uniform_pointer(base != nullptr ? base + at * kState : nullptr);
    }
    f32x4 decay[4];  // read at the end of the step
    {
      const float* src = p.tiles +
                         (static_cast<int64_t>(walk.first + i) * heads + head) * L::kForward +
                         L::kG + key0;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) decay[kb] = *reinterpret_cast<const f32x4*>(src + 16 * kb);
    }
    // Loads and stores are unconditional (the last piece again at the end; a
    // null resource drops its stores): past a branch the compiler waits for
    // everything in flight instead of the loads it needs.
    load(next, following, e);
    if constexpr (kTrain) store_state(boundary);
    spread_loads();
    // The chain is rhs -> SA -> S; everything else is placed where it fills
    // the chain's waits (the exchange of the key sums, the triangle products).
    f32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = to_f32<T>(o.v[j]);
    auto pick = [&](f32x4 x, int j) {  // x[step0 + j]
      return kKeyWaves == 1 ? x[j] : pick4(x, lane_step0 + j);
    };
    f32x4 rhs = over_keys(o.at, S);
#pragma unroll
    for (int j = 0; j < kSteps; ++j) rhs = mfma4(o.lak[j], pick(v, j), rhs);
    if constexpr (kKeyWaves > 1) part[i & 1][wave][0][lane] = rhs;
    f32x4 y = over_keys(o.rt, S);
#pragma unroll
    for (int j = 0; j < kSteps; ++j) y = mfma4(o.ark[j], pick(v, j), y);
    if constexpr (kKeyWaves > 1) {
      // Double-buffered by piece: the next barrier separates these reads from
      // the writes after it.
      __syncthreads();
      const int first = wave - kq;
      rhs = part[i & 1][first][0][lane];
#pragma unroll
      for (int q = 1; q < kKeyWaves; ++q) rhs += part[i & 1][first + q][0][lane];
    }
    add_columns(o.kt, v, S);
    const f32x4 sa = mm16(o.t, rhs, zero4());
    add_columns(o.bt, sa, S);
#pragma unroll
    for (int j = 0; j < kSteps; ++j) y = mfma4(o.arb[j], pick(sa, j), y);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) S[kb] *= decay[kb];
    if constexpr (kKeyWaves > 1) {
      finish_y(i - 1, done_start, done_ntok);
      done_start = o.start;
      done_ntok = o.ntok;
      part[i & 1][wave][1][lane] = y;  // read after the next barrier
    } else {
      const float rows[4] = {y[0], y[1], y[2], y[3]};
      store_y(o.start, o.ntok, rows);
    }
    if constexpr (kTrain) {
      const auto sas = buffer_rsrc(
          p.state_dot_a + (static_cast<int64_t>(o.start) * heads + head) * D,
          static_cast<uint32_t>(o.ntok) * 2 * row_bytes);
#pragma unroll
      for (int j = 0; j < kSteps; ++j) {
        __builtin_amdgcn_raw_buffer_store_b32(
            __float_as_uint(pick(sa, j)), sas,
            static_cast<uint32_t>(4 * g + step0 + j) * 2 * row_bytes + 4 * col, 0, 0);
      }
    }
  };

  // At wide heads the first piece's loads fly while the flags are looked at (1%
  // of a pass); at D = 64 that costs registers and 10%.
  Ops even{}, odd;
  if (kKeyWaves > 1 && walk.count > 0) load(even, 0, piece_at(p, walk, 0));
  if (unit_flagged(p, walk, head, lane)) {
    token_form<T, D, kTrain>(p, walk, seq, head, col, S, &part[0][0][0][0], store_state);
    if (state != nullptr) store_state(state);
    return;
  }
  if (walk.count > 0) {
    if (kKeyWaves == 1) load(even, 0, piece_at(p, walk, 0));
    for (int i = 0;; i += 2) {
      step(even, odd, i);
      if (i + 1 >= walk.count) break;
      step(odd, even, i + 1);
      if (i + 2 >= walk.count) break;
    }
    if constexpr (kKeyWaves > 1) {
      __syncthreads();
      finish_y(walk.count - 1, done_start, done_ntok);
    }
  }
  if (state != nullptr) store_state(state);
}

// The adjoint chain (head size 256), pieces in reverse. Same wave layout as the
// forward: dS[kb][j] is dL/dS of key 64q + 16kb + 4g + j, column col0 + n, at
// the end of the current piece; it goes to p.adjoints for the gradient kernel.
// Per piece, with dU = g o dS and dYs = scale dY:
//   dSA = Bh dU + Arb^T dYs,  dZ = T^T dSA,
//   dV  = Kh dU + Ark^T dYs + Lak^T dZ,  dS <- dU + Rt^T dYs + At^T dZ.
// Bound like the forward chain: 32 pieces in 16 units 106 us (the per-token
// backward, which also forms the gradients, takes 3330).
template <typename T, int D>
__global__ __launch_bounds__(256, 1) void piece32_adjoint_kernel(Piece32Params p) {
  using L = Tiles<D>;
  constexpr int kKeyWaves = D / 64;
  static_assert(kKeyWaves == 4, "one column slab per workgroup");
  using S16 = typename IoTraits<T>::storage;
  __shared__ f32x4 part[2][kKeyWaves][2][64];
  const int heads = p.num_heads;
  const int units = p.num_sequences * heads;
  const int unit = static_cast<int>(blockIdx.x) % units;
  const int seq = unit / heads, head = unit % heads;
  const int kq = uniform(static_cast<int>(threadIdx.x) >> 6);
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4, n = lane & 15;
  const int col = 16 * (static_cast<int>(blockIdx.x) / units) + n;
  const int key0 = 64 * kq + 4 * g;
  const Walk walk = walk_of(p, seq);
  constexpr uint32_t kState = D * D;
  const uint32_t s_off = static_cast<uint32_t>(key0 * D + col) * 4;
  auto state_rs = [&](const float* base, int64_t index) {
    return buffer_rsrc(base != nullptr ? base + index * kState : nullptr,
                       base != nullptr ? kState * 4 : 0u);
  };
  f32x4 dS[4];
  {
    const auto rs = state_rs(p.dstate_final, unit);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        dS[kb][j] = __uint_as_float(
            __builtin_amdgcn_raw_buffer_load_b32(rs, s_off, (16 * kb + j) * D * 4, 0));
      }
    }
  }
  auto store_adjoint = [&](float* base, int64_t index) {
    const auto rs = state_rs(base, index);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(dS[kb][j]), rs, s_off,
                                              (16 * kb + j) * D * 4, 0);
      }
    }
  };

  struct Ops {
    f32x4 bh[4], kh[4], at[4], rt[4], decay[4], t;
    float lak, arb, ark;  // the wave's step of the triangles' products
    uint16_t dy[4];       // dY[4g + j][col]
    int start, ntok;
  };
  const uint32_t row_bytes = static_cast<uint32_t>(heads) * D * 2;
  auto load = [&](Ops& o, int i, const int4& e) {
    o.start = e.x;
    o.ntok = e.y;
    const float* tiles =
        p.tiles + (static_cast<int64_t>(walk.first + i) * heads + head) * L::kBackward;
    auto at4 = [&](int offset) { return *reinterpret_cast<const f32x4*>(tiles + offset); };
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      o.bh[kb] = at4(L::kBh + n * D + key0 + 16 * kb);
      o.kh[kb] = at4(L::kKh + n * D + key0 + 16 * kb);
      o.decay[kb] = at4(L::kBackG + key0 + 16 * kb);
    }
    const bool ok = p.dy != nullptr;
    const auto ds = buffer_rsrc(ok ? static_cast<const S16*>(p.dy) +
                                         (static_cast<int64_t>(e.x) * heads + head) * D
                                   : nullptr,
                                ok ? static_cast<uint32_t>(e.y) * row_bytes : 0u);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      o.dy[j] = __builtin_amdgcn_raw_buffer_load_b16(
          ds, static_cast<uint32_t>(4 * g + j) * row_bytes + 2 * col, 0, 0);
    }
    const int tri = L::kBackTri + n * kPiece + 4 * g;
    o.lak = tiles[tri + kTriElems + kq];
    o.arb = tiles[tri + 2 * kTriElems + kq];
    o.ark = tiles[tri + 3 * kTriElems + kq];
    o.t = at4(tri);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const int key = 64 * kq + 16 * kb + n;
      o.rt[kb] = at4(L::kRtT + key * kPiece + 4 * g);
      o.at[kb] = at4(L::kAtT + key * kPiece + 4 * g);
    }
  };

  // The wave's rows (4g + kq) of dV of piece i from the key waves' sums, after
  // the barrier that follows them.
  auto finish_dv = [&](int i, int start, int ntok) {
    float dv = 0.0f;
#pragma unroll
    for (int q = 0; q < kKeyWaves; ++q) {
      dv += reinterpret_cast<const float*>(&part[i & 1][q][1][lane])[kq];
    }
    const auto vs = buffer_rsrc(static_cast<S16*>(p.dv) +
                                    (static_cast<int64_t>(start) * heads + head) * D,
                                static_cast<uint32_t>(ntok) * row_bytes);
    __builtin_amdgcn_raw_buffer_store_b16(
        from_f32<T>(dv), vs, static_cast<uint32_t>(4 * g + kq) * row_bytes + 2 * col, 0, 0);
  };
  int done_start = 0, done_ntok = 0;  // the piece whose dV is still in LDS
  auto step = [&](const Ops& o, Ops& next, int i) {
    const int following = max(i - 1, 0);
    const int4 e = piece_at(p, walk, following);
    const int64_t ph = static_cast<int64_t>(walk.first + i) * heads + head;
    load(next, following, e);  // unconditional, as in the forward
    store_adjoint(p.adjoints, ph);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) dS[kb] *= o.decay[kb];  // dU
    spread_loads();
    // The chain is dSA -> dZ -> dS; the rest fills its waits (see the forward).
    f32x4 dy;
#pragma unroll
    for (int j = 0; j < 4; ++j) dy[j] = p.scale * to_f32<T>(o.dy[j]);
    auto pick = [&](f32x4 x) { return pick4(x, static_cast<int>(threadIdx.x) >> 6); };
    const float dyq = pick(dy);
    f32x4 dsa = mfma4(o.arb, dyq, over_keys(o.bh, dS));
    part[i & 1][kq][0][lane] = dsa;
    f32x4 dv = mfma4(o.ark, dyq, over_keys(o.kh, dS));
    __syncthreads();
    dsa = part[i & 1][0][0][lane];
#pragma unroll
    for (int q = 1; q < kKeyWaves; ++q) dsa += part[i & 1][q][0][lane];
    add_columns(o.rt, dy, dS);
    const f32x4 dz = mm16(o.t, dsa, zero4());
    add_columns(o.at, dz, dS);
    const float dzq = pick(dz);
    dv = mfma4(o.lak, dzq, dv);
    finish_dv(i + 1, done_start, done_ntok);
    done_start = o.start;
    done_ntok = o.ntok;
    part[i & 1][kq][1][lane] = dv;  // read after the next barrier
    p.dz[ph * (kPiece * D) + (4 * g + kq) * D + col] = dzq;
  };

  // The first loads fly while the flags are looked at.
  Ops even{}, odd;
  if (walk.count > 0) load(even, walk.count - 1, piece_at(p, walk, walk.count - 1));
  if (unit_flagged(p, walk, head, lane)) return;  // train_recurrent.hip
  if (walk.count > 0) {
    for (int i = walk.count - 1;; i -= 2) {
      step(even, odd, i);
      if (i < 1) break;
      step(odd, even, i - 1);
      if (i < 2) break;
    }
    __syncthreads();
    finish_dv(0, done_start, done_ntok);
  }
  if (p.dstate0 != nullptr) store_adjoint(p.dstate0, unit);
}

// The gradients of a (piece, head) from its start state S0, the adjoint dS at
// its end, SA and dZ; every piece at once (head size 256), one workgroup each:
//   dRt = dYs S0^T + dArb Bh + dArk Kh    dAt = dZ S0^T + dLab Bh + dLak Kh
//   dBh = dLab^T At + dArb^T Rt           dKh = dLak^T At + dArk^T Rt
//   dBt = SA dS^T    dKt = V dS^T    dg = rowsum(S0 o dS)
// and the elementwise chain rules of chunk_bwd.hip. Wave w owns keys 32w ..
// 32w + 31; products come out with lane (g, n) holding token n, keys 4g .. +3
// of a 16-key block, the layout of the rows. Bound by reading S0 and dS (512
// KiB per piece and head) once: 512 of them in 82 us, 3.3 TB/s.
constexpr int kGradThreads = 512;
constexpr int kGradStride = 260;  // floats per LDS row: 16-byte aligned, rows 4 banks apart
constexpr int kGradTriStride = 20;

template <typename T, int D>
__global__ __launch_bounds__(kGradThreads, 2) void piece32_gradient_kernel(Piece32Params p) {
  using L = Tiles<D>;
  static_assert(D == 256, "eight waves of 32 keys");
  using S16 = typename IoTraits<T>::storage;
  __shared__ float rows[4][kPiece * kGradStride];         // dYs, dZ, SA, V [t][v]
  __shared__ float tri[4][kPiece * kGradTriStride];       // dArb, dArk, dLab, dLak [t][i]
  __shared__ float dgs[D];
  const int heads = p.num_heads;
  const int head = static_cast<int>(blockIdx.x) % heads;
  const int slot = static_cast<int>(blockIdx.x) / heads;
  const int64_t ph = static_cast<int64_t>(slot) * heads + head;
  constexpr int64_t kState = static_cast<int64_t>(D) * D;
  int start, ntok;
  const float* s0;
  if (p.seg_offsets != nullptr) {
    const int4 e = p.table[slot];
    start = uniform(e.x);
    ntok = uniform(e.y);
    const int chunk = uniform(e.z), index = uniform(e.w);
    s0 = index == 0 ? p.boundary + (static_cast<int64_t>(chunk) * heads + head) * kState
                    : p.interior + (static_cast<int64_t>(start / kPiece) * heads + head) * kState;
  } else {
    const int per = p.dense_t / kPiece;
    const int seq = slot / per, i = slot % per;
    start = seq * p.dense_t + kPiece * i;
    ntok = kPiece;
    s0 = p.boundary + ((static_cast<int64_t>(seq) * heads + head) * per + i) * kState;
  }
  if (ntok <= 0) return;
  const float* const ds = p.adjoints + ph * kState;
  const int tid = threadIdx.x;
  const int wave = uniform(tid >> 6);
  const int lane = tid & 63;
  const int g = lane >> 4, n = lane & 15;
  const bool on = n < ntok;
  const uint32_t row_bytes = static_cast<uint32_t>(heads) * D * 2;
  const int64_t row0 = (static_cast<int64_t>(start) * heads + head) * D;
  auto row_rs = [&](const void* x) {
    return buffer_rsrc(x != nullptr ? static_cast<const S16*>(x) + row0 : nullptr,
                       x != nullptr ? static_cast<uint32_t>(ntok) * row_bytes : 0u);
  };

  {
    // Row t = tid / 32, eight columns: dYs, V; dZ and SA as fp32.
    const int t = tid >> 5, c = 8 * (tid & 31);
    const uint32_t off = static_cast<uint32_t>(t) * row_bytes + 2 * c;
    const auto dys = row_rs(p.dy), vs = row_rs(p.v);
    const auto sas = buffer_rsrc(p.state_dot_a + row0, static_cast<uint32_t>(ntok) * 2 * row_bytes);
    const float* dz = p.dz + ph * (kPiece * D) + t * D + c;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int at = t * kGradStride + c + 4 * h;
      *reinterpret_cast<f32x4*>(&rows[0][at]) = widen4<T>(load4(dys, off + 8 * h)) * p.scale;
      *reinterpret_cast<f32x4*>(&rows[1][at]) = *reinterpret_cast<const f32x4*>(dz + 4 * h);
      const u32x4 sa = __builtin_amdgcn_raw_buffer_load_b128(sas, 2 * off + 16 * h, 0, 0);
      *reinterpret_cast<f32x4*>(&rows[2][at]) = __builtin_bit_cast(f32x4, sa);
      *reinterpret_cast<f32x4*>(&rows[3][at]) = widen4<T>(load4(vs, off + 8 * h));
    }
  }
  __syncthreads();
  // Step j of half h of columns c .. c + 31 takes column c + 8g + 4h + j, so
  // that a lane reads 32 and a group of lanes 128 consecutive bytes of a row.
  auto row4 = [&](int m, int c) {
    return *reinterpret_cast<const f32x4*>(&rows[m][n * kGradStride + c + 8 * g]);
  };

  // Sums over the value columns, 16 at a time: S0 and dS rows as A operands.
  f32x4 acc_r[2], acc_a[2], acc_b[2], acc_k[2];
  float dg[2] = {0.0f, 0.0f};
#pragma unroll
  for (int kt = 0; kt < 2; ++kt) acc_r[kt] = acc_a[kt] = acc_b[kt] = acc_k[kt] = zero4();
  const float* const s_row = s0 + (32 * wave + n) * D + 8 * g;
  const float* const d_row = ds + (32 * wave + n) * D + 8 * g;
#pragma unroll 2
  for (int c = 0; c < D; c += 32) {
    f32x4 s[2][2], d[2][2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        s[kt][h] = *reinterpret_cast<const f32x4*>(s_row + 16 * kt * D + c + 4 * h);
        d[kt][h] = *reinterpret_cast<const f32x4*>(d_row + 16 * kt * D + c + 4 * h);
      }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x4 xdy = row4(0, c + 4 * h), xdz = row4(1, c + 4 * h);
      const f32x4 xsa = row4(2, c + 4 * h), xv = row4(3, c + 4 * h);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
          acc_r[kt] = mfma4(s[kt][h][j], xdy[j], acc_r[kt]);
          acc_a[kt] = mfma4(s[kt][h][j], xdz[j], acc_a[kt]);
          acc_b[kt] = mfma4(d[kt][h][j], xsa[j], acc_b[kt]);
          acc_k[kt] = mfma4(d[kt][h][j], xv[j], acc_k[kt]);
          dg[kt] += s[kt][h][j] * d[kt][h][j];
        }
      }
    }
  }
  // The gradient triangles: waves 0-3, X[t][i] = sum_v A[t][v] B[i][v].
  if (wave < 4) {
    f32x4 x = zero4();
    const int am = wave >> 1, bm = 2 + (wave & 1);
#pragma unroll 4
    for (int c = 0; c < D; c += 32) {
      x = mm16(row4(am, c), row4(bm, c), x);
      x = mm16(row4(am, c + 4), row4(bm, c + 4), x);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = 4 * g + j;
      const bool keep = n < t || (n == t && wave < 2);
      tri[wave][t * kGradTriStride + n] = keep ? x[j] : 0.0f;
    }
  }
  // dg of key 32w + 16kt + n: the lanes of the four column groups.
#pragma unroll
  for (int kt = 0; kt < 2; ++kt) {
    dg[kt] += __shfl_xor(dg[kt], 16);
    dg[kt] += __shfl_xor(dg[kt], 32);
    if (g == 0) dgs[32 * wave + 16 * kt + n] = dg[kt];
  }
  __syncthreads();

  auto tri_r = [&](int m) {  // [t = n][i = 4g + j]
    return *reinterpret_cast<const f32x4*>(&tri[m][n * kGradTriStride + 4 * g]);
  };
  auto tri_c = [&](int m) {  // [t = 4g + j][i = n]
    f32x4 x;
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = tri[m][(4 * g + j) * kGradTriStride + n];
    return x;
  };
  const float* const tiles = p.tiles + ph * L::kBackward;
  const auto rr = row_rs(p.r), rw = row_rs(p.decay), rk = row_rs(p.k), ra = row_rs(p.a),
             rb = row_rs(p.b);
#pragma unroll
  for (int kt = 0; kt < 2; ++kt) {
    const int keyt = 32 * wave + 16 * kt;
    auto col4 = [&](int tile) {  // [key = n][t or i = 4g + j]
      return *reinterpret_cast<const f32x4*>(tiles + tile + (keyt + n) * kPiece + 4 * g);
    };
    const f32x4 atT = col4(L::kAtT), rtT = col4(L::kRtT), bhT = col4(L::kBackBhT),
                khT = col4(L::kBackKhT);
    const int key = keyt + 4 * g;
    const uint32_t off = static_cast<uint32_t>(n) * row_bytes + 2 * key;
    const u32x2 qw = load4(rw, off), qr = load4(rr, off), qk = load4(rk, off),
                qa = load4(ra, off), qb = load4(rb, off);
    acc_r[kt] = mm16(bhT, tri_r(0), acc_r[kt]);
    acc_r[kt] = mm16(khT, tri_r(1), acc_r[kt]);
    acc_a[kt] = mm16(bhT, tri_r(2), acc_a[kt]);
    acc_a[kt] = mm16(khT, tri_r(3), acc_a[kt]);
    f32x4 db = mm16(atT, tri_c(2), zero4());
    db = mm16(rtT, tri_c(0), db);
    f32x4 dk = mm16(atT, tri_c(3), zero4());
    dk = mm16(rtT, tri_c(1), dk);
    const f32x4 total = *reinterpret_cast<const f32x4*>(tiles + L::kBackG + key);
    const f32x4 dgv = *reinterpret_cast<const f32x4*>(&dgs[key]);
    f32x4 x = widen4<T>(qw);
    if (p.bias != nullptr) {
      const S16* bias = static_cast<const S16*>(p.bias) + static_cast<int64_t>(head) * D + key;
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] += to_f32<T>(bias[j]);
    }
    const f32x4 rv = widen4<T>(qr), kv = widen4<T>(qk), av = widen4<T>(qa), bv = widen4<T>(qb);
    f32x4 gr, gw, gk, ga, gb;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const Decay dec = piece_decay(x[j], on);
      const float dbt = total[j] * acc_b[kt][j], dkt = total[j] * acc_k[kt][j];
      const float dbc = db[j] + dbt, dkc = dk[j] + dkt;
      gr[j] = acc_r[kt][j] * dec.incl;
      ga[j] = acc_a[kt][j] * dec.excl;
      gb[j] = dbc * dec.inv;
      gk[j] = dkc * dec.inv;
      // Lanes past the piece hold zero rows (their loads are out of range).
      const float bh = bv[j] * dec.inv, kh = kv[j] * dec.inv;
      const float e2 = ga[j] * av[j];
      const float e1 = gr[j] * rv[j] - dbc * bh - dkc * kh;
      const float e3 = dbt * bh + dkt * kh;
      const float later = suffix16(e1 + e2) - e2;
      // The sum of e3 over the tokens, in every lane of the row.
      const float all3 = __shfl(suffix16(e3), lane & 48);
      const float dlg = later + all3 + dgv[j] * total[j];
      gw[j] = dlg * (-kExpNegHalf) * dec.sig * (1.0f - dec.sig);
    }
    auto store = [&](void* dst, f32x4 y) {
      const auto rs = buffer_rsrc(static_cast<S16*>(dst) + row0,
                                  static_cast<uint32_t>(ntok) * row_bytes);
      __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack2<T>(y[0], y[1]), pack2<T>(y[2], y[3])}, rs,
                                            off, 0, 0);
    };
    store(p.dr, gr);
    store(p.ddecay, gw);
    store(p.dk, gk);
    store(p.da, ga);
    store(p.db, gb);
  }
}

constexpr size_t round256(size_t x) { return (x + 255) & ~static_cast<size_t>(255); }

int64_t lists_of(const Piece32Params& p) {
  return p.seg_offsets != nullptr ? p.num_segments : p.num_sequences;
}

size_t tile_bytes(int head_size, int64_t heads, int64_t slots, bool backward) {
  const int64_t floats = head_size == 64    ? Tiles<64>::kForward
                         : head_size == 128 ? Tiles<128>::kForward
                         : backward         ? Tiles<256>::kBackward
                                            : Tiles<256>::kForward;
  return round256(static_cast<size_t>(slots) * heads * floats * sizeof(float));
}

// Scratch: the piece table, the chunks' first pieces, the flags, the tiles, then the
// backward's adjoints and dZ.
size_t table_bytes(int64_t slots) { return round256(static_cast<size_t>(slots) * sizeof(int4)); }
size_t base_bytes(int64_t lists) {
  return round256((static_cast<size_t>(lists) + 2) * sizeof(int32_t));
}
size_t flag_bytes(int64_t heads, int64_t slots) {
  return round256(static_cast<size_t>(heads) * slots * sizeof(uint32_t));
}

void lay_out(Piece32Params& p, int head_size, bool backward, void* scratch) {
  const int64_t slots = piece32_slots(p.total_tokens, lists_of(p));
  char* at = static_cast<char*>(scratch);
  p.table = reinterpret_cast<int4*>(at);
  at += table_bytes(slots);
  p.base = reinterpret_cast<int32_t*>(at);
  at += base_bytes(lists_of(p));
  p.flags = reinterpret_cast<uint32_t*>(at);
  p.slots_total = static_cast<int32_t>(slots);
  at += flag_bytes(p.num_heads, slots);
  p.tiles = reinterpret_cast<float*>(at);
  at += tile_bytes(head_size, p.num_heads, slots, backward);
  p.adjoints = reinterpret_cast<float*>(at);
  at += static_cast<size_t>(slots) * p.num_heads * head_size * head_size * sizeof(float);
  p.dz = reinterpret_cast<float*>(at);
}

// Pieces the parallel kernels run, after the piece table where one is needed.
int launch_table(const Piece32Params& p, int& pieces, hipStream_t stream) {
  const int slots = static_cast<int>(piece32_slots(p.total_tokens, lists_of(p)));
  pieces = p.dense_t > 0 ? p.num_sequences * (p.dense_t / kPiece) : slots;
  if (p.seg_offsets == nullptr) return FRWKV_OK;
  hipLaunchKernelGGL(piece32_table, dim3(1), dim3(kTableThreads), 0, stream, p, slots);
  return check_launch("piece32_table");
}

template <typename T, int D>
int launch_forward(const Piece32Params& p, hipStream_t stream) {
  int pieces = 0;
  int rc = launch_table(p, pieces, stream);
  if (rc != FRWKV_OK) return rc;
  hipLaunchKernelGGL((piece32_prepare<T, D, false>), dim3(pieces * p.num_heads), dim3(D), 0,
                     stream, p);
  rc = check_launch("piece32_prepare");
  if (rc != FRWKV_OK) return rc;
  constexpr int kBlocks = D / 16 / (4 / (D / 64));  // workgroups per unit
  const dim3 grid(p.num_sequences * p.num_heads * kBlocks);
  if constexpr (D == 256) {
    if (p.boundary != nullptr) {
      hipLaunchKernelGGL((piece32_forward_kernel<T, D, true>), grid, dim3(256), 0, stream, p);
      return check_launch("piece32_forward_kernel");
    }
  }
  hipLaunchKernelGGL((piece32_forward_kernel<T, D, false>), grid, dim3(256), 0, stream, p);
  return check_launch("piece32_forward_kernel");
}

template <typename T>
int dispatch_forward(const Piece32Params& p, int head_size, hipStream_t stream) {
  switch (head_size) {
    case 64:
      return launch_forward<T, 64>(p, stream);
    case 128:
      return launch_forward<T, 128>(p, stream);
    default:
      return launch_forward<T, 256>(p, stream);
  }
}

template <typename T>
int launch_backward(const Piece32Params& p, hipStream_t stream) {
  constexpr int D = 256;
  int pieces = 0;
  int rc = launch_table(p, pieces, stream);
  if (rc != FRWKV_OK) return rc;
  hipLaunchKernelGGL((piece32_prepare<T, D, true>), dim3(pieces * p.num_heads), dim3(D), 0,
                     stream, p);
  rc = check_launch("piece32_prepare");
  if (rc != FRWKV_OK) return rc;
  hipLaunchKernelGGL((piece32_adjoint_kernel<T, D>), dim3(p.num_sequences * p.num_heads * (D / 16)),
                     dim3(256), 0, stream, p);
  rc = check_launch("piece32_adjoint_kernel");
  if (rc != FRWKV_OK) return rc;
  hipLaunchKernelGGL((piece32_gradient_kernel<T, D>), dim3(pieces * p.num_heads),
                     dim3(kGradThreads), 0, stream, p);
  return check_launch("piece32_gradient_kernel");
}

// The flagged units' gradients, token by token; their sums over value columns
// go through the adjoints' area (at least 16 * 256 floats a token and head).
TrainParams redo_params(const Piece32Params& p) {
  TrainParams q{};
  q.num_heads = p.num_heads;
  q.total_tokens = p.total_tokens;
  q.num_sequences = p.num_sequences;
  q.seg_offsets = p.seg_offsets;
  q.seg_starts = p.seg_starts;
  q.seg_ends = p.seg_ends;
  q.num_chunks = p.num_segments;
  q.dense_t = p.dense_t;
  q.ckpt = p.boundary;
  q.interior = p.interior;
  q.r = p.r;
  q.decay = p.decay;
  q.bias = p.bias;
  q.k = p.k;
  q.v = p.v;
  q.a = p.a;
  q.b = p.b;
  q.dy = p.dy;
  q.dstate_final = p.dstate_final;
  q.dr = p.dr;
  q.ddecay = p.ddecay;
  q.dk = p.dk;
  q.dv = p.dv;
  q.da = p.da;
  q.db = p.db;
  q.dstate0 = p.dstate0;
  q.accum = p.adjoints;
  q.scale = p.scale;
  q.redo_flags = p.flags;
  q.redo_slots = p.slots_total;
  q.redo_base = p.seg_offsets != nullptr ? p.base : nullptr;
  return q;
}

}  // namespace

size_t piece32_forward_bytes(int head_size, int64_t heads, int64_t tokens, int64_t lists) {
  if (heads <= 0 || tokens <= 0 || lists <= 0) return 0;
  const int64_t slots = piece32_slots(tokens, lists);
  return table_bytes(slots) + base_bytes(lists) + flag_bytes(heads, slots) +
         tile_bytes(head_size, heads, slots, false);
}

size_t piece32_backward_bytes(int64_t heads, int64_t tokens, int64_t lists) {
  if (heads <= 0 || tokens <= 0 || lists <= 0) return 0;
  const int64_t slots = piece32_slots(tokens, lists);
  return table_bytes(slots) + base_bytes(lists) + flag_bytes(heads, slots) +
         tile_bytes(256, heads, slots, true) +
         static_cast<size_t>(slots) * heads * (256 + kPiece) * 256 * sizeof(float);
}

int piece32_forward(Piece32Params p, int head_size, int io_dtype, void* scratch,
                    hipStream_t stream) {
  lay_out(p, head_size, false, scratch);
  return io_dtype == FRWKV_DTYPE_BF16 ? dispatch_forward<Bf16>(p, head_size, stream)
                                      : dispatch_forward<F16>(p, head_size, stream);
}

int piece32_backward(Piece32Params p, int io_dtype, void* scratch, hipStream_t stream) {
  lay_out(p, 256, true, scratch);
  const int rc = io_dtype == FRWKV_DTYPE_BF16 ? launch_backward<Bf16>(p, stream)
                                              : launch_backward<F16>(p, stream);
  if (rc != FRWKV_OK) return rc;
  return launch_train_redo(redo_params(p), io_dtype, p.num_sequences * p.num_heads, stream);
}

}  // namespace frwkv
