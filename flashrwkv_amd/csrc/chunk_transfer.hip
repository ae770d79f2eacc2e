// Transfer states of sequence parts (chunk_parts.h): for a run of chunks of
// one (sequence, head), the map M and the offset N with
// S_end = M S_start + N.
//
// Per chunk, with the notation of the forward kernel (chunk_fwd_kernel.h), a state
// S (64 keys x any columns) moves by
//   SA = (I - Lab)^{-1} (At S + Lak V),  S' = diag(2^GC) (S + Bh^T SA + Kh^T V),
// so N follows it from 0 and M from the identity with V = 0. Neither needs r,
// Rt, Arb or Ark, and nothing is written per token.
//
// What bounds it: the serial chain of the part's chunks, as in the forward
// kernel. It uses eight waves where the forward uses four: the first four
// carry N's column slabs, the last four M's, and the preparation and the
// intra-chunk products (Lab, Lak and the diagonal inverses alone, about half
// the forward's) are spread over all eight, so a chunk of two states takes
// less time than the forward's chunk of one. 52 KB of LDS (60 KB in the
// split-precision variant) and at most 128 registers per lane leave two
// workgroups per CU. Measured: 5.2 us per chunk alone on a CU, 8.3 with two
// (the forward kernel 5.2 and 7.2); with up to 256 registers, one workgroup
// per CU, 128 units of 4 chunks took 42.4 us instead of 33.2.
#include "capi_internal.h"
#include "chunk_parts.h"
#include "wkv7_device.h"
#include "wkv7_mfma.h"

namespace frwkv {
namespace {

constexpr int kTransferThreads = 512;

template <bool kPrecise>
struct TransferSmem {
  uint16_t at[kOpTile];  // [t][k]
  uint16_t bh[kOpTile];  // [t][k]
  uint16_t kh[kOpTile];  // [t][k] (adjoint: Rt)
  uint16_t vt[kOpTile];  // [t][v] (adjoint: dYs)
  uint16_t kh_lo[kPrecise ? kOpTile : 4];  // low half of Kh (split_bf16x2)
  uint16_t lab[kTriBlocks * kTriBlock];    // [t][i]
  uint16_t lak[kTriBlocks * kTriBlock];    // [t][i] (adjoint: Arb)
  uint16_t tinv[4][kTriBlock];             // (I - Lab_pp)^{-1}, [t][i]
  float blk[4][kHead];  // decay product of each 16-token block
  float gc[kHead];      // 2^GC
};
static_assert(sizeof(TransferSmem<true>) <= 80 * 1024, "two workgroups per CU");

// A thread's token rows: token 16p + n, features 32h + 8g .. +7 of its wave
// (p = wave % 4, h = wave / 4, lane (g, n)).
struct TransferRows {
  uint4 w, a, b, k, v;  // adjoint: r and dy in place of k and v
};

// Decay-span verdicts of a prepared range (see chunk_fwd_kernel.h), uniform over
// the workgroup.
struct TransferSpans {
  bool whole;
  bool block[4];
  __device__ __forceinline__ bool block_ok(int q) const {
    return q == 0 ? block[0] : q == 1 ? block[1] : q == 2 ? block[2] : block[3];
  }
};

// Decodes the rows over tokens [lo, hi) of the chunk (others are zero rows),
// scans the decay and writes the operand tiles. The first barrier frees the
// tiles (every wave is past its previous state update) and publishes the
// block products; the second publishes the tiles.
template <typename T, DecayMode M, bool kPrecise, bool kAdjoint = false>
__device__ __forceinline__ TransferSpans transfer_prepare(TransferSmem<kPrecise>& sm,
                                                          const TransferRows& rows,
                                                          const float (&bias)[8], int lo,
                                                          int hi, float scale = 1.0f) {
  const int tid = lane_tid();
  const int wave = uniform(tid >> 6);
  const int lane = tid & 63;
  const int g = lane >> 4, n = lane & 15;
  const int p = wave & 3, h = wave >> 2;
  const int t = 16 * p + n;
  const int f0 = 32 * h + 8 * g;
  const bool on = t >= lo && t < hi;

  float up[8];  // inclusive decay product within the block
  {
    float x[8];
    unpack8<T>(rows.w, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if constexpr (M == DecayMode::kLogits) x[e] += bias[e];
      const float w = clamped_retention<M>(x[e]);
      up[e] = prefix16_mul(on ? w : 1.0f, n);
    }
  }
  if (n == 15) {
    *reinterpret_cast<float4*>(&sm.blk[p][f0]) = make_float4(up[0], up[1], up[2], up[3]);
    *reinterpret_cast<float4*>(&sm.blk[p][f0 + 4]) = make_float4(up[4], up[5], up[6], up[7]);
  }
  __syncthreads();

  float total[8], carry[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) total[e] = carry[e] = 1.0f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 x0 = *reinterpret_cast<const float4*>(&sm.blk[q][f0]);
    const float4 x1 = *reinterpret_cast<const float4*>(&sm.blk[q][f0 + 4]);
    const float xs[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if (q < p) carry[e] *= xs[e];
      total[e] *= xs[e];
    }
  }
  // Spans over all 64 features: lane l looks at feature l.
  TransferSpans spans;
  {
    float prod = 1.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float x = sm.blk[q][lane];
      prod *= x;
      spans.block[q] = __builtin_amdgcn_ballot_w64(!(x >= kSpanFloor)) == 0;
    }
    spans.whole = __builtin_amdgcn_ballot_w64(!(prod >= kSpanFloor)) == 0;
  }

  // 2^Gp and 2^-G, zero outside [lo, hi). The shift runs in all lanes: the
  // first token of a sub-range reads the lane before it, which is outside.
  float fa[8], fd[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float gp = exclusive16(up[e], n) * carry[e];
    fa[e] = on ? gp : 0.0f;
    fd[e] = on ? __builtin_amdgcn_rcpf(up[e] * carry[e]) : 0.0f;
  }
  const int o = t * kOpStride + f0;
  float x[8];
  unpack8<T>(rows.a, x);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] *= fa[e];
  store8_bf16(sm.at + o, x);
  unpack8<T>(rows.b, x);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] *= fd[e];
  store8_bf16(sm.bh + o, x);
  unpack8<T>(rows.k, x);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] *= kAdjoint ? (on ? up[e] * carry[e] : 0.0f) : fd[e];
  if constexpr (kPrecise) {
    store8_bf16_split(sm.kh + o, sm.kh_lo + o, x);
  } else {
    store8_bf16(sm.kh + o, x);
  }
  unpack8<T>(rows.v, x);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = on ? (kAdjoint ? scale * x[e] : x[e]) : 0.0f;
  store8_bf16(sm.vt + o, x);
  if (p == 0 && n == 0) {
    *reinterpret_cast<float4*>(&sm.gc[f0]) = make_float4(total[0], total[1], total[2], total[3]);
    *reinterpret_cast<float4*>(&sm.gc[f0 + 4]) =
        make_float4(total[4], total[5], total[6], total[7]);
  }
  __syncthreads();
  return spans;
}

// Lab, Lak ([t][i] blocks) and the diagonal inverses: waves 0-3 the diagonal
// block of their index and its inverse, waves 4-7 three of the twelve
// off-diagonal blocks each. Blocks are computed transposed (A operand = Y
// rows), as in chunk_fwd_kernel.h. The adjoint's second matrix is Arb (Rt Bh^T, with
// its diagonal) in place of Lak. Ends with a barrier.
template <bool kPrecise, bool kAdjoint = false>
__device__ __forceinline__ void transfer_intra(TransferSmem<kPrecise>& sm) {
  const int tid = lane_tid();
  const int wave = uniform(tid >> 6);
  const int lane = tid & 63;
  const int g = lane >> 4, n = lane & 15;

  auto block = [&](const uint16_t* x, const uint16_t* y, const uint16_t* y_lo, int p, int q) {
    f32x4 acc = zero4();
#pragma unroll
    for (int c = 0; c < 64; c += 32) {
      const i16x8 xa = lds_operand32<kOpStride>(x, 16 * p + n, c, g);
      acc = mfma32(lds_operand32<kOpStride>(y, 16 * q + n, c, g), xa, acc);
      if constexpr (kPrecise) {
        if (y_lo != nullptr) {
          acc = mfma32(lds_operand32<kOpStride>(y_lo, 16 * q + n, c, g), xa, acc);
        }
      }
    }
    return acc;
  };
  const uint16_t* kh_lo = kPrecise ? sm.kh_lo : nullptr;
  const uint16_t* x2 = kAdjoint ? sm.kh : sm.at;  // factors of the second matrix
  const uint16_t* y2 = kAdjoint ? sm.bh : sm.kh;
  if (wave < 4) {
    f32x4 l_r = zero4(), l_c = zero4();
#pragma unroll
    for (int c = 0; c < 64; c += 32) {
      const i16x8 xa = lds_operand32<kOpStride>(sm.at, 16 * wave + n, c, g);
      const i16x8 yb = lds_operand32<kOpStride>(sm.bh, 16 * wave + n, c, g);
      l_r = mfma32(yb, xa, l_r);  // lane (g, n): L[n][4g + j]
      l_c = mfma32(xa, yb, l_c);  // lane (g, n): L[4g + j][n]
    }
    f32x4 lak = block(x2, y2, kh_lo, wave, wave);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      l_r[j] = (4 * g + j < n) ? l_r[j] : 0.0f;
      lak[j] = (4 * g + j < n || (kAdjoint && 4 * g + j == n)) ? lak[j] : 0.0f;
    }
    const int at = tri_index(wave, wave) * kTriBlock;
    lds_store_transposed(sm.lab + at, kTriStride, g, n, l_r);
    lds_store_transposed(sm.lak + at, kTriStride, g, n, lak);
    lds_store_transposed(sm.tinv[wave], kTriStride, g, n, invert_unit_lower(l_r, l_c));
  } else {
    // Block pairs (1,0) (2,0) (2,1) (3,0) (3,1) (3,2), each for Lab and Lak.
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const int item = (wave - 4) + 4 * r;
      const int pair = item >> 1;
      const int p = pair < 1 ? 1 : (pair < 3 ? 2 : 3);
      const int q = pair - (p * (p - 1)) / 2;
      const bool with_k = (item & 1) != 0;
      const f32x4 acc =
          with_k ? block(x2, y2, kh_lo, p, q) : block(sm.at, sm.bh, nullptr, p, q);
      lds_store_transposed((with_k ? sm.lak : sm.lab) + tri_index(p, q) * kTriBlock, kTriStride,
                           g, n, acc);
    }
  }
  __syncthreads();
}

// One chunk's step of a column slab (C layout: S[kb][j] is row 16kb + 4g + j,
// column 16cs + n). kWithV: the slab belongs to N, else to M (V = 0).
template <bool kWithV, bool kPrecise>
__device__ __forceinline__ void transfer_step(const TransferSmem<kPrecise>& sm, f32x4 (&S)[4],
                                              int cs) {
  const int lane = lane_tid() & 63;
  const int g = lane >> 4, n = lane & 15;
  const i16x4 z4 = {0, 0, 0, 0};
  auto lo32 = [&](i16x4 x) { return cat(x, z4); };
  auto tri = [&](const uint16_t* m, int p, int q) {
    return lds_operand<kTriStride>(m + tri_index(p, q) * kTriBlock, n, 4 * g);
  };
  auto tri2 = [&](const uint16_t* m, int p, int q) { return cat(tri(m, p, q), tri(m, p, q + 1)); };
  auto tr32 = [&](const uint16_t* tile, int kb, int c) {
    return cat(lds_operand_tr<kOpStride>(tile, c, 16 * kb, g, n),
               lds_operand_tr<kOpStride>(tile, c + 16, 16 * kb, g, n));
  };
  i16x8 v01, v23;
  if constexpr (kWithV) {
    v01 = tr32(sm.vt, cs, 0);
    v23 = tr32(sm.vt, cs, 32);
  }

  f32x4 rhs[4];
  {
    const i16x8 s01 = cat(to_operand(S[0]), to_operand(S[1]));
    const i16x8 s23 = cat(to_operand(S[2]), to_operand(S[3]));
#pragma unroll
    for (int pb = 0; pb < 4; ++pb)
      rhs[pb] = mfma32(lds_operand32<kOpStride>(sm.at, 16 * pb + n, 0, g), s01, zero4());
#pragma unroll
    for (int pb = 0; pb < 4; ++pb)
      rhs[pb] = mfma32(lds_operand32<kOpStride>(sm.at, 16 * pb + n, 32, g), s23, rhs[pb]);
  }
  if constexpr (kWithV) {
    const i16x8 v0 = lo32(__builtin_shufflevector(v01, v01, 0, 1, 2, 3));
    const i16x8 v2 = lo32(__builtin_shufflevector(v23, v23, 0, 1, 2, 3));
    rhs[0] = mfma32(lo32(tri(sm.lak, 0, 0)), v0, rhs[0]);
    rhs[1] = mfma32(tri2(sm.lak, 1, 0), v01, rhs[1]);
    rhs[2] = mfma32(tri2(sm.lak, 2, 0), v01, rhs[2]);
    rhs[3] = mfma32(tri2(sm.lak, 3, 0), v01, rhs[3]);
    rhs[2] = mfma32(lo32(tri(sm.lak, 2, 2)), v2, rhs[2]);
    rhs[3] = mfma32(tri2(sm.lak, 3, 2), v23, rhs[3]);
  }

  // Block forward substitution SA_p = T_pp (rhs_p + sum_{q<p} Lab_pq SA_q).
  auto solve = [&](int pb) {
    return to_operand(mfma32(lo32(lds_operand<kTriStride>(sm.tinv[pb], n, 4 * g)),
                             lo32(to_operand(rhs[pb])), zero4()));
  };
  const i16x4 sa0 = solve(0);
  rhs[1] = mfma32(lo32(tri(sm.lab, 1, 0)), lo32(sa0), rhs[1]);
  const i16x4 sa1 = solve(1);
  const i16x8 sa01 = cat(sa0, sa1);
  rhs[2] = mfma32(tri2(sm.lab, 2, 0), sa01, rhs[2]);
  rhs[3] = mfma32(tri2(sm.lab, 3, 0), sa01, rhs[3]);
  const i16x4 sa2 = solve(2);
  rhs[3] = mfma32(lo32(tri(sm.lab, 3, 2)), lo32(sa2), rhs[3]);
  const i16x8 sa23 = cat(sa2, solve(3));

  f32x4 sn[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) sn[kb] = S[kb];
  if constexpr (kWithV) {
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) sn[kb] = mfma32(tr32(sm.kh, kb, 0), v01, sn[kb]);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) sn[kb] = mfma32(tr32(sm.kh, kb, 32), v23, sn[kb]);
    if constexpr (kPrecise) {
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) sn[kb] = mfma32(tr32(sm.kh_lo, kb, 0), v01, sn[kb]);
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) sn[kb] = mfma32(tr32(sm.kh_lo, kb, 32), v23, sn[kb]);
    }
  }
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) sn[kb] = mfma32(tr32(sm.bh, kb, 0), sa01, sn[kb]);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) sn[kb] = mfma32(tr32(sm.bh, kb, 32), sa23, sn[kb]);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const float4 gc = *reinterpret_cast<const float4*>(&sm.gc[16 * kb + 4 * g]);
    S[kb] = f32x4{sn[kb][0] * gc.x, sn[kb][1] * gc.y, sn[kb][2] * gc.z, sn[kb][3] * gc.w};
  }
}

template <typename T, DecayMode M, typename PoolT, bool kPrecise>
__global__ __launch_bounds__(kTransferThreads, 4) void chunk_transfer_kernel(ChunkFwdParams p) {
  __shared__ TransferSmem<kPrecise> sm;
  if (p.status != nullptr && p.status[0] != 0) return;
  const int tid = threadIdx.x;
  const int wave = uniform(tid >> 6);
  const int lane = tid & 63;
  const int g = lane >> 4, n = lane & 15;
  const int cs = wave & 3;        // column slab
  const bool map = wave >= 4;     // M's slab (else N's)
  const int heads = p.num_heads;
  const PartPlace place =
      p.part_slots > 0 ? packed_place<true>(p, lane) : unit_place<true>(p);
  const int part = place.part, seq = place.seq, head = place.head;
  const int slot = uniform(p.slots != nullptr ? p.slots[seq] : seq);
  if (slot < 0 || slot >= p.state_slots) return;

  // The part's segments (caller chunks), or its run of 64-token chunks.
  int seg = 0, seg_hi = 1, c0 = 0, c_end = 0;
  bool last;
  if (p.seg_offsets != nullptr) {
    const int lo = uniform(max(p.seg_offsets[seq], 0));
    const int hi = uniform(min(p.seg_offsets[seq + 1], p.num_segments));
    const PartRange r = part_range(p, max(hi - lo, 0), part);
    if (!r.exists) return;
    seg = lo + r.begin;
    seg_hi = lo + r.end;
    last = r.last;
  } else {
    int begin, end;
    if (p.dense_t > 0) {
      begin = seq * p.dense_t;
      end = begin + p.dense_t;
    } else {
      begin = p.cu_seqlens[seq];
      end = p.cu_seqlens[seq + 1];
    }
    begin = uniform(max(begin, 0));
    end = uniform(min(end, p.total_tokens));
    const PartRange r = part_range(p, (max(end - begin, 0) + kChunk - 1) / kChunk, part);
    if (!r.exists) return;
    c0 = begin + r.begin * kChunk;
    c_end = min(begin + r.end * kChunk, end);
    last = r.last;
  }
  if (last) return;  // no part follows
  auto next_segment = [&]() {    // the segment's tokens into [c0, c_end)
    if (p.seg_offsets == nullptr) return;
    c0 = uniform(max(p.seg_starts[seg], 0));
    c_end = uniform(min(p.seg_ends[seg], p.total_tokens));
  };

  // Start states, in C layout.
  f32x4 S[4];
  const uint32_t s_off = static_cast<uint32_t>((4 * g) * kHead + 16 * cs + n);
  if (part == 0 && p.state != nullptr) {
    using PS = typename IoTraits<PoolT>::storage;
    const PS* src = static_cast<const PS*>(p.state) +
                    (static_cast<int64_t>(slot) * heads + head) * kStateElems + s_off;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
      for (int j = 0; j < 4; ++j) S[kb][j] = to_f32<PoolT>(src[(16 * kb + j) * kHead]);
    }
  } else {
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        S[kb][j] = (part > 0 && map && 16 * kb + 4 * g + j == 16 * cs + n) ? 1.0f : 0.0f;
      }
    }
  }

  float bias[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) bias[e] = 0.0f;
  const int f0 = 32 * (wave >> 2) + 8 * g;
  if constexpr (M == DecayMode::kLogits) {
    if (p.bias != nullptr) {
      unpack8<T>(load_row8<T>(p.bias, static_cast<int64_t>(head) * kHead + f0), bias);
    }
  }

  using S16 = typename IoTraits<T>::storage;
  const uint32_t row_bytes = static_cast<uint32_t>(heads) * kHead * 2;
  const uint32_t row_off = static_cast<uint32_t>(16 * (wave & 3) + n) * row_bytes + 2 * f0;
  auto load = [&](const void* src, int first, int ntok) {
    const int64_t base = (static_cast<int64_t>(first) * heads + head) * kHead;
    const auto rs = buffer_rsrc(static_cast<const S16*>(src) + base,
                                static_cast<uint32_t>(ntok) * row_bytes);
    const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(rs, row_off, 0, 0);
    return make_uint4(x.x, x.y, x.z, x.w);
  };
  auto load_rows = [&](TransferRows& rows, int first, int ntok) {
    rows.w = load(p.decay, first, ntok);
    rows.a = load(p.a, first, ntok);
    rows.b = load(p.b, first, ntok);
    rows.k = load(p.k, first, ntok);
    rows.v = load(p.v, first, ntok);
  };

  bool more = seg < seg_hi;
  if (more) next_segment();
  while (more && c0 >= c_end) {  // empty segments
    more = ++seg < seg_hi;
    if (more) next_segment();
  }
  TransferRows rows;
  if (more) load_rows(rows, c0, min(kChunk, c_end - c0));
  while (more) {
    const int ntok = min(kChunk, c_end - c0);
    c0 += kChunk;
    while (more && c0 >= c_end) {
      more = ++seg < seg_hi;
      if (more) next_segment();
    }
    // One pass over the whole chunk, or, where its decay span exceeds the
    // limit, over 16- or 4-token sub-chunks (as in chunk_fwd_kernel.h).
    TransferSpans spans{};
    bool whole = true, probe = true;
    int lo = 0, hi = ntok;
    for (;;) {
      const TransferSpans cur = transfer_prepare<T, M, kPrecise>(sm, rows, bias, lo, hi);
      if (probe) {
        probe = false;
        spans = cur;
        whole = cur.whole;
        if (!whole) {
          hi = min(spans.block[0] ? 16 : 4, ntok);
          continue;
        }
        if (more) load_rows(rows, c0, min(kChunk, c_end - c0));
      }
      transfer_intra<kPrecise>(sm);
      if (!map) {
        transfer_step<true, kPrecise>(sm, S, cs);
      } else if (part > 0) {
        transfer_step<false, kPrecise>(sm, S, cs);
      }
      if (whole) break;
      lo = hi;
      if (lo >= ntok) break;
      const int q = lo >> 4;
      hi = min(lo + (spans.block_ok(q) ? 16 : 4), min(16 * q + 16, ntok));
    }
    if (!whole && more) load_rows(rows, c0, min(kChunk, c_end - c0));
  }

  store_part_state(place, part, map, s_off, S);
}

// One chunk's adjoint step of a column slab, dS at the chunk's end to dS at its
// start (C layout): with U = g o dS,
//   dSA = Bh U + Arb^T dYs,  dZ = T^T dSA,  dS0 = U + Rt^T dYs + At^T dZ
// (chunk_bwd.hip). kWithDy: the slab belongs to N, else to M (dY = 0).
template <bool kWithDy>
__device__ __forceinline__ void adjoint_step(const TransferSmem<false>& sm, f32x4 (&S)[4],
                                             int cs) {
  const int lane = lane_tid() & 63;
  const int g = lane >> 4, n = lane & 15;
  const i16x4 z4 = {0, 0, 0, 0};
  auto lo32 = [&](i16x4 x) { return cat(x, z4); };
  auto lt = [&](const uint16_t* m, int p, int q) {  // block (p, q) transposed
    return lds_operand_tr<kTriStride>(m + tri_index(p, q) * kTriBlock, 0, 0, g, n);
  };
  auto tr32 = [&](const uint16_t* tile, int kb, int t) {
    return cat(lds_operand_tr<kOpStride>(tile, t, 16 * kb, g, n),
               lds_operand_tr<kOpStride>(tile, t + 16, 16 * kb, g, n));
  };
  auto half = [](const i16x8& x, int h) {
    return h == 0 ? __builtin_shufflevector(x, x, 0, 1, 2, 3)
                  : __builtin_shufflevector(x, x, 4, 5, 6, 7);
  };
  i16x8 y01, y23;
  if constexpr (kWithDy) {
    y01 = tr32(sm.vt, cs, 0);
    y23 = tr32(sm.vt, cs, 32);
  }
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const float4 gc = *reinterpret_cast<const float4*>(&sm.gc[16 * kb + 4 * g]);
    S[kb] = f32x4{S[kb][0] * gc.x, S[kb][1] * gc.y, S[kb][2] * gc.z, S[kb][3] * gc.w};
  }
  f32x4 dsa[4];
  {
    const i16x8 u01 = cat(to_operand(S[0]), to_operand(S[1]));
    const i16x8 u23 = cat(to_operand(S[2]), to_operand(S[3]));
#pragma unroll
    for (int pb = 0; pb < 4; ++pb)
      dsa[pb] = mfma32(lds_operand32<kOpStride>(sm.bh, 16 * pb + n, 0, g), u01, zero4());
#pragma unroll
    for (int pb = 0; pb < 4; ++pb)
      dsa[pb] = mfma32(lds_operand32<kOpStride>(sm.bh, 16 * pb + n, 32, g), u23, dsa[pb]);
  }
  if constexpr (kWithDy) {
    const uint16_t* arb = sm.lak;
    dsa[3] = mfma32(lo32(lt(arb, 3, 3)), lo32(half(y23, 1)), dsa[3]);
    dsa[2] = mfma32(cat(lt(arb, 2, 2), lt(arb, 3, 2)), y23, dsa[2]);
    dsa[1] = mfma32(lo32(lt(arb, 1, 1)), lo32(half(y01, 1)), dsa[1]);
    dsa[1] = mfma32(cat(lt(arb, 2, 1), lt(arb, 3, 1)), y23, dsa[1]);
    dsa[0] = mfma32(cat(lt(arb, 0, 0), lt(arb, 1, 0)), y01, dsa[0]);
    dsa[0] = mfma32(cat(lt(arb, 2, 0), lt(arb, 3, 0)), y23, dsa[0]);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) S[kb] = mfma32(tr32(sm.kh, kb, 0), y01, S[kb]);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) S[kb] = mfma32(tr32(sm.kh, kb, 32), y23, S[kb]);
  }
  // dZ_p = T_pp^T (dSA_p + sum_{q>p} Lab^T(q, p) dZ_q).
  auto solve = [&](int pb) {
    return to_operand(mfma32(lo32(lds_operand_tr<kTriStride>(sm.tinv[pb], 0, 0, g, n)),
                             lo32(to_operand(dsa[pb])), zero4()));
  };
  const i16x4 dz3 = solve(3);
  dsa[2] = mfma32(lo32(lt(sm.lab, 3, 2)), lo32(dz3), dsa[2]);
  const i16x4 dz2 = solve(2);
  const i16x8 dz23 = cat(dz2, dz3);
  dsa[1] = mfma32(cat(lt(sm.lab, 2, 1), lt(sm.lab, 3, 1)), dz23, dsa[1]);
  dsa[0] = mfma32(cat(lt(sm.lab, 2, 0), lt(sm.lab, 3, 0)), dz23, dsa[0]);
  const i16x4 dz1 = solve(1);
  dsa[0] = mfma32(lo32(lt(sm.lab, 1, 0)), lo32(dz1), dsa[0]);
  const i16x8 dz01 = cat(solve(0), dz1);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) S[kb] = mfma32(tr32(sm.at, kb, 32), dz23, S[kb]);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) S[kb] = mfma32(tr32(sm.at, kb, 0), dz01, S[kb]);
}

// The adjoint's transfer states: chunks from the last to the first, segments
// likewise (backward part 0 is a sequence's last run). Same bound, split and
// tiles as chunk_transfer_kernel. Measured: 1 chunk per part 10.6 us, 3 chunks
// 20.6, 5 chunks 30.4 (192 workgroups); the backward of 2 x 17 chunks in 32
// heads takes 95 us with it and 185 without, of 2 x 8 chunks in 12 heads 35
// and 88.
template <typename T, DecayMode M>
__global__ __launch_bounds__(kTransferThreads, 4) void chunk_adjoint_kernel(ChunkBwdParams p) {
  __shared__ TransferSmem<false> sm;
  const int tid = threadIdx.x;
  const int wave = uniform(tid >> 6);
  const int lane = tid & 63;
  const int g = lane >> 4, n = lane & 15;
  const int cs = wave & 3;
  const bool map = wave >= 4;
  const int heads = p.num_heads;
  const PartPlace place = unit_place<true>(p);
  const int part = place.part, seq = place.seq, head = place.head;

  // The part's segments, or its run of chunks of the dense sequence; chunks
  // start at c_begin + 64 j.
  int seg = 0, seg_lo = 0, c_begin = 0, c_end = 0;
  bool last;
  if (p.seg_offsets != nullptr) {
    const int lo = uniform(max(p.seg_offsets[seq], 0));
    const int hi = uniform(min(p.seg_offsets[seq + 1], p.num_segments));
    const PartRange r = part_range(p, max(hi - lo, 0), part);
    if (!r.exists) return;
    seg = hi - r.begin;
    seg_lo = hi - r.end;
    last = r.last;
  } else {
    const int count = (p.dense_t + kChunk - 1) / kChunk;
    const PartRange r = part_range(p, count, part);
    if (!r.exists) return;
    c_begin = seq * p.dense_t + (count - r.end) * kChunk;
    c_end = seq * p.dense_t + min((count - r.begin) * kChunk, p.dense_t);
    seg = r.end > r.begin ? 1 : 0;
    last = r.last;
  }
  if (last) return;  // no part follows

  f32x4 S[4];
  const uint32_t s_off = static_cast<uint32_t>((4 * g) * kHead + 16 * cs + n);
  {
    const float* src = part == 0 ? p.dstate_final : nullptr;
    if (src != nullptr) src += (static_cast<int64_t>(seq) * heads + head) * kStateElems + s_off;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        S[kb][j] = src != nullptr ? src[(16 * kb + j) * kHead]
                   : (part > 0 && map && 16 * kb + 4 * g + j == 16 * cs + n) ? 1.0f
                                                                             : 0.0f;
      }
    }
  }

  float bias[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) bias[e] = 0.0f;
  const int f0 = 32 * (wave >> 2) + 8 * g;
  if constexpr (M == DecayMode::kLogits) {
    if (p.bias != nullptr) {
      unpack8<T>(load_row8<T>(p.bias, static_cast<int64_t>(head) * kHead + f0), bias);
    }
  }

  using S16 = typename IoTraits<T>::storage;
  const uint32_t row_bytes = static_cast<uint32_t>(heads) * kHead * 2;
  const uint32_t row_off = static_cast<uint32_t>(16 * (wave & 3) + n) * row_bytes + 2 * f0;
  auto load = [&](const void* src, int first, int ntok) {
    const int64_t base = (static_cast<int64_t>(first) * heads + head) * kHead;
    const auto rs = buffer_rsrc(static_cast<const S16*>(src) + base,
                                src != nullptr ? static_cast<uint32_t>(ntok) * row_bytes : 0u);
    const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(rs, row_off, 0, 0);
    return make_uint4(x.x, x.y, x.z, x.w);
  };
  auto load_rows = [&](TransferRows& rows, int first, int ntok) {
    rows.w = load(p.decay, first, ntok);
    rows.a = load(p.a, first, ntok);
    rows.b = load(p.b, first, ntok);
    rows.k = load(p.r, first, ntok);
    rows.v = load(p.dy, first, ntok);
  };

  // The chunk before: [c0, c_end) within the current segment, else the last
  // one of the nearest earlier segment with tokens.
  int c0 = c_end;
  auto previous = [&]() {
    c_end = c0;
    while (c0 <= c_begin) {
      if (--seg < seg_lo) return false;
      if (p.seg_offsets != nullptr) {
        c_begin = uniform(max(p.seg_starts[seg], 0));
        c0 = c_end = uniform(min(p.seg_ends[seg], p.total_tokens));
      }
    }
    c0 = c_begin + (c_end - c_begin - 1) / kChunk * kChunk;
    return true;
  };
  bool more = seg > seg_lo && previous();
  TransferRows rows;
  if (more) load_rows(rows, c0, c_end - c0);
  while (more) {
    const int ntok = c_end - c0;
    more = previous();
    // As in the transfer kernel, sub-chunks from the last to the first.
    TransferSpans spans{};
    bool whole = true, probe = true;
    int lo = 0, hi = ntok;
    for (;;) {
      const TransferSpans cur =
          transfer_prepare<T, M, false, true>(sm, rows, bias, lo, hi, p.scale);
      if (probe) {
        probe = false;
        spans = cur;
        whole = cur.whole;
        if (!whole) {
          lo = (hi - 1) & (spans.block_ok((hi - 1) >> 4) ? ~15 : ~3);
          continue;
        }
        if (more) load_rows(rows, c0, c_end - c0);
      }
      transfer_intra<false, true>(sm);
      if (!map) {
        adjoint_step<true>(sm, S, cs);
      } else if (part > 0) {
        adjoint_step<false>(sm, S, cs);
      }
      if (whole || lo == 0) break;
      hi = lo;
      lo = (hi - 1) & (spans.block_ok((hi - 1) >> 4) ? ~15 : ~3);
    }
    if (!whole && more) load_rows(rows, c0, c_end - c0);
  }

  store_part_state(place, part, map, s_off, S);
}

}  // namespace

template <typename T, DecayMode M, typename PoolT, bool kPrecise>
int launch_chunk_transfer(const ChunkFwdParams& p, int units, hipStream_t stream) {
  hipLaunchKernelGGL((chunk_transfer_kernel<T, M, PoolT, kPrecise>),
                     dim3(p.part_slots > 0 ? p.part_slots * p.num_heads : units * (p.parts - 1)),
                     dim3(kTransferThreads), 0, stream, p);
  return check_launch("chunk_transfer_kernel");
}

template <typename T, DecayMode M>
int launch_chunk_adjoint(const ChunkBwdParams& p, int units, hipStream_t stream) {
  hipLaunchKernelGGL((chunk_adjoint_kernel<T, M>), dim3(units * (p.parts - 1)),
                     dim3(kTransferThreads), 0, stream, p);
  return check_launch("chunk_adjoint_kernel");
}
template int launch_chunk_adjoint<Bf16, DecayMode::kLogits>(const ChunkBwdParams&, int,
                                                            hipStream_t);
template int launch_chunk_adjoint<Bf16, DecayMode::kRawW>(const ChunkBwdParams&, int,
                                                          hipStream_t);
template int launch_chunk_adjoint<F16, DecayMode::kLogits>(const ChunkBwdParams&, int,
                                                           hipStream_t);
template int launch_chunk_adjoint<F16, DecayMode::kRawW>(const ChunkBwdParams&, int,
                                                         hipStream_t);

#define FRWKV_TRANSFER(T, M, PoolT, P) \
  template int launch_chunk_transfer<T, M, PoolT, P>(const ChunkFwdParams&, int, hipStream_t);
FRWKV_TRANSFER(Bf16, DecayMode::kLogits, float, false)
FRWKV_TRANSFER(Bf16, DecayMode::kRawW, float, false)
FRWKV_TRANSFER(F16, DecayMode::kLogits, float, false)
FRWKV_TRANSFER(F16, DecayMode::kRawW, float, false)
FRWKV_TRANSFER(Bf16, DecayMode::kLogits, Bf16, false)
FRWKV_TRANSFER(Bf16, DecayMode::kRawW, Bf16, false)
FRWKV_TRANSFER(F16, DecayMode::kLogits, Bf16, false)
FRWKV_TRANSFER(F16, DecayMode::kRawW, Bf16, false)
FRWKV_TRANSFER(Bf16, DecayMode::kLogits, float, true)
FRWKV_TRANSFER(Bf16, DecayMode::kRawW, float, true)
#undef FRWKV_TRANSFER

}  // namespace frwkv
