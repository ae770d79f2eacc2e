// The bf16 instantiations of the chunked forward kernel (chunk_fwd_kernel.h)
// and the entries that run it: packed prefill, training and replay.
#include "chunk_fwd_kernel.h"
#include "piece32.h"

namespace frwkv {
namespace {

template <typename T, typename PoolT>
int dispatch_chunk_decay(const ChunkFwdParams& p, int decay_mode, int units,
                         hipStream_t stream) {
  if (decay_mode == FRWKV_DECAY_LOGITS) {
    return launch_chunk<T, DecayMode::kLogits, PoolT>(p, units, stream);
  }
  if (decay_mode == FRWKV_DECAY_RAW_W) {
    if (p.bias != nullptr) {
      return set_error(FRWKV_ERR_INVALID_ARGUMENT,
                       "decay_bias is only defined for the logits decay mode");
    }
    return launch_chunk<T, DecayMode::kRawW, PoolT>(p, units, stream);
  }
  return set_error(FRWKV_ERR_INVALID_ARGUMENT, "unknown decay mode %d", decay_mode);
}

template <typename PoolT>
int dispatch_chunk_io(const ChunkFwdParams& p, int io_dtype, int decay_mode, int units,
                      hipStream_t stream) {
  switch (io_dtype) {
    case FRWKV_DTYPE_BF16:
      return dispatch_chunk_decay<Bf16, PoolT>(p, decay_mode, units, stream);
    case FRWKV_DTYPE_F16:
      return dispatch_chunk_decay<F16, PoolT>(p, decay_mode, units, stream);
    default:
      return set_error(FRWKV_ERR_UNSUPPORTED,
                       "chunked kernels take float16 or bfloat16 tokens (io dtype %d)",
                       io_dtype);
  }
}

int check_token_pointers(const void* r, const void* decay, const void* k, const void* v,
                         const void* a, const void* b, const void* out) {
  if (!r || !decay || !k || !v || !a || !b || !out) {
    return set_error(FRWKV_ERR_INVALID_ARGUMENT, "null token pointer argument");
  }
  return FRWKV_OK;
}

}  // namespace
}  // namespace frwkv

extern "C" size_t frwkv_split_scratch_bytes(int kernel, int io_dtype, int decay_mode,
                                            int32_t num_sequences, int32_t num_heads,
                                            int32_t head_size, int32_t total, int32_t longest) {
  using namespace frwkv;
  if (num_sequences <= 0 || num_heads <= 0 || total <= 0) return 0;
  if (kernel == FRWKV_SPLIT_RECURRENT &&
      piece32_recurrent(io_dtype, decay_mode, head_size, num_sequences, num_heads, total,
                        longest)) {
    const size_t bytes = piece32_forward_bytes(head_size, num_heads, total, num_sequences);
    return bytes <= kPiece32RecurrentBytes ? bytes : 0;
  }
  if (kernel == FRWKV_SPLIT_RECURRENT && io_dtype != FRWKV_DTYPE_BF16) return 0;
  if (head_size == 256 && decay_mode == FRWKV_DECAY_LOGITS && kernel == FRWKV_SPLIT_CHUNK) {
    return piece32_forward_bytes(head_size, num_heads, total, num_sequences);
  }
  if (head_size == 256 && decay_mode == FRWKV_DECAY_LOGITS &&
      kernel == FRWKV_SPLIT_CALLER_CHUNKS) {
    return piece32_forward_bytes(head_size, num_heads, longest, total);
  }
  if (head_size == 256 && decay_mode == FRWKV_DECAY_LOGITS) {
    if (kernel == FRWKV_SPLIT_PRETRAIN_BACKWARD) {
      return piece32_backward_bytes(num_heads, total, num_sequences);
    }
    if (kernel == FRWKV_SPLIT_CALLER_CHUNKS_BACKWARD) {
      return piece32_backward_bytes(num_heads, longest, total);
    }
  }
  if (head_size != 64) return 0;
  const int64_t units = static_cast<int64_t>(num_sequences) * num_heads;
  switch (kernel) {
    case FRWKV_SPLIT_CHUNK:  // of equal sequences (pretraining): states by unit
      return packed_part_bytes(total, num_sequences, num_heads,
                               plan_packed_parts(num_sequences, num_heads, total, longest,
                                                 kForwardTime, kTransferTime));
    case FRWKV_SPLIT_RECURRENT:
      return packed_part_bytes(total, num_sequences, num_heads,
                               plan_packed_parts(num_sequences, num_heads, total, longest,
                                                 kPreciseTime, kTransferTime));
    case FRWKV_SPLIT_CALLER_CHUNKS:
      return unit_part_bytes(units, plan_caller_chunks(num_sequences, num_heads, total));
    case FRWKV_SPLIT_PRETRAIN_BACKWARD:
      return unit_part_bytes(units,
                             plan_parts(num_sequences, num_heads,
                                        num_sequences * chunks_of(total / num_sequences),
                                        chunks_of(total / num_sequences), kBackwardTime,
                                        kAdjointTime));
    case FRWKV_SPLIT_CALLER_CHUNKS_BACKWARD:
      return unit_part_bytes(units, plan_caller_chunks(num_sequences, num_heads, total,
                                                       kBackwardTime, kAdjointTime));
    default:
      return 0;
  }
}

extern "C" int frwkv_chunk_forward(
    int io_dtype, int decay_mode, int pool_dtype, int32_t num_sequences,
    int32_t num_heads, int32_t head_size, int32_t total_tokens, int32_t state_pool_size,
    const int32_t* cu_seqlens, const int32_t* state_indices,
    const int32_t* metadata_status, void* state_pool, const void* r, const void* decay,
    const void* decay_bias, const void* k, const void* v, const void* a, const void* b,
    void* output, float scale, void* stream) {
  return frwkv_chunk_forward_split(io_dtype, decay_mode, pool_dtype, num_sequences, num_heads,
                                   head_size, total_tokens, state_pool_size, cu_seqlens,
                                   state_indices, metadata_status, state_pool, r, decay,
                                   decay_bias, k, v, a, b, output, scale, /*max_seqlen=*/-1,
                                   nullptr, 0, stream);
}

extern "C" int frwkv_chunk_forward_split(
    int io_dtype, int decay_mode, int pool_dtype, int32_t num_sequences,
    int32_t num_heads, int32_t head_size, int32_t total_tokens, int32_t state_pool_size,
    const int32_t* cu_seqlens, const int32_t* state_indices,
    const int32_t* metadata_status, void* state_pool, const void* r, const void* decay,
    const void* decay_bias, const void* k, const void* v, const void* a, const void* b,
    void* output, float scale, int32_t max_seqlen, void* scratch, size_t scratch_bytes,
    void* stream) {
  using namespace frwkv;
  if (!cu_seqlens || !state_indices || !metadata_status || !state_pool) {
    return set_error(FRWKV_ERR_INVALID_ARGUMENT, "frwkv_chunk_forward: null pointer argument");
  }
  int rc = check_token_pointers(r, decay, k, v, a, b, output);
  if (rc != FRWKV_OK) return rc;
  if (head_size != 64) {
    return set_error(FRWKV_ERR_UNSUPPORTED, "chunked kernels support head size 64, got %d",
                     head_size);
  }
  if (num_sequences <= 0 || num_sequences > 65535 || num_heads <= 0 || total_tokens <= 0 ||
      state_pool_size <= 0) {
    return set_error(FRWKV_ERR_INVALID_ARGUMENT,
                     "frwkv_chunk_forward: sizes must be positive (B=%d, H=%d, N=%d, slots=%d)",
                     num_sequences, num_heads, total_tokens, state_pool_size);
  }
  if (!__builtin_isfinite(scale)) {
    return set_error(FRWKV_ERR_INVALID_ARGUMENT, "scale must be finite");
  }
  ChunkFwdParams p{};
  p.num_heads = num_heads;
  p.longest_first_sequences = num_sequences <= 64 ? num_sequences : 0;
  p.total_tokens = total_tokens;
  p.state_slots = state_pool_size;
  p.cu_seqlens = cu_seqlens;
  p.slots = state_indices;
  p.status = metadata_status;
  p.state = state_pool;
  p.r = r;
  p.decay = decay;
  p.bias = decay_bias;
  p.k = k;
  p.v = v;
  p.a = a;
  p.b = b;
  p.out = output;
  p.scale = scale;
  p.out_elems = static_cast<int64_t>(total_tokens) * num_heads * head_size;
  const int units = num_sequences * num_heads;
  use_packed_parts(p, num_sequences,
                   plan_packed_parts(num_sequences, num_heads, total_tokens, max_seqlen,
                                     kForwardTime, kTransferTime),
                   scratch, scratch_bytes);
  auto s = static_cast<hipStream_t>(stream);
  if (pool_dtype == FRWKV_DTYPE_F32) return dispatch_chunk_io<float>(p, io_dtype, decay_mode, units, s);
  if (pool_dtype == FRWKV_DTYPE_BF16) return dispatch_chunk_io<Bf16>(p, io_dtype, decay_mode, units, s);
  return set_error(FRWKV_ERR_UNSUPPORTED, "state pool must be float32 or bfloat16 (dtype %d)",
                   pool_dtype);
}

extern "C" int frwkv_statetune_forward(
    int io_dtype, int decay_mode, int32_t num_sequences, int32_t num_heads,
    int32_t head_size, int32_t total_tokens, int32_t num_chunks,
    const int32_t* sequence_chunk_offsets, const int32_t* chunk_token_starts,
    const int32_t* chunk_token_ends, float* state, const void* r, const void* decay,
    const void* decay_bias, const void* k, const void* v, const void* a, const void* b,
    void* output, float* boundary, float* state_dot_a, float* interior, float scale,
    void* stream) {
  return frwkv_statetune_forward_split(
      io_dtype, decay_mode, num_sequences, num_heads, head_size, total_tokens, num_chunks,
      sequence_chunk_offsets, chunk_token_starts, chunk_token_ends, state, r, decay, decay_bias,
      k, v, a, b, output, boundary, state_dot_a, interior, scale, nullptr, 0, stream);
}

extern "C" int frwkv_statetune_forward_split(
    int io_dtype, int decay_mode, int32_t num_sequences, int32_t num_heads,
    int32_t head_size, int32_t total_tokens, int32_t num_chunks,
    const int32_t* sequence_chunk_offsets, const int32_t* chunk_token_starts,
    const int32_t* chunk_token_ends, float* state, const void* r, const void* decay,
    const void* decay_bias, const void* k, const void* v, const void* a, const void* b,
    void* output, float* boundary, float* state_dot_a, float* interior, float scale,
    void* scratch, size_t scratch_bytes, void* stream) {
  using namespace frwkv;
  if (!sequence_chunk_offsets || !chunk_token_starts || !chunk_token_ends || !state ||
      !boundary || !state_dot_a) {
    return set_error(FRWKV_ERR_INVALID_ARGUMENT,
                     "frwkv_statetune_forward: null pointer argument");
  }
  int rc = check_token_pointers(r, decay, k, v, a, b, output);
  if (rc != FRWKV_OK) return rc;
  if (num_sequences <= 0 || num_heads <= 0 || total_tokens <= 0 || num_chunks <= 0) {
    return set_error(FRWKV_ERR_INVALID_ARGUMENT,
                     "frwkv_statetune_forward: sizes must be positive");
  }
  if (!__builtin_isfinite(scale)) {
    return set_error(FRWKV_ERR_INVALID_ARGUMENT, "scale must be finite");
  }
  if (head_size == 256 && decay_mode == FRWKV_DECAY_LOGITS && scratch != nullptr &&
      (io_dtype == FRWKV_DTYPE_BF16 || io_dtype == FRWKV_DTYPE_F16) &&
      scratch_bytes >= piece32_forward_bytes(head_size, num_heads, total_tokens, num_chunks)) {
    Piece32Params q{};
    q.num_heads = num_heads;
    q.num_sequences = num_sequences;
    q.total_tokens = total_tokens;
    q.seg_offsets = sequence_chunk_offsets;
    q.seg_starts = chunk_token_starts;
    q.seg_ends = chunk_token_ends;
    q.num_segments = num_chunks;
    q.state = state;
    q.state_slots = num_sequences;
    q.r = r;
    q.decay = decay;
    q.bias = decay_bias;
    q.k = k;
    q.v = v;
    q.a = a;
    q.b = b;
    q.out = output;
    q.boundary = boundary;
    q.interior = interior;
    q.state_dot_a = state_dot_a;
    q.scale = scale;
    return piece32_forward(q, head_size, io_dtype, scratch, static_cast<hipStream_t>(stream));
  }
  if (head_size == 128 || head_size == 256) {
    return frwkv_train_recurrent_forward(io_dtype, decay_mode, num_sequences, num_heads,
                                         head_size, total_tokens, sequence_chunk_offsets,
                                         chunk_token_starts, chunk_token_ends, num_chunks,
                                         /*dense_t=*/0,
                                         state, r, decay, decay_bias, k, v, a, b, output,
                                         boundary, state_dot_a, interior, /*fill_only=*/0,
                                         scale, stream);
  }
  if (head_size != 64) {
    return set_error(FRWKV_ERR_UNSUPPORTED, "head size must be 64, 128, or 256, got %d",
                     head_size);
  }
  ChunkFwdParams p{};
  p.num_heads = num_heads;
  p.total_tokens = total_tokens;
  p.state_slots = num_sequences;
  p.seg_offsets = sequence_chunk_offsets;
  p.seg_starts = chunk_token_starts;
  p.seg_ends = chunk_token_ends;
  p.num_segments = num_chunks;
  p.state = state;
  p.r = r;
  p.decay = decay;
  p.bias = decay_bias;
  p.k = k;
  p.v = v;
  p.a = a;
  p.b = b;
  p.out = output;
  p.boundary = boundary;
  p.state_dot_a = state_dot_a;
  p.interior = interior;
  p.scale = scale;
  p.out_elems = static_cast<int64_t>(total_tokens) * num_heads * head_size;
  use_unit_parts(p, static_cast<int64_t>(num_sequences) * num_heads,
                 plan_caller_chunks(num_sequences, num_heads, num_chunks), scratch,
                 scratch_bytes);
  return dispatch_chunk_io<float>(p, io_dtype, decay_mode, num_sequences * num_heads,
                                  static_cast<hipStream_t>(stream));
}

extern "C" size_t frwkv_statetune_interior_bytes(int32_t head_size, int32_t num_heads,
                                                 int32_t total_tokens) {
  if (num_heads <= 0 || total_tokens <= 0) return 0;
  const int64_t piece = head_size == 64 ? 64 : 16;
  const int64_t slots = (total_tokens + piece - 1) / piece;
  // Head size 128 keeps the states in bf16 (the piece kernels' own order).
  const int64_t bytes = head_size == 128 ? 2 : 4;
  return static_cast<size_t>(slots * num_heads * head_size * head_size * bytes);
}

extern "C" int frwkv_statetune_interior(int io_dtype, int decay_mode, int32_t num_heads,
                                        int32_t head_size, int32_t total_tokens,
                                        int32_t num_chunks, const int32_t* chunk_token_starts,
                                        const int32_t* chunk_token_ends, const float* boundary,
                                        const void* r, const void* decay, const void* decay_bias,
                                        const void* k, const void* v, const void* a,
                                        const void* b, float* interior, void* stream) {
  using namespace frwkv;
  if (!chunk_token_starts || !chunk_token_ends || !boundary || !interior || !r || !decay ||
      !k || !v || !a || !b) {
    return set_error(FRWKV_ERR_INVALID_ARGUMENT, "frwkv_statetune_interior: null pointer argument");
  }
  if (num_chunks <= 0 || num_heads <= 0 || total_tokens <= 0) {
    return set_error(FRWKV_ERR_INVALID_ARGUMENT,
                     "frwkv_statetune_interior: sizes must be positive");
  }
  if (head_size == 128 || head_size == 256) {
    return frwkv_train_recurrent_forward(io_dtype, decay_mode, num_chunks, num_heads, head_size,
                                         total_tokens, nullptr, chunk_token_starts,
                                         chunk_token_ends, num_chunks, /*dense_t=*/0,
                                         const_cast<float*>(boundary), r, decay, decay_bias, k,
                                         v, a, b, nullptr, nullptr, nullptr, interior,
                                         /*fill_only=*/1, 1.0f, stream);
  }
  if (head_size != 64) {
    return set_error(FRWKV_ERR_UNSUPPORTED, "head size must be 64, 128, or 256, got %d",
                     head_size);
  }
  ChunkFwdParams p{};
  p.num_heads = num_heads;
  p.total_tokens = total_tokens;
  p.state_slots = num_chunks;
  p.seg_starts = chunk_token_starts;
  p.seg_ends = chunk_token_ends;
  p.num_segments = num_chunks;
  p.state = const_cast<float*>(boundary);
  p.read_only_state = 1;
  p.r = r;
  p.decay = decay;
  p.bias = decay_bias;
  p.k = k;
  p.v = v;
  p.a = a;
  p.b = b;
  p.interior = interior;
  p.fill_only = 1;
  p.scale = 1.0f;
  return dispatch_chunk_io<float>(p, io_dtype, decay_mode, num_chunks * num_heads,
                                  static_cast<hipStream_t>(stream));
}

extern "C" int frwkv_pretrain_forward(int io_dtype, int decay_mode, int32_t batch,
                                      int32_t tokens, int32_t num_heads, int32_t head_size,
                                      const void* r, const void* decay, const void* k,
                                      const void* v, const void* a, const void* b,
                                      void* output, float* boundary, float* state_dot_a,
                                      void* stream) {
  return frwkv_pretrain_forward_split(io_dtype, decay_mode, batch, tokens, num_heads, head_size,
                                      r, decay, k, v, a, b, output, boundary, state_dot_a,
                                      nullptr, 0, stream);
}

extern "C" int frwkv_pretrain_forward_split(
    int io_dtype, int decay_mode, int32_t batch, int32_t tokens, int32_t num_heads,
    int32_t head_size, const void* r, const void* decay, const void* k, const void* v,
    const void* a, const void* b, void* output, float* boundary, float* state_dot_a,
    void* scratch, size_t scratch_bytes, void* stream) {
  using namespace frwkv;
  if (!boundary || !state_dot_a) {
    return set_error(FRWKV_ERR_INVALID_ARGUMENT, "frwkv_pretrain_forward: null pointer argument");
  }
  int rc = check_token_pointers(r, decay, k, v, a, b, output);
  if (rc != FRWKV_OK) return rc;
  if (batch <= 0 || tokens <= 0 || num_heads <= 0 || tokens % 16 != 0) {
    return set_error(FRWKV_ERR_INVALID_ARGUMENT,
                     "frwkv_pretrain_forward: B, H > 0 and T a positive multiple of 16 "
                     "(B=%d, T=%d, H=%d)", batch, tokens, num_heads);
  }
  if (static_cast<int64_t>(batch) * tokens > INT32_MAX) {
    return set_error(FRWKV_ERR_INVALID_ARGUMENT, "frwkv_pretrain_forward: B * T too large");
  }
  if (head_size == 256 && decay_mode == FRWKV_DECAY_LOGITS && scratch != nullptr &&
      (io_dtype == FRWKV_DTYPE_BF16 || io_dtype == FRWKV_DTYPE_F16) &&
      scratch_bytes >= piece32_forward_bytes(head_size, num_heads, batch * tokens, batch)) {
    Piece32Params q{};
    q.num_heads = num_heads;
    q.num_sequences = batch;
    q.total_tokens = batch * tokens;
    q.dense_t = tokens;
    q.r = r;
    q.decay = decay;
    q.k = k;
    q.v = v;
    q.a = a;
    q.b = b;
    q.out = output;
    q.boundary = boundary;
    q.state_dot_a = state_dot_a;
    q.scale = 1.0f;
    return piece32_forward(q, head_size, io_dtype, scratch, static_cast<hipStream_t>(stream));
  }
  if (head_size == 128 || head_size == 256) {
    return frwkv_train_recurrent_forward(io_dtype, decay_mode, batch, num_heads, head_size,
                                         batch * tokens, nullptr, nullptr, nullptr, 0, tokens,
                                         /*state=*/nullptr, r, decay, /*decay_bias=*/nullptr, k,
                                         v, a, b, output, boundary, state_dot_a,
                                         /*interior=*/nullptr, /*fill_only=*/0, 1.0f, stream);
  }
  if (head_size != 64) {
    return set_error(FRWKV_ERR_UNSUPPORTED, "head size must be 64, 128, or 256, got %d",
                     head_size);
  }
  ChunkFwdParams p{};
  p.num_heads = num_heads;
  p.total_tokens = batch * tokens;
  p.state_slots = batch;
  p.dense_t = tokens;
  p.boundary16 = 1;
  p.r = r;
  p.decay = decay;
  p.k = k;
  p.v = v;
  p.a = a;
  p.b = b;
  p.out = output;
  p.boundary = boundary;
  p.state_dot_a = state_dot_a;
  p.scale = 1.0f;
  p.out_elems = static_cast<int64_t>(batch) * tokens * num_heads * head_size;
  use_unit_parts(p, static_cast<int64_t>(batch) * num_heads,
                 plan_packed_parts(batch, num_heads, p.total_tokens, tokens, kForwardTime,
                                   kTransferTime),
                 scratch, scratch_bytes);
  return dispatch_chunk_io<float>(p, io_dtype, decay_mode, batch * num_heads,
                                  static_cast<hipStream_t>(stream));
}

extern "C" int frwkv_chunk_replay(int io_dtype, int decay_mode, int32_t num_chunks,
                                  int32_t num_heads, int32_t head_size, int32_t total_tokens,
                                  const int32_t* chunk_token_starts,
                                  const int32_t* chunk_token_ends, const float* boundary,
                                  const void* r, const void* decay, const void* decay_bias,
                                  const void* k, const void* v, const void* a, const void* b,
                                  void* output, float* state_dot_a, float scale,
                                  void* stream) {
  using namespace frwkv;
  if (!chunk_token_starts || !chunk_token_ends || !boundary || !state_dot_a) {
    return set_error(FRWKV_ERR_INVALID_ARGUMENT, "frwkv_chunk_replay: null pointer argument");
  }
  int rc = check_token_pointers(r, decay, k, v, a, b, output);
  if (rc != FRWKV_OK) return rc;
  if (num_chunks <= 0 || num_heads <= 0 || total_tokens <= 0) {
    return set_error(FRWKV_ERR_INVALID_ARGUMENT, "frwkv_chunk_replay: sizes must be positive");
  }
  if (!__builtin_isfinite(scale)) {
    return set_error(FRWKV_ERR_INVALID_ARGUMENT, "scale must be finite");
  }
  if (head_size != 64) {
    // Other head sizes: the fp32 per-token kernel, one unit per chunk.
    return frwkv_replay_recurrent(io_dtype, decay_mode, num_chunks, num_heads, head_size,
                                  total_tokens, chunk_token_starts, chunk_token_ends,
                                  boundary, r, decay, decay_bias, k, v, a, b, output,
                                  state_dot_a, scale, stream);
  }
  ChunkFwdParams p{};
  p.num_heads = num_heads;
  p.total_tokens = total_tokens;
  p.state_slots = num_chunks;
  p.seg_starts = chunk_token_starts;
  p.seg_ends = chunk_token_ends;
  p.num_segments = num_chunks;
  p.state = const_cast<float*>(boundary);
  p.read_only_state = 1;
  p.r = r;
  p.decay = decay;
  p.bias = decay_bias;
  p.k = k;
  p.v = v;
  p.a = a;
  p.b = b;
  p.out = output;
  p.state_dot_a = state_dot_a;
  p.scale = scale;
  p.out_elems = static_cast<int64_t>(total_tokens) * num_heads * head_size;
  return dispatch_chunk_io<float>(p, io_dtype, decay_mode, num_chunks * num_heads,
                                  static_cast<hipStream_t>(stream));
}
