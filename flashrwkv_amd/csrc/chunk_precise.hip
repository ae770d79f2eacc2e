// The split-precision instantiations of the chunked forward kernel
// (chunk_fwd_kernel.h): the recurrent operator's route for long sequences. A
// file of their own because they want another scheduler than the others (see
// _build.py).
#include "chunk_fwd_kernel.h"

// The recurrent operator's route for long sequences (called by
// frwkv_recurrent_forward): bf16 tokens, head size 64, fp32 pool, the
// split-precision variant of the chunk kernel. Arguments as there; the
// caller has checked pointers and sizes.
int frwkv_recurrent_chunked_forward(int decay_mode, int32_t num_sequences, int32_t num_heads,
                                    int32_t total_tokens, int32_t state_pool_size,
                                    const int32_t* cu_seqlens, const int32_t* state_indices,
                                    const int32_t* metadata_status, float* state_pool,
                                    const void* r, const void* decay, const void* decay_bias,
                                    const void* k, const void* v, const void* a, const void* b,
                                    void* output, float scale, int32_t max_seqlen, void* scratch,
                                    size_t scratch_bytes, void* stream) {
  using namespace frwkv;
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
  p.out_elems = static_cast<int64_t>(total_tokens) * num_heads * kHead;
  const int units = num_sequences * num_heads;
  use_packed_parts(p, num_sequences,
                   plan_packed_parts(num_sequences, num_heads, total_tokens, max_seqlen,
                                     kPreciseTime, kTransferTime),
                   scratch, scratch_bytes);
  auto s = static_cast<hipStream_t>(stream);
  if (decay_mode == FRWKV_DECAY_LOGITS) {
    return launch_chunk<Bf16, DecayMode::kLogits, float, true>(p, units, s);
  }
  if (decay_mode == FRWKV_DECAY_RAW_W) {
    if (decay_bias != nullptr) {
      return set_error(FRWKV_ERR_INVALID_ARGUMENT,
                       "decay_bias is only defined for the logits decay mode");
    }
    return launch_chunk<Bf16, DecayMode::kRawW, float, true>(p, units, s);
  }
  return set_error(FRWKV_ERR_INVALID_ARGUMENT, "unknown decay mode %d", decay_mode);
}
