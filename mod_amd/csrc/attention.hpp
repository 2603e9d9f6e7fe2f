// Dense attention over fp32 queries and fp32 or fp16 keys / values
// (attention.hip), shared by the drop-in op (model_ops.hip) and the batched
// prompt (prefill.hip).
#pragma once

#include "pio_common.hpp"

namespace pio {

struct AttnArgs {
    const float* q;       // row (b, s): q + b * q_b + s * q_s, head h at h * D
    const void* k;        // row (b, t) of kv head g: k + b * kv_b + t * kv_t + g * kv_h (elements)
    const void* v;        // as k
    float* out;           // row (b, s): out + b * o_b + s * o_s, head h at h * D (may be q itself)
    int8_t* planes;       // causal: instead of out, the planes of row s (wf_planes.hpp, K = H * D)
    int64_t q_b, o_b, kv_b;
    int q_s, o_s, kv_t;
    int64_t kv_h;
    int B, S, T, H, Hk, D;
    float scale;
    bool causal;          // query s sees keys 0 .. pos0 + s (T = pos0 + S), else all T
    int pos0;
    bool kv16;            // fp16 keys / values in the decoder's paired slots (D = 128)
    float m_seed;         // the running maximum starts here
};

// Whether attn_mfma takes these shapes and addresses (else: the caller's own
// kernel, or attn_mfma's error).
bool attn_mfma_supported(const AttnArgs& a);
int attn_mfma(const AttnArgs& a, hipStream_t st);

}  // namespace pio
