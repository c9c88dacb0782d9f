// prefill.h - launcher of the prompt attention (prefill.hip). Not installed.
#pragma once

#include "internal.h"

namespace sapphire {

constexpr int kPrefillPieces = 8;          // partials per (token, head) at most

// T tokens at positions pos0 .. pos0 + T - 1 of one sequence.
struct PrefillAttn {
    const float *qkv = nullptr;            // [T][nh*hd | nkv*hd | nkv*hd] as projected, 16-byte aligned
    const float *qn = nullptr, *kn = nullptr;
    const float *cos_t = nullptr, *sin_t = nullptr;
    float *kc = nullptr, *vc = nullptr;    // this layer's caches [nkv][max_ctx][hd]
    int T = 0, pos0 = 0, nh = 0, nkv = 0, hd = 0, max_ctx = 0, window = 0;
    float scale = 1.f, eps = 1e-6f;
    float *part = nullptr;                 // [pieces][T][nh][hd] (NULL: only the K/V rows are written)
    float2 *ms = nullptr;                  // [pieces][T][nh]
    int piece = 0;                         // set by the launch: positions per piece
};
bool prefill_attn_supported(int nh, int nkv, int hd);
// QK-norm, RoPE, the K/V rows, then the attention partials in *pieces pieces (the o
// projection's input pass merges them: launch_gemm_wide_prep_attn). q_rows: [T][nh*hd] scratch.
int launch_prefill_attention(PrefillAttn a, float *q_rows, int *pieces, hipStream_t s);

}  // namespace sapphire
