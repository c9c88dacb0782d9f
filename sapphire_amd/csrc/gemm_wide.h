// gemm_wide.h - launchers of the many-token quantized GEMM (gemm_wide.hip). Not installed.
#pragma once

#include "internal.h"

namespace sapphire {

constexpr int kWideBm = 32;       // tokens of a workgroup tile (operands are padded to it)
constexpr int kWideMaxK = 8192;
constexpr int kWideMaxSplit = 8;     // K splits at most

bool gemm_wide_supported(int K);
// Bytes of the prepared operands of T tokens (256-byte aligned device memory).
size_t gemm_wide_operand_bytes(int T, int K);
// K splits a launch with out.parts takes: parts holds splits * T * M floats.
int gemm_wide_splits(int dt, int M, int K, int T);
// Weight rows of its workgroups' tile.
int gemm_wide_tile_rows(int dt, int M, int K, int T);
// Bytes of the partial sums at most.
size_t gemm_wide_parts_bytes(int M, int T);
// The operands of T tokens from `in` (GemmIn's transform, sums of squares as trees).
int launch_gemm_wide_prep(int dt, const GemmIn &in, int K, int T, void *operand, hipStream_t s);

// The same from the attention's partials (prefill.h), K = nh * hd.
int launch_gemm_wide_prep_attn(int dt, const float *part, const void *ms, int pieces, int nh, int hd, int T,
                               void *operand, hipStream_t s);

// y[t * ldy + r], or with geglu y[t * ldy + j] = gelu(gate_j) * up_j of rows interleaved by
// eight; parts set: the K splits' partial sums [split][T][M] instead (gemm_wide_splits of them).
struct WideOut {
    float *y = nullptr;
    int ldy = 0;
    bool geglu = false;
    float *parts = nullptr;
};
int launch_gemm_wide(int dt, const void *w_tiled, int M, int K, int T, const void *operand, const WideOut &out,
                     hipStream_t s);

}  // namespace sapphire
