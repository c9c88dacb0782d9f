// prefill.hip - the attention of a prompt's tokens (many consecutive positions of one sequence)
// on the fp32 matrix cores: every K/V row of the chunk is written first (attention.c:292-309),
// then each token attends to the cache up to its own position (attention.c:93-163).
//
// v_mfma_f32_16x16x4_f32 multiplies fp32 operands as they are, so q, K, V, the weights and every
// sum stay fp32. A row of the tiles is one (token, query head) pair of a K/V head: G heads share
// it, so 16 rows are 16 / G tokens. Scores are formed transposed, S^T = K q^T, which leaves each
// lane one row's scores of four positions: exactly the B operand of O^T = V^T P^T, so the
// weights go from one product to the next without leaving their registers.
#include "decode_device.h"
#include "gemm_wide.h"
#include "prefill.h"

namespace sapphire {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
constexpr int kRows = 16;                  // (token, head) rows of a workgroup
constexpr int kWaves = kThreads / kWave;
constexpr int kPos = 16;                   // positions of a tile

// grid (tokens): q rows with QK-norm and RoPE, and the K/V rows of the cache (the K rows by
// norm_rope_heads, as every other writer of them, so bit-identical).
__global__ __launch_bounds__(kThreads) void prefill_qkv_kernel(PrefillAttn a, float *__restrict__ q_out) {
    __shared__ float raw[kAttnMaxQ + kAttnMaxKV];
    __shared__ float rot[kAttnMaxQ + kAttnMaxKV];
    __shared__ float part8[8 * 16];
    __shared__ float ss[16];
    const int t = blockIdx.x, pos = a.pos0 + t, hd = a.hd, nq = a.nh * hd, nk = a.nkv * hd;
    const float *src = a.qkv + (size_t)t * (nq + 2 * nk);
    const float *cs = a.cos_t + (size_t)pos * hd, *sn = a.sin_t + (size_t)pos * hd;
    for (int i = threadIdx.x; i < (nq + nk) / 4; i += kThreads)
        reinterpret_cast<float4 *>(raw)[i] = reinterpret_cast<const float4 *>(src)[i];
    for (int i = threadIdx.x; i < nk / 4; i += kThreads) {
        const int h = i * 4 / hd, d = i * 4 - h * hd;
        *reinterpret_cast<float4 *>(a.vc + ((size_t)h * a.max_ctx + pos) * hd + d) =
            reinterpret_cast<const float4 *>(src + nq + nk)[i];
    }
    __syncthreads();
    norm_rope_heads(raw, a.nh, hd, a.qn, cs, sn, a.eps, rot, part8, ss);
    norm_rope_heads(raw + nq, a.nkv, hd, a.kn, cs, sn, a.eps, rot + nq, part8, ss);
    for (int i = threadIdx.x; i < nq / 4; i += kThreads)
        reinterpret_cast<float4 *>(q_out + (size_t)t * nq)[i] = reinterpret_cast<const float4 *>(rot)[i];
    for (int i = threadIdx.x; i < nk / 4; i += kThreads) {
        const int h = i * 4 / hd, d = i * 4 - h * hd;
        *reinterpret_cast<float4 *>(a.kc + ((size_t)h * a.max_ctx + pos) * hd + d) =
            reinterpret_cast<const float4 *>(rot + nq)[i];
    }
}

// grid (row tiles, K/V heads, pieces): rows [16 x, 16 x + 16) of K/V head y over piece z of
// their positions. The four waves take the piece's 16-position tiles in turn, each with a running
// (max, sum, O) per row, merged at the end; the partial goes to a.part (O, unnormalised) and
// a.ms (max in log2 units, sum). A piece without positions of its rows leaves (-inf, 0).
// Two register buffers of half a tile's K or V rows each are refilled as soon as they are used (K
// low half, K high half, V of two positions per lane, V of the other two), so that with O a wave of
// head_dim 256 stays under 256 registers and two waves share a SIMD. (Whole tiles of K and V took
// 512, the moves between their two halves costing as much as the products: 48 us per layer of 1000
// tokens, now 36.)
template <int DPL, int G>
__global__ __launch_bounds__(kThreads, 2) void prefill_attn_kernel(PrefillAttn a, const float *__restrict__ q_rows) {
    constexpr int HD = kWave * DPL, NJ = HD / 16, TOK = kRows / G, LD = HD + 4;
    __shared__ __attribute__((aligned(16))) float buf[kWaves * kRows * LD];   // q, later the waves' O
    __shared__ float wm[kWaves][kRows], wsum[kWaves][kRows];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wid = tid / kWave;
    const int c = lane & 15, m = lane >> 4, hk = blockIdx.y;
    // later tokens attend to more positions: they go first
    const int tile = gridDim.x - 1 - blockIdx.x, t0 = tile * TOK;
    const int tl = min(t0 + TOK, a.T) - 1;             // last token of the tile
    const int nq = a.nh * HD;
    auto start_of = [&](int pos) { return a.window > 0 && pos + 1 > a.window ? pos + 1 - a.window : 0; };
    const int lo = start_of(a.pos0 + t0) + blockIdx.z * a.piece;
    const int hi = min(a.pos0 + tl + 1, lo + a.piece);
    // this lane's row: token, head, positions [r_lo, r_hi)
    const int tok = t0 + c / G, head = hk * G + c % G;
    const bool row_on = tok < a.T;
    const int rpos = a.pos0 + min(tok, tl);
    const int r_lo = max(lo, start_of(rpos)), r_hi = min(hi, rpos + 1);
    const size_t slot = (size_t)blockIdx.z * a.T * a.nh + (size_t)tok * a.nh + head;
    if (lo >= hi) {
        if (wid == 0 && m == 0 && row_on) a.ms[slot] = make_float2(-INFINITY, 0.f);
        return;
    }
    // q of the 16 rows into LDS (rows past the chunk repeat its last token)
    for (int i = tid; i < kRows * HD / 4; i += kThreads) {
        const int r = i / (HD / 4), d = i % (HD / 4) * 4;
        *reinterpret_cast<float4 *>(buf + r * LD + d) = *reinterpret_cast<const float4 *>(
            q_rows + (size_t)min(t0 + r / G, tl) * nq + (hk * G + r % G) * HD + d);
    }
    const float *kc = a.kc + (size_t)hk * a.max_ctx * HD, *vc = a.vc + (size_t)hk * a.max_ctx * HD;
    constexpr int HALF = NJ / 2;
    static_assert(HALF == 2 * DPL, "half a tile's K rows and half its V rows are the same size");
    f4 bufs[2][HALF];
    // K of position tb + c, dims 16 j + 4 m .. + 3 for j in half h; positions past the piece repeat
    // its last one (masked)
    auto load_k = [&](int tb, int h) {
        const float *p = kc + (size_t)min(tb + c, hi - 1) * HD + 4 * m + 16 * HALF * h;
#pragma unroll
        for (int j = 0; j < HALF; ++j) bufs[h][j] = *reinterpret_cast<const f4 *>(p + 16 * j);
    };
    // V of positions tb + 4 m + r, r = 2 h and 2 h + 1, dims 64 q + 4 c .. + 3
    auto load_v = [&](int tb, int h) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const float *p = vc + (size_t)min(tb + 4 * m + 2 * h + r, hi - 1) * HD + 4 * c;
#pragma unroll
            for (int q = 0; q < DPL; ++q) bufs[h][r * DPL + q] = *reinterpret_cast<const f4 *>(p + 64 * q);
        }
    };
    f4 o[DPL][4];                                      // o[q][e][r']: dim 64 q + 16 m + 4 r' + e of row c
#pragma unroll
    for (int q = 0; q < DPL; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[q][e] = f4{0.f, 0.f, 0.f, 0.f};
    float mx = -INFINITY, sum = 0.f;                   // sum: this lane's positions only
    const float sl2 = __fmul_rn(a.scale, 1.44269504088896341f);
    int tb = lo + wid * kPos;
    if (tb < hi) {
        load_k(tb, 0);
        load_k(tb, 1);
    }
    __syncthreads();
    for (; tb < hi; tb += kWaves * kPos) {
        // a score is the sum of short chains (the weight's relative error is its absolute one)
        constexpr int CH = HALF < 4 ? HALF : 4;
        f4 st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int j0 = 0; j0 < HALF; j0 += CH) {
                f4 s4[4] = {};
#pragma unroll
                for (int j = j0; j < j0 + CH; ++j) {
                    const f4 qv = *reinterpret_cast<const f4 *>(buf + c * LD + 16 * (HALF * h + j) + 4 * m);
#pragma unroll
                    for (int e = 0; e < 4; ++e) s4[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(bufs[h][j][e], qv[e], s4[e], 0, 0, 0);
                }
                st += (s4[0] + s4[1]) + (s4[2] + s4[3]);
            }
            load_v(tb, h);
        }
        float sc[4], mt = -INFINITY;
        bool on[4], edge = false;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = tb + 4 * m + r;
            on[r] = t >= r_lo && t < r_hi;
            edge |= !on[r];
            sc[r] = on[r] ? __fmul_rn(st[r], sl2) : -INFINITY;
            mt = fmaxf(mt, sc[r]);
        }
        mt = fmaxf(mt, __shfl_xor(mt, 16, kWave));
        mt = fmaxf(mt, __shfl_xor(mt, 32, kWave));
        const float mn = fmaxf(mx, mt);
        const float f = mx == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mx - mn);
        float p[4];
        sum = __fmul_rn(sum, f);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            // masked, or a score of -inf (also where every score so far is, mn included)
            p[r] = sc[r] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(sc[r] - mn);
            sum = __fadd_rn(sum, p[r]);
        }
        mx = mn;
        if (__any(f != 1.0f))
#pragma unroll
            for (int q = 0; q < DPL; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) o[q][e] *= f;
        // A masked position's weight is 0, and 0 times a NaN or infinite V is NaN: a tile that
        // has both takes its positions one by one and leaves the masked ones out (rare).
        bool slow = false;
        if (__any(edge)) {
            uint32_t ex = 0;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < HALF; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) ex = max(ex, __float_as_uint(bufs[h][j][e]) & 0x7f800000u);
            slow = __any(ex == 0x7f800000u) != 0;
        }
        const int tn = tb + kWaves * kPos;
        if (slow) {
            for (int k = 0; k < kPos; ++k) {
                const int t = tb + k;
                const float pk = k & 2 ? (k & 1 ? p[3] : p[2]) : (k & 1 ? p[1] : p[0]);
                const float w = __shfl(pk, (k >> 2) * 16 + c, kWave);
                if (t < r_lo || t >= r_hi) continue;
                const float *v = vc + (size_t)t * HD + 16 * m;
#pragma unroll
                for (int q = 0; q < DPL; ++q)
#pragma unroll
                    for (int r2 = 0; r2 < 4; ++r2)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            o[q][e][r2] = __builtin_fmaf(w, v[64 * q + 4 * r2 + e], o[q][e][r2]);
            }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (!slow)
#pragma unroll
                for (int r = 0; r < 2; ++r)
#pragma unroll
                    for (int q = 0; q < DPL; ++q)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            o[q][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(bufs[h][r * DPL + q][e], p[2 * h + r], o[q][e], 0, 0, 0);
            load_k(tn, h);                             // past the end: the last row again
        }
    }
    sum += __shfl_xor(sum, 16, kWave);
    sum += __shfl_xor(sum, 32, kWave);
    if (m == 0) {
        wm[wid][c] = mx;
        wsum[wid][c] = sum;
    }
    __syncthreads();                                   // every wave is past its reads of q
    float top = wm[0][c];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) top = fmaxf(top, wm[w][c]);
    // a wave without positions of the row, or with scores of -inf only, has sum 0 and O 0; its
    // factor must not be NaN
    const float fw = sum == 0.f ? 0.f : __builtin_amdgcn_exp2f(mx - top);
    float *mine = buf + (size_t)(wid * kRows + c) * LD + 16 * m;
#pragma unroll
    for (int q = 0; q < DPL; ++q)
#pragma unroll
        for (int r2 = 0; r2 < 4; ++r2)
#pragma unroll
            for (int e = 0; e < 4; ++e) mine[64 * q + 4 * r2 + e] = sum == 0.f ? 0.f : __fmul_rn(o[q][e][r2], fw);
    __syncthreads();
    for (int i = tid; i < kRows * HD / 4; i += kThreads) {
        const int r = i / (HD / 4), d = i % (HD / 4) * 4;
        if (t0 + r / G > tl) continue;
        f4 v = *reinterpret_cast<const f4 *>(buf + r * LD + d);
#pragma unroll
        for (int w = 1; w < kWaves; ++w) v += *reinterpret_cast<const f4 *>(buf + (w * kRows + r) * LD + d);
        const size_t sl = (size_t)blockIdx.z * a.T * a.nh + (size_t)(t0 + r / G) * a.nh + hk * G + r % G;
        *reinterpret_cast<f4 *>(a.part + sl * HD + d) = v;
    }
    if (wid == 0 && m == 0 && row_on) {
        float tot = 0.f;
        for (int w = 0; w < kWaves; ++w)
            if (wsum[w][c] != 0.f) tot += __fmul_rn(wsum[w][c], __builtin_amdgcn_exp2f(wm[w][c] - top));
        a.ms[slot] = make_float2(top, tot);
    }
}

int cu_count() {
    int dev = 0, c = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || c <= 0)
        return 256;
    return c;
}

}  // namespace

bool prefill_attn_supported(int nh, int nkv, int hd) {
    const int g = nkv > 0 ? nh / nkv : 0;
    return nkv > 0 && nkv <= 2 && nh % nkv == 0 && (g == 2 || g == 4 || g == 8) && (hd == 64 || hd == 128 || hd == 256) &&
           nh * hd <= kAttnMaxQ && nkv * hd <= kAttnMaxKV && nh + nkv <= 16;
}

int launch_prefill_attention(PrefillAttn a, float *q_rows, int *pieces, hipStream_t s) {
    if (!prefill_attn_supported(a.nh, a.nkv, a.hd) || a.T <= 0 || a.pos0 < 0 || a.pos0 + a.T > a.max_ctx) {
        set_error("prefill attention: unsupported shape (heads %d/%d, head_dim %d, %d tokens)", a.nh, a.nkv, a.hd, a.T);
        return -1;
    }
    hipLaunchKernelGGL(prefill_qkv_kernel, dim3(a.T), dim3(kThreads), 0, s, a, q_rows);
    if (!hip_ok(hipGetLastError(), "prefill qkv launch")) return -1;
    if (!a.part) {                                     // only the rows of the cache are wanted
        *pieces = 0;
        return 0;
    }
    // Positions are cut into pieces while the workgroups number fewer than four per CU (the
    // rows of late tokens attend to many more positions than those of early ones), pieces of at
    // least one tile per wave.
    const int g = a.nh / a.nkv, tok = kRows / g, tiles = (a.T + tok - 1) / tok;
    int len = a.pos0 + a.T;
    if (a.window > 0) len = std::min(len, a.window + tok);
    const int want = std::max(1, std::min(kPrefillPieces, (4 * cu_count() + tiles * a.nkv - 1) / (tiles * a.nkv)));
    const int unit = kWaves * kPos;
    a.piece = std::max(unit, ((len + want - 1) / want + unit - 1) / unit * unit);
    *pieces = (len + a.piece - 1) / a.piece;
    const dim3 grid(tiles, a.nkv, *pieces), block(kThreads);
#define SPH_PA(DPLV, GV) \
    if (a.hd == kWave * DPLV && g == GV) hipLaunchKernelGGL((prefill_attn_kernel<DPLV, GV>), grid, block, 0, s, a, q_rows); else
    SPH_PA(1, 2) SPH_PA(1, 4) SPH_PA(1, 8) SPH_PA(2, 2) SPH_PA(2, 4) SPH_PA(2, 8) SPH_PA(4, 2) SPH_PA(4, 4) SPH_PA(4, 8) {
        set_error("prefill attention: not instantiated");
        return -1;
    }
#undef SPH_PA
    return hip_ok(hipGetLastError(), "prefill attention launch") ? 0 : -1;
}

}  // namespace sapphire
