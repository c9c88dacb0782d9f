// gemm_wide.hip - Q4_0 / Q8_0 weights (TILED) times many activation vectors (a prompt's tokens)
// on the CDNA4 matrix cores: Y[t][r] = sum_k W[r][k] X[t][k] for t < T. The operands are those
// of the 16-sequence GEMM (gemm_mfma.hip): the integer weights exactly in fp16, each activation
// as fp16 hi + lo terms under one power-of-two range scale per token and 32 blocks, v_mfma_f32_16x16x32_f16
// per 32-weight block and term, the block's weight scale by one fp32 FMA per value.
//
// Two launches: gemm_wide_prep_kernel forms the A operands of every token once, in the order
// in which the matrix cores read them (2 KiB per 16 tokens and block: hi, lo); gemm_wide_kernel
// brings them into LDS by DMA (no registers; three stages of four blocks, two for the larger stages
// of Q4_0's 256-row and Q8_0's 128-row tile) and every workgroup
// multiplies BM tokens by BN weight rows, so that a weight is read and expanded once per BM
// tokens instead of once per 16. Q4_0 6912 x 1152 x 300: 166 us in passes of 16 (19 of them,
// each reading all the weights and bound by its staging and latency) -> 29 us.
#include "gemm_body.h"
#include "gemm_wide.h"
#include "prefill.h"

namespace sapphire {

namespace {

using namespace gemmb;

constexpr int kThreads = 256, kWavesWg = kThreads / kWave;
constexpr int kXcds = 8;

// The operand buffer of T tokens and K activations: [T / 16 tiles][K / 32 blocks][hi, lo][64]
// h8, then the range scales [chunk of 32 blocks][token], and per token the flags (1: a NaN or infinity, 2: a NaN) and, for a
// flagged token only, [2][K / 32] masks of its +inf and -inf elements. Tokens are padded to the
// widest workgroup tile: the padding is read and multiplied, never stored.
constexpr int kChunk = 32;
__host__ __device__ constexpr int chunks_of(int K) { return (K + kChunk * kBlock - 1) / (kChunk * kBlock); }
struct Operand {
    h8 *a;
    float *xsc;
    int tokens;                    // padded: the stride of the chunks' scales
    int *flag;
    uint32_t *inf;
};
int padded(int T) { return (T + kWideBm - 1) / kWideBm * kWideBm; }
Operand operand_at(void *buf, int T, int K) {
    const size_t p = (size_t)padded(T);
    Operand o;
    o.a = static_cast<h8 *>(buf);
    o.xsc = reinterpret_cast<float *>(static_cast<char *>(buf) + p * K * 4);
    o.tokens = (int)p;
    o.flag = reinterpret_cast<int *>(o.xsc + p * chunks_of(K));
    o.inf = reinterpret_cast<uint32_t *>(o.flag + p);
    return o;
}

struct AttnParts {
    const float *part;             // [pieces][T][nh][hd], unnormalised
    const float2 *ms;              // [pieces][T][nh]: maximum (log2 units), sum
    int pieces, hd;
};

// grid (tokens): token t's input transform (GemmIn's: sum of parts, rmsnorm_delta, residual,
// pre-norm; sums of squares as trees), the range scale over the finite values, the non-finite
// record and the hi / lo split. Thread p takes the pairs p + 256 i (8 activations each).
// ATTN: the input is the merge of the attention's partials instead (nh = K / hd heads).
template <int DT, int NP, bool ATTN = false>
__global__ __launch_bounds__(kThreads) void gemm_wide_prep_kernel(GemmIn in, int K, Operand op, AttnParts at = {}) {
    __shared__ float wsq[2][kWavesWg];
    __shared__ float wmx[NP][kWavesWg];
    __shared__ int wfl[kWavesWg];
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & (kWave - 1), wid = tid / kWave;
    const int nb = K / kBlock, pairs = K / 8;
    float v[NP][8], xv[NP][8], wd[NP][8], wn[NP][8];
#pragma unroll
    for (int i = 0; i < NP; ++i) {                     // every independent load goes out first
        const int p = tid + i * kThreads, k = p * 8;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = xv[i][e] = wd[i][e] = wn[i][e] = 0.f;
        if (p < pairs) {
            if (in.x) load8(in.x + (size_t)t * in.ldx + k, in.parts ? xv[i] : v[i]);
            if (in.parts) load8(in.parts + (size_t)t * in.ldp + k, v[i]);
            if (in.w_delta && in.parts) load8(in.w_delta + k, wd[i]);
            if (in.w_norm) load8(in.w_norm + k, wn[i]);
        }
    }
    // 1 / rms of the token's K values: each thread's squares, one wave sum each, then the waves
    // in a fixed order
    auto rms_inv = [&](int slot) {
        float sq = 0.f;
#pragma unroll
        for (int i = 0; i < NP; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) sq = __builtin_fmaf(v[i][e], v[i][e], sq);
        sq = lanes::wave_sum(sq);
        if (lane == 0) wsq[slot][wid] = sq;
        __syncthreads();
        float tot = 0.f;
#pragma unroll
        for (int w = 0; w < kWavesWg; ++w) tot += wsq[slot][w];
        return devmath::rms_inv_of(tot, K, in.eps);
    };
    auto scaled = [&](float r, const float (&w)[NP][8]) {
#pragma unroll
        for (int i = 0; i < NP; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) v[i][e] = __fmul_rn(__fmul_rn(v[i][e], r), __fadd_rn(1.0f, w[i][e]));
    };
    if (in.parts) {
        for (int c = 1; c < in.nparts; ++c)
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                const int p = tid + i * kThreads;
                if (p < pairs) {
                    float q[8];
                    load8(in.parts + c * in.part_stride + (size_t)t * in.ldp + p * 8, q);
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[i][e] = __fadd_rn(v[i][e], q[e]);
                }
            }
        if (in.w_delta) scaled(rms_inv(0), wd);
        if (in.x)
#pragma unroll
            for (int i = 0; i < NP; ++i)
#pragma unroll
                for (int e = 0; e < 8; ++e) v[i][e] = __fadd_rn(xv[i][e], v[i][e]);
    }
    if constexpr (ATTN) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int p = tid + i * kThreads;
            if (p >= pairs) continue;
            const int nh = K / at.hd, h = p * 8 / at.hd, d = p * 8 - h * at.hd;
            const size_t row = (size_t)t * nh + h, rows = (size_t)gridDim.x * nh;
            // every piece's loads first; a piece without positions (-inf, 0) has no O
            float2 ms[kPrefillPieces];
            float ov[kPrefillPieces][8];
#pragma unroll
            for (int c = 0; c < kPrefillPieces; ++c) {
                ms[c] = make_float2(-INFINITY, 0.f);
                if (c < at.pieces) {
                    ms[c] = at.ms[c * rows + row];
                    load8(at.part + (c * rows + row) * at.hd + d, ov[c]);
                }
            }
            float top = -INFINITY, sum = 0.f;
#pragma unroll
            for (int c = 0; c < kPrefillPieces; ++c)
                if (ms[c].y != 0.f) top = fmaxf(top, ms[c].x);
#pragma unroll
            for (int c = 0; c < kPrefillPieces; ++c)
                if (ms[c].y != 0.f) {
                    const float f = __builtin_amdgcn_exp2f(ms[c].x - top);
                    sum = __fadd_rn(sum, __fmul_rn(ms[c].y, f));
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[i][e] = __builtin_fmaf(ov[c][e], f, v[i][e]);
                }
#pragma unroll
            for (int e = 0; e < 8; ++e) v[i][e] = __fdiv_rn(v[i][e], sum);
        }
    }
    if (in.resid_out)
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int p = tid + i * kThreads;
            if (p < pairs) {
                float4 *dst = reinterpret_cast<float4 *>(in.resid_out + (size_t)t * in.ldr + p * 8);
                dst[0] = make_float4(v[i][0], v[i][1], v[i][2], v[i][3]);
                dst[1] = make_float4(v[i][4], v[i][5], v[i][6], v[i][7]);
            }
        }
    if (in.w_norm) scaled(rms_inv(1), wn);
    // a chunk's 128 pairs sit in two waves of one round
    bool nan = false, nf = false;
    uint32_t inf[NP][2];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        float mx = 0.f;
        inf[i][0] = inf[i][1] = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float x = v[i][e];
            nan |= x != x;
            inf[i][0] |= (x == INFINITY ? 1u : 0u) << e;
            inf[i][1] |= (x == -INFINITY ? 1u : 0u) << e;
            const bool bad = nonfinite::is_nf(x);
            nf |= bad;
            v[i][e] = bad ? 0.f : x;
            mx = fmaxf(mx, fabsf(v[i][e]));
        }
        mx = lanes::wave_max(mx);
        if (lane == 0) wmx[i][wid] = mx;
    }
    const int fl = (__any(nf) ? 1 : 0) | (__any(nan) ? 2 : 0);
    if (lane == 0) wfl[wid] = fl;
    __syncthreads();
    int flags = 0, ex[NP];
#pragma unroll
    for (int w = 0; w < kWavesWg; ++w) flags |= wfl[w];
    // the chunk's largest |x| * 2^-ex in [2^14, 2^15)
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const float mx = fmaxf(wmx[i][wid & ~1], wmx[i][wid | 1]);
        ex[i] = 0;
        if (mx > 0.f) {
            int f;
            frexpf(mx, &f);
            ex[i] = f - 15;
        }
        const int p = tid + i * kThreads;
        if ((p & (kChunk * 4 - 1)) == 0 && p < pairs) op.xsc[(size_t)(p / (kChunk * 4)) * op.tokens + t] = ldexpf(1.0f, ex[i]);
    }
    if (tid == 0) op.flag[t] = flags;
    h8 *row = op.a + (size_t)(t >> 4) * nb * 2 * kWave + (t & 15);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int p = tid + i * kThreads;
        if (p >= pairs) continue;
        const int bl = p >> 2, m = p & 3;
        h8 hv, lv;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float s = ldexpf(v[i][k_order<DT>(k)], -ex[i]) * k_factor<DT>(k);
            const _Float16 h = (_Float16)s;
            hv[k] = h;
            lv[k] = (_Float16)(s - (float)h);
        }
        row[(bl * 2 + 0) * kWave + m * 16] = hv;
        row[(bl * 2 + 1) * kWave + m * 16] = lv;
    }
    if (flags)                                         // rare: the token's masks
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int p = tid + i * kThreads;
            for (int sg = 0; sg < 2; ++sg) {
                const uint32_t w = lanes::quad_or(inf[i][sg] << (8 * (p & 3)));
                if ((p & 3) == 0 && p < pairs) op.inf[((size_t)t * 2 + sg) * nb + (p >> 2)] = w;
            }
        }
}

// Row `row`'s share of the non-finite activations of token t (chunk_fold over all of K).
template <int DT>
__device__ float token_fold(const Operand &op, int flags, const uint8_t *__restrict__ wq,
                            const uint8_t *__restrict__ wsc, int nb, int row, int t) {
    if (flags & 2) return __builtin_nanf("");
    float a = 0.f;
    for (int bl = 0; bl < nb; ++bl)
        for (int sg = 0; sg < 2; ++sg)
            for (uint32_t m = op.inf[((size_t)t * 2 + sg) * nb + bl]; m != 0; m &= m - 1) {
                const float w = nonfinite::weight_at<DT, LAYOUT_TILED>(wq, wsc, nb, row, bl * kBlock + __builtin_ctz(m));
                a = __fadd_rn(a, __fmul_rn(w, sg ? -INFINITY : INFINITY));
            }
    return a;
}

struct WideArgs {
    const uint8_t *wq;
    const uint8_t *wsc;
    Operand op;
    int M, K, T;
    int nt, nm, ks;                // workgroup tiles over the tokens / the rows, K splits
    bool rows_fast;                // consecutive workgroups walk the rows first
    float *y;                      // ks > 1: [ks][T][M] partial sums
    int ldy;
    bool geglu;
};

static_assert(kChunk == 8 * kGroupBlocks, "a chunk's range scale covers 8 groups");

// One workgroup of NW waves: each multiplies the workgroup's WT tiles of 16 tokens by WN tiles of 16
// weight rows of its own. A stage is one TILED group (four blocks) of the workgroup's operands,
// weights and scales, brought into LDS by DMA (no registers in flight) D - 1 groups ahead. One
// barrier per group: a stage is refilled after the barrier that ends its reads.
// The sums run in three levels (a group, a chunk, the row) so that no fp32 chain is longer than
// the K chunks and wave shares of the 16-vector GEMM make it there; four row tiles per wave
// leave registers for two (two groups, the row), enough up to kMaxTwoLevelK.
template <int DT, int WN, int WT, int NW, int D>
__global__ __launch_bounds__(NW *kWave, 2) void gemm_wide_kernel(WideArgs p) {
    constexpr int NQ = DT == DT_Q8_0 ? 2 : 1;
    constexpr int BN = WN * NW;                        // tiles of 16 rows
    constexpr int kA = WT * 8 * 1024, kQ = BN * NQ * 1024, kS = BN * 256, kStage = kA + kQ + kS;
    constexpr int kDma = WT * 8 / NW + BN * (NQ + 1) / NW;   // DMA instructions of a wave per stage
    static_assert(WT * 8 % NW == 0 && BN % NW == 0, "every wave issues the same number");
    __shared__ __attribute__((aligned(16))) char lds[D][kStage];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wid = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int n = lane & 15, m = lane >> 4;
    // Workgroups go to the XCDs round robin: each XCD takes a contiguous range of the tiles, so
    // that its L2 holds one side's share once instead of both sides whole.
    const int total = gridDim.x, per = total / kXcds, rem = total % kXcds, xcd = blockIdx.x % kXcds;
    int lin = xcd * per + min(xcd, rem) + (int)blockIdx.x / kXcds;
    const int kz = lin % p.ks;
    lin /= p.ks;
    const int bt = p.rows_fast ? lin / p.nm : lin % p.nt, bm = p.rows_fast ? lin % p.nm : lin / p.nt;
    const int nb = p.K / kBlock, G = nb / kGroupBlocks;
    const int g0 = kz * G / p.ks, g1 = (kz + 1) * G / p.ks;
    const int ntiles = (p.M + kTileRows - 1) / kTileRows;
    BConst bk = {0x000F000Fu, 0x00F000F0u, 0x64086408u, 0x64806480u};
    asm volatile("" : "+v"(bk.lo_mask), "+v"(bk.hi_mask), "+v"(bk.lo_bits), "+v"(bk.hi_bits));

    auto dma16 = [&](const void *src, char *dst) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                         (__attribute__((address_space(3))) void *)dst, 16, 0, 0);
    };
    auto issue = [&](int slot, int g) {
        char *st = lds[slot];
#pragma unroll
        for (int i = 0; i < WT * 8 / NW; ++i) {        // a tile of 16 tokens: 8 KiB in one piece
            const int c = i * NW + wid;
            dma16(p.op.a + ((size_t)(bt * WT + (c >> 3)) * nb + g * kGroupBlocks) * 2 * kWave + (c & 7) * kWave + lane,
                  st + c * 1024);
        }
#pragma unroll
        for (int i = 0; i < BN / NW; ++i) {            // tiles past the matrix read its last one
            const int c = i * NW + wid;
            const size_t gb = (size_t)min(bm * BN + c, ntiles - 1) * G + g;
#pragma unroll
            for (int h = 0; h < NQ; ++h) dma16(p.wq + (gb * NQ + h) * 1024 + lane * 16, st + kA + (c * NQ + h) * 1024);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(p.wsc + gb * 256 + lane * 4),
                                             (__attribute__((address_space(3))) void *)(st + kA + kQ + c * 256), 4, 0, 0);
        }
    };
    constexpr bool kMid = WN < 4;
    constexpr int kFlush = kMid ? 1 : 2;               // groups per first-level sum
    f4 acc[WN][WT], mid[WN][WT], tot[WN][WT];
#pragma unroll
    for (int i = 0; i < WN; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j) acc[i][j] = mid[i][j] = tot[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const char *st) {
        const h8 *x = reinterpret_cast<const h8 *>(st);
        Unit u[WN];
#pragma unroll
        for (int i = 0; i < WN; ++i) {
            const int c = wid * WN + i;
#pragma unroll
            for (int h = 0; h < NQ; ++h) u[i].a[h] = *reinterpret_cast<const u32x4 *>(st + kA + (c * NQ + h) * 1024 + lane * 16);
#pragma unroll
            for (int j = 0; j < 4; ++j) u[i].s[j] = *reinterpret_cast<const float *>(st + kA + kQ + c * 256 + j * 64 + n * 4);
        }
        // JB blocks at a time: every operand read first, then the MFMAs of all their chains, then
        // the scales, so that neither the reads nor the MFMAs wait for each other one by one
        constexpr int JB = WN * WT <= 4 ? kGroupBlocks : 2;
#pragma unroll
        for (int j0 = 0; j0 < kGroupBlocks; j0 += JB) {
            h8 hi[JB][WT], lo[JB][WT], b[JB][WN];
            f4 C[JB][WN][WT];
#pragma unroll
            for (int j = 0; j < JB; ++j)
#pragma unroll
                for (int q = 0; q < WT; ++q) {
                    const h8 *a = x + (q * kGroupBlocks + j0 + j) * 2 * kWave + lane;
                    hi[j][q] = a[0];
                    lo[j][q] = a[kWave];
                }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < JB; ++j) {
#pragma unroll
                for (int i = 0; i < WN; ++i) b[j][i] = b_operand<DT>(u[i].a, j0 + j, bk.lo_mask, bk.hi_mask, bk.lo_bits, bk.hi_bits);
#pragma unroll
                for (int q = 0; q < WT; ++q)
#pragma unroll
                    for (int i = 0; i < WN; ++i)
                        C[j][i][q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[j][q], b[j][i], f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            }
#pragma unroll
            for (int j = 0; j < JB; ++j)
#pragma unroll
                for (int q = 0; q < WT; ++q)
#pragma unroll
                    for (int i = 0; i < WN; ++i)
                        C[j][i][q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[j][q], b[j][i], C[j][i][q], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < JB; ++j)
#pragma unroll
                for (int q = 0; q < WT; ++q)
#pragma unroll
                    for (int i = 0; i < WN; ++i)
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[i][q][r] = __builtin_fmaf(C[j][i][q][r], u[i].s[j0 + j], acc[i][q][r]);
        }
    };
    // Past the end the issue repeats the last group, so that the wait always leaves the same
    // number of loads in flight (they complete in issue order).
#pragma unroll
    for (int d = 0; d < D - 1; ++d) issue(d, min(g0 + d, g1 - 1));
    f4 sc[WT];                                         // the current chunk's range scales (padded tokens: read, not used)
    for (int g = g0, slot = 0; g < g1; ++g) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 2) * kDma) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (g == g0 || (g & 7) == 0)
#pragma unroll
            for (int j = 0; j < WT; ++j)
                sc[j] = *reinterpret_cast<const f4 *>(p.op.xsc + (size_t)(g >> 3) * p.op.tokens + (bt * WT + j) * 16 + 4 * m);
        asm volatile("" ::: "memory");
        issue(slot == 0 ? D - 1 : slot - 1, min(g + D - 1, g1 - 1));
        multiply(lds[slot]);
        const bool end = (g & 7) == 7 || g + 1 == g1;  // the chunk ends: its range scale
        if ((g & (kFlush - 1)) == kFlush - 1 || end)
#pragma unroll
            for (int j = 0; j < WT; ++j)
#pragma unroll
                for (int i = 0; i < WN; ++i) {
                    if constexpr (kMid) {
                        mid[i][j] += acc[i][j];
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r) tot[i][j][r] = __builtin_fmaf(acc[i][j][r], sc[j][r], tot[i][j][r]);
                    }
                    acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
                }
        if (kMid && end)
#pragma unroll
            for (int j = 0; j < WT; ++j)
#pragma unroll
                for (int i = 0; i < WN; ++i) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) tot[i][j][r] = __builtin_fmaf(mid[i][j][r], sc[j][r], tot[i][j][r]);
                    mid[i][j] = f4{0.f, 0.f, 0.f, 0.f};
                }
        slot = slot == D - 1 ? 0 : slot + 1;
        // this wave's reads of the stage are done before the barrier that lets it be refilled
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no DMA outlives the workgroup's LDS

    int4 flags[WT];                                    // padded tokens': read, not used
#pragma unroll
    for (int q = 0; q < WT; ++q)
        flags[q] = *reinterpret_cast<const int4 *>(p.op.flag + (bt * WT + q) * 16 + 4 * m);
    float *dst = p.y + (p.ks > 1 ? (size_t)kz * p.T * p.M : 0);
#pragma unroll
    for (int q = 0; q < WT; ++q) {
        const int t0 = (bt * WT + q) * 16 + 4 * m;
#pragma unroll
        for (int i = 0; i < WN; ++i) {
            const int ti = bm * BN + wid * WN + i, row = ti * kTileRows + n;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float val = tot[i][q][r];
                // the fold of the whole row goes to the first K split
                const int fl = r == 0 ? flags[q].x : r == 1 ? flags[q].y : r == 2 ? flags[q].z : flags[q].w;
                if (fl && kz == 0 && row < p.M && t0 + r < p.T) val += token_fold<DT>(p.op, fl, p.wq, p.wsc, nb, row, t0 + r);
                if (p.geglu) {
                    // lanes n < 8 hold gate rows 8 ti + n, lanes n + 8 the matching up rows
                    const float up = __shfl_xor(val, 8, kWave);
                    const int c = ti * 8 + n;
                    if (n < 8 && t0 + r < p.T && 2 * c < p.M)
                        dst[(size_t)(t0 + r) * p.ldy + c] = __fmul_rn(devmath::gelu_ref(val), up);
                } else if (row < p.M && t0 + r < p.T) {
                    dst[(size_t)(t0 + r) * p.ldy + row] = val;
                }
            }
        }
    }
}

int cu_count() {
    int dev = 0, c = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || c <= 0)
        return 256;
    return c;
}

struct Shape {
    int bm, bn;                    // tokens and rows of a workgroup
};
constexpr Shape kShapes[] = {{32, 256}, {32, 128}, {32, 64}};
constexpr int kNumShapes = 3, kSmallest = kNumShapes - 1;
constexpr int kMaxTwoLevelK = 2304;
constexpr int kSplitPerCu = 2;     // workgroups per CU up to which K is split

// The workgroup tile and K split of a GEMM. An A operand read from LDS feeds the MFMAs of the rows of
// one wave, so a wider tile has fewer LDS reads and waits per product, and the widest one that still
// gives every CU a workgroup is the fastest (Q4_0 16384 x 6912 x 512: 278 us at 256 rows, 309 at 128,
// 385 at 64; 640 x 1024 x 512, where only the last one covers the CUs: 20, 15 and 12 us; Q8_0's
// 256-row stage leaves one workgroup per CU and loses). The last round of workgroups is not looked
// at: just past the CUs every tile takes the same (Q4_0 6912 x 1152 x 300, 270 workgroups of 256
// rows: 30.8 us, 128 rows 30.0, 64 rows 30.0; 288 tokens, where 243 would not cover the CUs: 23.8,
// 21.9 and 25.2). Where the smallest tile leaves CUs
// idle, K is split until two workgroups per CU: 1152 x 6912 x 300 takes 37 us in two parts against 48
// (three per CU: 640 x 2048 x 500 23 us against 20, the partial sums' traffic), but 640 x 1024 x 300
// 12.7 against 12.0, the partial sums costing more than the shorter chains save, so not below 12
// groups.
void plan(int dt, int M, int K, int T, bool may_split, int *shape, int *ks) {
    const int cus = cu_count(), G = K / (kGroupBlocks * kBlock);
    auto grid = [&](int i) { return ((T + kShapes[i].bm - 1) / kShapes[i].bm) * ((M + kShapes[i].bn - 1) / kShapes[i].bn); };
    int s = dt == DT_Q8_0 || K > kMaxTwoLevelK ? 1 : 0, k = 1;
    while (s < kSmallest && grid(s) < cus) ++s;
    if (may_split && s == kSmallest && G >= 12)
        while (k < kWideMaxSplit && grid(s) * (k + 1) <= kSplitPerCu * cus && G / (k + 1) >= 4) ++k;
    *shape = s;
    *ks = k;
}

}  // namespace

bool gemm_wide_supported(int K) { return K > 0 && K % (kGroupBlocks * kBlock) == 0 && K <= kWideMaxK; }

size_t gemm_wide_operand_bytes(int T, int K) {
    const size_t p = (size_t)padded(T);
    return (p * K * 4 + p * chunks_of(K) * 4 + p * 4 + p * (K / kBlock) * 8 + 255) & ~size_t(255);
}

// K is split only while the smallest tile's workgroups number at most two per CU, which bounds
// the partial sums
size_t gemm_wide_parts_bytes(int M, int T) {
    return std::min((size_t)kWideMaxSplit * T * M, (size_t)kSplitPerCu * cu_count() * kShapes[kSmallest].bm * kShapes[kSmallest].bn) * sizeof(float);
}

int gemm_wide_splits(int dt, int M, int K, int T) {
    int s, k;
    plan(dt, M, K, T, true, &s, &k);
    return k;
}

int gemm_wide_tile_rows(int dt, int M, int K, int T) {
    int s, k;
    plan(dt, M, K, T, true, &s, &k);
    return kShapes[s].bn;
}

int launch_gemm_wide_prep(int dt, const GemmIn &in, int K, int T, void *operand, hipStream_t st) {
    auto al = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15u) == 0; };
    if (!gemm_wide_supported(K) || T <= 0 || !operand || in.x_blocked || (!in.x && !in.parts) ||
        (in.x && (!al(in.x) || in.ldx % 4 != 0 || in.ldx < K)) ||
        (in.parts && (!al(in.parts) || in.nparts < 1 || in.ldp % 4 != 0 || in.ldp < K || in.part_stride % 4 != 0)) ||
        (in.w_delta && (!in.parts || !al(in.w_delta))) || (in.w_norm && !al(in.w_norm)) ||
        (in.resid_out && (!al(in.resid_out) || in.ldr % 4 != 0))) {
        set_error("wide GEMM input: unsupported arguments (T=%d K=%d)", T, K);
        return -1;
    }
    const Operand op = operand_at(operand, T, K);
    const bool small = K <= 8 * kThreads;
    auto kern = dt == DT_Q4_0 ? (small ? gemm_wide_prep_kernel<DT_Q4_0, 1> : gemm_wide_prep_kernel<DT_Q4_0, 4>)
                              : (small ? gemm_wide_prep_kernel<DT_Q8_0, 1> : gemm_wide_prep_kernel<DT_Q8_0, 4>);
    hipLaunchKernelGGL(kern, dim3(T), dim3(kThreads), 0, st, in, K, op, AttnParts{});
    return hip_ok(hipGetLastError(), "gemm_wide prep launch") ? 0 : -1;
}

int launch_gemm_wide_prep_attn(int dt, const float *part, const void *ms, int pieces, int nh, int hd, int T,
                               void *operand, hipStream_t st) {
    const int K = nh * hd;
    if (!gemm_wide_supported(K) || K > 8 * kThreads || T <= 0 || pieces < 1 || pieces > kPrefillPieces || hd % 8 != 0) {
        set_error("wide GEMM attention input: unsupported arguments (T=%d, %d heads of %d, %d pieces)", T, nh, hd, pieces);
        return -1;
    }
    const AttnParts at{part, static_cast<const float2 *>(ms), pieces, hd};
    auto kern = dt == DT_Q4_0 ? gemm_wide_prep_kernel<DT_Q4_0, 1, true> : gemm_wide_prep_kernel<DT_Q8_0, 1, true>;
    hipLaunchKernelGGL(kern, dim3(T), dim3(kThreads), 0, st, GemmIn{}, K, operand_at(operand, T, K), at);
    return hip_ok(hipGetLastError(), "gemm_wide attention prep launch") ? 0 : -1;
}

int launch_gemm_wide(int dt, const void *w, int M, int K, int T, const void *operand, const WideOut &out,
                     hipStream_t st) {
    if (!gemm_wide_supported(K) || !tiled_layout_ok(dt, M, K) || M <= 0 || T <= 0 || !operand || !(out.y || out.parts) ||
        (out.geglu && (out.parts || M % 16 != 0)) || (!out.parts && out.ldy < (out.geglu ? M / 2 : M))) {
        set_error("wide GEMM: unsupported arguments (M=%d K=%d T=%d)", M, K, T);
        return -1;
    }
    int s, ks;
    plan(dt, M, K, T, out.parts != nullptr, &s, &ks);
    const size_t so = q_tiled_scales_offset(dt, M, K);
    WideArgs a;
    a.wq = static_cast<const uint8_t *>(w);
    a.wsc = a.wq + so;
    a.op = operand_at(const_cast<void *>(operand), T, K);
    a.M = M;
    a.K = K;
    a.T = T;
    a.nt = (T + kShapes[s].bm - 1) / kShapes[s].bm;
    a.nm = (M + kShapes[s].bn - 1) / kShapes[s].bn;
    a.ks = ks;
    // the smaller side is the one every XCD reads whole
    a.rows_fast = (size_t)M * block_bytes(dt) / 8 < (size_t)T * 16;
    a.y = out.parts ? out.parts : out.y;
    a.ldy = out.parts ? M : out.ldy;
    a.geglu = out.geglu;
    const dim3 grid((unsigned)(a.nt * a.nm * ks));
    // stages: as many as leave two workgroups per CU
    if (dt == DT_Q4_0 && s == 0) hipLaunchKernelGGL((gemm_wide_kernel<DT_Q4_0, 4, 2, 4, 2>), grid, dim3(256), 0, st, a);
    else if (dt == DT_Q4_0 && s == 1) hipLaunchKernelGGL((gemm_wide_kernel<DT_Q4_0, 2, 2, 4, 3>), grid, dim3(256), 0, st, a);
    else if (dt == DT_Q4_0) hipLaunchKernelGGL((gemm_wide_kernel<DT_Q4_0, 1, 2, 4, 3>), grid, dim3(256), 0, st, a);
    else if (s == 1) hipLaunchKernelGGL((gemm_wide_kernel<DT_Q8_0, 2, 2, 4, 2>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((gemm_wide_kernel<DT_Q8_0, 1, 2, 4, 3>), grid, dim3(256), 0, st, a);
    return hip_ok(hipGetLastError(), "gemm_wide launch") ? 0 : -1;
}

}  // namespace sapphire
