// sample.hip - the next token as perform_inference draws it (inference.c:262-266, 297), for a
// batch of logit rows: temperature <= 0 is sample_greedy (utils.c:145-156); otherwise the
// logits are scaled by 1/T (vec_scale, utils.c:87-92) and sample_temperature (utils.c:158-180)
// draws: max seeded with logits[0] (strict >), w_i = expf((l_i - max) / T) in place, sum the
// w_i left to right in float, then walk cumsum += w_i / sum (float) and return the first i with
// r <= cumsum, n - 1 if there is none. r is the caller's draw in place of rand() / RAND_MAX.
//
// The token is the reference's bit for bit, so both float chains (the sum, and the running sum
// the draw is compared with) are reproduced exactly, in parallel:
// * while a chain v <- fl(v + x) (x >= 0) stays inside one binade [2^e, 2^(e+1)), whose
//   spacing is u, it is integer arithmetic on M = v / u: fl(v + x) = (M + k) u with k = x / u
//   rounded to nearest, and on a tie (x / u = f + 1/2) the even one of M + f and M + f + 1.
//   Each element is the map M -> M + d[M & 1] (k and the tie read from the element's float
//   bits in integer arithmetic); maps compose (associatively), so a sub-chunk of kSub elements
//   is one pair (d0, d1) for a given binade. The binades a chain can occupy at a sub-chunk's
//   start are fixed to at most two by the exact prefix sum and the error bound of recursive
//   summation (|fl-sum - sum| <= n 2^-24 sum for nonnegative terms);
// * the maps are kept for groups of 64 elements as well, each for the binades of its own start;
// * one wave per row walks the sub-chunks with these maps, 64 at a time; in a sub-chunk where
//   the binade changes or the draw is reached it scans the 16 groups' maps, and the group where
//   that happens is added element by element with real float adds (the reference's own
//   operation), whatever binades it crosses. (Composing 16 elements' maps per lane in the walk
//   instead, once per binade change, took 107 us per walk of 262144 weights; a group's 64 adds
//   take a third of a microsecond, and the walk 31 us.)
// The weights come from libm_expf, glibc's expf bit for bit.
#include "internal.h"
#include "libm_expf.h"

#include <cmath>

namespace sapphire {
namespace {

constexpr int kWave = 64;
constexpr int kThreads = 256;
constexpr int kPer = 4;                         // elements per thread in the grid kernels
constexpr int kSub = kThreads * kPer;           // elements per sub-chunk (one grid workgroup)
constexpr int kGroup = kWave;                   // elements per group
constexpr int kGroups = kSub / kGroup;          // groups per sub-chunk: one per row of 16 lanes
static_assert(kGroup == 16 * kPer && kGroups == 16, "a group is a row of 16 lanes of the grid kernels");
constexpr int kMaxSubs = 2048;                  // n <= 2^21 keeps the error bound below 1/4
constexpr int kSlots = 12;                      // sub-chunks a walk fetches ahead
constexpr int kShortSubs = 4;                   // rows up to this long take the walk with little LDS
constexpr int kCap = 1 << 28;                   // saturation of map increments
constexpr int kZero = -1000, kSub_ = -127;      // binade ids of 0 and of the subnormals

struct SubStat {         // per row and sub-chunk
    float max;           // largest non-NaN scaled logit (+-inf included)
    int arg;             // its first index, -1 if the sub-chunk is all NaN
    int nan;             // whether the sub-chunk holds a NaN
    int nan0;            // sub-chunk 0 only: whether the row's first scaled logit is NaN
    double wsum;         // sum of the sub-chunk's weights (exact enough for the bounds)
};
struct SubMaps {         // per row and sub-chunk or group: its map for its (up to) two binades
    int reg[2];
    int d[2][2];
};
struct RowInfo {
    float m;             // the reference's max (NaN when logits[0] is NaN)
    int bad;             // a NaN weight (or an all -inf row): the token is n - 1
    float sum;           // the float sum of the weights
    int pad;
};

struct Reg {
    int id, uexp, mlim;  // binade id, exponent of its spacing, 2^24 (2^23 subnormal, 1 for zero)
};

__device__ __forceinline__ Reg reg_zero() { return {kZero, 0, 1}; }
__device__ __forceinline__ Reg reg_id(int id) {
    if (id == kZero) return reg_zero();
    if (id == kSub_) return {kSub_, -149, 1 << 23};
    return {id, id - 23, 1 << 24};
}
__device__ __forceinline__ Reg reg_of(float v) {               // v >= +0, finite
    const int e = (int)(__float_as_uint(v) >> 23);
    return v == 0.0f ? reg_zero() : reg_id(e == 0 ? kSub_ : e - 127);
}
__device__ __forceinline__ Reg reg_of_bound(double x) {
    if (!(x > 0.0)) return reg_zero();
    if (x < 0x1p-126) return reg_id(kSub_);
    return reg_id(min(ilogb(x), 127));
}
__device__ __forceinline__ int m_of(float v, const Reg &R) {    // v in R
    const int f = (int)(__float_as_uint(v) & 0x7fffffu);
    return R.id == kZero ? 0 : R.id == kSub_ ? f : f | 0x800000;
}
__device__ __forceinline__ float val_of(int M, const Reg &R) {   // exact for M < R.mlim
    const uint32_t f = (uint32_t)M & 0x7fffffu;
    return R.id == kZero ? 0.0f : __uint_as_float(R.id == kSub_ ? f : (uint32_t)(R.id + 127) << 23 | f);
}

struct Map {
    int d0, d1;
};
__device__ __forceinline__ Map map_id() { return {0, 0}; }
// a then b
__device__ __forceinline__ Map compose(Map a, Map b) {
    const int e = a.d0 + ((a.d0 & 1) ? b.d1 : b.d0);
    const int o = a.d1 + ((a.d1 & 1) ? b.d0 : b.d1);
    return {min(e, kCap), min(o, kCap)};
}
__device__ __forceinline__ int apply(int M, Map m) { return M + min((M & 1) ? m.d1 : m.d0, kCap); }

// The map of element x (bits xb of a float >= +0) in binade R: k = x / u rounded to nearest,
// a tie to the even sum. x = mx 2^e2, so x / u = mx 2^(e2 - uexp) in integers.
__device__ __forceinline__ Map elem_map(uint32_t xb, const Reg &R) {
    if (R.id == kZero) return xb ? Map{kCap, kCap} : map_id();
    const uint32_t ex = xb >> 23;
    const uint32_t mx = ex ? (xb & 0x7fffffu) | 0x800000u : xb;
    const int sh = (ex ? (int)ex - 150 : -149) - R.uexp;
    if (sh >= 0) {
        const uint64_t k = (uint64_t)mx << min(sh, 40);
        if (k >= (1u << 25)) return {kCap, kCap};
        return {(int)k, (int)k};
    }
    const int s = -sh;
    if (s >= 26) return map_id();              // x / u < 2^24 2^-26
    const uint32_t f = mx >> s, rem = mx & ((1u << s) - 1u), half = 1u << (s - 1);
    const int fi = (int)f;
    if (rem > half) return {fi + 1, fi + 1};
    if (rem < half) return {fi, fi};
    return {fi + (fi & 1), fi + ((fi & 1) ^ 1)};
}

__device__ __forceinline__ float scaled(float l, float inv_t, int scale) { return scale ? __fmul_rn(l, inv_t) : l; }

__device__ __forceinline__ bool better(float v, int i, float bv, int bi) {
    return bi < 0 || (i >= 0 && (v > bv || (v == bv && i < bi)));
}

// grid (sub-chunks, batch): SubStat of each sub-chunk of the (scaled) logits
__global__ __launch_bounds__(kThreads) void smp_stats(const float *__restrict__ logits, int n, size_t ld,
                                                      float inv_t, int scale, SubStat *__restrict__ stats) {
    __shared__ float sv[kThreads / kWave];
    __shared__ int si[kThreads / kWave], sn[kThreads / kWave];
    const int nsub = gridDim.x, q = blockIdx.x, b = blockIdx.y;
    const float *x = logits + (size_t)b * ld;
    const int i0 = q * kSub + threadIdx.x * kPer;
    float bv = -INFINITY;
    int bi = -1, nan = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const int i = i0 + k;
        if (i < n) {
            const float s = scaled(x[i], inv_t, scale);
            if (s != s) nan = 1;
            else if (bi < 0 || s > bv) {
                bv = s;
                bi = i;
            }
        }
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
        const float ov = __shfl_xor(bv, off, kWave);
        const int oi = __shfl_xor(bi, off, kWave);
        if (better(ov, oi, bv, bi)) {
            bv = ov;
            bi = oi;
        }
        nan |= __shfl_xor(nan, off, kWave);
    }
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    if (lane == 0) {
        sv[wid] = bv;
        si[wid] = bi;
        sn[wid] = nan;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kThreads / kWave; ++w) {
            if (better(sv[w], si[w], bv, bi)) {
                bv = sv[w];
                bi = si[w];
            }
            nan |= sn[w];
        }
        SubStat st;
        st.max = bv;
        st.arg = bi;
        st.nan = nan;
        st.nan0 = q == 0 ? (int)(scaled(x[0], inv_t, scale) != scaled(x[0], inv_t, scale)) : 0;
        st.wsum = 0.0;
        stats[(size_t)b * nsub + q] = st;
    }
}

// The reference's max and the row's status from the sub-chunk statistics (all threads).
__device__ void row_max(const SubStat *__restrict__ st, int nsub, float *m_out, int *bad_out) {
    __shared__ float sm[kThreads / kWave];
    __shared__ int sb[kThreads / kWave];
    float m = -INFINITY;
    int nan = 0;
    for (int q = threadIdx.x; q < nsub; q += blockDim.x) {
        m = fmaxf(m, st[q].max);
        nan |= st[q].nan;
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
        m = fmaxf(m, __shfl_xor(m, off, kWave));
        nan |= __shfl_xor(nan, off, kWave);
    }
    if ((threadIdx.x & (kWave - 1)) == 0) {
        sm[threadIdx.x / kWave] = m;
        sb[threadIdx.x / kWave] = nan;
    }
    __syncthreads();
    m = sm[0];
    nan = sb[0];
    for (int w = 1; w < (int)(blockDim.x / kWave); ++w) {
        m = fmaxf(m, sm[w]);
        nan |= sb[w];
    }
    __syncthreads();
    if (st[0].nan0) m = __int_as_float(0x7fc00000);
    *m_out = m;
    // NaN anywhere, or max = +inf (inf - inf) or -inf (every weight NaN): the sum is NaN
    *bad_out = nan || m != m || m == INFINITY || m == -INFINITY;
}

// grid (sub-chunks, batch): w = expf((s - m) / T) written to w (may alias the logits), the
// sub-chunk's weight sum into its SubStat, the row's RowInfo (sub-chunk 0)
__global__ __launch_bounds__(kThreads) void smp_weights(const float *logits, int n, size_t ld, float inv_t,
                                                        int scale, float t, float *w, size_t ldw,
                                                        SubStat *__restrict__ stats, RowInfo *__restrict__ rows) {
    __shared__ double sd[kThreads / kWave];
    const int nsub = gridDim.x, q = blockIdx.x, b = blockIdx.y;
    SubStat *st = stats + (size_t)b * nsub;
    float m;
    int bad;
    row_max(st, nsub, &m, &bad);
    const float *x = logits + (size_t)b * ld;
    float *wr = w + (size_t)b * ldw;
    const int i0 = q * kSub + threadIdx.x * kPer;
    double sum = 0.0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const int i = i0 + k;
        if (i < n) {
            const float v = libm_expf(__fdiv_rn(__fsub_rn(scaled(x[i], inv_t, scale), m), t));
            wr[i] = v;
            sum += (double)v;
        }
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0) sd[threadIdx.x / kWave] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < kThreads / kWave; ++k) sum += sd[k];
        st[q].wsum = sum;
        if (q == 0) {
            RowInfo ri;
            ri.m = m;
            ri.bad = bad;
            ri.sum = 0.0f;
            ri.pad = 0;
            rows[b] = ri;
        }
    }
}

// Element x of a chain, as float bits: the weight (chain 0) or the weight over the float sum
// (chain 1).
__device__ __forceinline__ uint32_t chain_elem(float wv, int chain, float sum) {
    return __float_as_uint(chain ? __fdiv_rn(wv, sum) : wv);
}

// One DPP move of both halves of a map; lanes without a source (and rows outside row_mask)
// read 0, the identity map.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ Map dpp_map(Map m) {
    return {__builtin_amdgcn_update_dpp(0, m.d0, CTRL, ROW_MASK, 0xf, true),
            __builtin_amdgcn_update_dpp(0, m.d1, CTRL, ROW_MASK, 0xf, true)};
}

// Inclusive scan of the maps of each row of 16 lanes.
__device__ __forceinline__ Map row_scan(Map m) {
    m = compose(dpp_map<0x111, 0xf>(m), m);   // row_shr:1
    m = compose(dpp_map<0x112, 0xf>(m), m);   // row_shr:2
    m = compose(dpp_map<0x114, 0xf>(m), m);   // row_shr:4
    return compose(dpp_map<0x118, 0xf>(m), m);   // row_shr:8
}

// Inclusive scan of the wave's maps in lane order (lane l gets m_0 ... m_l composed): shifts
// by 1, 2, 4, 8 within each 16-lane row, then the last lane of row 0 (and of row 2) into the
// next row, then lane 31 into rows 2 and 3.
__device__ __forceinline__ Map wave_scan(Map m) {
    m = row_scan(m);
    m = compose(dpp_map<0x142, 0xa>(m), m);   // row_bcast:15 into rows 1 and 3
    m = compose(dpp_map<0x143, 0xc>(m), m);   // row_bcast:31 into rows 2 and 3
    return m;
}

__device__ __forceinline__ int first_lane(unsigned long long bal) { return __builtin_ctzll(bal); }

// The binades a chain can be in after weights of exact sum p (chain 1: over the float sum), at
// most two. Recursive summation of n nonnegative floats: relative error below (n + 2) 2^-24
// (with margin); the quotients w / sum add 2^-24 relative each, and subnormal ones 2^-150.
__device__ __forceinline__ void chain_regs(double p, int n, int chain, float sum, Reg &lo, Reg &hi) {
    double rel = 2.0 * (n + 2) * 0x1p-24, abs_err = 0.0;
    if (chain) {
        p /= (double)sum;
        rel += 0x1p-22;
        abs_err = (double)n * 0x1p-149;
    }
    lo = reg_of_bound(p * (1.0 - rel) - abs_err);
    hi = reg_of_bound(p * (1.0 + rel) + abs_err);
}

// The map of binade id in a group or sub-chunk; one that cannot be applied (and ends the scan
// there) when it was not prepared.
__device__ __forceinline__ Map map_for(const SubMaps &c, int id) {
    const int k = c.reg[0] == id ? 0 : (c.reg[1] == id ? 1 : -1);
    return k < 0 ? Map{kCap, kCap} : Map{c.d[k][0], c.d[k][1]};
}

// grid (sub-chunks, batch): the maps (chain 0: the weight sum; chain 1: the running sum of the
// weights over the float sum) of each group for the binades the chain can be in at its start,
// and of the sub-chunk for those at its own. A sub-chunk that stays in one binade has that
// binade prepared in every group, so its map is the groups' maps composed.
__global__ __launch_bounds__(kThreads) void smp_maps(const float *__restrict__ w, int n, size_t ldw, int chain,
                                                     const SubStat *__restrict__ stats,
                                                     const RowInfo *__restrict__ rows, SubMaps *__restrict__ maps,
                                                     SubMaps *__restrict__ gmaps, int *__restrict__ cross) {
    __shared__ double sd[kThreads / kWave], sg[kGroups];
    __shared__ SubMaps gm[kGroups];
    const int nsub = gridDim.x, q = blockIdx.x, b = blockIdx.y;
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave, g = threadIdx.x / 16;
    const float *wr = w + (size_t)b * ldw;
    const int i0 = q * kSub + threadIdx.x * kPer;
    float wv[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) wv[k] = i0 + k < n ? wr[i0 + k] : 0.0f;
    const RowInfo ri = rows[b];
    if (ri.bad) return;
    const SubStat *st = stats + (size_t)b * nsub;
    // the exact sums of the weights before this sub-chunk, and of its groups
    double p = 0.0, gs = 0.0;
    for (int k = threadIdx.x; k < q; k += kThreads) p += st[k].wsum;
#pragma unroll
    for (int k = 0; k < kPer; ++k) gs += (double)wv[k];
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) p += __shfl_xor(p, off, kWave);
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) gs += __shfl_xor(gs, off, kWave);
    if (lane == 0) sd[wid] = p;
    if ((lane & 15) == 0) sg[g] = gs;
    __syncthreads();
    p = sd[0];
    for (int k = 1; k < kThreads / kWave; ++k) p += sd[k];
    double pg = p;
#pragma unroll
    for (int k = 0; k < kGroups - 1; ++k) pg += k < g ? sg[k] : 0.0;
    Reg lo, hi;
    chain_regs(pg, n, chain, ri.sum, lo, hi);
    Map m0 = map_id(), m1 = map_id();
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const uint32_t x = chain_elem(wv[k], chain, ri.sum);
        m0 = compose(m0, elem_map(x, lo));
        m1 = compose(m1, elem_map(x, hi));
    }
    // the row of 16 lanes composed in order, into its last lane
    m0 = row_scan(m0);
    m1 = row_scan(m1);
    if ((lane & 15) == 15) {
        SubMaps c;
        c.reg[0] = lo.id;
        c.d[0][0] = m0.d0;
        c.d[0][1] = m0.d1;
        c.reg[1] = hi.id;
        c.d[1][0] = m1.d0;
        c.d[1][1] = m1.d1;
        gm[g] = c;
        gmaps[((size_t)b * nsub + q) * kGroups + g] = c;
    }
    __syncthreads();
    if (threadIdx.x == 2) {
        // whether the exact sum changes binade in this sub-chunk (where the chain almost always
        // does too: the walk fetches it ahead)
        const double e = p + ((sg[0] + sg[1] + sg[2] + sg[3]) + (sg[4] + sg[5] + sg[6] + sg[7]) +
                              (sg[8] + sg[9] + sg[10] + sg[11]) + (sg[12] + sg[13] + sg[14] + sg[15]));
        const double k = chain ? 1.0 / (double)ri.sum : 1.0;
        cross[(size_t)b * nsub + q] = q == 0 || reg_of_bound(p * k).id != reg_of_bound(e * k).id;
    }
    if (threadIdx.x < 2) {
        Reg sl, sh;
        chain_regs(p, n, chain, ri.sum, sl, sh);
        const int id = threadIdx.x == 0 ? sl.id : sh.id;
        Map m = map_id();
        for (int k = 0; k < kGroups; ++k) m = compose(m, map_for(gm[k], id));
        SubMaps &c = maps[(size_t)b * nsub + q];
        c.reg[threadIdx.x] = id;
        c.d[threadIdx.x][0] = m.d0;
        c.d[threadIdx.x][1] = m.d1;
    }
}

// grid (batch), one wave per row walks (four fetch): the chain walk. chain 0 stores the float sum of the weights
// in RowInfo; chain 1 finds the first index whose running sum reaches the row's draw r
// (draws[step * batch + b], step = *d_step or 0) and writes the token (n - 1 if none, or for
// a bad row). The wave takes 64 sub-chunks at a time, one per lane: a scan of their maps in
// the chain's binade finds the first sub-chunk in which the binade changes or r is reached
// (or whose binades were not prepared). There a scan of the 16 groups' maps finds the first
// group where the same happens, and its elements are added one by one; the scan resumes after it.
// The sub-chunks expected to hold a change (cross) are brought into LDS by four waves before the
// walk, in one memory round trip instead of one each (37 -> 31 us per walk of 262144 weights).
// SUBS, SLOTS: the sub-chunks of the longest row and those fetched ahead. The maps and elements of
// kMaxSubs and kSlots fill most of a CU's LDS, so that 256 rows walk at a time; short rows come in
// larger batches and take a form of which seven share a CU (draws from 300 rows of 64: 38 us, 71 with
// the long form; 300 rows of 4096 77 and 115).
template <int SUBS, int SLOTS>
__global__ __launch_bounds__(kThreads) void smp_walk(const float *__restrict__ w, int n, size_t ldw, int chain,
                                                     int nsub, const SubMaps *__restrict__ maps,
                                                     const SubMaps *__restrict__ gmaps, const int *__restrict__ cross,
                                                     RowInfo *__restrict__ rows, const float *__restrict__ draws,
                                                     const int *__restrict__ d_step, int batch,
                                                     int *__restrict__ tokens) {
    __shared__ SubMaps cm[SUBS];
    __shared__ float xs[SLOTS + 1][kSub];              // the last slot: sub-chunks not fetched ahead
    __shared__ SubMaps gs[SLOTS + 1][kGroups];
    __shared__ int slot_q[SLOTS], nslots;
    const int b = blockIdx.x, lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    const RowInfo ri = rows[b];
    if (ri.bad) {
        if (chain && threadIdx.x == 0) tokens[b] = n - 1;
        return;
    }
    const float r = chain ? draws[(size_t)(d_step ? *d_step : 0) * batch + b] : INFINITY;
    const float *wr = w + (size_t)b * ldw;
    if (wid == 0) {
        int have = 0;
        for (int k = 0; k < nsub; k += kWave) {
            const bool c = k + lane < nsub && cross[(size_t)b * nsub + k + lane] != 0;
            const unsigned long long bal = __ballot(c);
            const int at = have + __popcll(bal & ((1ull << lane) - 1));
            if (c && at < SLOTS) slot_q[at] = k + lane;
            have += __popcll(bal);
        }
        if (lane == 0) nslots = min(have, SLOTS);
    } else {
        for (int k = threadIdx.x - kWave; k < nsub; k += kThreads - kWave) cm[k] = maps[(size_t)b * nsub + k];
    }
    __syncthreads();
    // sub-chunk sq's elements and group maps into a slot
    auto fetch = [&](int slot, int sq) {
        SubMaps gm;
        float x[kGroups];
        if (lane < kGroups) gm = gmaps[((size_t)b * nsub + sq) * kGroups + lane];
#pragma unroll
        for (int g = 0; g < kGroups; ++g) x[g] = wr[min(sq * kSub + g * kGroup + lane, n - 1)];
#pragma unroll
        for (int g = 0; g < kGroups; ++g) xs[slot][g * kGroup + lane] = sq * kSub + g * kGroup + lane < n ? x[g] : 0.0f;
        if (lane < kGroups) gs[slot][lane] = gm;
    };
    for (int k = wid; k < nslots; k += kThreads / kWave) fetch(k, slot_q[k]);
    __syncthreads();
    if (wid != 0) return;                              // one wave walks
    const int my_q = lane < nslots ? slot_q[lane] : -1;
    float v = 0.0f;
    int q = 0, found = -1;
    while (q < nsub && found < 0) {
        // sub-chunks q .. q + 63 in the current binade
        {
            const Reg R = reg_of(v);
            const int M0 = m_of(v, R), qi = q + lane;
            const Map m = qi < nsub ? map_for(cm[min(qi, nsub - 1)], R.id) : map_id();
            const int Me = apply(M0, wave_scan(m));
            const bool stop = qi < nsub && (Me >= R.mlim || r <= val_of(Me, R));
            const unsigned long long bal = __ballot(stop);
            if (bal == 0) {
                const int last = min(kWave, nsub - q) - 1;
                v = val_of(__builtin_amdgcn_readlane(Me, last), R);
                q += kWave;
                continue;
            }
            const int s = first_lane(bal);
            if (s > 0) v = val_of(__builtin_amdgcn_readlane(Me, s - 1), R);
            q += s;
        }
        // sub-chunk q: lane g < 16 holds group g's maps
        const int base = q * kSub;
        const unsigned long long hit = __ballot(my_q == q);
        const int slot = hit ? first_lane(hit) : SLOTS;
        if (!hit) fetch(SLOTS, q);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // one wave: its LDS accesses are in order
        const SubMaps gm = gs[slot][lane & (kGroups - 1)];
        int from = 0;                                  // the first group not yet added
        while (from < kGroups) {
            const Reg R = reg_of(v);
            const int M0 = m_of(v, R);
            const Map m = lane >= from && lane < kGroups ? map_for(gm, R.id) : map_id();
            const int Me = apply(M0, row_scan(m));
            const bool stop = lane >= from && lane < kGroups && (Me >= R.mlim || r <= val_of(Me, R));
            const unsigned long long bal = __ballot(stop);
            if (bal == 0) {                            // the rest of the sub-chunk stays in the binade
                v = val_of(__builtin_amdgcn_readlane(Me, kGroups - 1), R);
                break;
            }
            const int s = first_lane(bal);
            if (s > from) v = val_of(__builtin_amdgcn_readlane(Me, s - 1), R);
            // the group's 64 real adds (elements past the row are 0), every lane alike; if the
            // draw is reached, again with lane j keeping the sum after element j
            const int xb = (int)chain_elem(xs[slot][s * kGroup + lane], chain, ri.sum);
            const float v0 = v;
#pragma unroll
            for (int j = 0; j < kGroup; ++j) v = __fadd_rn(v, __int_as_float(__builtin_amdgcn_readlane(xb, j)));
            if (r <= v) {
                float c = v0, mine = 0.0f;
#pragma unroll
                for (int j = 0; j < kGroup; ++j) {
                    c = __fadd_rn(c, __int_as_float(__builtin_amdgcn_readlane(xb, j)));
                    mine = lane == j ? c : mine;
                }
                found = base + s * kGroup + first_lane(__ballot(r <= mine));
                break;
            }
            from = s + 1;
        }
        ++q;
    }
    if (lane == 0) {
        if (chain) tokens[b] = found >= 0 ? found : n - 1;
        else rows[b].sum = v;
    }
}

// grid (batch), one wave: sample_greedy from the sub-chunk statistics: the first maximum, 0
// when logits[0] is NaN
__global__ __launch_bounds__(kWave) void smp_greedy(const SubStat *__restrict__ stats, int nsub,
                                                    int *__restrict__ tokens) {
    const SubStat *st = stats + (size_t)blockIdx.x * nsub;
    float bv = -INFINITY;
    int bi = -1;
    for (int q = threadIdx.x; q < nsub; q += kWave)
        if (better(st[q].max, st[q].arg, bv, bi)) {
            bv = st[q].max;
            bi = st[q].arg;
        }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
        const float ov = __shfl_xor(bv, off, kWave);
        const int oi = __shfl_xor(bi, off, kWave);
        if (better(ov, oi, bv, bi)) {
            bv = ov;
            bi = oi;
        }
    }
    if (threadIdx.x == 0) tokens[blockIdx.x] = st[0].nan0 || bi < 0 ? 0 : bi;
}

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

int subs_of(int n) { return (n + kSub - 1) / kSub; }

}  // namespace

size_t sample_workspace_bytes(int n, int batch) {
    const size_t cells = (size_t)subs_of(n) * batch;
    return align256(cells * sizeof(SubStat)) + align256(cells * sizeof(SubMaps)) +
           align256(cells * kGroups * sizeof(SubMaps)) + align256(cells * sizeof(int)) +
           align256((size_t)batch * sizeof(RowInfo));
}

bool sample_supported(int n, int batch) { return n > 0 && batch > 0 && subs_of(n) <= kMaxSubs; }

int launch_sample(const float *logits, int n, int batch, size_t ld, float temperature, float *w, size_t ldw,
                  const float *draws, const int *d_step, int *tokens, void *ws, hipStream_t s) {
    if (!sample_supported(n, batch)) {
        set_error("sampling supports 1..%d logits per row", kMaxSubs * kSub);
        return -1;
    }
    const int nsub = subs_of(n);
    const size_t cells = (size_t)nsub * batch;
    char *p = static_cast<char *>(ws);
    auto *stats = reinterpret_cast<SubStat *>(p);
    p += align256(cells * sizeof(SubStat));
    auto *maps = reinterpret_cast<SubMaps *>(p);       // of one chain, then of the other
    p += align256(cells * sizeof(SubMaps));
    auto *gmaps = reinterpret_cast<SubMaps *>(p);
    p += align256(cells * kGroups * sizeof(SubMaps));
    auto *cross = reinterpret_cast<int *>(p);
    p += align256(cells * sizeof(int));
    auto *rows = reinterpret_cast<RowInfo *>(p);
    const dim3 grid(nsub, batch);
    if (temperature <= 0.0f) {
        hipLaunchKernelGGL(smp_stats, grid, dim3(kThreads), 0, s, logits, n, ld, 1.0f, 0, stats);
        if (!hip_ok(hipGetLastError(), "sample stats launch")) return -1;
        hipLaunchKernelGGL(smp_greedy, dim3(batch), dim3(kWave), 0, s, stats, nsub, tokens);
        return hip_ok(hipGetLastError(), "sample greedy launch") ? 0 : -1;
    }
    // vec_scale skips s == 1.0f; a product with 1.0f changes no value either way. A NaN
    // temperature (not scaled there) makes every weight NaN either way: token n - 1.
    const float inv_t = 1.0f / temperature;
    const int scale = inv_t != 1.0f;
    hipLaunchKernelGGL(smp_stats, grid, dim3(kThreads), 0, s, logits, n, ld, inv_t, scale, stats);
    if (!hip_ok(hipGetLastError(), "sample stats launch")) return -1;
    hipLaunchKernelGGL(smp_weights, grid, dim3(kThreads), 0, s, logits, n, ld, inv_t, scale, temperature, w, ldw,
                       stats, rows);
    if (!hip_ok(hipGetLastError(), "sample weights launch")) return -1;
    auto walk = nsub <= kShortSubs ? smp_walk<kShortSubs, kShortSubs> : smp_walk<kMaxSubs, kSlots>;
    for (int chain = 0; chain < 2; ++chain) {
        hipLaunchKernelGGL(smp_maps, grid, dim3(kThreads), 0, s, w, n, ldw, chain, stats, rows, maps, gmaps, cross);
        if (!hip_ok(hipGetLastError(), "sample maps launch")) return -1;
        hipLaunchKernelGGL(walk, dim3(batch), dim3(kThreads), 0, s, w, n, ldw, chain, nsub, maps, gmaps, cross, rows, draws,
                           d_step, batch, tokens);
        if (!hip_ok(hipGetLastError(), "sample walk launch")) return -1;
    }
    return 0;
}

}  // namespace sapphire
