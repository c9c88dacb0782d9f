// quantize.hip - the producer of Q4_0 / Q8_0 weights: F32 / BF16 rows [M][K] into the
// reference's block arrays [M][ceil(K/32)] (include/kernels.h:29-38), elements past K in the
// last block of a row taken as zeros.
//
// The reference has no quantizer (it only reads blocks: tensor.c:108-110,
// safetensors_reader.c:406-414); its block structs are ggml's, and this follows ggml's
// published reference quantizer (quantize_row_q8_0_ref / quantize_row_q4_0_ref) with the
// reference's fp32 scale and its Q4_0 nibble order (element 2j in the low nibble of byte j,
// 2j+1 in the high nibble, q4_0_avx.c:61-66):
//   Q8_0: amax = max|x|; d = amax / 127; id = d ? 1/d : 0; q = roundf(x * id).
//   Q4_0: max = the first x of largest |x| (+0 when all are zero); d = max / -8;
//         id = d ? 1/d : 0; q = min(15, trunc(x * id + 8.5)).
// Each product and sum is rounded on its own (the library is built without contraction) and
// divisions are correctly rounded. Inputs must be finite; a block whose scale is subnormal
// (1/d overflows) saturates infinite products and codes NaN ones (0 * inf) as zero.
//
// The codes are a few operations per element: the block's largest and smallest value give its
// maximum and (Q4_0) the sign of the first element that has it, unless both signs do; roundings
// are conversions, their saturation covering the clamps. What those forms get wrong (a NaN or
// infinite element, a scale whose reciprocal overflows) goes through the plain ones, a wave at a
// time. Before, with the index of the first maximum tracked and every code clamped by compares,
// the arithmetic alone took about as long as the memory (262144 x 640 BF16 to Q4_0 110 us, now 98;
// 262144 x 1151, rows starting anywhere, 349 us with single-element loads, now 177). With the bytes
// stored through LDS instead of a dword per lane they take 90 and 155 us, 4.9-5.1 TB/s, the rate of
// a device copy.
//
// Layout of the work: four lanes per block, lane l holding elements 8l..8l+7 (two 16-byte
// fp32 loads or one 16-byte bf16 load, consecutive lanes on consecutive bytes; rows that start
// anywhere by the same loads, unaligned); the block's
// maximum goes through two DPP steps inside the quad. Each lane loads 64 or 128 bytes of source
// (4 fp32 or 8 bf16 blocks) before it quantizes any of them; a wave's blocks are consecutive, and
// their bytes go out through LDS, 16 per lane.
#include <algorithm>

#include "internal.h"
#include "lanes.h"

namespace sapphire {

namespace {

constexpr int kQThreads = 256, kWave = 64;
constexpr int kLanes = 4;   // lanes per block, eight elements each
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

template <int CTRL>
__device__ __forceinline__ int dpp_int(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}

// max / min over the 4 lanes of a quad (quad_perm [1,0,3,2], then [2,3,0,1])
__device__ __forceinline__ float max4(float v) {
    v = fmaxf(v, lanes::dpp_mov<0xB1>(v));
    return fmaxf(v, lanes::dpp_mov<0x4E>(v));
}
__device__ __forceinline__ float min4(float v) {
    v = fminf(v, lanes::dpp_mov<0xB1>(v));
    return fminf(v, lanes::dpp_mov<0x4E>(v));
}
__device__ __forceinline__ int min4(int v) {
    v = min(v, dpp_int<0xB1>(v));
    return min(v, dpp_int<0x4E>(v));
}

// Integer codes of the rounded values: ggml's conversions for blocks of normal scale; for a
// subnormal scale (1/d overflows) an infinite product saturates and a NaN one (0 * inf)
// gives the code of zero.
__device__ __forceinline__ int q8_code(float v) {
    return v != v ? 0 : v > 127.0f ? 127 : v < -127.0f ? -127 : (int)v;
}
__device__ __forceinline__ int q4_code(float v) { return v != v ? 8 : v > 15.0f ? 15 : v < 0.0f ? 0 : (int)v; }

// How a lane reads its eight elements: 16-byte aligned (K % 8 == 0 and an aligned source), at any
// alignment (K >= 8), or one by one.
enum Access { kAligned = 0, kUnaligned = 1, kSingle = 2 };

// Elements e0..e0+7 of a row (zeros past K), without branches around the loads: the eight are
// loaded at an address clamped into the row and zeroed (kUnaligned: shifted into place) past it.
template <int SRC, int ACC>
__device__ __forceinline__ void load8(const void *__restrict__ src, size_t base, int e0, int K, float (&x)[8]) {
    const bool in = e0 < K;
    if constexpr (ACC != kSingle) {
        const int at = ACC == kAligned ? (in ? e0 : 0) : min(e0, K - 8);
        const size_t off = base + at;
        float v[8];
        if constexpr (SRC == DT_F32) {
            const float *p = static_cast<const float *>(src) + off;
            f32x4 a, b;
            if constexpr (ACC == kAligned) {
                a = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(p));
                b = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(p) + 1);
            } else {
                __builtin_memcpy(&a, p, 16);
                __builtin_memcpy(&b, p + 4, 16);
            }
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
            v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        } else {
            const uint16_t *p = static_cast<const uint16_t *>(src) + off;
            u32x4 t;
            if constexpr (ACC == kAligned) t = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p));
            else __builtin_memcpy(&t, p, 16);
            const uint32_t w[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[2 * i] = __uint_as_float(w[i] << 16);
                v[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
            }
        }
        if constexpr (ACC == kAligned) {
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = in ? v[i] : 0.f;
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = v[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int e = e0 + i;
            const size_t at = base + (size_t)min(e, K - 1);
            float v;
            if constexpr (SRC == DT_F32) v = static_cast<const float *>(src)[at];
            else v = __uint_as_float((uint32_t) static_cast<const uint16_t *>(src)[at] << 16);
            x[i] = e < K ? v : 0.f;
        }
    }
}

// kUnaligned: the eight elements loaded at min(e0, K - 8) moved down by what was clamped (8 and
// more: all zeros), for the lanes at a row's end.
__device__ __forceinline__ void shift_into_place(int e0, int K, float (&x)[8]) {
    const int sh = e0 - min(e0, K - 8);
    if (!__any(sh != 0)) return;
#pragma unroll
    for (int bit = 4; bit >= 1; bit >>= 1)
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = (sh & bit) ? (i + bit < 8 ? x[i + bit] : 0.f) : x[i];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = sh >= 8 ? 0.f : x[i];
}

// roundf(v) as an integer for |v| < 2^22: adding the float below 1/2 towards v's sign and
// truncating rounds halves away from zero and everything else to the nearest.
__device__ __forceinline__ int round_away(float v) { return (int)__fadd_rn(v, copysignf(0x1.fffffep-2f, v)); }

// Between a wave's LDS stores and its other lanes' loads of them (and the next trip's stores): the
// hardware keeps a wave's LDS accesses in order, the compiler reasons per lane and is told here.
// No instruction of it is left in the kernel.
__device__ __forceinline__ void wave_handover() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// DENSE: K % 32 == 0, so block b starts at element 32b. Otherwise row and block come from a
// 32-bit division (the launcher keeps such matrices below 2^31 blocks).
template <int DST, int SRC, int ACC, bool DENSE, int U>
__global__ __launch_bounds__(kQThreads) void quantize_kernel(const void *__restrict__ src, int K, int nb,
                                                            long nblocks, uint8_t *__restrict__ dst) {
    constexpr int BB = DST == DT_Q4_0 ? 20 : 36;
    constexpr int kRun = U * kWave / kLanes;           // consecutive blocks of a wave's trip
    constexpr int kWords = kRun * BB / 4;
    __shared__ __attribute__((aligned(16))) uint32_t stage[kQThreads / kWave][kWords];
    const int lq = threadIdx.x & (kLanes - 1), lane = threadIdx.x & (kWave - 1);
    uint32_t *mine = stage[threadIdx.x / kWave];
    const long wave = ((long)blockIdx.x * kQThreads + threadIdx.x) / kWave;
    const long stride = (long)gridDim.x * (kQThreads / kWave) * kRun;
    const bool wide = (reinterpret_cast<uintptr_t>(dst) & 15) == 0;   // runs are multiples of 16 bytes
    for (long r0 = wave * kRun; r0 < nblocks; r0 += stride) {
        const long b0 = r0 + lane / kLanes;
        // every lane loads U blocks (past the end: the last block again), then quantizes them
        float x[U][8];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const long b = min(b0 + u * (kWave / kLanes), nblocks - 1);
            if constexpr (DENSE) {
                load8<SRC, ACC>(src, (size_t)b * 32, lq * 8, 32, x[u]);
            } else {
                const uint32_t row = (uint32_t)b / (uint32_t)nb;
                const int blk = (int)((uint32_t)b - row * (uint32_t)nb);
                load8<SRC, ACC>(src, (size_t)row * K, blk * 32 + lq * 8, K, x[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const long b = b0 + u * (kWave / kLanes);
            uint32_t *out = mine + (u * (kWave / kLanes) + lane / kLanes) * (BB / 4);
            if constexpr (ACC == kUnaligned) {
                // the row's elements sit in row order in the row's blocks
                const uint32_t bb = (uint32_t)min(b, nblocks - 1);
                if constexpr (!DENSE) shift_into_place((int)(bb % (uint32_t)nb) * 32 + lq * 8, K, x[u]);
            }
            float top = x[u][0], low = x[u][0];
            bool nan = false;
#pragma unroll
            for (int i = 1; i < 8; ++i) {
                top = fmaxf(top, x[u][i]);
                low = fminf(low, x[u][i]);
            }
#pragma unroll
            for (int i = 0; i < 8; i += 2) nan |= __builtin_isunordered(x[u][i], x[u][i + 1]);
            top = max4(top);
            low = min4(low);
            const float amax = fmaxf(fmaxf(top, -low), 0.f);   // NaN elements never count
            float d, id;
            if constexpr (DST == DT_Q8_0) {
                d = amax / 127.0f;
                id = d != 0.f ? 1.0f / d : 0.f;
            } else {
                float mx = top > -low ? amax : -amax;
                // both signs reach the maximum: the first element (in block order) that does
                if (__any(top == -low)) {
                    int key = 0x7FFFFFFF;
#pragma unroll
                    for (int i = 7; i >= 0; --i)
                        key = fabsf(x[u][i]) == amax ? ((lq * 8 + i) << 1) | (int)(__float_as_uint(x[u][i]) >> 31) : key;
                    key = min4(key);
                    mx = top == -low ? ((key & 1) ? -amax : amax) : mx;
                }
                mx = amax == 0.f ? 0.f : mx;
                d = mx / -8.0f;
                id = d != 0.f ? 1.0f / d : 0.f;
            }
            // |id| overflows or the maximum is infinite (then id is 0): infinite and NaN products
            const bool plain = __any(nan || !(amax < INFINITY) || !(fabsf(id) < INFINITY)) != 0;
            if constexpr (DST == DT_Q8_0) {
                uint32_t w[2] = {0u, 0u};
                if (!plain) {
#pragma unroll
                    for (int i = 0; i < 8; i += 4) {
                        uint32_t q[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) q[e] = (uint32_t)round_away(__fmul_rn(x[u][i + e], id));
                        w[i >> 2] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(q[3], q[2], 0x0C0C0400u),
                                                          __builtin_amdgcn_perm(q[1], q[0], 0x0C0C0400u), 0x05040100u);
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        w[i >> 2] |= (uint32_t)(q8_code(roundf(__fmul_rn(x[u][i], id))) & 0xFF) << (8 * (i & 3));
                }
                out[1 + 2 * lq] = w[0];
                out[2 + 2 * lq] = w[1];
            } else {
                uint32_t w = 0;
                if (!plain) {
                    // every value is at least 0.5: only the upper clamp is left
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        w |= min((uint32_t)__fadd_rn(__fmul_rn(x[u][i], id), 8.5f), 15u) << (4 * i);
                } else {
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        w |= (uint32_t)q4_code(__fadd_rn(__fmul_rn(x[u][i], id), 8.5f)) << (4 * i);
                }
                out[1 + lq] = w;
            }
            if (lq == 0) out[0] = __float_as_uint(d);
        }
        wave_handover();
        // the run's bytes, contiguous, by whole lanes
        uint32_t *o = reinterpret_cast<uint32_t *>(dst + (size_t)r0 * BB);
        if (wide && r0 + kRun <= nblocks) {
#pragma unroll
            for (int k = 0; k < (kWords / 4 + kWave - 1) / kWave; ++k)
                if (k * kWave + lane < kWords / 4)
                    reinterpret_cast<u32x4 *>(o)[k * kWave + lane] = reinterpret_cast<const u32x4 *>(mine)[k * kWave + lane];
        } else {
            const int words = (int)min((long)kRun, nblocks - r0) * (BB / 4);
            for (int k = lane; k < words; k += kWave) o[k] = mine[k];
        }
        wave_handover();
    }
}

int device_cus_q() {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
        return 256;
    return n;
}

template <int DST, int SRC>
int launch_typed(const void *src, int M, int K, void *dst, hipStream_t st) {
    constexpr int U = SRC == DT_F32 ? 4 : 8;   // 128 bytes of source per lane in flight
    const int nb = (K + 31) / 32;
    const long nblocks = (long)M * nb;
    const bool vec = K % 8 == 0 && (reinterpret_cast<uintptr_t>(src) & 15) == 0;
    if (K % 32 != 0 && nblocks >= (1L << 31)) {
        set_error("quantize: rows of a partial block need fewer than 2^31 blocks per call");
        return -1;
    }
    const long per_wg = (long)(kQThreads / kLanes) * U;
    static int cus = device_cus_q();
    const long grid = std::max(1L, std::min((nblocks + per_wg - 1) / per_wg, 8L * cus));
    uint8_t *d = static_cast<uint8_t *>(dst);
    const dim3 g((unsigned)grid), t(kQThreads);
    if (vec && K % 32 == 0)
        hipLaunchKernelGGL((quantize_kernel<DST, SRC, kAligned, true, U>), g, t, 0, st, src, K, nb, nblocks, d);
    else if (vec)
        hipLaunchKernelGGL((quantize_kernel<DST, SRC, kAligned, false, U>), g, t, 0, st, src, K, nb, nblocks, d);
    else if (K % 32 == 0)
        hipLaunchKernelGGL((quantize_kernel<DST, SRC, kUnaligned, true, U>), g, t, 0, st, src, K, nb, nblocks, d);
    else if (K >= 8)
        hipLaunchKernelGGL((quantize_kernel<DST, SRC, kUnaligned, false, U>), g, t, 0, st, src, K, nb, nblocks, d);
    else
        hipLaunchKernelGGL((quantize_kernel<DST, SRC, kSingle, false, U>), g, t, 0, st, src, K, nb, nblocks, d);
    return 0;
}

}  // namespace

int launch_quantize(int dst_dtype, int src_dtype, const void *src, int M, int K, void *blocks, hipStream_t st) {
    if ((dst_dtype != DT_Q4_0 && dst_dtype != DT_Q8_0) || (src_dtype != DT_F32 && src_dtype != DT_BF16) || !src ||
        !blocks || M <= 0 || K <= 0) {
        set_error("quantize: source must be F32 or BF16, destination Q4_0 or Q8_0, with positive shape");
        return -1;
    }
    if (reinterpret_cast<uintptr_t>(blocks) & 3) {
        set_error("quantize: the block array must be 4-byte aligned");
        return -1;
    }
    int rc;
    if (dst_dtype == DT_Q4_0 && src_dtype == DT_F32) rc = launch_typed<DT_Q4_0, DT_F32>(src, M, K, blocks, st);
    else if (dst_dtype == DT_Q4_0) rc = launch_typed<DT_Q4_0, DT_BF16>(src, M, K, blocks, st);
    else if (src_dtype == DT_F32) rc = launch_typed<DT_Q8_0, DT_F32>(src, M, K, blocks, st);
    else rc = launch_typed<DT_Q8_0, DT_BF16>(src, M, K, blocks, st);
    if (rc != 0) return -1;
    return hip_ok(hipGetLastError(), "quantize launch") ? 0 : -1;
}

}  // namespace sapphire
