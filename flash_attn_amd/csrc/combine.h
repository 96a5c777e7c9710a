// Merging the partial results of a split key range: the row-wise merge itself, used by combine_kernel and by split
// kernels that merge their own results, and what the latter need to agree on who does it.
#pragma once
#include "common.h"

namespace fa {

template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
// sum over the LPK consecutive lanes that share a key; every lane of the group ends with the total
template <int LPK>
__device__ __forceinline__ float group_sum(float v)
{
    v += dpp_mov<0xB1>(v);                          // quad_perm [1,0,3,2]
    v += dpp_mov<0x4E>(v);                          // quad_perm [2,3,0,1]
    if constexpr (LPK >= 8) v += dpp_mov<0x141>(v);   // row_half_mirror
    if constexpr (LPK >= 16) v += dpp_mov<0x140>(v);  // row_mirror
    return v;
}

// Reductions over the 64 lanes of a wave without LDS: DPP inside the rows of 16 lanes, v_permlane32_swap between the
// halves, v_readlane for the last two rows; the result is wave-uniform.
__device__ __forceinline__ float wave_sum(float v)
{
    v = xhalf_sum(group_sum<16>(v));  // lanes of rows r and r ^ 2 now hold the total of both rows
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0)) +
           __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
}
__device__ __forceinline__ float wave_max(float v)
{
    v = fmaxf(v, dpp_mov<0xB1>(v));
    v = fmaxf(v, dpp_mov<0x4E>(v));
    v = fmaxf(v, dpp_mov<0x141>(v));
    v = fmaxf(v, dpp_mov<0x140>(v));
    v = xhalf_max(v);
    return fmaxf(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0)),
                 __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16)));
}

// Split launches that merge their own results (a.counters): the S work-groups that share a few rows store their partial
// results, count themselves in at one counter, and the last one to arrive merges the rows, which saves the combine launch
// behind the split launch and the gap between the two.  Nobody waits for anybody.  The work-groups run on different XCDs
// with an L2 each, so partial results are stored and loaded at agent scope (written through, read past the L2): a
// cache write-back and invalidation per work-group would do as well and costs more than a few KiB of such accesses.
// The last one leaves the counter at zero for the next launch on the stream.
// Two launches -> one, GPU time per call: decode B1 H4 Nk487 d128 in 4 splits 7.1 -> 5.5 us, B3 H12 Nk1152 d64 in 5 splits
// 7.8 -> 6.6, B1 H32 Nk4096 d128 in 8 splits 15.4 -> 14.7 (the arrival costs a store, an atomic and a load from memory in a
// row, about 2 us).  Of the tiled kernels those for few rows do it, for up to four rows in up to eight splits (rows_form_merges in fwd_kernel.h); the others
// have many rows, whose partial results, written through piece by piece, took longer than the second launch (B3 H8 H_kv1 Nk7296 d64: 9.7 -> 14.2 us).
__device__ __forceinline__ void store_partial(float* p, float v, bool shared)
{
    if (shared) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *p = v;
}
// four columns on a 16-byte boundary
__device__ __forceinline__ void store_partial4(float* p, v4f v, bool shared)
{
    if (shared) {
        union { v4f f; uint64_t u[2]; } r;
        r.f = v;
        uint64_t* const q = reinterpret_cast<uint64_t*>(p);
        __hip_atomic_store(q, r.u[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(q + 1, r.u[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        *reinterpret_cast<v4f*>(p) = v;
    }
}
// Called by every thread of the work-group, behind its last store_partial; `flag` is an LDS word nobody else uses.
__device__ __forceinline__ bool last_to_arrive(uint32_t* counter, int num_splits, int* flag)
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's stores are where the others will look
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t before = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool last = before == (uint32_t)num_splits - 1u;
        if (last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *flag = last ? 1 : 0;
    }
    __syncthreads();
    return *flag != 0;
}

// kHere: the partial results come from work-groups of the same launch (see above).
template <bool kHere>
__device__ __forceinline__ float load_partial(const float* p)
{
    if constexpr (kHere) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return *p;
}
template <bool kHere>
__device__ __forceinline__ float4 load_partial4(const float* p)
{
    if constexpr (kHere) {
        union { uint64_t u[2]; float4 f; } r;
        const uint64_t* q = reinterpret_cast<const uint64_t*>(p);
        r.u[0] = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        r.u[1] = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return r.f;
    }
    return *reinterpret_cast<const float4*>(p);
}
// One query row: LSE = logsumexp_s LSE_s, O = sum_s exp(LSE_s - LSE) O_s
// (same value as m = max M_s, l = sum e^{M_s-m} L_s, O = sum (L_s e^{M_s-m} / l) O_s of splitkv.h:359-397), by W waves
// that call this together (W = 1, or all four of a work-group) and take every W-th pair of splits each, the even one on
// the lower half of the wave.  What bounds it is the latency of the partial rows, of which a half-wave has U in flight:
// up to kSplitsPerWave splits are one batch of one wave, more are spread over four (grouped decode B3 H8 H_kv1 Nk7296
// d64, 57 splits: 9.7 -> 7.8 us).
// With d % 8 == 0 a lane holds four consecutive columns, and the first partial rows are requested before the
// log-sum-exp values they will be weighted with.  Every wave works out the weights of all splits for itself (s_w,
// FLASH_MAX_SPLITS_K floats of LDS of its own).
constexpr int kSplitsPerWave = 16;
// rows = rows that one work-group merges (1 behind a launch of its own): a wave each, batch after batch, or all waves one
// row after the other, whichever takes fewer batches in a row
inline int combine_waves_for(int num_splits, int rows)
{
    const int one = (num_splits + kSplitsPerWave - 1) / kSplitsPerWave * ((rows + 3) / 4);
    const int four = (num_splits + 4 * kSplitsPerWave - 1) / (4 * kSplitsPerWave) * rows;
    return four < one ? 4 : 1;
}
constexpr int kCombineLds = 4 * FLASH_MAX_SPLITS_K + 4 * 128;  // floats: weights of four waves, then their sums over d <= 128
template <bool kHere, int W>
__device__ __forceinline__ void combine_row(const float* __restrict__ O_partial, const float* __restrict__ LSE_partial,
                                            half_t* __restrict__ O, float* __restrict__ LSE, int bh, int i, int Nq, int d, int S,
                                            float* lds)
{
    const int lane = threadIdx.x & 63;
    const int wave = wave_uniform(threadIdx.x >> 6);
    const int part = W == 1 ? 0 : wave;
    float* const s_w = lds + wave * FLASH_MAX_SPLITS_K;
    float* const s_o = lds + 4 * FLASH_MAX_SPLITS_K;
    const float* lp = LSE_partial + (size_t)bh * S * Nq + i;  // stride Nq between splits
    const size_t sstride = (size_t)Nq * d;                     // floats between the partial rows of two splits
    const float* op = O_partial + ((size_t)bh * S * Nq + i) * d;
    const bool vec = (d & 7) == 0;  // rows of the partials and of O are 16-byte aligned (the host checks the bases)
    constexpr int U = kSplitsPerWave / 2;
    const int c4 = (lane & 31) * 4, grp = 2 * part + (lane >> 5);
    const bool act = c4 < d;
    auto request = [&](int s0, float4 (&v)[U]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = s0 + 2 * W * u;
            v[u] = (act && s < S) ? load_partial4<kHere>(op + s * sstride + c4) : float4{0.f, 0.f, 0.f, 0.f};
        }
    };
    float4 pre[U];
    if (vec) request(grp, pre);
    // (at most two splits per lane: FLASH_MAX_SPLITS_K is 128)
    const float l0 = lane < S ? load_partial<kHere>(lp + (size_t)lane * Nq) : -INFINITY;
    const float l1 = lane + 64 < S ? load_partial<kHere>(lp + (size_t)(lane + 64) * Nq) : -INFINITY;
    const float mx = wave_max(fmaxf(l0, l1));
    const float mu = (mx == -INFINITY) ? 0.0f : mx;
    const float w0 = __expf(l0 - mu), w1 = __expf(l1 - mu);
    if (lane < S) s_w[lane] = w0;
    if (lane + 64 < S) s_w[lane + 64] = w1;
    const float sum = wave_sum(w0 + w1);  // (lanes past S add exp(-inf))
    const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
    if (part == 0 && lane == 0) LSE[(size_t)bh * Nq + i] = sum > 0.0f ? mx + __logf(sum) : -INFINITY;
    half_t* const orow = O + ((size_t)bh * Nq + i) * d;
    if (vec) {
        float4 acc = {0.f, 0.f, 0.f, 0.f};
        auto add = [&](int s0, const float4 (&v)[U]) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int s = s0 + 2 * W * u;
                const float w = s < S ? s_w[s] : 0.0f;
                acc.x += w * v[u].x, acc.y += w * v[u].y, acc.z += w * v[u].z, acc.w += w * v[u].w;
            }
        };
        add(grp, pre);
        for (int s0 = grp + 2 * W * U; s0 < S; s0 += 2 * W * U) {  // (one wave: never more than one batch)
            float4 nxt[U];
            request(s0, nxt);
            __builtin_amdgcn_sched_barrier(0);
            add(s0, nxt);
        }
        acc.x = xhalf_sum(acc.x), acc.y = xhalf_sum(acc.y), acc.z = xhalf_sum(acc.z), acc.w = xhalf_sum(acc.w);
        if constexpr (W > 1) {
            if (lane < 32) *reinterpret_cast<float4*>(s_o + part * 128 + c4) = acc;
            __syncthreads();
            if (part == 0) {
#pragma unroll
                for (int w = 1; w < W; ++w) {
                    const float4 v = *reinterpret_cast<const float4*>(s_o + w * 128 + c4);
                    acc.x += v.x, acc.y += v.y, acc.z += v.z, acc.w += v.w;
                }
            }
            __syncthreads();  // (the next row of a caller that merges several)
        }
        if (act && part == 0 && lane < 32) {
            union { v2h h[2]; uint2 u; } r;
            r.h[0] = pack_f16(acc.x * inv, acc.y * inv);
            r.h[1] = pack_f16(acc.z * inv, acc.w * inv);
            *reinterpret_cast<uint2*>(orow + c4) = r.u;
        }
    } else {
        // rows at any alignment: column by column, the columns of a row spread over the lanes of all waves
        for (int dc = 64 * part + lane; dc < d; dc += 64 * W) {
            float o = 0.0f;
            for (int s0 = 0; s0 < S; s0 += U) {  // U requests at a time, added in order
                float v[U];
#pragma unroll
                for (int u = 0; u < U; ++u) v[u] = s0 + u < S ? load_partial<kHere>(op + (s0 + u) * sstride + dc) : 0.0f;
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < U; ++u) o += (s0 + u < S ? s_w[s0 + u] : 0.0f) * v[u];
            }
            orow[dc] = (half_t)(o * inv);
        }
    }
}

}  // namespace fa
