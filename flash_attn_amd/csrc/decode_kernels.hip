// Split-KV decode (one query row per head), split combine, and the stand-alone dropout keep-mask kernel.
//
// decode_split_kernel and decode_stream_kernel (the same with longer arguments) replace forward_kernel_splitkv (src/flash_forward_splitkv.h:14-344)
// for Nq == 1, where the reference's 128-row MMA tile would waste 127 of 128 rows: the work is a pure stream over K and V, bound by HBM.
//   * one work-group per (head slice, split) -- per (G query heads of one K/V head, split) under grouped-query
//     attention, so that K and V are streamed once per K/V head; its 4 waves take blocks of the split's keys in turn
//   * a key row is spread over LPK lanes (16 bytes each), so one wave instruction reads 1 KiB of consecutive bytes
//   * q.k: v_dot2_f32_f16 per lane, then a DPP butterfly over the LPK lanes of the key (no LDS, no shuffles)
//   * online softmax per key group; p * V accumulated in fp32 per lane (8 head-dim columns per lane)
//   * key groups and waves are merged once at the end through LDS; partial O (normalised, fp32) and
//     LSE_s = m_s + log l_s go to the workspace (reference: O_tmp, M, L; src/flash_forward_splitkv.h:313-338)
// combine_kernel replaces forward_kernel_splitkv_combine (src/flash_forward_splitkv.h:347-399) with one wave per
// query row and coalesced reads of the partials (the reference uses one thread per row).
#include "combine.h"
#include "common.h"
#include "decode_kernels.h"

namespace fa {

// Arguments of the decode kernel.  What every address depends on has words of its own where there is room, without ALiBi: cut out of
// `shifts`, d and num_splits cost each launch 0.04 us of GPU time that nothing hides.  112 bytes are what the host passes on fastest
// (see Packed in common.h), but launches of a busy GPU follow each other 0.15-0.2 us faster where the arguments take more than 128
// (120 and 128 like 112; 192, 256 and 272 alike): so launches that the GPU bounds, from 4 MiB of K and V on, get 192.  112 / 192 bytes: 2 MiB B1
// H8 Nk512 d128 5.48 / 5.56 us, 0.3 MiB B1 H4 Nk300 d64 5.41 / 5.53, 4 MiB B1 H16 Nk512 d128 5.90 / 5.90, 6 MiB Nk768 6.55 / 6.42, 10 MiB B4 H8 Nk640
// 6.70 / 6.48, 7.8 MiB B2 H8 Nk2000 d64 7.75 / 7.74, 9.4 MiB B1 H32 Nk1200 d64 6.55 / 6.36, Nk2048 d128 9.94 / 9.75, Nk4096 d128 14.59 / 14.41.
struct DecodeOwn {
    int d, num_splits;
};
struct DecodeHeads {
    int H;
    uint32_t mul_heads;
};
template <bool kAlibi>
struct DecodeArgs {
    uint32_t mul_slices, mul_kv;
    uint32_t shifts;  // of by_slices, by_kv_group, by_heads: five bits each; d, num_splits: eight bits each; bit 31: combine_waves is 4
    int slices;       // groups of G query heads
    std::conditional_t<kAlibi, DecodeHeads, DecodeOwn> own;
    int Nk, wl, keys_per_split;
    float scale_log2;
    const half_t *Q, *K, *V;
    half_t* O;
    float *LSE, *O_partial, *LSE_partial;
    uint32_t* counters;
    const float* alibi;
};
template <bool kAlibi>
struct DecodeStreamArgs : DecodeArgs<kAlibi> {
    uint32_t unused[20];
};
static_assert(sizeof(DecodeStreamArgs<true>) == 192 && sizeof(DecodeStreamArgs<false>) == 192, "more than 128 bytes");
static_assert(sizeof(DecodeArgs<true>) <= kCheapArgs && sizeof(DecodeArgs<false>) <= kCheapArgs, "cheap launches");
template <bool kAlibi>
static DecodeArgs<kAlibi> decode_args(const FwdArgs& a, int slices)
{
    DecodeArgs<kAlibi> p{};
    p.mul_slices = a.by_slices.mul, p.mul_kv = a.by_kv_group.mul, p.slices = slices;
    p.shifts = a.by_slices.shift | a.by_kv_group.shift << 5 | a.by_heads.shift << 10 | (uint32_t)a.d << 15 | (uint32_t)a.num_splits << 23 |
               (a.combine_waves == 4 ? 1u << 31 : 0u);
    if constexpr (kAlibi) p.own = {a.H, a.by_heads.mul};
    else p.own = {a.d, a.num_splits};
    p.Nk = a.Nk, p.wl = a.wl, p.keys_per_split = a.keys_per_split, p.scale_log2 = a.scale_log2;
    p.Q = a.Q, p.K = a.K, p.V = a.V, p.O = a.O, p.LSE = a.LSE, p.O_partial = a.O_partial, p.LSE_partial = a.LSE_partial;
    p.counters = a.counters, p.alibi = a.alibi;
    return p;
}
template <bool kAlibi>
__device__ __forceinline__ FwdArgs unpacked(const DecodeArgs<kAlibi>& p)
{
    FwdArgs a{};
    auto div = [&](uint32_t mul, int k) __attribute__((always_inline)) { return FastDiv{mul, p.shifts >> (5 * k) & 31u}; };
    a.by_slices = div(p.mul_slices, 0), a.by_kv_group = div(p.mul_kv, 1);
    a.combine_waves = p.shifts >> 31 ? 4 : 1;
    if constexpr (kAlibi) {
        a.d = p.shifts >> 15 & 255u, a.num_splits = p.shifts >> 23 & 255u;
        a.H = p.own.H, a.by_heads = div(p.own.mul_heads, 2), a.alibi = p.alibi;
    } else {
        a.d = p.own.d, a.num_splits = p.own.num_splits;
    }
    a.Nk = p.Nk, a.wl = p.wl, a.keys_per_split = p.keys_per_split, a.scale_log2 = p.scale_log2;
    a.Q = p.Q, a.K = p.K, a.V = p.V, a.O = p.O, a.LSE = p.LSE, a.O_partial = p.O_partial, a.LSE_partial = p.LSE_partial;
    a.counters = p.counters;
    return a;
}

// G = query heads served by one work-group: the G consecutive heads share one K/V head (grouped-query attention), so
// the K/V stream is read once for all of them.  G == 1 is the plain one-K/V-head-per-query-head case.
template <int LPK, int G, bool kAlibi>
__device__ __forceinline__ void decode_split(const DecodeArgs<kAlibi>& packed_args)
{
    const FwdArgs a = unpacked(packed_args);
    constexpr int KPI = 64 / LPK;      // keys per wave instruction
    constexpr int U = G > 2 ? 4 : 8;   // load instructions in flight per tensor
    constexpr int KB = U * KPI;        // keys per wave block
    constexpr int NG = 4 * KPI;        // key groups per work-group
    constexpr int DB = LPK * 8;        // head-dim bucket
    __shared__ __attribute__((aligned(16))) float s_acc[NG][DB];
    __shared__ float s_m[NG], s_l[NG];
    __shared__ int s_last;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = wave_uniform(tid >> 6);
    const int c = lane % LPK;
    const int kg = lane / LPK;
    const int split = a.by_slices.quotient(blockIdx.x);
    const int bh0 = (blockIdx.x - split * packed_args.slices) * G;  // first of the G query slices of this work-group
    const int d = a.d, Nk = a.Nk;
    // Rows of any length from eight elements on, at any 2-byte alignment: a lane behind the row's whole chunks works
    // on the row's last 16 bytes, columns d - 8 ... d - 1 (no load leaves the row), with q zeroed where the lane before
    // has covered a column already; lanes past the row do the same with q = 0.
    const int col = 8 * c;
    const int colc = col + 8 <= d ? col : d - 8;

    union U8 { v4u u; v8h h; v2h p[4]; };
    U8 qv[G];
#pragma unroll
    for (int gq = 0; gq < G; ++gq)
        qv[gq].h = mask_q_chunk_anyalign(*reinterpret_cast<const v4u_anyalign*>(a.Q + (size_t)(bh0 + gq) * d + colc), col, d);

    // the single query row sits at position ii = Nk - 1 (row index i + Nk - Nq): causal / right window never cut
    const int ii = Nk - 1;
    int kstart = a.wl >= 0 ? max(0, ii - a.wl) : 0;
    int kend = Nk;
    if (a.num_splits > 1) {
        kstart = max(kstart, split * a.keys_per_split);
        kend = min(kend, (split + 1) * a.keys_per_split);
    }
    const int kvs = a.kv_slice(bh0);
    const half_t* __restrict__ Kbh = a.K + (size_t)kvs * Nk * d + colc;
    const half_t* __restrict__ Vbh = a.V + (size_t)kvs * Nk * d + colc;
    const float c2 = a.scale_log2;
    float slope2[G];
#pragma unroll
    for (int gq = 0; gq < G; ++gq) {
        slope2[gq] = 0.0f;
        if constexpr (kAlibi) slope2[gq] = a.alibi ? a.alibi[a.head(bh0 + gq)] * kLog2e : 0.0f;
    }

    float m[G], l[G];
    float acc[G][8];
#pragma unroll
    for (int gq = 0; gq < G; ++gq) {
        m[gq] = -INFINITY;
        l[gq] = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[gq][e] = 0.0f;
    }

    // The key loop is double-buffered by hand: the 2 U loads of the wave's next block (16 bytes per lane each) are issued
    // before the current block is consumed, and a scheduling fence keeps them there.  Left to the compiler the loop
    // waited for every K row before requesting the next one (eight memory round trips in series per block: a lone
    // work-group streamed 13 GB/s).
    auto load_block = [&](int kb, U8 (&kr)[U], U8 (&vr)[U]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int j = kb + i * KPI + kg;
            const size_t off = (size_t)(j < kend ? j : kend - 1) * d;
            // (non-temporal: K and V are read once; as ordinary loads they measured 5.9 instead of 6.8 TB/s)
            kr[i].u = __builtin_nontemporal_load(reinterpret_cast<const v4u_anyalign*>(Kbh + off));
        }
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int j = kb + i * KPI + kg;
            const size_t off = (size_t)(j < kend ? j : kend - 1) * d;
            vr[i].u = __builtin_nontemporal_load(reinterpret_cast<const v4u_anyalign*>(Vbh + off));
        }
    };
    auto consume = [&](int kb, const U8 (&kr)[U], const U8 (&vr)[U]) __attribute__((always_inline)) {
#pragma unroll
        for (int gq = 0; gq < G; ++gq) {
            float t[U];
            float mb = -INFINITY;
#pragma unroll
            for (int i = 0; i < U; ++i) {
                float s = 0.0f;
#pragma unroll
                for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_fdot2(qv[gq].p[e], kr[i].p[e], s, false);
                s = group_sum<LPK>(s);
                const int j = kb + i * KPI + kg;
                float tv = s * c2;
                if constexpr (kAlibi) tv -= slope2[gq] * (float)(ii - j);
                if (j >= kend) tv = -INFINITY;
                t[i] = tv;
                mb = fmaxf(mb, tv);
            }
            const float m_new = fmaxf(m[gq], mb);
            const float m_use = (m_new == -INFINITY) ? 0.0f : m_new;
            const float alpha = fast_exp2(m[gq] - m_use);
            m[gq] = m_new;
            float rs = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[gq][e] *= alpha;
#pragma unroll
            for (int i = 0; i < U; ++i) {
                const float p = fast_exp2(t[i] - m_use);
                rs += p;
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[gq][e] = __builtin_fmaf(p, (float)vr[i].h[e], acc[gq][e]);
            }
            l[gq] = l[gq] * alpha + rs;
        }
    };
    {
        U8 k0[U], v0[U], k1[U], v1[U];
        int kb = kstart + wave * KB;  // wave-uniform
        if (kb < kend) load_block(kb, k0, v0);
        while (kb < kend) {
            const int kb1 = kb + 4 * KB;
            if (kb1 < kend) load_block(kb1, k1, v1);
            __builtin_amdgcn_sched_barrier(0);
            consume(kb, k0, v0);
            if (kb1 >= kend) break;
            const int kb2 = kb1 + 4 * KB;
            if (kb2 < kend) load_block(kb2, k0, v0);
            __builtin_amdgcn_sched_barrier(0);
            consume(kb1, k1, v1);
            kb = kb2;
        }
    }

    // ---- merge the NG key groups of the work-group, one query head after the other through the same LDS buffer
    const int grp = wave * KPI + kg;
#pragma unroll
    for (int gq = 0; gq < G; ++gq) {
        if (gq > 0) __syncthreads();
#pragma unroll
        for (int e = 0; e < 8; ++e) s_acc[grp][col + e] = acc[gq][e];
        if (c == 0) {
            s_m[grp] = m[gq];
            s_l[grp] = l[gq];
        }
        __syncthreads();
        if (tid < DB) {
            const int bh = bh0 + gq;
            float M = -INFINITY;
#pragma unroll
            for (int gI = 0; gI < NG; ++gI) M = fmaxf(M, s_m[gI]);
            const float Mu = (M == -INFINITY) ? 0.0f : M;
            float L = 0.0f, o = 0.0f;
#pragma unroll
            for (int gI = 0; gI < NG; ++gI) {
                const float w = fast_exp2(s_m[gI] - Mu);
                L += w * s_l[gI];
                o += w * s_acc[gI][tid];
            }
            const float inv = L > 0.0f ? 1.0f / L : 0.0f;
            const float lse = L > 0.0f ? __builtin_fmaf(M, kLn2, fast_log2(L) * kLn2) : -INFINITY;
            // column of position tid: the eight positions behind the row's whole chunks hold columns d - 8 ... d - 1, of
            // which the first 8 - d % 8 were written by the positions before
            const int c0 = d & ~7, rem = d & 7;
            const int tcol = tid < c0 ? tid : tid - (8 - rem);
            const bool ok = tid < c0 || (rem != 0 && tid < c0 + 8 && tcol >= c0);
            if (a.num_splits > 1) {
                const size_t prow = (size_t)bh * a.num_splits + split;  // Nq == 1
                const bool here = a.counters != nullptr;
                if (ok) store_partial(a.O_partial + prow * d + tcol, o * inv, here);
                if (tid == 0) store_partial(a.LSE_partial + prow, lse, here);
            } else {
                if (ok) a.O[(size_t)bh * d + tcol] = (half_t)(o * inv);
                if (tid == 0) a.LSE[bh] = lse;
            }
        }
    }
    if (a.counters != nullptr && last_to_arrive(a.counters + bh0 / G, a.num_splits, &s_last)) {
        static_assert(NG * DB >= kCombineLds, "the merge fits the buffer of the key groups");
        float* const lds = &s_acc[0][0];
        if (a.combine_waves == 1) {
            for (int gq = wave; gq < G; gq += 4)
                combine_row<true, 1>(a.O_partial, a.LSE_partial, a.O, a.LSE, bh0 + gq, 0, 1, d, a.num_splits, lds);
        } else {
            for (int gq = 0; gq < G; ++gq)
                combine_row<true, 4>(a.O_partial, a.LSE_partial, a.O, a.LSE, bh0 + gq, 0, 1, d, a.num_splits, lds);
        }
    }
}

template <int LPK, bool kAlibi, int G>
__global__ void __launch_bounds__(256) decode_split_kernel(const DecodeArgs<kAlibi> args)
{
    decode_split<LPK, G>(args);
}
template <int LPK, bool kAlibi, int G>
__global__ void __launch_bounds__(256) decode_stream_kernel(const DecodeStreamArgs<kAlibi> args)
{
    decode_split<LPK, G, kAlibi>(args);
}

// one wave per query row, or one work-group (W = 4)
template <int W>
__global__ void __launch_bounds__(256) combine_kernel(const float* __restrict__ O_partial,
                                                      const float* __restrict__ LSE_partial, half_t* __restrict__ O,
                                                      float* __restrict__ LSE, int rows, int Nq, FastDiv by_Nq, int d, int S)
{
    __shared__ __attribute__((aligned(16))) float lds[kCombineLds];
    const int row = W == 1 ? blockIdx.x * 4 + wave_uniform(threadIdx.x >> 6) : blockIdx.x;
    if (row >= rows) return;
    const int bh = by_Nq.quotient(row);
    combine_row<false, W>(O_partial, LSE_partial, O, LSE, bh, row - bh * Nq, Nq, d, S, lds);
}

// keep[b,h,i,j] = (16-bit field dropout_field(j) of the Philox call dropout_call(j) of row (b*H + h, i)) >= threshold;
// one thread per call, i.e. per eight keys: 16*(c >> 1) + 8*r2 + 4*(c & 1) + e
__global__ void __launch_bounds__(256) keep_mask_kernel(uint8_t* __restrict__ mask, long long rows, int Nq, int Nk,
                                                        uint32_t thr, uint32_t seed_lo, uint32_t seed_hi,
                                                        uint32_t off_lo)
{
    const int calls = 2 * ((Nk + 15) >> 4);
    const long long total = rows * calls;
    for (long long idx = (long long)blockIdx.x * 256 + threadIdx.x; idx < total; idx += (long long)gridDim.x * 256) {
        const long long r = idx / calls;
        const int c = (int)(idx % calls);
        const uint32_t bh = (uint32_t)(r / Nq), i = (uint32_t)(r % Nq);
        const v4u w = philox4x32_10((uint32_t)c, i, bh, off_lo, seed_lo, seed_hi);
        uint8_t* mrow = mask + (size_t)r * Nk;
#pragma unroll
        for (int f = 0; f < 8; ++f) {
            const int j = 16 * (c >> 1) + 8 * (f >> 2) + 4 * (c & 1) + (f & 3);
            if (j < Nk) mrow[j] = philox_field16(w, f) >= thr ? 1 : 0;
        }
    }
}

int decode_heads_per_group(int kv_group) { return kv_group % 8 == 0 ? 8 : kv_group % 4 == 0 ? 4 : kv_group % 2 == 0 ? 2 : 1; }

template <int LPK, int G>
static hipError_t launch_decode_instance(const FwdArgs& a, hipStream_t st)
{
    const long long slices = (long long)a.B * a.H / G;
    const unsigned groups = (unsigned)(slices * a.num_splits);
    FwdArgs b = a;
    set_divisors(b, slices);
    const long long keys = a.wl >= 0 && a.wl < a.Nk ? a.wl + 1 : a.Nk;
    const bool stream = keys * a.B * a.Hk >= ((1 << 20) + a.d - 1) / a.d;  // 4 MiB of K and V, 4 d bytes a key
    auto launch = [&](auto alibi) {
        constexpr bool kAlibi = decltype(alibi)::value;
        const DecodeArgs<kAlibi> args = decode_args<kAlibi>(b, (int)slices);
        if (stream) return launch_kernel(decode_stream_kernel<LPK, kAlibi, G>, dim3(groups), dim3(256), 0, st, DecodeStreamArgs<kAlibi>{args, {}});
        return launch_kernel(decode_split_kernel<LPK, kAlibi, G>, dim3(groups), dim3(256), 0, st, args);
    };
    return a.alibi != nullptr ? launch(std::true_type{}) : launch(std::false_type{});
}

template <int LPK>
static hipError_t launch_decode_bucket(const FwdArgs& a, hipStream_t st)
{
    // as many of the query heads of a K/V head per work-group as divide the group (up to 8)
    switch (decode_heads_per_group(a.kv_group)) {
        case 8: return launch_decode_instance<LPK, 8>(a, st);
        case 4: return launch_decode_instance<LPK, 4>(a, st);
        case 2: return launch_decode_instance<LPK, 2>(a, st);
        default: return launch_decode_instance<LPK, 1>(a, st);
    }
}

int launch_decode_split(const FwdArgs& a, hipStream_t st)
{
    if (a.d > 64) return (int)launch_decode_bucket<16>(a, st);
    if (a.d > 32) return (int)launch_decode_bucket<8>(a, st);
    return (int)launch_decode_bucket<4>(a, st);
}

int launch_combine(const FwdArgs& a, hipStream_t st)
{
    const int rows = (int)((long long)a.B * a.H * a.Nq);  // < 2^31: validate_shape
    const FastDiv by_Nq = fast_div(a.Nq);
    if (a.combine_waves == 1)
        return (int)launch_kernel(combine_kernel<1>, dim3((unsigned)(rows + 3) / 4), dim3(256), 0, st, a.O_partial, a.LSE_partial, a.O,
                                  a.LSE, rows, a.Nq, by_Nq, a.d, a.num_splits);
    return (int)launch_kernel(combine_kernel<4>, dim3((unsigned)rows), dim3(256), 0, st, a.O_partial, a.LSE_partial, a.O, a.LSE, rows,
                              a.Nq, by_Nq, a.d, a.num_splits);
}

int launch_keep_mask(uint8_t* mask, int B, int H, int Nq, int Nk, uint32_t thr, uint64_t seed, uint64_t offset,
                     hipStream_t st)
{
    const long long rows = (long long)B * H * Nq;
    const long long total = rows * (2 * ((Nk + 15) / 16));  // one thread per Philox call
    long long groups = (total + 255) / 256;
    if (groups > 65536) groups = 65536;
    if (groups < 1) groups = 1;
    return (int)launch_kernel(keep_mask_kernel, dim3((unsigned)groups), dim3(256), 0, st, mask, rows, Nq, Nk, thr,
                              (uint32_t)seed, (uint32_t)(seed >> 32), (uint32_t)offset);
}

}  // namespace fa
