// Shared definitions for the gfx950 FlashAttention-forward kernels: launch-argument structs, vector types,
// wave64 helpers and the counter-based Philox used for dropout.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <atomic>

#define FLASH_MAX_SPLITS_K 128  // must equal FLASH_MAX_SPLITS of the public header

namespace fa {

typedef _Float16 half_t;
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
// 16 bytes at any 2-byte / 4-byte boundary (the hardware runs in unaligned access mode): rows of d % 8 != 0 elements
typedef v4u __attribute__((aligned(2))) v4u_anyalign;
typedef v4f __attribute__((aligned(4))) v4f_anyalign;
typedef v4h __attribute__((aligned(2))) v4h_anyalign;
// operand type of the ds_read_b64_tr_b16 builtin
typedef __fp16 v4hp __attribute__((__vector_size__(4 * sizeof(__fp16))));

#define FA_LDS __attribute__((address_space(3)))

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// Division of an index 0 <= n < 2^31 by a divisor that the host knows: n / d = floor(2n M / 2^32) / 2^l with
// l = ceil(log2 d) and M = ceil(2^(31+l) / d) < 2^32 (exact: M d exceeds 2^(31+l) by less than 2^l, which adds less than
// 1/d to the quotient).  On the scalar unit that is a shift, a multiply and a shift, where the compiler's division by
// a run-time divisor is a chain of some thirty instructions through the vector unit's reciprocal.  With the five or six
// divisions in front of a work-group's first request replaced (315 -> 169 instructions at d = 64), a launch is over 0.3 us
// earlier (B1 H2 N128 d64 5.1 -> 4.8 us, decode B15 H2 Nk3200 d64 8.9 -> 8.5 us, B2 H8 N2560 d40 causal 34.1 -> 33.6).
struct FastDiv {
    uint32_t mul, shift;
    __host__ __device__ __forceinline__ int quotient(int n) const { return (int)((uint32_t)(((uint64_t)(2u * (uint32_t)n) * mul) >> 32) >> shift); }
};
inline FastDiv fast_div(long long divisor)
{
    const uint64_t d = divisor > 1 ? (uint64_t)divisor : 1u;
    uint32_t l = 0;
    while ((1ull << l) < d) ++l;
    return {(uint32_t)(((1ull << (31 + l)) + d - 1) / d), l};
}

__host__ __device__ __forceinline__ constexpr FastDiv fast_div_by_one() { return {0x80000000u, 0u}; }

// Arguments of the tiled forward kernel and of the decode/combine kernels, filled by the host from flash_params
// (which is itself the superset of the reference's mykernelParamType, include/utils.h:21-44).
struct FwdArgs {
    const half_t* Q;
    const half_t* K;
    const half_t* V;
    half_t* O;
    float* LSE;
    float* O_partial;    // [B,H,S,Nq,d] fp32, normalised per split (reference O_tmp)
    float* LSE_partial;  // [B,H,S,Nq]   fp32, m_s + log l_s   (reference M, L)
    const float* alibi;  // [H] or nullptr
    uint8_t* keep_out;   // [B,H,Nq,Nk] or nullptr
    float* scores_out;   // [B,H,Nq,Nk] or nullptr (element-wise instance of the 4-wave kernel only)
    uint64_t* stamps;    // [work-groups][kStampWords] or nullptr (instrumented instances only)
    int B, H, Nq, Nk, d;
    int Hk, kv_group;    // K/V heads and query heads per K/V head (H = Hk * kv_group)
    int causal, wl, wr;  // wl / wr < 0: unbounded
    float scale_log2;    // softmax_scale * log2(e)
    uint32_t drop_thr;   // keep iff 16-bit philox field >= drop_thr
    uint32_t drop_sub2;  // drop_thr - 1 in both 16-bit halves (vector instances; they are launched with drop_thr >= 1)
    float drop_rscale;   // 1 / (1 - p)
    uint32_t seed_lo, seed_hi, off_lo;
    int kernel_hint;     // 0: by shape, 1: 4-wave kernel, 2: 8-wave kernel where it can serve the call
    int num_splits;      // 1: write O/LSE; > 1: write the partial workspace
    int keys_per_split;  // multiple of 128
    int Tr;              // number of query row blocks
    int slice_chunk;     // head slices per chunk of the work-group order (set by the kernel's launcher)
    int snake_end;       // work-groups below this index sit on the GPU together; odd 256-blocks of them run reversed (launcher)
    int group_xcd;       // query heads per K/V head where the slice order keeps the heads of a K/V head on one XCD (launcher):
    int group_span;      // for the first so many slices of a chunk, 0: for none (slice_of_position)
    int split_rotate;    // 1: the split index of a work-group is rotated by its row block (launcher; split_of_rest)
    // divisions of the work-group index and of the head slice (launcher: set_divisors)
    FastDiv by_chunk, by_slices, by_splits, by_xcd_group, by_kv_group, by_heads;
    int fold_rows;       // > 0: the query heads of a K/V head are the rows of one problem, this many rows each (see RowSpan)
    int fold_group;      // query heads folded into one
    FastDiv by_fold, by_row_blocks;
    uint32_t* counters;  // nullptr, or where the work-groups of a split launch count themselves in (combine.h)
    int combine_waves;   // waves that merge a row's partial results: 1 or 4 (combine_waves_for)
    int alibi_left;      // ALiBi and no visible key lies right of its row (causal, or right window 0)

    // index of the K/V slice [Nk,d] read by query slice bh = b * H + h: H is a multiple of the heads per K/V head
    __device__ __forceinline__ int kv_slice(int bh) const { return by_kv_group.quotient(bh); }
    __device__ __forceinline__ int head(int bh) const { return bh - by_heads.quotient(bh) * H; }
};

// Divisors of a launch, once its slice order is set (the decode kernel, whose order has no chunks, deals out
// `slices` groups of query heads per split)
inline void set_divisors(FwdArgs& b, long long slices)
{
    b.by_chunk = fast_div(slices * b.Tr * b.num_splits);
    b.by_slices = fast_div(slices);
    b.by_splits = fast_div(b.num_splits);
    b.by_xcd_group = fast_div(b.group_xcd);
    b.by_kv_group = fast_div(b.kv_group);
    b.by_heads = fast_div(b.H);
    b.by_fold = fast_div(b.fold_rows);
    b.by_row_blocks = fast_div(b.Tr);
}

// ---- FwdArgs as the tiled kernels get it.  A launch takes the host the longer the more its arguments are: back to back an empty
// kernel takes 2.6 us with 32 ... 112 bytes, 3.5-3.7 with 120 ... 272 (sizes in random order).  So the kernels get 112 bytes,
// narrow fields packed, and unpack them at their start; what only ALiBi, dropout and debug outputs need follows in
// PackedMore, 184 bytes.  FwdArgs (272 bytes) -> packed: B1 H2 N64 d64 3.65 -> 3.44 us, N128 d32 3.75 -> 3.55, B1 H8 N200 d64 4.5 -> 4.3 (medians; the runs spread by 10-20 %);
// where the GPU is the bound a launch of up to 128 bytes starts 0.15-0.2 us later behind the one before than a longer
// one (the decode kernel goes by that, decode_kernels.hip), 1 % of a launch of 20 us.  Split launches find their partial
// results where the others have O and LSE.
// (The words that tell a work-group its place in the order come first: one scalar load.)
struct Packed {
    int snake_end, slice_chunk, Tr;
    uint32_t shifts;  // of by_chunk, by_slices, by_splits, by_xcd_group, by_kv_group (folded: by_fold): five bits each; bit 25: split_rotate, bit 26: causal
    uint32_t sizes;   // d, num_splits: eight bits each; group_xcd: sixteen
    uint32_t mul_chunk, mul_slices, mul_splits;
    int group_span_or_fold_rows;      // folded launches have one query head per K/V head
    uint32_t mul_xcd_or_fold_group;
    uint32_t mul_kv_or_fold;
    int Nq, Nk, wl, wr, keys_per_split;
    const half_t *Q, *K, *V;
    void *O, *LSE;
    float scale_log2;
};
struct PackedMore : Packed {
    int H;
    FastDiv by_heads;
    uint32_t drop_thr, drop_sub2;
    float drop_rscale;
    uint32_t seed_lo, seed_hi, off_lo;
    const float* alibi;
    uint8_t* keep_out;
    float* scores_out;
    uint64_t* stamps;
};
constexpr size_t kCheapArgs = 112;  // bytes up to which a launch costs its least
static_assert(offsetof(Packed, scale_log2) + sizeof(float) <= kCheapArgs && sizeof(Packed) <= kCheapArgs, "cheap launches");
static_assert(FLASH_MAX_SPLITS_K < 256, "eight bits");

// Arguments of launches of few rows per slice (kVarRows of fwd_kernel.h), whose last work-groups may merge the partial results: 112 bytes
// hold results and partial results both.  Up to 32 rows, or folded: one query head per K/V head; order of the work-groups: rows_item.
constexpr int kRowsLimit = 32;  // rows of a work-group
struct PackedRows {
    uint32_t mul_slices, mul_row_blocks;
    int slices;
    uint32_t shifts;  // of by_slices, by_row_blocks, by_kv_group (folded: by_fold): five bits each; bit 15: causal, bit 16: combine_waves is 4 (the kernel merges with one wave per row whatever it says: up to eight splits are one batch); fold_rows (64 at most, kFoldRows): eight bits from 24 on
    uint32_t sizes;   // d, num_splits: eight bits each; fold_group: sixteen
    int Nq, Nk, keys_per_split, wl, wr;
    const half_t *Q, *K, *V;
    half_t* O;
    float *LSE, *O_partial, *LSE_partial;
    uint32_t* counters;
    uint32_t mul_kv_or_fold;
    float scale_log2;
};
struct PackedRowsMore : PackedRows {
    uint64_t* stamps;
};
static_assert(sizeof(PackedRows) <= kCheapArgs, "cheap launches");

inline PackedRowsMore packed_rows(const FwdArgs& a)
{
    PackedRowsMore p{};
    p.mul_slices = a.by_slices.mul, p.mul_row_blocks = a.by_row_blocks.mul, p.slices = a.B * a.H;
    p.shifts = a.by_slices.shift | a.by_row_blocks.shift << 5 | (a.fold_rows ? a.by_fold : a.by_kv_group).shift << 10 | (a.causal ? 1u << 15 : 0u) | (a.combine_waves == 4 ? 1u << 16 : 0u) |
               (uint32_t)a.fold_rows << 24;
    p.sizes = (uint32_t)a.d | (uint32_t)a.num_splits << 8 | (uint32_t)a.fold_group << 16;
    p.Nq = a.Nq;
    p.Nk = a.Nk, p.keys_per_split = a.keys_per_split, p.wl = a.wl, p.wr = a.wr;
    p.Q = a.Q, p.K = a.K, p.V = a.V, p.O = a.O, p.LSE = a.LSE, p.O_partial = a.O_partial, p.LSE_partial = a.LSE_partial;
    p.counters = a.counters, p.mul_kv_or_fold = (a.fold_rows ? a.by_fold : a.by_kv_group).mul, p.scale_log2 = a.scale_log2;
    p.stamps = a.stamps;
    return p;
}
template <bool kFold, typename P>
__host__ __device__ __forceinline__ FwdArgs unpacked_rows(const P& p)
{
    FwdArgs a{};
    a.by_slices = FastDiv{p.mul_slices, p.shifts & 31u}, a.by_row_blocks = FastDiv{p.mul_row_blocks, p.shifts >> 5 & 31u};
    (kFold ? a.by_fold : a.by_kv_group) = FastDiv{p.mul_kv_or_fold, p.shifts >> 10 & 31u};
    if (kFold) a.by_kv_group = fast_div_by_one();
    a.causal = p.shifts >> 15 & 1u, a.combine_waves = p.shifts >> 16 & 1u ? 4 : 1, a.fold_rows = p.shifts >> 24;
    a.d = p.sizes & 255u, a.num_splits = p.sizes >> 8 & 255u, a.fold_group = p.sizes >> 16;
    a.Nq = p.Nq, a.Tr = (p.Nq + 31) / 32, a.slice_chunk = p.slices;
    a.Nk = p.Nk, a.keys_per_split = p.keys_per_split, a.wl = p.wl, a.wr = p.wr;
    a.Q = p.Q, a.K = p.K, a.V = p.V, a.O = p.O, a.LSE = p.LSE, a.O_partial = p.O_partial, a.LSE_partial = p.LSE_partial;
    a.counters = p.counters, a.scale_log2 = p.scale_log2;
    if constexpr (sizeof(P) > sizeof(PackedRows)) a.stamps = p.stamps;
    return a;
}

inline PackedMore packed(const FwdArgs& a)
{
    PackedMore p{};
    const bool fold = a.fold_rows > 0, xcd = a.group_xcd < 65536;  // (more heads per K/V head than that keep the plain order)
    p.snake_end = a.snake_end, p.slice_chunk = a.slice_chunk, p.Tr = a.Tr;
    p.shifts = a.by_chunk.shift | a.by_slices.shift << 5 | a.by_splits.shift << 10 | (fold || !xcd ? 0u : a.by_xcd_group.shift) << 15 |
               (fold ? a.by_fold : a.by_kv_group).shift << 20 | (a.split_rotate ? 1u << 25 : 0u) | (a.causal ? 1u << 26 : 0u);
    p.sizes = (uint32_t)a.d | (uint32_t)a.num_splits << 8 | (xcd ? (uint32_t)a.group_xcd : 1u) << 16;
    p.mul_chunk = a.by_chunk.mul, p.mul_slices = a.by_slices.mul, p.mul_splits = a.by_splits.mul;
    p.group_span_or_fold_rows = fold ? a.fold_rows : xcd ? a.group_span : 0;
    p.mul_xcd_or_fold_group = fold ? (uint32_t)a.fold_group : a.by_xcd_group.mul;
    p.mul_kv_or_fold = (fold ? a.by_fold : a.by_kv_group).mul;
    p.Nq = a.Nq, p.Nk = a.Nk, p.wl = a.wl, p.wr = a.wr, p.keys_per_split = a.keys_per_split;
    p.Q = a.Q, p.K = a.K, p.V = a.V;
    p.O = a.num_splits > 1 ? static_cast<void*>(a.O_partial) : a.O;
    p.LSE = a.num_splits > 1 ? a.LSE_partial : a.LSE;
    p.scale_log2 = a.scale_log2;
    p.H = a.H, p.by_heads = a.by_heads;
    p.drop_thr = a.drop_thr, p.drop_sub2 = a.drop_sub2, p.drop_rscale = a.drop_rscale;
    p.seed_lo = a.seed_lo, p.seed_hi = a.seed_hi, p.off_lo = a.off_lo;
    p.alibi = a.alibi, p.keep_out = a.keep_out, p.scores_out = a.scores_out, p.stamps = a.stamps;
    return p;
}

// what packed() was given, as far as the kernels ask for it
template <bool kFold, typename P>
__host__ __device__ __forceinline__ FwdArgs unpacked(const P& p)
{
    FwdArgs a{};
    auto div = [&](uint32_t mul, int k) __attribute__((always_inline)) { return FastDiv{mul, p.shifts >> (5 * k) & 31u}; };
    a.snake_end = p.snake_end, a.slice_chunk = p.slice_chunk, a.Tr = p.Tr;
    a.by_chunk = div(p.mul_chunk, 0), a.by_slices = div(p.mul_slices, 1), a.by_splits = div(p.mul_splits, 2);
    a.split_rotate = p.shifts >> 25 & 1u, a.causal = p.shifts >> 26 & 1u;
    a.d = p.sizes & 255u, a.num_splits = p.sizes >> 8 & 255u;
    a.by_kv_group = fast_div_by_one();
    if constexpr (kFold) {
        a.fold_rows = p.group_span_or_fold_rows, a.fold_group = (int)p.mul_xcd_or_fold_group;
        a.by_fold = div(p.mul_kv_or_fold, 4);
    } else {
        a.group_span = p.group_span_or_fold_rows, a.group_xcd = p.sizes >> 16;
        a.by_xcd_group = div(p.mul_xcd_or_fold_group, 3), a.by_kv_group = div(p.mul_kv_or_fold, 4);
    }
    a.Nq = p.Nq, a.Nk = p.Nk, a.wl = p.wl, a.wr = p.wr, a.keys_per_split = p.keys_per_split;
    a.Q = p.Q, a.K = p.K, a.V = p.V;
    a.O = static_cast<half_t*>(p.O), a.O_partial = static_cast<float*>(p.O);
    a.LSE = a.LSE_partial = static_cast<float*>(p.LSE);
    a.scale_log2 = p.scale_log2;
    if constexpr (sizeof(P) > sizeof(Packed)) {
        a.H = p.H, a.by_heads = p.by_heads;
        a.drop_thr = p.drop_thr, a.drop_sub2 = p.drop_sub2, a.drop_rscale = p.drop_rscale;
        a.seed_lo = p.seed_lo, a.seed_hi = p.seed_hi, a.off_lo = p.off_lo;
        a.alibi = p.alibi, a.keep_out = p.keep_out, a.scores_out = p.scores_out, a.stamps = p.stamps;
    }
    return a;
}

// Folded launches: the G query heads of a K/V head, n rows each, are one problem of G n rows over that K/V head -- in
// memory they are just that, Q [B,H,n,d] is [B,H_kv,G n,d] -- in which row r is query r % n.
// (kFold: in the instances for such launches.  As a run-time choice in every instance the same code cost each launch
// 0.15 us.)
// Position among the queries of row r, and those of rows r0 ... r1 as a range (`straight`: one after the other)
template <bool kFold>
__device__ __forceinline__ int row_position(const FwdArgs& a, int r)
{
    if constexpr (kFold) return r - a.by_fold.quotient(r) * a.fold_rows;
    return r;
}
struct RowSpan {
    int first, last;
    bool straight;
};
template <bool kFold>
__device__ __forceinline__ RowSpan row_span(const FwdArgs& a, int r0, int r1)
{
    if constexpr (kFold) {
        const int h0 = a.by_fold.quotient(r0), h1 = a.by_fold.quotient(r1);
        if (h0 != h1) return {0, a.fold_rows - 1, false};
        return {r0 - h0 * a.fold_rows, r1 - h0 * a.fold_rows, true};
    }
    return {r0, r1, true};
}
// row of the split workspace [B,H,S,n] of row r of slice bh
template <bool kFold>
__device__ __forceinline__ size_t partial_row(const FwdArgs& a, int bh, int split, int r)
{
    if constexpr (kFold) {
        const int hq = a.by_fold.quotient(r);
        return (((size_t)bh * a.fold_group + hq) * a.num_splits + split) * a.fold_rows + (r - hq * a.fold_rows);
    }
    return ((size_t)bh * a.num_splits + split) * a.Nq + r;
}

// Index of this lane in its wave, worked out where it is asked for: in rare branches and behind loops, so that nothing made of
// it occupies a register throughout a loop (as an ordinary expression the compiler moves it, and whatever follows from it,
// in front of the loop).
__device__ __forceinline__ int lane_here()
{
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
}

__device__ __forceinline__ int wave_uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Q chunk for the chunk position at column col (a multiple of 8) of a row of d >= 8 elements at any alignment, where the
// position behind the row's whole chunks stands for columns d - 8 ... d - 1 and v holds what was loaded from there (see
// fwd_kernel.h): the columns that the chunk before has covered already are zeroed, and so are positions past the row.
__device__ __forceinline__ v8h mask_q_chunk_anyalign(v4u v, int col, int d)
{
    union { v4u u; v8h h; } t;
    t.u = v;
    const int covered = col + 8 <= d ? 0 : col < d ? 8 - (d & 7) : 8;  // leading elements that must not count
#pragma unroll
    for (int e = 0; e < 8; ++e) t.h[e] = e >= covered ? t.h[e] : (half_t)0.0f;
    return t.h;
}

// A work-group whose rows see no key at all (rows above a causal diagonal that starts below them, a split of the key
// range beyond their mask): O = 0 and LSE = -inf for rows [r0, r1) of head slice bh, or the same in the slice's partial
// results of split `split`.  The rows are one contiguous piece of memory; it is filled with 16-byte stores at whatever
// alignment the piece has, the last one ending with the piece.  Called by every thread of the group, before anything else
// is requested: such a group is done in the time of its stores.
template <bool kFold = false>
__device__ __forceinline__ void store_empty_rows(const FwdArgs& a, int bh, int split, int r0, int r1, int tid, int nthreads)
{
    char* base;
    float* lse;
    size_t bytes;
    if (kFold && a.num_splits > 1) {  // one piece per head
        for (int r = r0; r < r1; ++r) {
            const size_t prow = partial_row<kFold>(a, bh, split, r);
            for (int i = tid; i < a.d; i += nthreads) a.O_partial[prow * a.d + i] = 0.0f;
            if (tid == 0) a.LSE_partial[prow] = -INFINITY;
        }
        return;
    }
    if (a.num_splits > 1) {
        const size_t prow = ((size_t)bh * a.num_splits + split) * a.Nq + r0;
        base = reinterpret_cast<char*>(a.O_partial + prow * a.d);
        lse = a.LSE_partial + prow;
        bytes = (size_t)(r1 - r0) * a.d * sizeof(float);
    } else {
        const size_t row = (size_t)bh * a.Nq + r0;
        base = reinterpret_cast<char*>(a.O + row * a.d);
        lse = a.LSE + row;
        bytes = (size_t)(r1 - r0) * a.d * sizeof(half_t);
    }
    const v4u z = {0u, 0u, 0u, 0u};
    const size_t whole = bytes / 16;
    for (size_t i = tid; i < whole; i += nthreads) __builtin_nontemporal_store(z, reinterpret_cast<v4u_anyalign*>(base + 16 * i));
    if (tid == 0 && (bytes & 15) != 0) {
        if (whole > 0) {
            *reinterpret_cast<v4u_anyalign*>(base + bytes - 16) = z;
        } else {
            for (size_t i = 0; i < bytes; i += 2) *reinterpret_cast<uint16_t*>(base + i) = 0;
        }
    }
    for (int i = tid; i < r1 - r0; i += nthreads) lse[i] = -INFINITY;
}

// Position of a work-group in the launch's work order.  The order is "heaviest first", which balances a launch that
// makes several rounds: whichever place frees up takes the heaviest work-group left.  But the work-groups of the first
// round are not placed by load: the dispatcher deals work-group i to XCD i % 8 and there to CU (i / 8) % 32, so that with
// r places per CU work-groups i, i + 256, ..., i + 256 (r - 1) share a CU whatever they weigh (measured: a causal launch
// of 512 work-groups at two per CU left the CUs with 2 ... 32 key tiles each).  Inside that resident part (indices below
// snake_end = min(work-groups, places), a multiple of 8) every second block of 256 therefore takes its items in reverse
// CU order -- the CU with the heaviest item of one block gets the lightest of the next -- while i % 8, the XCD and with it
// the L2 that a head slice's K and V sit in, stays as it is.
__host__ __device__ __forceinline__ int work_position(int block, int snake_end)
{
    if (block < snake_end && (block & 256)) {
        const int base = block & ~255;
        const int size = snake_end - base < 256 ? snake_end - base : 256;  // a multiple of 8
        const int pos = block - base;
        return base + ((size >> 3) - 1 - (pos >> 3)) * 8 + (pos & 7);
    }
    return block;
}

// Head slice of position `local` in a chunk of the slice order.  Position p runs on XCD p % 8 (slices vary fastest over
// the work-groups).  With grouped K/V heads the G = group_xcd query heads of a K/V head are G consecutive slices and would
// land on G different XCDs, each pulling the same K and V into its own L2 (measured on B4 H32 H_kv4 N4096 d128 causal:
// 3.7 times the K/V/Q bytes fetched).  Instead position (x, y) = (p % 8, p / 8) takes query head y % G of K/V slice
// 8 (y / G) + x: the heads of a K/V head share an XCD and follow each other there.  A bijection on the first multiple of 8 G
// positions; what is left of a chunk that is no such multiple keeps the plain order.
// Split index and row-block index of the position `rest` inside a slice (splits fastest).  Where the slices of a chunk
// are not a multiple of 8, the XCD of a work-group depends on its split: with 4 slices and 2 splits, XCDs 0-3 get
// every first split and XCDs 4-7 every second one, and under a causal mask, whose first splits are the long ones, half the
// chip then carries three quarters of the work (measured B1 H4 N16384 d32 causal, 2 splits: 201 us, against 160 us
// unsplit and 158 us with 5 splits).  Rotating the split index by the row-block index deals every split to every XCD.
// The launcher asks for it exactly where the plain order aliases: work-group x + 8 n of XCD x has split
// (x / c + (8 / c) n) % S for c = 1, 2 or 4 slices per chunk, which reaches every split only if S is odd; other chunk
// sizes mix by themselves, and rotating an order that already mixes measured 0 ... -14 %.
__host__ __device__ __forceinline__ int split_of_rest(const FwdArgs& a, int rest, int* row_block_index)
{
    const int mi = a.by_splits.quotient(rest), s0 = rest - mi * a.num_splits;
    *row_block_index = mi;
    if (!a.split_rotate) return s0;
    const int s = s0 + mi;
    return s - a.by_splits.quotient(s) * a.num_splits;
}
inline int split_rotate_for(int num_splits, int slice_chunk)
{
    return num_splits > 1 && num_splits % 2 == 0 && (slice_chunk == 1 || slice_chunk == 2 || slice_chunk == 4) ? 1 : 0;
}

__host__ __device__ __forceinline__ int slice_of_position(const FwdArgs& a, int local)
{
    if (local < a.group_span) {
        const int x = local & 7, y = local >> 3, yg = a.by_xcd_group.quotient(y);
        return (yg * 8 + x) * a.group_xcd + y - yg * a.group_xcd;
    }
    return local;
}

// Work-group -> head slice, split and row block.  Slices vary fastest, so that with B*H a multiple of 8 a slice always
// lands on the same XCD (and L2); the heaviest causal row blocks (largest index) are dispatched first.  Slices are dealt
// out in chunks of a.slice_chunk (the launcher's choice: all of them unless the problem has far more work-groups than the
// GPU holds at once), chunk after chunk, so that the row blocks of a slice run closer together in time and find its K
// and V in the caches.
struct WorkItem {
    int bh, split, m_block;
};
__host__ __device__ __forceinline__ WorkItem work_item(const FwdArgs& a, int block)
{
    const int pos = work_position(block, a.snake_end);
    const int ch = a.by_chunk.quotient(pos), w = pos - ch * (a.slice_chunk * a.Tr * a.num_splits);
    const int rest = a.by_slices.quotient(w);
    WorkItem it;
    it.bh = ch * a.slice_chunk + slice_of_position(a, w - rest * a.slice_chunk);
    int mi;
    it.split = split_of_rest(a, rest, &mi);
    it.m_block = a.Tr - 1 - mi;
    return it;
}

// The same of PackedRows: slices vary fastest, then splits, and the row blocks of a split, which read the same keys, run on one XCD (its
// L2 sees them once): position p of eight neighbours takes indices 8 Tr (p / 8) + p % 8 + 8 m, the last few, that are no eight, plain order.  With
// the row blocks slowest they were on as many XCDs as the split count made it: causal B3 H2 Nq128 Nk8000 d128 in 9 splits 20.9 -> 16.4 us.
template <bool kOneBlock>
__host__ __device__ __forceinline__ WorkItem rows_item(const FwdArgs& a, int block)
{
    int p = block, m = 0;
    if constexpr (!kOneBlock) {
        const int pairs = a.slice_chunk * a.num_splits, whole = pairs & ~7, q = a.by_row_blocks.quotient(block >> 3);
        p = 8 * q + (block & 7), m = (block >> 3) - q * a.Tr;
        if (block >= whole * a.Tr) {
            p = block - whole * a.Tr;
            for (m = 0; p >= pairs - whole; ++m) p -= pairs - whole;
            p += whole;
        }
    }
    const int split = a.by_slices.quotient(p);
    return {p - split * a.slice_chunk, split, a.Tr - 1 - m};
}

// snake_end for a launch of `groups` work-groups with `resident` places on the GPU
inline int snake_end_for(long long groups, int resident)
{
    const long long n = groups < resident ? groups : resident;
    return (int)(n & ~7LL);
}

// Exchange between lane l and lane l^32 (v_permlane32_swap): result[0] holds the low half's value in both halves,
// result[1] the high half's.
__device__ __forceinline__ float xhalf_max(float v)
{
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xhalf_sum(float v)
{
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Debug time stamps of the instrumented kernel instances: readings of the constant 100 MHz counter, taken by every wave
// (they are scalar) and stored by the first lane of the work-group in the epilogue with an ordinary vector store.
// Beside stages 3 and 5 the shader-clock counter is read as well: their difference over the time between the two stages
// is the clock the work-group ran at in its key-tile loop.
constexpr int kStampTimes = 7;
constexpr int kStampWords = 9;  // FLASH_STAMP_WORDS of the public header
template <bool kOn>
struct Stamps {
    uint64_t t[kOn ? kStampTimes : 1];
    uint64_t cyc[kOn ? 2 : 1];
    // stage 0 also presets the later stages: one that a work-group never reaches (no key tile) is stored as the time
    // of the stage before it
    __device__ __forceinline__ void take(int i)
    {
        if constexpr (kOn) {
            const uint64_t now = __builtin_amdgcn_s_memrealtime();
            if (i == 0) {
#pragma unroll
                for (int k = 0; k < kStampTimes; ++k) t[k] = now;
                cyc[0] = cyc[1] = 0;
            } else {
                t[i] = now;
                if (i == 3) cyc[0] = __builtin_amdgcn_s_memtime();
                if (i == 5) cyc[1] = __builtin_amdgcn_s_memtime();
            }
        }
    }
    // word 7: tiles << 32 | XCC id << 16 | low half of HW_ID (wave, SIMD, pipe, CU, SH, SE); word 8: shader-clock cycles
    // between stages 3 and 5
    __device__ __forceinline__ void store(uint64_t* out, int ntiles) const
    {
        if constexpr (kOn) {
            if (out != nullptr && threadIdx.x == 0) {
                const uint32_t hw = __builtin_amdgcn_s_getreg((31 << 11) | 4);    // HW_REG_HW_ID
                const uint32_t xcc = __builtin_amdgcn_s_getreg((31 << 11) | 20);  // HW_REG_XCC_ID
                uint64_t* o = out + (size_t)blockIdx.x * kStampWords;
                uint64_t last = t[0];
#pragma unroll
                for (int i = 0; i < kStampTimes; ++i) {
                    last = t[i] > last ? t[i] : last;
                    o[i] = last;
                }
                o[kStampTimes] = ((uint64_t)(uint32_t)ntiles << 32) | ((uint64_t)(xcc & 0xfu) << 16) | (hw & 0xffffu);
                o[kStampTimes + 1] = cyc[1] > cyc[0] ? cyc[1] - cyc[0] : 0;
            }
        }
    }
};

// two fp32 -> packed fp16, round to nearest even, in one instruction (v_cvt_pk_f16_f32)
__device__ __forceinline__ v2h pack_f16(float a, float b)
{
    const v2f t = {a, b};
    return __builtin_convertvector(t, v2h);
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float fast_log2(float x) { return __builtin_amdgcn_logf(x); }

// Philox4x32-10.  Dropout contract: one call yields eight 16-bit fields (field f = bits 16*(f&1).. of output word f>>1)
// and serves eight keys of one query row: key = (lo32(seed), hi32(seed)), counter = (call(j), i, b*H + h, lo32(offset)),
// element (i, j) reads field(j) and is kept iff that field >= floor(p * 2^16).  Of every 16 consecutive keys the call
// with even index serves keys 0-3 and 8-11, the odd one keys 4-7 and 12-15: the eight keys whose scores one lane of the
// tiled kernels holds (32x32 MFMA accumulator layout), so that a lane uses every bit it computes.  Replaces the
// stateful curandStatePhilox4_32_10_t draw of the reference (src/flash_forward.h:50-54,227).
__host__ __device__ __forceinline__ uint32_t dropout_call(uint32_t j) { return 2u * (j >> 4) + ((j >> 2) & 1u); }
__host__ __device__ __forceinline__ uint32_t dropout_field(uint32_t j) { return 4u * ((j >> 3) & 1u) + (j & 3u); }
// 32 x 32 -> 64-bit product in one instruction (v_mad_u64_u32; integer multiplies run at a quarter of the VALU rate,
// and the compiler would issue two of them, v_mul_hi_u32 and v_mul_lo_u32, per product)
__device__ __forceinline__ void mul_wide_u32(uint32_t m, uint32_t x, uint32_t& hi, uint32_t& lo)
{
    uint64_t r;
    asm("v_mad_u64_u32 %0, vcc, %1, %2, 0" : "=v"(r) : "s"(m), "v"(x) : "vcc");
    hi = (uint32_t)(r >> 32);
    lo = (uint32_t)r;
}

// Both products of a Philox round in one statement: between two of the above the compiler puts a wait state, in case the first ends with
// an instruction that writes part of a register, whose result the next instruction must not read.  v_mad_u64_u32 writes whole
// registers, and neither of the two reads what the other writes (vcc is carry out alone).
__device__ __forceinline__ void mul_wide_pair(uint32_t m0, uint32_t x0, uint32_t m1, uint32_t x1, uint32_t& hi0, uint32_t& lo0,
                                              uint32_t& hi1, uint32_t& lo1)
{
    uint64_t r0, r1;
    asm("v_mad_u64_u32 %0, vcc, %2, %3, 0\n\tv_mad_u64_u32 %1, vcc, %4, %5, 0"
        : "=&v"(r0), "=v"(r1)
        : "s"(m0), "v"(x0), "s"(m1), "v"(x1)
        : "vcc");
    hi0 = (uint32_t)(r0 >> 32), lo0 = (uint32_t)r0;
    hi1 = (uint32_t)(r1 >> 32), lo1 = (uint32_t)r1;
}

// Element masks of a tile: two 32 x 32 score blocks (keys 0 ... 31 and 32 ... 63 of the tile).  In the accumulator layout lane
// (l32 = lane % 32, g = lane / 32) holds in register r the score of query row l32 and key 8 (r / 4) + r % 4 + 4 g of the
// block.  A block's mode is a sum of
//   kMaskRight, kMaskLeft   the boundary runs along the block's diagonal, and the keys right of it (key > row) or left of it
//                           (key < row) go: a fixed set of lanes per register, in either half of the lanes the first so many
//                           rows or all but these, which s_bfm makes; one v_cndmask per score
//   kMaskAbove, kMaskBelow  keys above `hi` or below `lo` go (the lane's own bounds, counted from the tile's first key plus the
//                           lane's 4 g): a comparison and a v_cndmask per score
//   kMaskWhole              all of it goes
// and 0 leaves the block alone; `modes` holds the first block's in bits 0-7, the second one's in bits 8-15.
// One statement with its branches inside, and a block's sixteen registers as one operand, on purpose: with branches that the
// compiler sees, or with an operand per register, one path or the other ends in copies of the accumulators, 64 v_mov per
// boundary tile and as many registers to copy into, which cost the instances for d <= 96 a work-group per CU.  The assembler
// takes the number of the first register out of the operand's name.
// (The wait states at the head: whoever produced the scores may have been an MFMA right in front, which the compiler does not
// account for where it cannot see who reads them.)
constexpr int kMaskRight = 1, kMaskLeft = 2, kMaskAbove = 4, kMaskBelow = 8, kMaskWhole = 16;
// SYM: the first number of the operand's "v[first:last]"; anything but sixteen vector registers is an error
#define FA_FIRST_REGISTER(SYM, OPERAND) \
    ".set " SYM ", 0\n\t.set fa_last, 0\n\t.set fa_in, 0\n\t.irpc fa_c, \"" OPERAND "\"\n\t" \
    ".ifc \\fa_c,:\n\t.set fa_in, 2\n\t.endif\n\t.ifc \\fa_c,]\n\t.set fa_in, 3\n\t.endif\n\t" \
    ".if fa_in == 1\n\t.set " SYM ", " SYM " * 10 + \\fa_c\n\t.endif\n\t" \
    ".if fa_in == 2\n\t.ifnc \\fa_c,:\n\t.set fa_last, fa_last * 10 + \\fa_c\n\t.endif\n\t.endif\n\t" \
    ".ifc \\fa_c,[\n\t.set fa_in, 1\n\t.endif\n\t.endr\n\t" \
    ".if fa_last - " SYM " - 15\n\t.error \"an accumulator of sixteen registers\"\n\t.endif\n\t"
// register, its key in the lower half of the lanes and in the upper half
#define FA_MASK_16A(X) X("fa_a+0", 0, 4) X("fa_a+1", 1, 5) X("fa_a+2", 2, 6) X("fa_a+3", 3, 7) X("fa_a+4", 8, 12) \
    X("fa_a+5", 9, 13) X("fa_a+6", 10, 14) X("fa_a+7", 11, 15) X("fa_a+8", 16, 20) X("fa_a+9", 17, 21) \
    X("fa_a+10", 18, 22) X("fa_a+11", 19, 23) X("fa_a+12", 24, 28) X("fa_a+13", 25, 29) X("fa_a+14", 26, 30) \
    X("fa_a+15", 27, 31)
#define FA_MASK_16B(X) X("fa_b+0", 0, 4) X("fa_b+1", 1, 5) X("fa_b+2", 2, 6) X("fa_b+3", 3, 7) X("fa_b+4", 8, 12) \
    X("fa_b+5", 9, 13) X("fa_b+6", 10, 14) X("fa_b+7", 11, 15) X("fa_b+8", 16, 20) X("fa_b+9", 17, 21) \
    X("fa_b+10", 18, 22) X("fa_b+11", 19, 23) X("fa_b+12", 24, 28) X("fa_b+13", 25, 29) X("fa_b+14", 26, 30) \
    X("fa_b+15", 27, 31)
#define FA_MASK_RIGHT(R, K, K4) \
    "s_bfm_b32 vcc_lo, " #K ", 0\n\ts_bfm_b32 vcc_hi, " #K4 ", 0\n\tv_cndmask_b32_e32 v[" R "], v[" R "], %[ninf], vcc\n\t"
#define FA_MASK_LEFT(R, K, K4) \
    "s_bfm_b64 vcc, " #K4 "+1, 32\n\ts_bfm_b32 vcc_lo, " #K "+1, 0\n\tv_cndmask_b32_e32 v[" R "], %[ninf], v[" R "], vcc\n\t"
// (A v_cndmask wants two wait states behind the vector instruction that wrote its scalar operand, and inside a statement nobody but
// the statement provides them.  Comparisons into vcc and into a scalar pair take turns, two of a block's scores ahead of their
// selections: the instructions between are the neighbours' and cost nothing, where an s_nop 1 per score takes half as long again.)
#define FA_MASK_CMP0(CMP, BOUND, T) CMP "_e32 vcc, " #T ", " BOUND "\n\t"
#define FA_MASK_CMP1(CMP, BOUND, T) CMP "_e64 %[pair], " #T ", " BOUND "\n\t"
#define FA_MASK_SEL0(A, R) "v_cndmask_b32_e32 v[" A "+" #R "], v[" A "+" #R "], %[ninf], vcc\n\t"
#define FA_MASK_SEL1(A, R) "v_cndmask_b32_e64 v[" A "+" #R "], v[" A "+" #R "], %[ninf], %[pair]\n\t"
#define FA_MASK_NEXT(CMP, BOUND, A, R0, R1, T0, T1) \
    FA_MASK_SEL0(A, R0) FA_MASK_CMP0(CMP, BOUND, T0) FA_MASK_SEL1(A, R1) FA_MASK_CMP1(CMP, BOUND, T1)
#define FA_MASK_BOUND(CMP, BOUND, A, T0, T1, T2, T3, T4, T5, T6, T7, T8, T9, T10, T11, T12, T13, T14, T15) \
    FA_MASK_CMP0(CMP, BOUND, T0) FA_MASK_CMP1(CMP, BOUND, T1) "s_nop 0\n\t" \
    FA_MASK_NEXT(CMP, BOUND, A, 0, 1, T2, T3) FA_MASK_NEXT(CMP, BOUND, A, 2, 3, T4, T5) FA_MASK_NEXT(CMP, BOUND, A, 4, 5, T6, T7) \
    FA_MASK_NEXT(CMP, BOUND, A, 6, 7, T8, T9) FA_MASK_NEXT(CMP, BOUND, A, 8, 9, T10, T11) FA_MASK_NEXT(CMP, BOUND, A, 10, 11, T12, T13) \
    FA_MASK_NEXT(CMP, BOUND, A, 12, 13, T14, T15) FA_MASK_SEL0(A, 14) "s_nop 0\n\t" FA_MASK_SEL1(A, 15)
#define FA_MASK_BOUND_A(CMP, BOUND) FA_MASK_BOUND(CMP, BOUND, "fa_a", 0, 1, 2, 3, 8, 9, 10, 11, 16, 17, 18, 19, 24, 25, 26, 27)
#define FA_MASK_BOUND_B(CMP, BOUND) FA_MASK_BOUND(CMP, BOUND, "fa_b", 32, 33, 34, 35, 40, 41, 42, 43, 48, 49, 50, 51, 56, 57, 58, 59)
#define FA_MASK_ABOVE(BOUNDS) BOUNDS("v_cmp_gt_i32", "%[hi]")
#define FA_MASK_BELOW(BOUNDS) BOUNDS("v_cmp_lt_i32", "%[lo]")
#define FA_MASK_WHOLE(R, K, K4) "v_mov_b32 v[" R "], %[ninf]\n\t"
// (a taken branch costs some twenty cycles: whole groups of modes are passed by together)
#define FA_MASK_IF(BIT, NAME, BODY) "s_bitcmp1_b32 %[modes], " #BIT "\n\ts_cbranch_scc0 .Lfa_" NAME "%=\n\t" BODY ".Lfa_" NAME "%=:\n\t"
#define FA_MASK_BLOCK(B, ANY, WHOLE, B0, B1, REGS) \
    "s_and_b32 vcc_lo, %[modes], " ANY "\n\ts_cbranch_scc0 .Lfa_" B "z%=\n\t" \
    FA_MASK_IF(B0, B "r", REGS(FA_MASK_RIGHT)) FA_MASK_IF(B1, B "l", REGS(FA_MASK_LEFT)) \
    "s_and_b32 vcc_lo, %[modes], " WHOLE "\n\ts_cbranch_scc0 .Lfa_" B "z%=\n\t" REGS(FA_MASK_WHOLE) ".Lfa_" B "z%=:\n\t"
// (The comparisons of both blocks stand together behind everything else, one taken branch away: in a launch of few tiles they are
// code that nobody has fetched yet.  With the blocks' other modes between them -> like this, unmasked: B1 H2 N100 d32 4.08 -> 3.91
// us, d64 4.76 -> 4.58, B8 H16 N130 d64 5.98 -> 5.79, N230 d128 9.08 -> 8.92.)
template <bool kDiagonals>
__device__ __forceinline__ void mask_tile(v16f& s0, v16f& s1, int modes, int lo, int hi, float ninf)
{
    uint64_t pair;
    if constexpr (kDiagonals)
        asm(FA_FIRST_REGISTER("fa_a", "%[s0]") FA_FIRST_REGISTER("fa_b", "%[s1]") "s_nop 15\n\t"
            "s_bitcmp1_b32 %[modes], 3\n\ts_cbranch_scc1 .Lfa_below%=\n\ts_bitcmp1_b32 %[modes], 2\n\ts_cbranch_scc1 .Lfa_above%=\n\t"
            FA_MASK_BLOCK("a", "19", "16", 0, 1, FA_MASK_16A) FA_MASK_BLOCK("b", "19*256", "16*256", 8, 9, FA_MASK_16B)
            "s_branch .Lfa_end%=\n\t"
            ".Lfa_below%=:\n\t" FA_MASK_BELOW(FA_MASK_BOUND_A) FA_MASK_BELOW(FA_MASK_BOUND_B)
            "s_bitcmp1_b32 %[modes], 2\n\ts_cbranch_scc0 .Lfa_end%=\n\t"
            ".Lfa_above%=:\n\t" FA_MASK_ABOVE(FA_MASK_BOUND_A) FA_MASK_ABOVE(FA_MASK_BOUND_B) ".Lfa_end%=:\n\t"
            : [s0] "+v"(s0), [s1] "+v"(s1), [pair] "=&s"(pair)
            : [modes] "s"(modes), [lo] "v"(lo), [hi] "v"(hi), [ninf] "v"(ninf)
            : "vcc", "scc");
    else
        asm(FA_FIRST_REGISTER("fa_a", "%[s0]") FA_FIRST_REGISTER("fa_b", "%[s1]") "s_nop 15\n\t"
            FA_MASK_IF(2, "a", FA_MASK_ABOVE(FA_MASK_BOUND_A) FA_MASK_ABOVE(FA_MASK_BOUND_B))
            FA_MASK_IF(3, "b", FA_MASK_BELOW(FA_MASK_BOUND_A) FA_MASK_BELOW(FA_MASK_BOUND_B))
            : [s0] "+v"(s0), [s1] "+v"(s1), [pair] "=&s"(pair)
            : [modes] "s"(modes), [lo] "v"(lo), [hi] "v"(hi), [ninf] "v"(ninf)
            : "vcc", "scc");
}
// 1 where x is negative / zero, in integers alone: as comparisons the scalar conditions end up in vector instructions
__device__ __forceinline__ int is_negative(int x) { return (int)((unsigned)x >> 31); }
__device__ __forceinline__ int is_zero(int x) { return 1 - is_negative(x | -x); }
// Which ends of the interval cross the tile at key kb0, for rows that see keys from lo_max (the last first one) on and up to hi_min:
// bit 0 the first key, bit 1 the last one
__device__ __forceinline__ int mask_sides(int kb0, int lo_max, int hi_min) { return is_negative(kb0 - lo_max) | is_negative(hi_min - 63 - kb0) << 1; }
// Which of the wave's bounds run along block diagonals, same bits: first row lo_min / hi_min, last row lo_max / hi_max
__device__ __forceinline__ int diagonal_sides(bool straight, int lo_min, int lo_max, int hi_min, int hi_max)
{
    return (straight && lo_max - lo_min == 31 && (lo_min & 31) == 0 ? 1 : 0) | (straight && hi_max - hi_min == 31 && (hi_min & 31) == 0 ? 2 : 0);
}
// Modes of a tile; general (the bounds of the lane's own row are asked for) where a crossing end does not run along a diagonal
__device__ __forceinline__ bool mask_is_general(int sides, int diagonals) { return (sides & ~diagonals) != 0; }
__device__ __forceinline__ int mask_modes_general(int sides) { return ((sides & 1) * kMaskBelow + (sides >> 1) * kMaskAbove) * 0x101; }
__device__ __forceinline__ int mask_modes_diagonal(int kb0, int sides, int lo_min, int hi_min)
{
    // last / first visible key of the wave's first row, in blocks from the tile's first one
    const int th = (sides & 2) ? (hi_min - kb0) >> 5 : 2, tl = (sides & 1) ? (lo_min - kb0) >> 5 : -1;
    int modes = 0;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
        const int whole = is_negative(th - kb) | is_negative(kb - tl);
        modes |= (whole * kMaskWhole + (1 - whole) * (is_zero(th - kb) * kMaskRight + is_zero(tl - kb) * kMaskLeft)) << (8 * kb);
    }
    return modes;
}

// three-input exclusive or in one instruction (v_bitop3_b32, truth table 0x96)
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) { return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96); }

__device__ __forceinline__ v4u philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0, uint32_t k1)
{
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        uint32_t hi0, lo0, hi1, lo1;
        mul_wide_u32(0xD2511F53u, c0, hi0, lo0);
        mul_wide_u32(0xCD9E8D57u, c2, hi1, lo1);
        c0 = xor3(hi1, c1, k0);
        c1 = lo1;
        c2 = xor3(hi0, c3, k1);
        c3 = lo0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    v4u o = {c0, c1, c2, c3};
    return o;
}

// The same function for the tiled kernels, where a work-group holds one head slice, a lane one query row, and all lanes of a
// half wave ask for the same call.  Written out, the words that the first three rounds leave depend on the row alone (the
// first-round word that holds the row number, and its product), on the call and the head slice alone (every other
// product up to the third round's first), or on both by an exclusive-or -- so a wave works out the call's part for 64 calls
// at once, a lane each, into LDS (CallTable below), and a call is left with 15 of its 20 integer multiplies, which are what
// bounds a launch with dropout.  Causal with dropout, 19 multiplies per call -> 15 (and the rounds interleaved with the MFMAs
// of the second product, see pv in fwd_kernel.h): B8 H16 N1300 d80 77.3 -> 69.4 us, B16 H16 N2048 d64 265 -> 250, B2 H4 N1986 d96
// (paired) 38.4 -> 35.0, B4 H16 N900 d31 20.5 -> 18.7, B8 H32 N1000 d96 92 -> 89, B4 H16 N2048 d128 (8-wave kernel) 99.7 -> 97.2.
//   round 1   A0 = hi(M1 bh) ^ i ^ k0   A1 = lo(M1 bh)            A2 = hi(M0 c) ^ off ^ k1    A3 = lo(M0 c)
//   round 2   B0 = hi(M1 A2) ^ A1 ^ k0' B1 = lo(M1 A2)            B2 = hi(M0 A0) ^ A3 ^ k1'   B3 = lo(M0 A0)
//   round 3   hi(M1 B2) ^ B1 ^ k0"      lo(M1 B2)                 hi(M0 B0) ^ B3 ^ k1"        lo(M0 B0)
constexpr uint32_t kPhiloxM0 = 0xD2511F53u, kPhiloxM1 = 0xCD9E8D57u, kPhiloxW0 = 0x9E3779B9u, kPhiloxW1 = 0xBB67AE85u;
struct PhiloxRow {
    uint32_t hi, lo;  // M0 A0
};
__device__ __forceinline__ PhiloxRow philox_row_part(uint32_t i, uint32_t bh, uint32_t k0)
{
    PhiloxRow r;
    mul_wide_u32(kPhiloxM0, (uint32_t)(((uint64_t)kPhiloxM1 * bh) >> 32) ^ i ^ k0, r.hi, r.lo);
    return r;
}
// {A3 ^ k1', B1 ^ k0", hi(M0 B0) ^ k1", lo(M0 B0)}
__device__ __forceinline__ v4u philox_call_part(uint32_t c, uint32_t bh, uint32_t off, uint32_t k0, uint32_t k1)
{
    uint32_t hi, a3, b1, lo;
    mul_wide_u32(kPhiloxM0, c, hi, a3);
    mul_wide_u32(kPhiloxM1, hi ^ (off ^ k1), hi, b1);
    mul_wide_u32(kPhiloxM0, hi ^ (kPhiloxM1 * bh ^ (k0 + kPhiloxW0)), hi, lo);
    const v4u r = {a3 ^ (k1 + kPhiloxW1), b1 ^ (k0 + 2 * kPhiloxW0), hi ^ (k1 + 2 * kPhiloxW1), lo};
    return r;
}
__device__ __forceinline__ v4u philox_from_parts(const PhiloxRow& row, const v4u& call, uint32_t k0, uint32_t k1)
{
    uint32_t hi0, lo0, hi1, lo1;
    mul_wide_u32(kPhiloxM1, row.hi ^ call[0], hi1, lo1);
    uint32_t c0 = hi1 ^ call[1], c1 = lo1, c2 = call[2] ^ row.lo, c3 = call[3];
#pragma unroll
    for (int r = 3; r < 10; ++r) {
        const uint32_t q0 = k0 + r * kPhiloxW0, q1 = k1 + r * kPhiloxW1;
        mul_wide_pair(kPhiloxM0, c0, kPhiloxM1, c2, hi0, lo0, hi1, lo1);
        c0 = xor3(hi1, c1, q0);
        c1 = lo1;
        c2 = xor3(hi0, c3, q1);
        c3 = lo0;
    }
    const v4u o = {c0, c1, c2, c3};
    return o;
}

// The call parts of 64 calls (512 keys, eight tiles) in LDS, one table per wave: nobody else reads it, so nothing but the
// order of the wave's own LDS operations stands between a refill and the reads.
template <int kWaves>
__device__ __forceinline__ v4u* call_table_memory()
{
    __shared__ v4u t[kWaves * 64];
    return t;
}
struct CallTable {
    v4u* mem;    // of the wave
    int chunk;   // calls 64 chunk ... 64 chunk + 63 are in it
    // in front of the reads of the tile at key kb0 (wave-uniform)
    __device__ __forceinline__ void cover(int kb0, int lane, uint32_t bh, uint32_t off, uint32_t k0, uint32_t k1)
    {
        if ((kb0 >> 9) != chunk) {
            chunk = kb0 >> 9;
            mem[lane] = philox_call_part((uint32_t)(64 * chunk + lane), bh, off, k0, k1);
        }
    }
    // call of the keys jg + 4 g ... (jg a multiple of 16): index 2 (jg / 16) + g
    __device__ __forceinline__ v4u at(int kb0, int within, int g) const { return mem[((kb0 >> 3) & 63) + (within >> 3) + g]; }
};

// Keep decisions of two scores at once: p2 holds their probabilities as packed fp16, w the two 16-bit Philox fields in the
// same halves, sub2 = threshold - 1 in both halves (threshold >= 1).  A saturating subtraction leaves a half non-zero
// iff field >= threshold; clipped to 1 it multiplies the fp16 bit pattern as an integer: the pattern, or zero.  Three
// packed instructions for two scores instead of a comparison and a select for each.
// (inline asm: from the same thing written with vector types the compiler recovers the comparison and emits a compare,
// a select and a byte permute per score)
__device__ __forceinline__ uint32_t keep_pair(uint32_t p2, uint32_t w, uint32_t sub2)
{
    uint32_t x;
    asm("v_pk_sub_u16 %0, %1, %2 clamp\n\tv_pk_min_u16 %0, %0, %3\n\tv_pk_mul_lo_u16 %0, %4, %0"
        : "=&v"(x)
        : "v"(w), "s"(sub2), "v"(0x00010001u), "v"(p2));
    return x;
}

// An MFMA reads a register two wait states after the vector instruction that wrote it at the earliest; the compiler, which keeps
// that distance in its own code, does not see which instruction a statement like keep_pair's ends with.  To stand between
// operands that come out of such a statement and the MFMA.
__device__ __forceinline__ void settle_for_mfma(v8h& p) { asm("s_nop 1" : "+v"(p)); }

// 16-bit field f (0..7) of a Philox output
__device__ __forceinline__ uint32_t philox_field16(const v4u& w, int f) { return (w[f >> 1] >> (16 * (f & 1))) & 0xffffu; }

// One KiB from global memory straight into LDS: lane l fetches 16 bytes at base + off (its own offset) and the wave
// writes them to lds_dst + 16 l.  Issued as inline asm on purpose: the compiler models the builtin form as a FLAT
// access that may touch LDS, and from then on degrades every LDS wait of the loop to "wait for everything".  The
// caller waits with s_waitcnt vmcnt(0) before the barrier that publishes the tile.
__device__ __forceinline__ void dma_kib(const char* base, uint32_t off, FA_LDS char* lds_dst)
{
    const uint32_t m0v = (uint32_t)(uintptr_t)lds_dst;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(m0v), "v"(off), "s"(base)
                 : "memory", "m0");
}
// A float at an address that is the same in all lanes, which nobody writes during the launch: a load of the scalar unit.
__device__ __forceinline__ float read_uniform(const float* p)
{
    return *reinterpret_cast<const __attribute__((address_space(4))) float*>(reinterpret_cast<uintptr_t>(p));
}
// The same request marked non-temporal, for data that no other work-group will ask for (the K/V stream of a decode
// launch): measured 5.4 -> 6.3 TB/s on grouped-query decode with eight query heads per K/V head.
__device__ __forceinline__ void dma_kib_nt(const char* base, uint32_t off, FA_LDS char* lds_dst)
{
    const uint32_t m0v = (uint32_t)(uintptr_t)lds_dst;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"
                 :
                 : "s"(m0v), "v"(off), "s"(base)
                 : "memory", "m0");
}

// Launch with the error of THIS launch as the return value (hipGetLastError would also hand back whatever an
// unrelated earlier call of the process left behind).
template <typename T>
struct same_type { typedef T type; };
template <typename... P>
inline hipError_t launch_kernel(void (*kern)(P...), dim3 grid, dim3 block, size_t smem, hipStream_t st,
                                typename same_type<P>::type... args)
{
    void* argv[] = {static_cast<void*>(&args)...};
    return hipLaunchKernel(reinterpret_cast<const void*>(kern), grid, block, argv, smem, st);
}

// Raises the dynamic-LDS limit of a kernel once per device (the attribute belongs to the device's copy of the kernel).
// `done` is the caller's per-kernel flag array.  Concurrent first calls from several threads may both set the
// attribute, which is harmless; the flags are atomics so that such calls do not race in the language's sense either.
constexpr int kMaxDevices = 64;
typedef std::atomic<bool> DeviceFlags[kMaxDevices];
inline hipError_t ensure_dynamic_lds(const void* kern, int bytes, DeviceFlags& done)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) dev = kMaxDevices - 1;  // beyond the table: set it on every launch
    if (dev != kMaxDevices - 1 && done[dev].load(std::memory_order_acquire)) return hipSuccess;
    e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess) done[dev].store(true, std::memory_order_release);
    return e;
}

}  // namespace fa
