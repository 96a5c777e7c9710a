// Tiled FlashAttention forward for gfx950 (wave64, MFMA 32x32x16 f16 -> f32).
//
// Replaces forward_kernel / forward_kernel_splitkv of the reference (src/flash_forward.h:13-306,
// src/flash_forward_splitkv.h:14-344); the math contract is the one of the reference's CPU verifier
// (src/main.cu:309-383).  The structure is specific to CDNA4:
//
//  * One work-group = 4 waves; wave w owns 32*NB query rows, the group 128*NB.  KV tiles hold 64 keys.
//  * Scores are computed transposed, S^T = K Q^T: the MFMA A operand is a K fragment read from LDS
//    (ds_read_b128), the B operand a Q fragment that stays in registers for the whole kernel.  In the 32x32
//    accumulator layout every lane then holds 16 keys of ONE query row (row = lane % 32), so the online-softmax
//    max / sum are in-lane reductions plus one v_permlane32_swap between lane l and l^32.
//  * The probabilities, rounded to fp16 where the reference rounds them (include/utils.h:47-55), already sit in
//    the B-operand layout of O^T += V^T P^T; no LDS round trip for P.  The V^T A operand needs four keys of one
//    head-dim column per lane: that is what ds_read_b64_tr_b16 delivers from the row-major V tile.
//  * O^T accumulates in registers (fp32) and is normalised once in the epilogue; the reference keeps O in shared
//    memory and renormalises it every tile (src/flash_forward.h:284-289).
//  * K and V tiles are double-buffered in LDS and requested straight into it (global_load_lds_dwordx4), tile t+1
//    while tile t is computed, one barrier per tile; only the instance that serves every request (rows of fewer than
//    eight elements among them) stages its tiles through registers.
//  * Small unsplit problems take the narrow instances: 32 query rows per work-group, held by all four waves, each of
//    which walks every fourth key tile with LDS stages of its own; the four results are merged through LDS.
//  * Every mask of the family (causal, sliding window, key bound for ragged Nk) is one per-row interval
//    [lo_i, hi_i] of allowed keys; tiles entirely inside the interval of every row of the wave skip the
//    element test.  The KV tile range of the group is pruned like src/flash_forward.h:39-48.
//  * Ragged Nq / Nk: row indices of loads are clamped, stores are predicated, keys >= Nk are masked (the
//    reference zero-fills them and leaves them unmasked).  Head dims that are not a multiple of 8 use the
//    instances for rows at any alignment (kVec = false).
#pragma once
#include <type_traits>

#include "combine.h"
#include "common.h"

namespace fa {

template <int D, int NB, bool kNarrow = false, bool kShort = false>
struct FwdCfg {
    static constexpr int kWaves = 4;
    static constexpr int RW = 32 * NB;        // query rows per wave
    static constexpr int BR = kWaves * RW;    // query rows per work-group
    static constexpr int BC = 64;             // keys per tile
    static constexpr int CH = D / 8;          // 16-byte chunks per row
    // Rows of at most D - 16 elements (kShort: d = 40 in 64 columns, 72 and 80 in 96, 100 and 112 in 128) leave out the last k-step,
    // its share of K in LDS and of the requests for it: a tile is bound by what it issues and moves, and one in twelve of its MFMAs at D = 96
    // met zeroes of Q.  With the k-step -> without: causal B3 H12 N1777 d80 34.7 -> 32.9 us, B4 H16 N2048 d80 106.8 -> 101.0, d72 causal
    // 60.1 -> 57.6, B10 H16 H_kv8 N1216 d40 74.7 -> 70.3, B15 H16 N1536 d100 causal 187 -> 178 (8-wave), B1 H4 N2048 d100 16.8 -> 15.6
    // (narrow), causal with dropout B8 H32 N1000 d80 91.0 -> 86.3; split over 8409 keys B3 H16 Nq192 d72, bound by HBM, +-0.  (At run time, one branch around the
    // MFMAs, it gave 1-3 % there and cost the other rows 0.3-1 %.)
    static constexpr int KS = D / 16 - (kShort ? 1 : 0);  // k-steps of the QK^T contraction
    static constexpr int CHK = 2 * KS;        // 16-byte chunks per K row
    static constexpr int MB = D / 32;         // 32-wide head-dim blocks of O^T
    // LDS rows.  K rows are read 16 bytes per lane by 32 consecutive rows, which have to be spread over all banks.
    // Either the rows are padded by one 16-byte chunk (kPadK: stride / 16 odd), or the chunks of row r are permuted by
    // exclusive-or with kswz(r), which gives any 16 consecutive rows 16 different places among the 64 banks.  A
    // request of permuted rows is one KiB of whole consecutive rows, and a tile takes one request less than with padded
    // ones, whose requests begin and end anywhere in a row; but a fragment address takes a register per k-step where
    // padded rows have immediate offsets.  Measured, padded -> permuted: causal with dropout B8 H32 N1000 d96 104.0 -> 95.5
    // us, B8 H1 N1920 d32 causal 9.96 -> 9.83, B2 H4 N960 d40 causal 9.53 -> 9.36, d = 64 +-1 %; d = 128, eight k-steps, 10
    // registers more and 1-4 % slower, keeps its padding, except in the narrow instances, where a wave requests whole
    // tiles and the period of the permutation saves offsets (NPX below).
    // V rows are read by ds_read_b64_tr_b16, four consecutive rows of 64 bytes per half wave: a stride of 64 (mod 128)
    // puts the four rows on disjoint bank groups.
    static constexpr bool kPadK = D == 128 && !kNarrow;
    static constexpr int CK = CHK + (kPadK ? 1 : 0);  // chunks of a K row in LDS
    static constexpr int SK = CK * 16;
    static constexpr int SV = D * 2;
    static constexpr __host__ __device__ int kswz(int r)
    {
        if (kPadK) return 0;
        if (kShort) return (r >> 3) & 1;  // rows of 224 / 160 / 96 bytes, an odd multiple of 32: eight rows spread by themselves
        return D == 128 ? r & 15 : D == 64 ? (r >> 1) & 7 : (r >> 2) & 3;  // rows of 256 / 128 / 192 or 64 bytes
    }
    // Where the row length is a multiple of 128 bytes, the two 64-byte halves of each 128 bytes are exchanged in rows
    // 2, 3 (mod 4), which has the same effect without padding.
    static constexpr bool VSWZ = (D * 2) % 128 == 0;
    static constexpr int KBUF = BC * SK;
    static constexpr int VBUF = BC * SV;
    static constexpr bool kQApart = kNarrow && D <= 64;  // Q has a place of its own behind the four waves' stages
    static constexpr int kTiles = 2 * KBUF + 2 * VBUF, kOut = 4 * NB * 32 * (2 * D + 16);
    static constexpr int SMEM = kTiles > kOut ? kTiles : kOut;
    static constexpr int NSTG = 2;
    static constexpr int SMEM_DMA = NSTG * (KBUF + VBUF);
    static constexpr int NKX = (CK + 3) / 4;      // 1 KiB blocks of a K tile (CK of them) per wave, rounded up
    static constexpr int NVX = CH / 4;            // 1 KiB blocks of a V tile (CH of them) per wave
    static constexpr int NLD = BC * CH / 256;  // 16-byte chunks per thread per tile (K and V each)
    static_assert(D % 32 == 0 && D <= 128 && (!kShort || D >= 64), "head-dim bucket");
    static_assert((BC * CH) % 256 == 0, "tile chunks must divide over the group");
};

// 8 fp16 of one row starting at column col (multiple of 8); columns >= d read as zero.
// kVec: rows are 16-byte aligned (d % 8 == 0); kFullD: d equals the bucket width, no column test at all.
template <bool kVec, bool kFullD>
__device__ __forceinline__ v4u load_chunk(const half_t* __restrict__ rowp, int col, int d)
{
    if constexpr (kFullD) {
        return *reinterpret_cast<const v4u*>(rowp + col);
    } else if constexpr (kVec) {
        const int cc = col < d ? col : d - 8;  // stay inside the row, discard below
        v4u v = *reinterpret_cast<const v4u*>(rowp + cc);
        const v4u z = {0u, 0u, 0u, 0u};
        return col < d ? v : z;
    } else {
        union { v8h h; v4u u; } r;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int c = col + e;
            const half_t x = rowp[c < d ? c : d - 1];
            r.h[e] = c < d ? x : (half_t)0.0f;
        }
        return r.u;
    }
}

// Rows that start at any 2-byte boundary (d % 8 != 0), d >= 8: a chunk is still one 16-byte load -- the hardware runs in
// unaligned access mode -- taken at the chunk's own column, or, for the row's last, partial chunk and for chunks past the
// row, at column d - 8, so that no load ever leaves the row.  Nothing is moved into place afterwards: the last chunk
// position of a row simply stands for the columns d - 8 ... d - 1 instead of 8 (d / 8) ... 8 (d / 8) + 7.
//   Q   the columns that the chunk before has covered already (the first 8 - d % 8 of the partial chunk) are zeroed, and so
//       are chunks past the row (mask_q_chunk_anyalign): every product with them is 0 times finite data of the K row itself.
//   K   as loaded.
//   V   as loaded: the chunk position yields O's columns d - 8 ... d - 1, of which the epilogue stores the row's last 16
//       bytes; chunks past the row yield columns that are never stored.
// Element by element, a 64 x 32 tile took 16 two-byte loads per thread with an address computation each, where this takes
// two loads and no arithmetic on the data.
__device__ __forceinline__ v4u load_chunk_anyalign(const half_t* __restrict__ rowp, int col, int d)
{
    return *reinterpret_cast<const v4u_anyalign*>(rowp + (col + 8 <= d ? col : d - 8));
}

// Running maximum is only raised when some row of the wave outgrows it by more than this many powers of two;
// until then probabilities are taken relative to the stale maximum (bounded by 2^kLazyTau, exact in the end
// because numerator and denominator carry the same factor).  Saves the per-tile rescale of the O accumulators.
constexpr float kLazyTau = 8.0f;
// Running maximum (log2 units) of a row that has seen no key: the lowest finite number, relative to which a masked score is
// still 2^-inf = 0 and every visible one raises it; -inf would need a case of its own wherever it is subtracted.
constexpr float kNothingSeen = -3.402823466e38f;

// variant bits of the kernel template
// kVarStamp: debug time stamps.  kVarAlibiLeft (with kVarAlibi, kVarVec): every visible key lies at or left of its row
// (causal mask or a right window of 0), which lets the bias ride in the MFMA accumulator (see calib below).
// kVarKvOnce (with kVarVec, kVarFullD, no other feature but kVarFold): every K/V tile is requested by this work-group alone --
// one row block per slice and one query head (folded: all the query heads) per K/V head, the shape of a decode launch -- and
// its requests are non-temporal.
// kVarEvery (with kVarAlibi and kVarDropout, without kVarVec): the instance that serves every request, see kEvery below.
// kVarNarrow (unsplit launches; in splits with kVarRows): the four waves of a work-group share 32 query rows and take every fourth key tile
// each, see kNarrow below.
// kVarPair (with ALiBi: keys at or left of the row alone, no dropout): eight waves in two halves that take every other tile each, see kPair below.
// kVarFold (no other feature): the rows are the query heads of a K/V head, see row_position in common.h.
// kVarShort (D >= 64, not kVarFullD, kVarEvery or kVarFold): rows of at most D - 16 elements, see FwdCfg::kShort.
// kVarRows (with kVarNarrow; no other feature but kVarFold): launches of few rows per slice, whole or in splits, see kRows below.
// kVarManyRows (with kVarRows): more than 32 rows, whose row blocks ask for the same tiles, or rows of d < 32: ordinary requests.
constexpr int kVarVec = 1, kVarAlibi = 2, kVarDropout = 4, kVarFullD = 8, kVarStamp = 16, kVarAlibiLeft = 32, kVarKvOnce = 64,
              kVarEvery = 128, kVarNarrow = 256, kVarFold = 512, kVarPair = 1024, kVarShort = 2048, kVarRows = 4096, kVarManyRows = 8192;

// arguments of an instance
template <int VAR>
using KernelArgs = std::conditional_t<(VAR & kVarRows) != 0, std::conditional_t<(VAR & kVarStamp) != 0, PackedRowsMore, PackedRows>,
                                      std::conditional_t<(VAR & (kVarAlibi | kVarDropout | kVarStamp | kVarEvery)) != 0, PackedMore, Packed>>;

// The arguments take up two lines of 64 bytes, PackedMore three.  Left to the compiler nothing of the last one is asked for before the
// work-group knows its place -- with ALiBi or dropout, before Q is on its way --, and the first tile requests wait until it has come from memory; so
// one word of it is asked for with what the work-group needs first.  Late -> with the first: B1 H8 N640 d96 causal with dropout 8.77 -> 8.47
// us, B2 H8 N900 d96 14.71 -> 14.45, B8 H16 N256 d32 6.90 -> 6.71, B1 H4 N600 d96 causal with bias 7.85 -> 7.61, B4 H8 N1000 d64 15.26 -> 15.16,
// long launches +-0.  (With both features the seeds are asked for early as it is: d31, d64, d100 +-0, d40 1.5 % slower.)
template <int VAR>
__device__ __forceinline__ void ask_for_all_arguments(const FwdArgs& a)
{
    if constexpr (((VAR & kVarAlibi) != 0) != ((VAR & kVarDropout) != 0)) asm volatile("" : : "s"(a.off_lo));
    if constexpr ((VAR & kVarFold) != 0) asm volatile("" : : "s"(a.scale_log2));
}

// work-groups per CU (narrow: one or two by their LDS; held to 256 VGPRs all the same, without which the compiler keeps more
// than there are and moves them to and from accumulation registers): three up to D = 96 (168 VGPRs), except for the instance that
// serves every request, which stages its tiles through registers, and at D = 96 those with sixteen registers of bias constants
// and dropout, which would spill (bias and dropout without those constants, two per CU -> three: B8 H32 N1000 d96 168 -> 158 us, B16 H16
// N512 d80 47.8 -> 46.8, but B4 H12 N777 d88 32.4 -> 33.5).  Four at D = 64 without either (128 VGPRs: B32 H32 N512 d64 in 128-row blocks 100.3 -> 91.1 us
// together with the shorter chunks below); with the bias constants four spill in the loop (window of 256 keys with ALiBi B2
// H16 N4096 d64 22.9 -> 24.4).
constexpr int fwd_groups_per_cu(int D, int NB, int VAR)
{
    if ((VAR & (kVarNarrow | kVarPair)) != 0) return 2;
    if (D == 96 && (VAR & kVarAlibiLeft) != 0 && (VAR & kVarDropout) != 0) return 2;
    if (NB == 1 && D == 64 && (VAR & (kVarEvery | kVarDropout | kVarAlibiLeft)) == 0) return 4;
    return NB == 1 && D <= 96 && (VAR & kVarEvery) == 0 ? 3 : 2;
}

// Arguments of fwd_kernel.  Two groups of instances got slower by what the compiler makes of the packed fields:
//  * D = 96 without features: told that d and num_splits are eight bits wide it orders the work around the loop otherwise, at the same
//    number of instructions in the loop.  Known -> not: causal B1 H64 H_kv8 N448 d96 9.64 -> 9.44 us, B8 H8 N200 7.26 -> 7.10, N192 6.23 -> 6.16,
//    B14 H4 N120 d80 5.14 -> 5.07.  Narrow instances, other buckets, ALiBi and dropout stay or lose up to 3 %.
//  * D = 32 at any alignment with ALiBi and dropout: 209 of the 321 8-byte instructions of its loop lay off 8-byte boundaries, with
//    one more word in front of them 112: causal B2 H8 N2000 d31 41.6 -> 40.45 us.
template <int D, int VAR>
__device__ __forceinline__ FwdArgs fwd_arguments(const KernelArgs<VAR>& packed_args)
{
    if constexpr ((VAR & kVarRows) != 0) {
        const FwdArgs a = unpacked_rows<(VAR & kVarFold) != 0>(packed_args);
        asm volatile("" : : "s"(a.scale_log2));  // (the second line of the arguments with the first)
        return a;
    } else {
        FwdArgs a = unpacked<(VAR & kVarFold) != 0>(packed_args);
        ask_for_all_arguments<VAR>(a);
        if constexpr (D == 96 && (VAR & (kVarAlibi | kVarDropout | kVarNarrow)) == 0) asm("" : "+s"(a.d), "+s"(a.num_splits));
        if constexpr (D == 32 && (VAR & ~kVarStamp) == (kVarAlibi | kVarDropout)) asm volatile("s_nop 0");
        return a;
    }
}

template <int D, int NB, int VAR>
__global__ void __launch_bounds__((VAR & kVarPair) != 0 ? 512 : 256, fwd_groups_per_cu(D, NB, VAR)) fwd_kernel(const KernelArgs<VAR> packed_args)
{
    const FwdArgs a = fwd_arguments<D, VAR>(packed_args);
    constexpr bool kVec = (VAR & kVarVec) != 0, kAlibi = (VAR & kVarAlibi) != 0, kDropout = (VAR & kVarDropout) != 0,
                   kFullD = (VAR & kVarFullD) != 0, kStamp = (VAR & kVarStamp) != 0, kKvOnce = (VAR & kVarKvOnce) != 0;
    using C = FwdCfg<D, NB, (VAR & kVarNarrow) != 0, (VAR & kVarShort) != 0>;
    static_assert((VAR & kVarShort) == 0 || (VAR & (kVarFullD | kVarEvery | kVarFold)) == 0, "shorter rows");
    Stamps<kStamp> stamps;
    stamps.take(0);
    constexpr int BC = C::BC, KS = C::KS, MB = C::MB, CH = C::CH, SK = C::SK, SV = C::SV, NLD = C::NLD;
    // Tiles go from global memory straight into LDS (global_load_lds_dwordx4) instead of through registers: measured
    // +6-12 % at D = 128, +1-4 % at D = 64 and 96.  The request takes global addresses at any 2-byte boundary, so rows of
    // any length from eight elements on are served; only the instance that also serves shorter rows stages through
    // registers (kEvery, defined below).
    constexpr bool kDma = (VAR & kVarEvery) == 0;
    // Rows at any alignment (kVec false) have the same four instances as rows of whole chunks: plain, ALiBi, dropout, both.
    // They count on d >= 8, a positive scale, a slope table where ALiBi is compiled in and a dropout threshold of at least
    // 1 like the vector instances do.  One more instance, with both features compiled in, serves every request (kEvery:
    // slope 0 / threshold 0 make the features identities), a non-positive scale, rows of fewer than eight elements and
    // the score dump among them.
    constexpr bool kEvery = (VAR & kVarEvery) != 0;
    static_assert(!kEvery || (!kVec && kAlibi && kDropout), "the instance that serves every request");
    // Problems of few work-groups are bound by the chain of tiles that a work-group walks through one after the other
    // (fwd_uses_narrow says which).  The narrow instances cut that chain to a quarter: a work-group owns
    // 32 query rows, all four waves hold those rows, and wave w takes the key tiles w, w + 4, w + 8, ... of the range on
    // its own: it requests them into LDS stages of its own (no work-group barrier inside the loop, every wave waits
    // for its own requests only), and the four partial results are merged through LDS at the end like the partial results
    // of a split -- in the same launch, where a split count of four would need the combine launch behind it.
    constexpr bool kNarrow = (VAR & kVarNarrow) != 0;
    static_assert(!kNarrow || (kDma && NB == 1 && !kKvOnce), "narrow instances");
    // The narrow form for launches of few rows per slice (fwd_uses_rows says which), in splits too: their partial results leave the merge
    // as whole rows of floats, and where a caller has brought counters (combine.h) and the rows are four or fewer, the last work-group
    // of a slice merges the splits.  With up to 32 rows nobody else asks for the tiles, and the requests are non-temporal.
    // Ordinary / non-temporal, time over time, over 1000 random launches: K and V that no cache holds, up to 8 MiB 1.02 ... 1.04, 40 MiB 1.03 ... 1.05, 128 MiB 1.05 ... 1.09, more
    // 1.11; called again and again with the same K and V, up to 20 MiB 0.99 ... 1.00, 20-40 MiB (the L2 holds 32) 0.94 ... 0.99, more 0.98 ... 1.06 (whole launches 0.88 ... 1.12).
    // Not with d < 32 (launch_fwd_bucket_st).
    constexpr bool kRows = (VAR & kVarRows) != 0, kRowsOnce = kRows && (VAR & kVarManyRows) == 0;
    static_assert(!kRows || (kNarrow && !kAlibi && !kDropout), "few rows");
    constexpr bool kFold = (VAR & kVarFold) != 0;
    static_assert(!kFold || (!kAlibi && !kDropout), "folded instances");
    // A launch of one work-group per CU leaves a SIMD one wave, whose score, softmax and output phases follow one another:
    // a paired work-group has eight waves.  Waves 0 ... 3 walk the even tiles of the range, waves 4 ... 7, which hold the same
    // rows and have LDS stages of their own, the odd ones, and the two partial results are merged through LDS at the end.
    constexpr bool kPair = (VAR & kVarPair) != 0;
    static_assert(!kPair || (kDma && NB == 1 && !kNarrow), "paired instances");
    // (narrow: two stages per wave up to D = 64, one above: four waves' tiles of 26 / 33 KiB)
    constexpr int NSTG = kNarrow ? (D <= 64 ? 2 : 1) : kDma ? C::NSTG : 2;
    constexpr int BRW = kNarrow ? 32 : C::BR;  // query rows per work-group
    // Narrow: Q is fetched like the first 32 rows of a K tile, so that the wave's first wait is for Q and tile 0 alone.  Loaded into
    // registers -> so: B1 H8 N1021 d31 8.0 -> 7.3 us, d63 11.5 -> 10.2, N1024 d64 7.2 -> 7.0, N2048 causal d64 14.4 -> 13.9, N1024
    // d128 10.8 -> 10.1, N300 d128 7.3 -> 6.75, B1 H2 N3000 d111 33.1 -> 31.9, d72, d80 and one or two tiles per wave +-1 %.  Whole rows of 96
    // without bias keep the loads (kQLoads), with V of tile 0 requested at once: the other way it leaves only once Q is there, which costs launches
    // of few tiles more than the rest gain (Q like a tile / loads: causal B14 H4 N120 4.89 / 4.73 us, B3 H3 N194 4.80 / 4.71, B1 H8 N400 6.00 / 5.94,
    // with dropout N640 8.48 / 8.42; unmasked N120 4.84 / 4.68, N256 4.75 / 4.81, N1024 7.87 / 7.83, B1 H4 N2000 12.16 / 12.29).  With a bias the
    // scalar load of the slope gains by the shorter first wait: causal B1 H4 N600 7.60 against 7.84.  With few rows (kRows) at D = 128, too, V goes
    // out at once, its tiles coming from HBM: B4 H32 H_kv8 Nk8192 25.8 -> 25.4, B1 Nk32768 26.1 -> 25.8 (shorter rows, loaded piece by piece: 12.7 -> 14.8).
    constexpr bool kQLoads = kNarrow && kFullD && ((D == 96 && !kAlibi) || (D == 128 && kRows));
    // Where to, and bytes from one wave's to the next one's
    constexpr bool kQApart = C::kQApart;
    constexpr int kQWave = kQApart ? 32 * C::SK : NSTG * (C::KBUF + C::VBUF);
    constexpr int kQLds = kQApart ? 4 * NSTG * (C::KBUF + C::VBUF) : NSTG * C::KBUF + (NSTG - 1) * C::VBUF;
    extern __shared__ __attribute__((aligned(16))) char smem[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = wave_uniform(kPair ? (tid >> 6) & 3 : tid >> 6);
    const int half = kPair ? wave_uniform(tid >> 8) : 0;
    // tile buffers: of the work-group, or (narrow) of the wave, or (paired) of four waves
    constexpr int kWaveLds = NSTG * (C::KBUF + C::VBUF);
    const int lds_base = kNarrow ? wave * kWaveLds : kPair ? half * kWaveLds : 0;
    char* const Ks = smem + lds_base;
    char* const Vs = Ks + NSTG * C::KBUF;
    const int l32 = lane & 31;
    const int g = lane >> 5;

    WorkItem item;
    if constexpr (kRows) item = rows_item<kRowsOnce>(a, blockIdx.x);
    else item = work_item(a, blockIdx.x);
    const int bh = item.bh, split = item.split, m_block = item.m_block;
    const int Nq = a.Nq, Nk = a.Nk, d = kFullD ? D : a.d;
    const int shift = Nk - (kFold ? a.fold_rows : Nq);
    const int q0 = m_block * BRW;
    const int wave_row0 = kNarrow ? 0 : wave * C::RW;  // first row of the wave inside the work-group's block

    // ---- key range of the work-group (block pruning, src/flash_forward.h:39-48; split range, splitkv.h:40-43)
    int kmin = 0, kmax = Nk;
    {
        const RowSpan rows = row_span<kFold>(a, q0, q0 + BRW - 1 < Nq ? q0 + BRW - 1 : Nq - 1);
        const int last_row = rows.last + shift;
        if (a.wl >= 0) kmin = max(0, rows.first + shift - a.wl);
        if (a.causal) kmax = min(kmax, last_row + 1);
        if (a.wr >= 0) kmax = min(kmax, last_row + a.wr + 1);
        if (a.num_splits > 1) {
            const int s0 = split * a.keys_per_split;
            kmin = max(kmin, s0);
            kmax = min(kmax, s0 + a.keys_per_split);
        }
    }
    const int tile_begin = kmin / BC;
    const int ntiles = kmax > kmin ? (kmax + BC - 1) / BC - tile_begin : 0;
    if (!kStamp && !kRows && ntiles == 0) {  // (the instrumented twins take the long way and report their stages, kRows to count itself in)
        store_empty_rows<kFold>(a, bh, split, q0, q0 + BRW < Nq ? q0 + BRW : Nq, tid, kPair ? 512 : 256);
        return;
    }

    // ---- per-lane rows, and what the masks leave of the keys.  Nothing in front of the first score needs the bounds: they
    // are worked out behind the first requests (set_bounds, called below), like everything else that can wait.  A
    // launch of few tiles is bound by its instructions up to there, fetched through a cold instruction cache: 0.1 us per
    // launch (B3 H4 N73 d64 4.92 -> 4.83 us), and B32 H32 N512 d64, whose work-groups have eight tiles each, 107.4 -> 105.9.
    int row_i[NB];
    float iif[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) row_i[nb] = q0 + wave_row0 + nb * 32 + l32;
    // first and last key that row i sees (asked for in boundary tiles, and worked out there: two registers less in the loop)
    auto row_bounds = [&](int i, int* lo, int* hi) __attribute__((always_inline)) {
        const int ii = row_position<kFold>(a, i < Nq ? i : Nq - 1) + shift;
        int l_ = 0, h_ = Nk - 1;
        if (a.wl >= 0) l_ = max(0, ii - a.wl);
        if (a.causal) h_ = min(h_, ii);
        if (a.wr >= 0) h_ = min(h_, ii + a.wr);
        if (a.num_splits > 1) {
            l_ = max(l_, kmin);
            h_ = min(h_, kmax - 1);
        }
        *lo = l_;
        *hi = h_;
    };
    // wave-uniform bounds: [lo_max, hi_min] is visible to every row of the wave (a tile inside it needs no element
    // test), nothing outside [lo_min, hi_max] is visible to any of them (a tile outside it is skipped by the wave)
    int lo_max, hi_min, lo_min, hi_max;
    int diagonals;  // which of the bounds run along diagonals of 32 x 32 score blocks (diagonal_sides)
    // the same in tiles of the work-group's range: first one and number of those that some row of the wave sees, and of those
    // that every row sees whole
    int live0, nlive, clean0, nclean;
    auto set_bounds = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const int i = row_i[nb];
            iif[nb] = (float)(row_position<kFold>(a, i < Nq ? i : Nq - 1) + shift);
        }
        bool straight;
        {
            const int first = q0 + wave_row0, last = first + C::RW - 1;
            const RowSpan rows = row_span<kFold>(a, first < Nq ? first : Nq - 1, last < Nq ? last : Nq - 1);
            const int iif_ = rows.first + shift, iil_ = rows.last + shift;
            straight = rows.straight;
            lo_max = lo_min = 0;
            hi_min = hi_max = Nk - 1;
            if (a.wl >= 0) lo_max = max(0, iil_ - a.wl), lo_min = max(0, iif_ - a.wl);
            if (a.causal) hi_min = min(hi_min, iif_), hi_max = min(hi_max, iil_);
            if (a.wr >= 0) hi_min = min(hi_min, iif_ + a.wr), hi_max = min(hi_max, iil_ + a.wr);
            if (a.num_splits > 1) {
                lo_max = max(lo_max, kmin);
                lo_min = max(lo_min, kmin);
                hi_min = min(hi_min, kmax - 1);
                hi_max = min(hi_max, kmax - 1);
            }
        }
        diagonals = diagonal_sides(straight, lo_min, lo_max, hi_min, hi_max);
        // (At D = 96 with bias and dropout this one register of the vector unit was one too many and lived in scratch memory.  On the scalar
        // unit everywhere: B2 H8 N2000 causal with bias d31 28.1 -> 29.0 us, d31 with dropout as well 41.9 -> 40.7.)
        if constexpr (D == 96 && kAlibi && kDropout) diagonals = wave_uniform(diagonals);
        // (a wave whose rows all lie past Nq sees nothing: it only helps to stage the tiles)
        live0 = (lo_min >> 6) - tile_begin;
        nlive = q0 + wave_row0 < Nq ? max(0, (hi_max >> 6) - tile_begin - live0 + 1) : 0;
        clean0 = ((lo_max + 63) >> 6) - tile_begin;
        nclean = max(0, ((hi_min - 63) >> 6) - tile_begin - clean0 + 1);
    };

    const half_t* __restrict__ Qbh = a.Q + (size_t)bh * Nq * d;
    const int kvs = a.kv_slice(bh);
    const half_t* __restrict__ Kbh = a.K + (size_t)kvs * Nk * d;
    const half_t* __restrict__ Vbh = a.V + (size_t)kvs * Nk * d;

    // ---- Q fragments (B operand of S^T = K Q^T): lane holds row l32, columns 16*ks + 8*g .. +7
    v8h qf[NB][KS];
#pragma unroll
    for (int nb = 0; nb < NB && (!kNarrow || kQLoads); ++nb) {
        const int ic = row_i[nb] < Nq ? row_i[nb] : Nq - 1;
        const half_t* qrow = Qbh + (size_t)ic * d;
        if constexpr (kVec) {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                union { v4u u; v8h h; } t;
                t.u = load_chunk<kVec, kFullD>(qrow, 16 * ks + 8 * g, d);
                qf[nb][ks] = t.h;
            }
        } else {
            // rows at any alignment: every load of the row block first, then the zero padding and the packing (written as
            // one chunk after the other, each 2-byte load was waited for before the next was issued)
            if (!kEvery || d >= 8) {
                v4u raw[KS];
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) raw[ks] = load_chunk_anyalign(qrow, 16 * ks + 8 * g, d);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    qf[nb][ks] = mask_q_chunk_anyalign(raw[ks], 16 * ks + 8 * g, d);
                }
            } else {
                half_t raw[KS][8];
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const int c = 16 * ks + 8 * g + e;
                        raw[ks][e] = qrow[c < d ? c : d - 1];
                    }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                    for (int e = 0; e < 8; ++e) qf[nb][ks][e] = 16 * ks + 8 * g + e < d ? raw[ks][e] : (half_t)0.0f;
            }
        }
    }

    // ---- tile staging through registers (the instance that serves every request; all others request their tiles
    // straight into LDS, below): thread handles chunk ids tid + 256*x  ->  (row, chunk) of the 64 x CH tile.  The
    // loads of tile t+1 are issued in front of the arithmetic of tile t and waited for where their data is written to
    // LDS behind it: nothing is computed on what was loaded (a select on it would drag the wait for the whole tile in
    // front of the arithmetic).
    int ld_row[NLD], ld_col[NLD];
#pragma unroll
    for (int x = 0; x < NLD; ++x) {
        const int cid = tid + 256 * x;
        ld_row[x] = cid / CH;
        ld_col[x] = (cid % CH) * 8;
    }
    // A staged chunk: the 16 bytes as loaded (chunk positions past the row's whole chunks hold the row's last elements:
    // load_chunk_anyalign), except that rows of fewer than eight elements are fetched element by element and padded
    // with zeroes.
    v4u kreg[NLD], vreg[NLD];
    auto gload = [&](const half_t* __restrict__ base, int tile, v4u (&reg)[NLD]) {
        const int kb0 = tile * BC;
#pragma unroll
        for (int x = 0; x < NLD; ++x) {
            const int r = kb0 + ld_row[x];
            const half_t* __restrict__ rowp = base + (size_t)(r < Nk ? r : Nk - 1) * d;
            reg[x] = d >= 8 ? load_chunk_anyalign(rowp, ld_col[x], d) : load_chunk<false, false>(rowp, ld_col[x], d);
        }
    };
    auto put_k = [&](int buf) {
#pragma unroll
        for (int x = 0; x < NLD; ++x)
            *reinterpret_cast<v4u*>(Ks + buf * C::KBUF + ld_row[x] * SK + ((ld_col[x] * 2) ^ (C::kswz(ld_row[x]) << 4))) = kreg[x];
    };
    auto put_v = [&](int buf) {
#pragma unroll
        for (int x = 0; x < NLD; ++x)
            *reinterpret_cast<v4u*>(Vs + buf * C::VBUF + ld_row[x] * SV +
                                    ((ld_col[x] * 2) ^ (C::VSWZ ? ((ld_row[x] >> 1) & 1) << 6 : 0))) = vreg[x];
    };

    // ---- direct global -> LDS path: the tile buffers keep their layout (K rows padded or permuted, V rows with the
    // 64-byte halves exchanged in rows 2, 3 mod 4), and a request fills 64 consecutive 16-byte chunks of a buffer: lane l of
    // block x fetches whatever belongs into chunk 64 x + l (the pad chunk of a K row gets a copy of its neighbour).
    // Blocks go round the four waves; the odd K block goes to the waves that still have a block index left for it.
    // Rows shorter than the bucket: chunk positions past the row's whole chunks fetch the row's last 16 bytes (see
    // load_chunk_anyalign): for K they meet zero columns of Q, for V they only reach rows of O^T that are never stored.
    const int row_bytes = kFullD ? D * 2 : d * 2;
    const int whole_tiles = Nk / BC;  // tiles of the sequence that hold BC keys
    auto chunk_offset = [&](int c) { return kFullD ? c * 16 : (c * 8 + 8 <= d ? c * 16 : (d - 8) * 2); };
    // (narrow: every block of a tile is the wave's own, and so is the buffer; both permutations repeat every 16 rows, which are
    // CH / 4 blocks, so that only the first CH / 4 requests need offsets of their own and all others are the same some
    // multiple of 16 rows further on, which goes into the scalar base address: 66 registers less at D = 128; where 16 rows
    // of K are no whole number of blocks, 32 are)
    constexpr int NKX = kNarrow ? C::CHK : C::NKX, NVX = kNarrow ? CH : C::NVX;
    constexpr int kKeyRows = C::CHK % 4 == 0 ? 16 : 32;  // rows of K after which the offsets repeat
    constexpr int NKO = kNarrow ? C::CHK * kKeyRows / 64 : NKX, NVO = kNarrow ? CH / 4 : NVX;  // offsets held
    auto block_of = [&](int i) { return kNarrow ? i : wave + 4 * i; };
    uint32_t koff[NKO], voff[NVO];
    int krow[NKO], vrow[NVO];
    auto k_offset = [&](int i) __attribute__((always_inline)) {
        const int q = 64 * block_of(i) + lane;
        krow[i] = q / C::CK;
        const int c = q % C::CK;
        koff[i] = (uint32_t)(krow[i] * row_bytes + chunk_offset((c < C::CHK ? c : C::CHK - 1) ^ C::kswz(krow[i])));
    };
    if constexpr (kDma) {
#pragma unroll
        for (int i = 0; i < NKO && (!kNarrow || kQLoads); ++i) k_offset(i);  // (narrow: request by request, below)
#pragma unroll
        for (int i = 0; i < NVO; ++i) {
            const int q = 64 * block_of(i) + lane;
            vrow[i] = q / CH;
            const int c = q % CH;
            voff[i] = (uint32_t)(vrow[i] * row_bytes + chunk_offset(C::VSWZ ? c ^ (((vrow[i] >> 1) & 1) << 2) : c));
        }
    }
    const bool k_extra = kNarrow || C::CK % 4 == 0 || wave + 4 * (NKX - 1) < C::CK;  // the last round of K blocks exists for this wave
    auto dma_tile_parts = [&](int tile, int stage, auto k_part, auto v_part) {
        // The tile's offset joins the scalar base address, so that a request of a whole tile needs no vector
        // arithmetic at all; only the last tile of a ragged sequence adjusts rows: keys past Nk re-read key Nk - 1
        // (their scores are masked).
        const size_t tb = (size_t)tile * (size_t)(BC * row_bytes);
        const bool whole = tile < whole_tiles;
        FA_LDS char* const kst = (FA_LDS char*)smem + lds_base + stage * C::KBUF;
        FA_LDS char* const vst = (FA_LDS char*)smem + lds_base + NSTG * C::KBUF + stage * C::VBUF;
        const char* const Kb = reinterpret_cast<const char*>(Kbh) + tb;
        const char* const Vb = reinterpret_cast<const char*>(Vbh) + tb;
        auto issue = [&](auto ragged_c) {
            constexpr bool kRagged = decltype(ragged_c)::value;
            // (laundered: the compiler otherwise carries one running vector offset per request through every tile
            // for the sake of this one)
            int rows_left = Nk - tile * BC;
            if constexpr (kRagged) asm volatile("" : "+s"(rows_left));
            // request i of a tensor: offset i % n, i / n times 16 rows further on
            auto request = [&](const char* base, uint32_t off, int row, int further, FA_LDS char* dst) __attribute__((always_inline)) {
                if constexpr (kRagged) {  // (all of it in the offset, which is unsigned)
                    row += further;
                    off += (uint32_t)((further - (row >= rows_left ? row - rows_left + 1 : 0)) * row_bytes);
                } else {
                    base += (size_t)further * (size_t)row_bytes;
                }
                if constexpr (kKvOnce || kRowsOnce) dma_kib_nt(base, off, dst);
                else dma_kib(base, off, dst);
            };
#pragma unroll
            for (int i = 0; i < NKX; ++i) {
                if (!decltype(k_part)::value || (i == NKX - 1 && !k_extra)) break;
                request(Kb, koff[i % NKO], krow[i % NKO], i / NKO * kKeyRows, kst + block_of(i) * 1024);
            }
#pragma unroll
            for (int i = 0; i < NVX; ++i) {
                if (!decltype(v_part)::value) break;
                request(Vb, voff[i % NVO], vrow[i % NVO], i / NVO * 16, vst + block_of(i) * 1024);
            }
        };
        if (__builtin_expect(whole, 1)) issue(std::false_type{});
        else issue(std::true_type{});
    };
    auto dma_tile = [&](int tile, int stage) { dma_tile_parts(tile, stage, std::true_type{}, std::true_type{}); };
    // wait until every request has landed
    auto dma_wait = [&]() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };

    // Narrow at D = 64: the scores of a wave's next tile are worked out beside the exponentials of the present one
    // (tile_with_scores_ahead), since a wave alone on its SIMD otherwise leaves the vector unit idle for every MFMA and the matrix
    // unit for every exponential.  One tile after the other -> ahead: B1 H8 N1024 d64 7.8 -> 7.55 us, N2048 causal 15.1 -> 14.4, B2 H3 N1792
    // 19.2 -> 18.2, B1 H8 N1024 d40 7.45 -> 6.7, d63 causal with bias 13.7 -> 12.8; one tile per wave +-0.  At D = 32, where K Q^T is four
    // MFMAs and two work-groups share a CU, it is +1 ... -3 %; above D = 64 there is no second stage for K.  With dropout
    // the Philox rounds stand beside the MFMAs already.
    constexpr bool kAheadQk = kNarrow && D == 64 && !kDropout;

    // ---- accumulators
    v16f oacc[MB][NB];
    float m_ref[NB], m_thr[NB], l_run[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        m_ref[nb] = kNothingSeen;
        m_thr[nb] = -INFINITY;
        l_run[nb] = 0.0f;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[mb][nb][r] = 0.0f;
    }

    // Scores leave the MFMA unscaled.  With a positive scale the scaling commutes with the row maximum and is folded
    // into the exponent (one fma per score): cs = scale, and the ALiBi bias is added beforehand divided by the scale.
    // A non-positive scale is served by the kEvery instance alone (the host sends it there): then the scores are
    // scaled first and cs = 1.
    const float c2 = a.scale_log2;
    const bool scale_late = !kEvery || c2 > 0.0f;
    const float cs = scale_late ? c2 : 1.0f;
    const float inv_cs = __builtin_amdgcn_rcpf(cs);  // (of the raise threshold alone: whether a row is rescaled is no matter of its last bit)
    // The ALiBi slope of the head is read once the first tile requests are on their way (read_slope below): nothing before the
    // first softmax needs it.  Narrow: by the scalar unit, whose loads have a count of their own; the wait for a vector load takes in
    // every tile request, V(1) among them (causal B1 H8 N1021 d63 12.8 -> 10.9 us, d31 8.7 -> 7.7, B1 H4 N600 d80 9.3 -> 8.3 together with
    // what Q gains below).  The others wait for two tiles first anyway, and lose 1-3 % by a slope in a scalar register.
    float slope2 = 0.0f, nsig = 0.0f;

    // ALiBi where every visible key lies at or left of its row (causal mask, or a right window of 0: j <= i, keys right
    // of the row are masked anyway): |i - j| = i - j splits into a part that only depends on the accumulator register,
    // -nsig * (8 (r / 4) + r % 4), and a part per lane and 32-key block.  The first goes into the MFMA as the initial
    // accumulator value, the second into the addend of the exponent fma: no instruction per score is left.
    constexpr bool kFoldAlibi = kAlibi && kVec && (VAR & kVarAlibiLeft) != 0;
    static_assert(!kAheadQk || !kFoldAlibi, "scores worked out ahead start from zero");
    v16f calib;
    auto read_slope = [&]() {
        if constexpr (kAlibi) {
            // (only the kEvery instance is launched without a slope table)
            slope2 = (!kEvery || a.alibi) ? (kNarrow ? read_uniform(a.alibi + a.head(bh)) : a.alibi[a.head(bh)]) * kLog2e : 0.0f;
            nsig = scale_late ? -slope2 / c2 : 0.0f;
            if constexpr (kFoldAlibi) {
#pragma unroll
                for (int r = 0; r < 16; ++r) calib[r] = -nsig * (float)(8 * (r >> 2) + (r & 3));
            }
        }
    };

    // dropout: the parts of the Philox calls that depend on the row alone and on the call alone (common.h)
    PhiloxRow drop_row[NB];
    CallTable calls;
    v4u first_part;  // of the tile at hand
    if constexpr (kDropout) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) drop_row[nb] = philox_row_part((uint32_t)row_i[nb], (uint32_t)bh, a.seed_lo);
        constexpr int kWaves = kPair ? 8 : 4;
        calls.mem = call_table_memory<kWaves>() + 64 * (kPair ? 4 * half + wave : wave);
        calls.chunk = -1;
    }

    // debug dump of the tile's keep decisions: the words once more, so that the ordinary path need not keep them
    auto dump_keep = [&](int kb0) {
        if constexpr (kDropout) {
            if (__builtin_expect(a.keep_out == nullptr, 1)) return;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const int ln = lane_here(), g = ln >> 5, row = q0 + wave_row0 + nb * 32 + (ln & 31);
                if (row >= Nq) continue;
                uint8_t* const kout = a.keep_out + ((size_t)bh * Nq + row) * Nk;
#pragma unroll 1
                for (int jg = 0; jg < BC; jg += 16) {
                    const v4u w = philox_from_parts(drop_row[nb], calls.at(kb0, jg, g), a.seed_lo, a.seed_hi);
#pragma unroll
                    for (int f = 0; f < 8; ++f) {
                        const int j = kb0 + jg + 8 * (f >> 2) + 4 * g + (f & 3);
                        if (j < Nk) kout[j] = philox_field16(w, f) >= a.drop_thr ? 1 : 0;
                    }
                }
            }
        }
    };

    // LDS read offsets of this lane
    const int k_rd = l32 * SK + (C::kPadK ? g * 16 : 0);                         // + kb*32*SK + k_step(ks)
    const int k_ch = C::kPadK ? 0 : (g ^ C::kswz(l32)) << 4;
    auto k_step = [&](int ks) { return (ks * 32) ^ k_ch; };
    const int v_rd = (4 * g + ((lane & 15) >> 2)) * SV + (((lane >> 4) & 1) * 16 + (lane & 3) * 4) * 2;  // + row/col blocks
    const int v_sw = C::VSWZ ? ((lane >> 3) & 1) << 6 : 0;

    // S^T = K Q^T of the tile in K buffer `buf`
    auto qk = [&](int buf, v16f (&s)[2][NB]) {
        constexpr bool folded = kFoldAlibi;
        constexpr bool kInOrder = NB == 1 && (folded || (D == 32 && !kAlibi && !kDropout && !kNarrow && !kPair && !kFullD) ||
                                              (D == 96 && kNarrow && kAlibi && kDropout));
        const char* kbase = Ks + buf * C::KBUF + k_rd;
        // Written out in issue order, fenced step by step -- three fragments ahead, then MFMA and read in turn -- where the issue-order
        // groups at the end of this function do not do:
        //  * with the bias in the accumulator the first k-step's MFMAs are inline asm (below), which the groups cannot name: with
        //    them in the stream the compiler fell back to waiting for every fragment right behind its request;
        //  * at D = 32, where there are four MFMAs, the groups are lost in the plain instances as soon as what is around them changes,
        //    and the compiler requests two fragments, waits for both, and does the same again.  So -> written out: causal B5 H2 Nq60 Nk5905 d31
        //    (split) 11.0 -> 10.85 us, B1 H8 Nq200 Nk8000 d31 (split) 13.85 -> 13.5, B8 H16 N2000 d31 window of 128 keys 20.4 -> 20.2, causal B4
        //    H16 N700 d24 9.40 -> 9.27.  Rows of the bucket's width hide the waits behind other waves, and lose 1-2 % by the
        //    fences (B15 H64 H_kv8 N107 d32 7.25 -> 7.39, B4 H8 N2000 32.1 -> 32.5); the paired and narrow ones have their order;
        //  * nor, for the same reason, in the narrow instance of D = 96 with ALiBi and dropout: causal B1 H8 N640 9.72 -> 9.39 us, B1 H4 N1000
        //    11.74 -> 11.31, B1 H8 N1021 without a mask 11.98 -> 11.56.
        if constexpr (kInOrder) {
            constexpr int n = 2 * KS, kAhead = 3;  // step i: k-step i / 2, key block i % 2
            v8h af[n];
#pragma unroll
            for (int i = 0; i < kAhead; ++i) af[i] = *reinterpret_cast<const v8h*>(kbase + (i & 1) * 32 * SK + k_step(i >> 1));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < n; ++i) {
                const int ks = i >> 1, kb = i & 1;
                const v16f z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
                if constexpr (folded) {
                    if (ks == 0) asm("v_mfma_f32_32x32x16_f16 %0, %1, %2, %3" : "=&v"(s[kb][0]) : "v"(af[i]), "v"(qf[0][ks]), "v"(calib));
                }
                if (ks == 0 && !folded) s[kb][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], qf[0][ks], z, 0, 0, 0);
                if (ks > 0) s[kb][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], qf[0][ks], s[kb][0], 0, 0, 0);
                if (i + kAhead < n)
                    af[i + kAhead] = *reinterpret_cast<const v8h*>(kbase + ((i + kAhead) & 1) * 32 * SK + k_step((i + kAhead) >> 1));
                __builtin_amdgcn_sched_barrier(0);
            }
            return;
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                const v8h af = *reinterpret_cast<const v8h*>(kbase + kb * 32 * SK + k_step(ks));
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    if (ks == 0) {
                        // first k-step: the accumulator starts from zero (an inline constant) or, with the ALiBi bias
                        // folded in, from the per-register bias constants, which stay where they are
                        if constexpr (folded) {
                            // written out: the compiler only knows the form whose result overwrites the addend and would
                            // copy the sixteen constants for every tile.  Hazards of an MFMA the compiler cannot see as
                            // one: its operands are ready (the asm's inputs: af comes with the wait for its LDS read,
                            // qf and calib were written long before); its result is next read as the addend of the
                            // second k-step's MFMA on the same registers, a dependency the hardware interlocks -- hence
                            // at least two k-steps -- and by VALU code only after that one.
                            static_assert(!folded || KS >= 2, "the score accumulator is first read by a following MFMA");
                            asm("v_mfma_f32_32x32x16_f16 %0, %1, %2, %3" : "=&v"(s[kb][nb]) : "v"(af), "v"(qf[nb][ks]), "v"(calib));
                        } else {
                            const v16f z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
                            s[kb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af, qf[nb][ks], z, 0, 0, 0);
                        }
                    } else {
                        s[kb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af, qf[nb][ks], s[kb][nb], 0, 0, 0);
                    }
                }
            }
        }
        // issue order: kQkAhead fragment reads first, then read and MFMA in turn (left to itself the compiler waits
        // for each fragment right after requesting it)
        if constexpr (NB == 1) {
            constexpr int kQkAhead = 3, n = 2 * KS;
            __builtin_amdgcn_sched_group_barrier(0x100, kQkAhead, 0);
#pragma unroll
            for (int i = 0; i < n - kQkAhead; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, kQkAhead, 0);
        }
    };

    // online softmax of one tile (per query row = per lane); leaves P^T packed to fp16 in pf
    // masked: some row of the wave does not see all of the tile (wave-uniform)
    // ahead: stops in front of the exponentials (tile_with_scores_ahead below has them)
    auto softmax = [&](bool masked, int kb0, v16f (&s)[2][NB], v8h (&pf)[2][2][NB], auto ahead) __attribute__((always_inline)) {
        constexpr bool folded = kFoldAlibi;
        if constexpr (kDropout) calls.cover(kb0, lane, (uint32_t)bh, a.off_lo, a.seed_lo, a.seed_hi);
        if constexpr (kDropout && !kEvery) first_part = calls.at(kb0, 0, g);  // (in time for pv)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            // folded ALiBi: bias of 32-key block kb that is common to the lane's 16 scores there (score units)
            float abias[2] = {0.0f, 0.0f};
            if constexpr (folded) {
                abias[0] = nsig * (iif[nb] - (float)(kb0 + 4 * g));
                abias[1] = abias[0] - nsig * 32.0f;
            }
            if constexpr (kAlibi && !folded) {
                // score*scale - slope*|i - j|  (src/main.cu:315,324), in the log2 domain
                const float jb = (float)(kb0 + 4 * g) - iif[nb];
                if (scale_late) {
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            s[kb][nb][r] = __builtin_fmaf(nsig, __builtin_fabsf(jb + (float)(32 * kb + 8 * (r >> 2) + (r & 3))), s[kb][nb][r]);
                } else {
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            s[kb][nb][r] = s[kb][nb][r] * c2 - slope2 * __builtin_fabsf(jb + (float)(32 * kb + 8 * (r >> 2) + (r & 3)));
                }
            }
            if (__builtin_expect(masked, 0)) {
                // (common.h: mask_tile.)  The bounds of the wave's rows run along block diagonals when they move by one key per
                // row and start at a multiple of 32: causal masks and windows whose offsets are multiples of 32, rows not
                // clipped by a sequence or split end.
                // (kb0 is laundered: the compiler otherwise carries what it makes of it here through every tile)
                asm volatile("" : "+s"(kb0));
                const int sides = mask_sides(kb0, lo_max, hi_min);
                int modes, lo_rel, hi_rel;
                if (NB != 1 || mask_is_general(sides, diagonals)) {
                    const int ln = lane_here();
                    int lo, hi;
                    row_bounds(q0 + wave_row0 + nb * 32 + (ln & 31), &lo, &hi);
                    lo_rel = lo - kb0 - 4 * (ln >> 5);
                    hi_rel = hi - kb0 - 4 * (ln >> 5);
                    modes = mask_modes_general(sides);
                } else {
                    asm("" : "=v"(lo_rel), "=v"(hi_rel));  // (not read)
                    modes = mask_modes_diagonal(kb0, sides, lo_min, hi_min);
                }
                mask_tile<NB == 1>(s[0][nb], s[1][nb], wave_uniform(modes), lo_rel, hi_rel, -INFINITY);
            }
            if constexpr (kEvery) {
                if (a.scores_out != nullptr && row_i[nb] < Nq) {  // debug dump of the visible scores, natural-log units
                    float* srow = a.scores_out + ((size_t)bh * Nq + row_i[nb]) * Nk;
                    int lo, hi;
                    row_bounds(row_i[nb], &lo, &hi);
                    const float unit = (scale_late ? cs : 1.0f) * kLn2;
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const int j = kb0 + 4 * g + 32 * kb + 8 * (r >> 2) + (r & 3);
                            if (j >= lo && j <= hi) srow[j] = s[kb][nb][r] * unit;
                        }
                }
            }
            // Row maximum of the lane's own scores (half of the row's keys: the other half sits in lane l ^ 32), two chains side
            // by side.  Whether some row outgrows the running maximum is asked without the exchange between the two lanes and
            // in score units, against a threshold that is worked out where the maximum is raised: one comparison per tile,
            // where exchange, scaling and sum took ten dependent instructions.
            float mk[2] = {-INFINITY, -INFINITY};
#pragma unroll
            for (int r = 0; r < 16; ++r)
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) mk[kb] = fmaxf(mk[kb], s[kb][nb][r]);
            float mx = folded ? fmaxf(mk[0] + abias[0], mk[1] + abias[1]) : fmaxf(mk[0], mk[1]);
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(mx > m_thr[nb]) != 0ull, 0)) {
                const float m_new = fmaxf(m_ref[nb], xhalf_max(mx) * cs);  // cs > 0
                float alpha = fast_exp2(m_ref[nb] - m_new);
                asm volatile("; raise running max" : "+v"(alpha));  // keeps the rescale inside this rare branch
                m_ref[nb] = m_new;
                m_thr[nb] = (m_new + kLazyTau) * inv_cs;
                l_run[nb] *= alpha;
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                    for (int r = 0; r < 16; ++r) oacc[mb][nb][r] *= alpha;
            }
            if constexpr (decltype(ahead)::value) continue;
            float rs = 0.0f;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                const float addend = folded ? __builtin_fmaf(abias[kb], cs, -m_ref[nb]) : -m_ref[nb];
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float p = fast_exp2(__builtin_fmaf(s[kb][nb][r], cs, addend));
                    rs = kb == 0 && r == 0 ? p : rs + p;
                    s[kb][nb][r] = p;
                }
            }
            l_run[nb] += rs;  // per-lane partial; the two half-waves are added in the epilogue
            if constexpr (kDropout && kEvery) {  // (the other instances: pv below)
                // drop iff field < threshold, row sum left undropped (src/flash_forward.h:221-237); the survivors' factor
                // 1/(1-p) is common to the whole row and multiplies O once in the epilogue instead of every score here
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        // the lane's eight keys among the 16 from kb0 + 32 kb + 16 q on: field f belongs to the (8*(f>>2) + 4*g + (f&3))th
                        const v4u w = philox_from_parts(drop_row[nb], calls.at(kb0, 32 * kb + 16 * q, g), a.seed_lo, a.seed_hi);
#pragma unroll
                        for (int f = 0; f < 8; ++f) {
                            const int r = 8 * q + f;
                            s[kb][nb][r] = philox_field16(w, f) >= a.drop_thr ? s[kb][nb][r] : 0.0f;
                        }
                    }
            }
            if constexpr (!(kDropout && !kEvery)) {  // (there pv packs them)
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                        for (int e = 0; e < 8; e += 2) {
                            const v2h h2 = pack_f16(s[kb][nb][8 * tt + e], s[kb][nb][8 * tt + e + 1]);
                            pf[kb][tt][nb][e] = h2[0];
                            pf[kb][tt][nb][e + 1] = h2[1];
                        }
            }
        }
    };

    // V^T fragment of the tile in V buffer `buf`: keys 32 kb + 16 tt ... + 15, columns of block mb
    // (a lane's rows all share bit 1 of the row index: the swizzle is one per-lane choice between two bases)
    auto v_frags = [&](int buf) __attribute__((always_inline)) {
        const char* const b0 = Vs + buf * C::VBUF + v_rd + v_sw;
        const char* const b1 = Vs + buf * C::VBUF + v_rd + (v_sw ^ (C::VSWZ ? 64 : 0));
        return [=](int kb, int tt, int mb) __attribute__((always_inline)) {
            const char* p0 = C::VSWZ ? ((mb & 1) ? b1 : b0) + (32 * kb + 16 * tt) * SV + (mb >> 1) * 128 : b0 + (32 * kb + 16 * tt) * SV + mb * 64;
            union { v4hp p[2]; v8h v; } af;
            af.p[0] = __builtin_amdgcn_ds_read_tr16_b64_v4f16((FA_LDS v4hp*)(p0));
            af.p[1] = __builtin_amdgcn_ds_read_tr16_b64_v4f16((FA_LDS v4hp*)(p0 + 8 * SV));
            return af.v;
        };
    };

    // O^T += V^T P^T with the tile in V buffer `buf`
    auto pv = [&](int buf, int kb0, v16f (&s)[2][NB], v8h (&pf)[2][2][NB]) {
        auto v_frag = v_frags(buf);
        if constexpr (kDropout && !kEvery) {
            // Dropout, 16 keys at a time (a step): drop iff field < threshold, row sum left undropped
            // (src/flash_forward.h:221-237); the survivors' factor 1/(1-p) is common to the whole row and multiplies O once in
            // the epilogue.  The steps are fenced off from each other, so that the matrix units work on one step while the
            // vector unit is at the next one's Philox rounds: left to itself the compiler put all MFMAs behind all rounds.
            static_assert(NB == 1, "one row per lane");
            v4u part = first_part;
#pragma unroll
            for (int st = 0; st < 4; ++st) {
                const int kb = st >> 1, q = st & 1;
                v8h af[MB];
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) af[mb] = v_frag(kb, q, mb);
                const v4u mine = part;
                if (st < 3) part = calls.at(kb0, 16 * (st + 1), g);
                __builtin_amdgcn_sched_barrier(0);
                // the lane's eight keys among the step's 16: field f belongs to the (8*(f>>2) + 4*g + (f&3))th.  Registers 8q + 2k
                // and 8q + 2k + 1 become one packed fp16 word, fields 2k and 2k + 1 are the halves of Philox word k: the
                // decisions are applied to the packed word (keep_pair)
                const v4u w = philox_from_parts(drop_row[0], mine, a.seed_lo, a.seed_hi);
                v8h p;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    union { v2h h; uint32_t u; } pk;
                    pk.h = pack_f16(s[kb][0][8 * q + 2 * k], s[kb][0][8 * q + 2 * k + 1]);
                    pk.u = keep_pair(pk.u, w[k], a.drop_sub2);
                    p[2 * k] = pk.h[0];
                    p[2 * k + 1] = pk.h[1];
                }
                settle_for_mfma(p);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) oacc[mb][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[mb], p, oacc[mb][0], 0, 0, 0);
            }
            return;
        }
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) {
                    const v8h af = v_frag(kb, tt, mb);
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb)
                        oacc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af, pf[kb][tt][nb], oacc[mb][nb], 0, 0, 0);
                }
            }
        }
    };

    // A wave alone on its SIMD: what softmax leaves to do of the tile whose scores (rows raised) are in s, and P V with it, while the
    // matrix unit is at the scores of the tile to come, K in buffer kbuf.  The exponents leave the score registers first, so that
    // the next scores take their place; then the MFMAs of K Q^T stand between the exponentials of the first 32 keys, and those of
    // their P V between the exponentials of the others, step by step behind fences.  (The last tile has no successor: what is
    // in the buffer then is multiplied all the same, and not looked at.)
    auto tile_with_scores_ahead = [&](int vbuf, int kbuf, v16f (&s)[2][NB]) __attribute__((always_inline)) {
        constexpr int n = 2 * KS, kAhead = 3;  // step i: k-step i / 2, key block i % 2
        const char* const kbase = Ks + kbuf * C::KBUF + k_rd;
        auto v_frag = v_frags(vbuf);
        // (the fences order nothing that only computes; what passes through here is worked out by then)
        auto pin = [](auto& v) __attribute__((always_inline)) { asm volatile("" : "+v"(v)); };
        auto k_frag = [&](int i) { return *reinterpret_cast<const v8h*>(kbase + (i & 1) * 32 * SK + k_step(i >> 1)); };
        v8h kf[n], vf[2 * 2 * MB];
        union { uint32_t u[4]; v8h h; } p[2][2];
        float x[2][16], rs = 0.0f;
#pragma unroll
        for (int i = 0; i < kAhead; ++i) kf[i] = k_frag(i);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                x[kb][r] = __builtin_fmaf(s[kb][0][r], cs, -m_ref[0]);
                pin(x[kb][r]);
            }
        __builtin_amdgcn_sched_barrier(0);
        // exponentials of scores r0 ... r0 + count - 1 of a key block, each pair packed
        auto exps = [&](int kb, int r0, int count) __attribute__((always_inline)) {
#pragma unroll
            for (int r = r0; r < r0 + count; r += 2) {
                const float p0 = fast_exp2(x[kb][r]), p1 = fast_exp2(x[kb][r + 1]);
                rs = kb == 0 && r == 0 ? p0 + p1 : rs + p0 + p1;
                union { v2h h; uint32_t u; } two;
                two.h = pack_f16(p0, p1);
                pin(two.u);
                pin(rs);
                p[kb][r >> 3].u[(r & 7) >> 1] = two.u;
            }
        };
        constexpr int kPer = 16 / n & ~1;  // scores per step of K Q^T
#pragma unroll
        for (int i = 0; i < n; ++i) {
            const v16f z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
            s[i & 1][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[i], qf[0][i >> 1], i < 2 ? z : s[i & 1][0], 0, 0, 0);
            if (i + kAhead < n) kf[i + kAhead] = k_frag(i + kAhead);
            // the first fragments of V behind the last ones of K
            else if (i + kAhead - n < 2 * MB) vf[i + kAhead - n] = v_frag(0, (i + kAhead - n) / MB, (i + kAhead - n) % MB);
            exps(0, kPer * i, i == n - 1 ? 16 - kPer * i : kPer);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = kAhead; i < 2 * MB; ++i) vf[i] = v_frag(0, i / MB, i % MB);
        constexpr int kPerV = 16 / (2 * MB);
#pragma unroll
        for (int i = 0; i < 2 * MB; ++i) {
            oacc[i % MB][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[i], p[0][i / MB].h, oacc[i % MB][0], 0, 0, 0);
            vf[2 * MB + i] = v_frag(1, i / MB, i % MB);
            exps(1, kPerV * i, kPerV);
            __builtin_amdgcn_sched_barrier(0);
        }
        l_run[0] += rs;
#pragma unroll
        for (int i = 0; i < 2 * MB; ++i)
            oacc[i % MB][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[2 * MB + i], p[1][i / MB].h, oacc[i % MB][0], 0, 0, 0);
    };

    // The Q fragments must have landed before the loop starts: a load still counted as outstanding at the loop
    // header makes the compiler guard every use of qf inside the loop with a vmcnt wait, and since vmcnt counts in
    // order, that wait would also drain the K/V prefetch of the same iteration.
    auto pin_q = [&]() {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qf[nb][ks]));
    };

    // ---- loop over the key tiles
    // A wave whose rows all lie past Nq (fewer than 128 query rows: short prompts, or the heads of one K/V head decoding
    // together) only helps to stage the tiles, and so does any wave for a tile that none of its rows can see (the far
    // end of the causal diagonal block, the near end of a sliding window).
    auto tile_live = [&](int t) { return (unsigned)(t - live0) < (unsigned)nlive; };
    auto tile_masked = [&](int t) { return (unsigned)(t - clean0) >= (unsigned)nclean; };
    auto tile_math = [&](int t, int buf) {
        if (__builtin_expect(tile_live(t), 1)) {
            v16f s[2][NB];
            v8h pf[2][2][NB];
            const int kb0 = (tile_begin + t) * BC;
            qk(buf, s);
            softmax(tile_masked(t), kb0, s, pf, std::false_type{});
            pv(buf, kb0, s, pf);
            dump_keep(kb0);
        }
    };
    if constexpr (kNarrow) {
        // Wave w walks the tiles w, w + 4, ... with two stages of its own: tile n + 2 is requested into the stage of
        // tile n as soon as that tile's fragments have been read, and before tile n + 1 is touched its requests (older
        // than those of tile n + 2) have been waited for.  No other wave reads or writes these buffers.
        const int nt = wave < ntiles ? (ntiles - wave + 3) / 4 : 0;
        static_assert(NKX + NVX <= 63, "vmcnt immediate");
        // In front of tile 0 the wave waits for no more than Q, K(0) and, with two stages, V(0).  Q comes straight into LDS too: loaded
        // into registers, it is waited for by a count that takes in every younger request, and comes in 16-byte pieces of 32 rows
        // where these are whole ones.  With one stage it lies where V will be, whose request follows once Q is in registers (an
        // area of its own and V requested at once: d96 -2 %, all waves' K then arrive behind some V).  With two stages V(1) goes
        // out with the rest where rows are aligned; requests at 2-byte alignment take 15 ns per KiB and CU to issue where others take
        // 5, so there it waits for its turn.
        auto request = [&](int n, int stage, auto k_part) {
            if (n < nt) dma_tile_parts(tile_begin + wave + 4 * n, stage, k_part, std::integral_constant<bool, !decltype(k_part)::value>{});
        };
        constexpr std::true_type k_part{};
        constexpr std::false_type v_part{};
        if constexpr (kQLoads) {
            // (written as for any number of stages: as one statement the compiler puts the address arithmetic between the
            // requests, and N1024 takes 8.12 us instead of 7.83)
#pragma unroll
            for (int u = 0; u < NSTG; ++u)
                if (u < nt) dma_tile(tile_begin + wave + 4 * u, u);
        } else if (nt > 0) {
            const char* const Qb = reinterpret_cast<const char*>(Qbh) + (size_t)q0 * (size_t)row_bytes;
            const int rows_left = Nq - q0;
            static_assert(NKO <= C::CHK / 2, "offsets");
            // (each offset is worked out right in front of its request; rows past Nq re-read the last one)
#pragma unroll
            for (int i = 0; i < C::CHK / 2; ++i) {
                if (i < NKO) k_offset(i);
                asm volatile("" : "+v"(koff[i % NKO]));
                const int further = i / NKO * kKeyRows;
                const int over = max(krow[i % NKO] + further - (rows_left - 1), 0);
                dma_kib(Qb, koff[i % NKO] + (uint32_t)__mul24(further - over, row_bytes), (FA_LDS char*)smem + kQLds + wave * kQWave + i * 1024);
            }
            request(0, 0, k_part);
            if constexpr (NSTG == 2) {
                request(0, 0, v_part);
                request(1, 1, k_part);
                if constexpr (kVec) request(1, 1, v_part);
            }
        }
        stamps.take(1);
        if constexpr (kStamp) __builtin_amdgcn_sched_barrier(0);  // (ahead of the work on Q, whose wait drains the requests too)
        set_bounds();
        read_slope();
        if (NSTG == 2 && nt > 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NKX + (kVec ? NVX : 0)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if constexpr (!kQLoads) {
            const char* const qbase = smem + kQLds + wave * kQWave + k_rd;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const v4u raw = *reinterpret_cast<const v4u*>(qbase + k_step(ks));
                const int col = 16 * ks + 8 * g;
                const v4u z = {0u, 0u, 0u, 0u};
                union { v4u u; v8h h; } t;
                t.u = kFullD || 16 * ks + 16 <= D - 32 || col < d ? raw : z;
                // (d > D - 32: the columns before are all there)
                qf[0][ks] = kVec || 16 * ks + 16 <= D - 32 ? t.h : mask_q_chunk_anyalign(raw, col, d);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        pin_q();
        if constexpr (!kQLoads && (NSTG == 1 || !kVec)) request(NSTG - 1, NSTG - 1, v_part);
        stamps.take(2);
        stamps.take(3);  // (no barrier in front of the loop)
        if constexpr (kAheadQk) {
            // K runs one tile ahead of V.  At the end of tile n the stage buffers K(n + 1) and V(n) have been read, K(n + 2) and V(n + 1)
            // are on their way, K(n + 3) and V(n + 2) are requested.
            v16f s[2][NB];
            v8h none[2][2][NB];
            if (nt == 1) {  // (no successor whose scores could be worked out)
                tile_math(wave, 0);
                stamps.take(4);
            } else if (nt > 1) {
                qk(0, s);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                request(2, 0, k_part);
                if (nt > 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NVX + NKX) : "memory");  // K(1)
                else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NVX) : "memory");
                int buf = 0, n = 0;
                do {
                    const int t = wave + 4 * n;
                    softmax(tile_masked(t), (tile_begin + t) * BC, s, none, std::true_type{});
                    tile_with_scores_ahead(buf, buf ^ 1, s);
                    if (kStamp && n == 0) stamps.take(4);
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    request(n + 2, buf, v_part);
                    request(n + 3, buf ^ 1, k_part);
                    if (n + 3 < nt) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NKX + NVX) : "memory");
                    else if (n + 2 < nt) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NVX) : "memory");
                    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    buf ^= 1;
                } while (++n < nt);
            }
        } else if constexpr (NSTG == 2) {
            int buf = 0;
            for (int n = 0; n < nt; ++n) {
                tile_math(wave + 4 * n, buf);
                if (kStamp && n == 0) stamps.take(4);
                if (n + 2 < nt) {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the stage has been read
                    dma_tile(tile_begin + wave + 4 * (n + 2), buf);
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NKX + NVX) : "memory");
                } else {
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                }
                buf ^= 1;
            }
        } else {
            // One stage: K(n + 1) is requested as soon as the scores of tile n are out of the K buffer, V(n + 1) as soon
            // as the V buffer has been read; each is waited for right before its first use, the younger request of the
            // other tensor staying in flight.
            // (One body per kind of tile: with the scores' two halves each under a condition of their own the compiler copied
            // the 32 scores once per tile, and a wave alone on its SIMD hides none of that: B1 H8 Nq280 Nk9850 d128 62.3 us, with bodies apart
            // 49.5; d96 54.1 and 42.2; causal B1 H4 N640 d128 9.5 and 8.5.)
            auto step = [&](int n, auto live_c) {
                constexpr bool kLive = decltype(live_c)::value;
                const int t = wave + 4 * n;
                const bool more = n + 1 < nt;
                v16f s[2][NB];
                v8h pf[2][2][NB];
                if constexpr (kLive) qk(0, s);
                if (more) {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    dma_tile_parts(tile_begin + wave + 4 * (n + 1), 0, std::true_type{}, std::false_type{});
                }
                if constexpr (kLive) softmax(tile_masked(t), (tile_begin + t) * BC, s, pf, std::false_type{});
                // V(n): older than the K request just issued
                if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NKX) : "memory");
                else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                if constexpr (kLive) {
                    pv(0, (tile_begin + t) * BC, s, pf);
                    dump_keep((tile_begin + t) * BC);
                }
                if (kStamp && n == 0) stamps.take(4);
                if (more) {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    dma_tile_parts(tile_begin + wave + 4 * (n + 1), 0, std::false_type{}, std::true_type{});
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NVX) : "memory");  // K(n + 1) is there
                }
            };
            for (int n = 0; n < nt; ++n) {
                if (tile_live(wave + 4 * n)) step(n, std::true_type{});
                else step(n, std::false_type{});
            }
        }
    } else if constexpr (kDma) {
        // Tile t + 2 is requested when tile t is done (its stage has been read, behind a barrier); before the barrier that ends
        // tile t, the requests of tile t + 1 have landed.
        // Before tile 0 every stage is free: the prologue requests one tile per stage, so that the request which
        // tile 0 would issue is already on its way (a work-group with few tiles otherwise pays the memory latency a
        // second time at the end of its first tile).
        // With ALiBi and every visible key at or left of its row the tiles are walked from the last to the first: the bias
        // grows towards the row, so in rising order the row maximum outgrew kLazyTau, and O was rescaled, in tile after
        // tile.  Causal window of 1650 keys B9 H3 N5649 d72: 112.3 -> 104.4 us, B4 H4 N3392 d128 with 704 keys 32.8 -> 31.0,
        // B2 H16 N4096 d64 with 256 keys (a third of whose heads rescaled per tile) 23.8 -> 23.3.
        auto nth = [&](int t) {
            const int i = kPair ? 2 * t + half : t;
            return kFoldAlibi ? ntiles - 1 - i : i;
        };
        // (paired: both halves go round as often, for the barrier; the second one's last tile may not exist)
        auto there = [&](int t) { return !kPair || 2 * t + half < ntiles; };
        const int rounds = kPair ? (ntiles + 1) / 2 : ntiles;
        static_assert(NSTG == 2, "a stage that is read and one that is filled");
        // (Launches whose every tile has one reader take them from HBM, all work-groups at once: they request the second tile only
        // when the first one is there, since both at once arrive in twice the time of one.  B8 H32 H_kv8 Nq1 Nk5003 d128 30.6 -> 29.4
        // us, B1 H32 H_kv8 Nq16 Nk8192 d128 17.3 -> 16.8, B16 H32 H_kv4 Nq3 Nk6000 d80 24.4 -> 23.9; other split launches +-1 %, paired
        // work-groups, whose halves have a tile each on its way, -2 %.)
        constexpr bool late = (kFold || kKvOnce) && !kPair;
        auto second_tile = [&](bool now) {
            if (now && 1 < rounds && there(1)) dma_tile(tile_begin + nth(1), 1);
        };
        if (0 < rounds && there(0)) dma_tile(tile_begin + nth(0), 0);
        second_tile(!late);
        set_bounds();
        read_slope();
        stamps.take(1);
        dma_wait();
        pin_q();
        stamps.take(2);
        second_tile(late);
        __syncthreads();
        stamps.take(3);
        int buf = 0;  // stage of tile t
        for (int t = 0; t < rounds; ++t) {
            if (there(t)) tile_math(nth(t), buf);
            if (kStamp && t == 0) stamps.take(4);
            dma_wait();
            __syncthreads();
            // (the request stands at the end so that the first tile, whose successor is on its way already, is no case of its own:
            // a copy of the tile's code costs a launch of few tiles its way through a cold instruction cache)
            if (kPair ? there(t + 2) : t + 2 < ntiles) dma_tile(tile_begin + nth(t + 2), buf);
            buf ^= 1;
        }
    } else {
        // double-buffered through registers: tile t+1 is fetched from global memory while tile t is computed
        if (ntiles > 0) {
            gload(Kbh, tile_begin, kreg);
            gload(Vbh, tile_begin, vreg);
        }
        set_bounds();
        read_slope();
        if (ntiles > 0) {
            stamps.take(1);
            put_k(0);
            put_v(0);
        }
        pin_q();
        stamps.take(2);
        __syncthreads();
        stamps.take(3);
        for (int t = 0; t < ntiles; ++t) {
            const int cur = t & 1;
            const bool has1 = t + 1 < ntiles;
            if (has1) {
                gload(Kbh, tile_begin + t + 1, kreg);
                gload(Vbh, tile_begin + t + 1, vreg);
            }
            tile_math(t, cur);
            if (kStamp && t == 0) stamps.take(4);
            if (has1) {
                put_k(cur ^ 1);
                put_v(cur ^ 1);
            }
            __syncthreads();
        }
    }

    stamps.take(5);
    auto store_stamps = [&]() {
        if constexpr (kStamp) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the result stores of this wave have left
            stamps.take(6);
            stamps.store(a.stamps, ntiles);
        }
    };

    if constexpr (kNarrow) {
        // ---------------- merge of the four waves' partial results (same rows, disjoint keys), then O and LSE.
        // Like the combine of split partials: weights 2^(m_w - M) on the row sums and on the unnormalised O.
        __syncthreads();  // every wave is done with its tile buffers
        float* const sm = reinterpret_cast<float*>(smem);  // [4][32] running maxima (log2 units)
        float* const sl = sm + 4 * 32;                      // [4][32] row sums
        // (Rows four floats apart from each other's banks, four columns per access and 8-byte stores of O: with a stride of D every
        // row of a store began at the same bank, and single floats and halves took 2 us of a launch.  B1 H8 N1021 d31 9.07 -> 8.45
        // us, B1 H8 N1024 d64 8.55 -> 7.76, d128 13.2 -> 11.6, B1 H4 N700 d100 causal 15.5 -> 11.4, B2 H4 N256 d64 5.47 -> 4.41.)
        constexpr int SM = D + 4;
        float* const so = sl + 4 * 32;                      // [4][32][SM] unnormalised O, by chunk position
        static_assert((2 * 4 * 32 + 4 * 32 * SM) * 4 <= 4 * kWaveLds, "merge buffers fit the tile buffers");
        const float l = xhalf_sum(l_run[0]);
        if (g == 0) {
            sm[wave * 32 + l32] = m_ref[0];
            sl[wave * 32 + l32] = l;
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int rg = 0; rg < 4; ++rg) {
                const v4f o = {oacc[mb][0][4 * rg], oacc[mb][0][4 * rg + 1], oacc[mb][0][4 * rg + 2], oacc[mb][0][4 * rg + 3]};
                *reinterpret_cast<v4f*>(so + (wave * 32 + l32) * SM + 32 * mb + 8 * rg + 4 * g) = o;
            }
        __syncthreads();
        // eight threads per row, four consecutive chunk positions at a time: 128 bytes of each partial result per row and read
        const int row = tid >> 3;
        float M = kNothingSeen;
#pragma unroll
        for (int w = 0; w < 4; ++w) M = fmaxf(M, sm[w * 32 + row]);
        float L = 0.0f, wgt[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            wgt[w] = fast_exp2(sm[w * 32 + row] - M);
            L += wgt[w] * sl[w * 32 + row];
        }
        const float inv = L > 0.0f ? (kDropout ? a.drop_rscale : 1.0f) / L : 0.0f;
        const int gi = q0 + row;
        if constexpr (kRows) {
            if (a.num_splits > 1) {
                const bool here = kFullD && a.counters != nullptr;
                if (gi < Nq) {
                    const size_t prow = partial_row<kFold>(a, bh, split, gi);
                    float* const op = a.O_partial + prow * d;
                    const int cfull = d & ~7, rem = d & 7;
#pragma unroll
                    for (int k = 0; k < D / 32; ++k) {
                        const int cc = 4 * ((tid & 7) + 8 * k);
                        v4f o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                        for (int w = 0; w < 4; ++w) {
                            const v4f p = *reinterpret_cast<const v4f*>(so + (w * 32 + row) * SM + cc);
#pragma unroll
                            for (int e = 0; e < 4; ++e) o[e] = __builtin_fmaf(wgt[w], p[e], o[e]);
                        }
#pragma unroll
                        for (int e = 0; e < 4; ++e) o[e] *= inv;
                        if constexpr (kVec) {
                            if (kFullD || cc < d) store_partial4(op + cc, o, here);
                        } else if (cc < cfull || (rem != 0 && cc < cfull + 8)) {
                            float* const oc = op + (cc < cfull ? cc : cc - (8 - rem));
#pragma unroll
                            for (int e = 0; e < 4; ++e) oc[e] = o[e];
                        }
                    }
                    if ((tid & 7) == 0) store_partial(a.LSE_partial + prow, L > 0.0f ? __builtin_fmaf(M, kLn2, fast_log2(L) * kLn2) : -INFINITY, here);
                }
                if constexpr (kFullD) {  // (no other instance gets counters: rows_form_merges)
                    if (here && last_to_arrive(a.counters + bh, a.num_splits, reinterpret_cast<int*>(smem))) {
                        float* const lds = reinterpret_cast<float*>(smem) + 64;
                        for (int r = wave; r < Nq; r += 4) {  // (a wave per row, whose splits are one batch)
                            const int hq = kFold ? a.by_fold.quotient(r) : 0;
                            combine_row<true, 1>(a.O_partial, a.LSE_partial, a.O, a.LSE, kFold ? bh * a.fold_group + hq : bh, kFold ? r - hq * a.fold_rows : r,
                                                 kFold ? a.fold_rows : Nq, d, a.num_splits, lds);
                        }
                    }
                }
                store_stamps();
                return;
            }
        }
        if (gi < Nq) {
            half_t* const op = a.O + ((size_t)bh * Nq + gi) * d;
            const int cfull = d & ~7, rem = d & 7;
#pragma unroll
            for (int k = 0; k < D / 32; ++k) {
                const int cc = 4 * ((tid & 7) + 8 * k);
                v4f o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const v4f p = *reinterpret_cast<const v4f*>(so + (w * 32 + row) * SM + cc);
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[e] = __builtin_fmaf(wgt[w], p[e], o[e]);
                }
                const v4h r = {(half_t)(o[0] * inv), (half_t)(o[1] * inv), (half_t)(o[2] * inv), (half_t)(o[3] * inv)};
                // (behind the row's whole chunks sit the columns d - 8 ... d - 1; those that a position before holds as well are
                // the same)
                if constexpr (kFullD) *reinterpret_cast<v4h*>(op + cc) = r;
                else if (cc < cfull || (rem != 0 && cc < cfull + 8)) *reinterpret_cast<v4h_anyalign*>(op + (cc < cfull ? cc : cc - (8 - rem))) = r;
            }
            if ((tid & 7) == 0)
                a.LSE[(size_t)bh * Nq + gi] = L > 0.0f ? __builtin_fmaf(M, kLn2, fast_log2(L) * kLn2) : -INFINITY;
        }
        store_stamps();
        return;
    }

    if constexpr (kPair) {
        // ---------------- merge of the two halves' partial results, register by register, as the merge above
        // (behind the loop's last barrier; the buffer lies behind the O staging of the epilogue, which other waves may be in)
        constexpr int kOut = 4 * 32 * (2 * D + 16);
        static_assert(kOut + 4 * (16 * MB + 2) * 256 <= 2 * kWaveLds, "merge buffer fits the tile buffers");
        // (four registers per access, a wave's 64 lanes one after the other)
        float* const mine = reinterpret_cast<float*>(smem + kOut) + wave * (16 * MB + 2) * 64;
        v4f* const mine_o = reinterpret_cast<v4f*>(mine) + lane;
        float* const mine_ml = mine + 16 * MB * 64 + lane;
        if (half == 1) {
            mine_ml[0] = m_ref[0];
            mine_ml[64] = l_run[0];
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int rg = 0; rg < 4; ++rg)
                    mine_o[(4 * mb + rg) * 64] = v4f{oacc[mb][0][4 * rg], oacc[mb][0][4 * rg + 1], oacc[mb][0][4 * rg + 2], oacc[mb][0][4 * rg + 3]};
        }
        __syncthreads();
        if (half == 1) return;
        const float m1 = mine_ml[0], M = fmaxf(m_ref[0], m1);
        const float w0 = fast_exp2(m_ref[0] - M), w1 = fast_exp2(m1 - M);
        m_ref[0] = M;
        l_run[0] = __builtin_fmaf(w1, mine_ml[64], w0 * l_run[0]);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int rg = 0; rg < 4; ++rg) {
                const v4f o = mine_o[(4 * mb + rg) * 64];
#pragma unroll
                for (int e = 0; e < 4; ++e) oacc[mb][0][4 * rg + e] = __builtin_fmaf(w1, o[e], w0 * oacc[mb][0][4 * rg + e]);
            }
    }

    // ---------------- epilogue: normalise once, store O (fp16) + LSE, or the fp32 split partials
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const float l = xhalf_sum(l_run[nb]);
        const float inv = l > 0.0f ? (kDropout ? a.drop_rscale : 1.0f) / l : 0.0f;
        const float lse = l > 0.0f ? __builtin_fmaf(m_ref[nb], kLn2, fast_log2(l) * kLn2) : -INFINITY;  // (one rounding at the size of m)
        const int i = q0 + wave_row0 + nb * 32 + (lane_here() & 31);
        if (i >= Nq) continue;
        if (a.num_splits > 1) {
            const size_t prow = partial_row<kFold>(a, bh, split, i);
            if (g == 0) a.LSE_partial[prow] = lse;
            float* op = a.O_partial + prow * d;
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int rg = 0; rg < 4; ++rg) {
                    const int dc = 32 * mb + 8 * rg + 4 * g;
                    if (kVec) {
                        if (kFullD || dc < d) {
                            v4f o = {oacc[mb][nb][4 * rg] * inv, oacc[mb][nb][4 * rg + 1] * inv,
                                     oacc[mb][nb][4 * rg + 2] * inv, oacc[mb][nb][4 * rg + 3] * inv};
                            *reinterpret_cast<v4f*>(op + dc) = o;
                        }
                    } else if (!kEvery || d >= 8) {
                        // rows at any alignment: the chunk position behind the row's whole chunks holds columns d - 8 ... d - 1
                        const int c0 = d & ~7, rem = d & 7;
                        if (dc < c0 || (rem != 0 && dc < c0 + 8)) {
                            v4f o = {oacc[mb][nb][4 * rg] * inv, oacc[mb][nb][4 * rg + 1] * inv,
                                     oacc[mb][nb][4 * rg + 2] * inv, oacc[mb][nb][4 * rg + 3] * inv};
                            *reinterpret_cast<v4f_anyalign*>(op + (dc < c0 ? dc : dc - (8 - rem))) = o;
                        }
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (dc + e < d) op[dc + e] = oacc[mb][nb][4 * rg + e] * inv;
                    }
                }
        } else {
            if (g == 0) a.LSE[(size_t)bh * Nq + i] = lse;
            if (kEvery && d < 8) {
                half_t* op = a.O + ((size_t)bh * Nq + i) * d;
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                    for (int rg = 0; rg < 4; ++rg) {
                        const int dc = 32 * mb + 8 * rg + 4 * g;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (dc + e < d) op[dc + e] = (half_t)(oacc[mb][nb][4 * rg + e] * inv);
                    }
            }
        }
    }
    if (!kEvery || d >= 8) {
        if (a.num_splits == 1) {
            // A lane holds 4 consecutive head-dim columns of one row at a time, which as a direct
            // store would be 32 rows x 8 bytes per instruction.  The wave's 32 x d block goes through LDS instead (the tile
            // buffers are free behind the last barrier; rows padded by 16 bytes) and leaves in consecutive 16-byte pieces
            // of whole rows.  The stores are non-temporal: O is not read again by this launch, and lines left dirty in L2
            // would only be written back when the kernel ends.
            constexpr int SO = 2 * D + 16;
            static_assert(4 * NB * 32 * SO <= C::SMEM, "O staging fits the tile buffers");
            char* const ost = smem + wave * (NB * 32 * SO);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const float l = xhalf_sum(l_run[nb]);
                const float inv = l > 0.0f ? (kDropout ? a.drop_rscale : 1.0f) / l : 0.0f;
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                    for (int rg = 0; rg < 4; ++rg) {
                        v4h o = {(half_t)(oacc[mb][nb][4 * rg] * inv), (half_t)(oacc[mb][nb][4 * rg + 1] * inv),
                                 (half_t)(oacc[mb][nb][4 * rg + 2] * inv), (half_t)(oacc[mb][nb][4 * rg + 3] * inv)};
                        *reinterpret_cast<v4h*>(ost + (nb * 32 + l32) * SO + (32 * mb + 8 * rg + 4 * g) * 2) = o;
                    }
            }
            char* const Ob = reinterpret_cast<char*>(a.O + (size_t)bh * Nq * d);
            constexpr int NP = NB * 32 * CH;  // 16-byte pieces of the wave's block, CH per row
#pragma unroll
            for (int p0 = 0; p0 < NP; p0 += 64) {
                const int p = p0 + lane;
                const int rl = p / CH, ch = p % CH;
                const int gi = q0 + wave * C::RW + rl;
                if (p < NP && gi < Nq && (kFullD || ch * 8 < d)) {
                    const v4u piece = *reinterpret_cast<const v4u*>(ost + rl * SO + ch * 16);
                    if constexpr (kVec)
                        __builtin_nontemporal_store(piece, reinterpret_cast<v4u*>(Ob + (size_t)gi * d * 2 + ch * 16));
                    else  // rows at any alignment: the last chunk position holds the row's last 16 bytes
                        __builtin_nontemporal_store(piece, reinterpret_cast<v4u_anyalign*>(Ob + (size_t)gi * d * 2 + (ch * 8 + 8 <= d ? ch * 16 : (d - 8) * 2)));
                }
            }
        }
    }
    store_stamps();
}

// Launcher of one head-dim bucket, defined in fwd_d{32,64,96,128}.hip.
// variant bits: kVarVec (d % 8 == 0), kVarAlibi, kVarDropout; kVarFullD is derived here (d == bucket width).
int launch_fwd_d32(const FwdArgs& a, int variant, int nb, hipStream_t st);
int launch_fwd_d64(const FwdArgs& a, int variant, int nb, hipStream_t st);
int launch_fwd_d96(const FwdArgs& a, int variant, int nb, hipStream_t st);
int launch_fwd_d128(const FwdArgs& a, int variant, int nb, hipStream_t st);
// whether launch_fwd_d128 takes the 8-wave kernel (256 query rows per work-group instead of 128)
// (slices = B * H * num_splits; hint = flash_params::kernel_hint)
bool fwd_uses_pingpong(int d, bool direct, int Nq, int Nk, int causal, int wl, int wr, long long slices, int hint);

// Head slices per chunk of the work-group order: the smallest divisor of the slice count (a multiple of 8, which keeps a
// slice on one XCD) whose chunk still holds twice the work-groups that run at once -- enough for "heaviest row blocks
// first" to balance the tail of a chunk; all slices when there is no such divisor below the slice count.
// Measured on causal + dropout B8 H32 N1000 d96 (256 slices, 8 row blocks, 512 work-groups at once): chunks of 128
// slices +3-5 %; 64: +-0; 32: -2 %; 16: -9 %; 96 and 192 (a ragged last chunk): -1 %.  With this rule, against all
// slices in one chunk: causal B16 H32 N1024 d128 +5 %, B8 H32 N2048 d64 +4 %, B8 H32 N4096 d128 (8-wave kernel) +16 %;
// once or four times the resident work-groups per chunk instead of twice: 0 ... -4 %.
// Where all work-groups weigh alike (no mask, one split) there is no tail to balance and the chunk is sixteen slices, whose
// row blocks follow each other closely enough to find the slices' K and V in L2.  Chunks of 8 / 16 / 32 / 64 / 128 / 256 /
// all: B32 H32 N512 d64 101.0 / 100.9 / 100.5 / 101.7 / 101.8 / 103.1 / 104.7 us, B8 H32 N1024 d96 118.9 / 118.1 / 119.0 / 119.8 /
// 119.9 / 133.7, B8 H32 N2048 d64 320 / 318 / 318 / 321 / 325 / 332, B16 H16 N1024 d128 161 / 163 / 162 / 163 / 164 / 170.
constexpr int kNumCus = 256;  // MI355X
inline int slice_chunk_for(int slices, int groups_per_slice, int resident, bool alike, int step = 8)
{
    if (slices <= 0 || groups_per_slice <= 0) return 1;
    const long long want = alike ? 16 : (2LL * resident + groups_per_slice - 1) / groups_per_slice;
    for (long long c = (want + step - 1) / step * step; c < slices; c += step)
        if (slices % c == 0) return (int)c;
    return slices;
}

// slice_chunk, group_xcd and group_span of a launch: with grouped K/V heads the chunks are multiples of 8 G slices where the
// slice count allows, so that the heads of every K/V head share an XCD (slice_of_position); otherwise the heads of as many
// K/V heads do as fill whole rounds of eight, and the chunks are the large ones, of which whole rounds are the most.
// Ragged slice counts, plain order -> like this: with dropout (heads not folded) B1 H596 H_kv149 Nq20 Nk14594 d64 349 -> 255 us,
// d128 893 -> 639, H600 H_kv150 in one chunk instead of 24 slices 323 -> 255; window of 500 B3 H56 H_kv7 N3000 d64 100 -> 92.5;
// causal B5 H28 H_kv7 N2048 d128 (8-wave kernel) 180 -> 172, B3 H40 H_kv10 N1777 d64 63.3 -> 62.5; unmasked B7 H24 H_kv6 N1000 d80 78.8
// -> 78.1, B17 H48 H_kv6 Nq100 Nk5000 d128 326 -> 295; 24 shapes, none slower.
inline void set_slice_order(FwdArgs& b, int groups_per_slice, int resident)
{
    const int slices = b.B * b.H, round = 8 * b.kv_group;
    const bool alike = !b.causal && b.wl < 0 && b.wr < 0 && b.num_splits == 1 && (b.kv_group == 1 || slices % round == 0);
    b.slice_chunk = slice_chunk_for(slices, groups_per_slice, resident, alike, slices % round == 0 ? round : 8);
    b.group_xcd = b.kv_group;
    b.group_span = b.kv_group > 1 && b.slice_chunk % b.kv_group == 0 ? b.slice_chunk / round * round : 0;
}

// order of the work-groups of launch_fwd_instance: slices, splits, places
template <int D, int NB, int VAR>
inline void set_work_order(FwdArgs& b)
{
    constexpr int kResident = ((VAR & kVarPair) != 0 ? 1 : NB == 1 ? fwd_groups_per_cu(D, NB, VAR) : 2) * kNumCus;
    // (chunks as for three work-groups per CU at D = 64, where four measured +-1 % causal)
    constexpr int kChunked = kResident < 3 * kNumCus ? kResident : 3 * kNumCus;
    // (D = 96: chunks as for two work-groups per CU.  For three, causal B8 H32 N1000 d96 takes all its 256 slices as one chunk
    // instead of 128 and finds fewer tiles in the caches: 74.9 -> 79.0 us, unmasked N = 1024 119.9 -> 133.7)
    set_slice_order(b, b.Tr * b.num_splits, D == 96 ? 2 * kNumCus : kChunked);
    b.split_rotate = split_rotate_for(b.num_splits, b.slice_chunk);
    // (All places, the fourth at D = 64 too: with two row blocks per slice, whose second one is nearly empty, three of a CU's four
    // work-groups were full ones on every other CU.  B32 H16 N130 d64 10.9 -> 9.9 us, B40 13.0 -> 12.3, B48 15.2 -> 14.8.)
    b.snake_end = snake_end_for((long long)b.Tr * b.B * b.H * b.num_splits, kResident);
    set_divisors(b, b.slice_chunk);
}

template <int D, int NB, int VAR>
inline hipError_t launch_fwd_instance(const FwdArgs& a, hipStream_t st)
{
    using C = FwdCfg<D, NB, false, (VAR & kVarShort) != 0>;
    auto kern = fwd_kernel<D, NB, VAR>;
    static DeviceFlags attr_done;  // per instantiation and device
    constexpr bool kPair = (VAR & kVarPair) != 0;
    constexpr int smem = (kPair ? 2 : 1) * (C::SMEM_DMA > C::SMEM ? C::SMEM_DMA : C::SMEM);  // (equal: both paths use two stages)
    if (hipError_t e = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), smem, attr_done); e != hipSuccess) return e;
    const long long groups = (long long)a.Tr * a.B * a.H * a.num_splits;
    FwdArgs b = a;
    set_work_order<D, NB, VAR>(b);
    return launch_kernel(kern, dim3((unsigned)groups), dim3(kPair ? 512 : 256), smem, st, packed(b));
}

// The instances of a bucket: {d == bucket, d % 8 == 0} x {plain, ALiBi, ALiBi with every visible key at or left of its
// row, dropout, both}, for rows at any alignment (d % 8 != 0) {plain, ALiBi, dropout, both}, and the one that serves
// every other request; those for shorter rows (all but the last) once more for d <= D - 16; the narrow, paired and folded ones below.  ST = kVarStamp selects their instrumented twins (debug
// time stamps).  Nothing else looks at the stamp pointer: a stamped call is launched as the same call without.
// The narrow instances (kNarrow in fwd_kernel; those of few rows have rules of their own, below) serve unsplit launches whose time is the chain of key tiles that a work-group
// walks through, which they cut to a quarter for a fixed cost of about 1 us (a wave's own requests, the merge of four).
// Measured against the 128-row instances, paired ones among them, on 1240 random launches of up to 1600 work-groups of 32 rows;
// the lines below lie where the ratio of the two crosses one:
//  * One round -- no more 32-row work-groups than places for them, one per CU by their LDS, two at D = 32 (from 4 tiles on): from 2
//    tiles on, 3 at 96 < d < 128 (N150, 3 tiles, d31 / 64 / 128 / 100 6.2 / 6.2 / 7.8 / 8.3 -> 5.1 / 5.2 / 6.6 / 7.6 us; N120, 2 tiles,
//    5.9 / 5.7 / 6.8 / 7.2 -> 5.2 / 5.2 / 6.3 / 7.4; window of 100 keys N600, 4 tiles, 8.0 / 8.1 / 10.1 / 10.3 -> 5.3 / 5.3 / 6.7 / 7.8).
//    Launches of up to 64 of them keep the 128-row form below 4 tiles, 5 under a window, at a cost (128 rows / narrow, d32 / 64 / 96 / 128: H8
//    N128 3.7 / 4.5 / 5.0 / 5.9 against 3.3 / 4.0 / 4.3 / 5.3 us, N190 4.6 / 5.6 / 6.3 / 7.4 against 3.6 / 4.4 / 4.7 / 5.8, H4 N300 under a window of
//    100 keys 6.1 / 7.3 / 8.1 / 9.4 against 3.7 / 4.5 / 4.8 / 5.9; back to back the first are at the host's rate of 4.9 us per call either way): a
//    stamped call runs as the call without, and readers of the stamps count on a row per 128 query rows there (test_stage_stamps).
//  * More rounds where the later work-groups are the light ones of a causal mask over about as many keys as rows, the more tiles the more
//    of them that see a key: D >= 96 from (groups - 256) / 16 tiles on, up to 640, 720 from 60 tiles, 800 from 100 on (narrow / 128 rows: B1
//    H5 N4105 d96, 645 of them, 36.7 / 44.7 us; H14 N1001 d96, 448, 13.0 / 15.6; H16 Nq586 d128, 304, 10.9 / 13.4; but H10 N2833 d80, 890, 37.2 / 33.7);
//    D = 64 from 8 + (groups - 256) / 12 tiles on up to 560, 640 from 36 on; d = 32: a tile for every 40 of them (B1 H11 N2402: 20.0 -> 15.8), shorter
//    rows, whose requests a wave alone hides less well, up to 640 from 16 on, 800 from 32 on; D = 64 with dropout like D >= 96 beyond 18 tiles
//    (B1 H11 N1267 21.9 -> 16.2), D = 32 with dropout from 10 tiles on.  With more keys than 5/4 of the rows (4/3 with dropout) the lightest ones
//    are heavy too: up to 512, from 8 + (groups - 256) / 16 tiles on, / 32 with dropout (1.9 keys per row, B1 H14 N1213 d112, 532 of them, 44 / 33 us).
//  * Short rows over many tiles in more rounds, any mask, where the 128-row work-groups are more than the CUs and so cannot be paired
//    (B5 H8 H_kv4 Nq785 Nk20772 d32, 260 of them: 270 -> 172 us), or the last rounds are light, or there are few rounds; while K and V, which
//    the narrow ones read once per 32 rows, stay in the 32 MiB of L2 (117 slices of 20695 keys d32, 310 MB, ten work-groups each:
//    266 us against 455), or so many share a slice that its tiles do, or the rows are so short that 6.8 TB/s brings them in time.  Odd d not without dropout (B1 H7 N4555 d31 37.5 against 67.7).
inline bool fwd_uses_narrow(const FwdArgs& a, bool every)
{
    if (every || a.num_splits != 1 || a.kernel_hint != 0) return false;
    const long long groups = (long long)a.B * a.H * ((a.Nq + 31) / 32);
    if (groups > 1280) return false;
    const int bucket = (a.d + 31) / 32;
    const bool whole = a.d == 32 * bucket;
    // keys that the rows of a 128-row work-group see, at most
    const long long left = a.wl >= 0 ? a.wl : a.Nk, right = a.causal ? 0 : a.wr >= 0 ? a.wr : a.Nk;
    const long long keys = left + right + 128 < a.Nk ? left + right + 128 : a.Nk;
    const int tiles = (int)((keys + 63) / 64);
    if (groups <= (bucket == 1 ? 2 * kNumCus : kNumCus)) {
        if (groups <= 64) return tiles >= (keys < a.Nk ? 5 : 4);
        return tiles >= (groups > kNumCus ? 4 : bucket == 4 && !whole ? 3 : 2);
    }
    if (keys < a.Nk) return false;  // a window: the later work-groups are as heavy as the first
    const bool dropout = a.drop_thr != 0;
    const long long rows = a.fold_rows ? a.fold_rows : a.Nq;
    if (a.causal && 2 * rows >= a.Nk) {
        if (bucket == 1) return (whole && 40 * tiles >= groups) || (groups <= (tiles >= 32 ? 800 : 640) && tiles >= (dropout ? 10 : 16));
        const long long seeing = rows > a.Nk ? groups * a.Nk / rows : groups;  // the others leave at once
        const bool to_nothing = (dropout ? 4 : 5) * rows >= (dropout ? 3 : 4) * (long long)a.Nk;  // the lightest work-groups see few keys
        if (seeing > (to_nothing ? 800 : 2 * kNumCus)) return false;
        if (bucket == 2 && !(dropout && tiles > 18)) return 12 * (tiles - 8) >= seeing - kNumCus && (seeing <= 560 || (seeing <= 640 && tiles >= 36));
        if (to_nothing) return 16 * tiles >= seeing - kNumCus && seeing <= (tiles >= 100 ? 800 : tiles >= 60 ? 720 : 640);
        return (dropout ? 32 : 16) * (tiles - 8) >= seeing - kNumCus;
    }
    if (bucket > 2 || (a.d % 2 != 0 && !dropout)) return false;
    const long long groups128 = (long long)a.Tr * a.B * a.H;
    const bool no_pair = groups128 > kNumCus;
    const bool lighter = (a.causal || a.wr >= 0) != (a.wl >= 0) && 5 * rows >= 2 * (long long)a.Nk;
    const long long kv_bytes = 4LL * a.d * a.Nk * a.B * a.Hk;
    const bool in_l2 = kv_bytes <= (32 << 20);
    if (bucket == 2) return groups <= 2 * kNumCus && tiles >= 24 && (no_pair || lighter || (in_l2 && (dropout || groups <= 384)));
    const bool rounds_pay = no_pair || lighter || groups <= (kv_bytes <= (8 << 20) ? 768 : 640);
    const bool fed = in_l2 || groups >= 45LL * a.B * a.Hk || groups * a.d <= 20480 || groups128 > 4 * kNumCus;
    return tiles >= (no_pair ? 32 : 64) && rounds_pay && fed;
}

// LDS of a narrow work-group: two stages per wave up to D = 64, one above
template <int D, int VAR>
constexpr int narrow_lds()
{
    using C = FwdCfg<D, 1, true, (VAR & kVarShort) != 0>;
    return 4 * (D <= 64 ? 2 : 1) * (C::KBUF + C::VBUF) + (C::kQApart ? 4 * 32 * C::SK : 0);
}

template <int D, int VAR>
inline hipError_t launch_fwd_narrow_instance(const FwdArgs& a, hipStream_t st)
{
    auto kern = fwd_kernel<D, 1, VAR | kVarNarrow>;
    static DeviceFlags attr_done;  // per instantiation and device
    constexpr int smem = narrow_lds<D, VAR>();
    if (hipError_t e = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), smem, attr_done); e != hipSuccess) return e;
    FwdArgs b = a;
    b.Tr = (a.Nq + 31) / 32;
    const long long groups = (long long)b.Tr * a.B * a.H;
    set_slice_order(b, b.Tr, kNumCus);
    b.split_rotate = 0;
    b.snake_end = snake_end_for(groups, kNumCus);
    set_divisors(b, b.slice_chunk);
    return launch_kernel(kern, dim3((unsigned)groups), dim3(256), smem, st, packed(b));
}

// Launches of few rows (kRows in fwd_kernel), no features, no window.  Old form (128-row work-groups, one wave of which has rows) / this one, each
// with its best split count, inputs that no cache holds, us:
//  * Up to 32 rows per slice (decode with heads as rows, folded heads, speculative tokens), whole, 128 ... 256 slices, one work-group
//    per CU: what the non-temporal requests give the narrow form.  B32 H32 H_kv8 Nk4096 d128 91.1 / 79.7, Nk1024 25.2 / 22.7, Nk512 14.4 / 13.0, B20
//    54.0 / 49.8, B32 d64 47.2 / 41.6, B64 H16 H_kv4 Nk3000 d96 51.0 / 44.7, B24 H64 H_kv8 d80 33.8 / 30.4, B30 H8 Nq8 Nk3000 d128 62.8 / 53.8; a second
//    round costs (320 slices 54.8 / 60.3, 512 77.9 / 81.7).
//  * Up to 32 rows in splits, four tiles or more each, at most 32 of them, up to eight tiles per wave: B1 H32 H_kv8 Nk1920 d64 8.8 / 7.3, B1 H16 H_kv4
//    Nk3584 d64 8.9 / 7.5, B4 H32 H_kv8 Nk8192 d128 26.2 / 25.2, B1 Nk32768 28.2 / 26.0, B12 H32 H_kv4 Nq3 Nk8396 d80 29.0 / 26.0, B4 H8 Nq16 Nk8192
//    d128 28.6 / 25.7.  Above d = 64, where Q of a short launch comes a memory latency ahead of V, only launches that fill the GPU gain (B1 H32 H_kv8
//    Nk2048 d128, 128 work-groups, 8.5 / 8.8; B5 H4 H_kv1 Nk7937 d96 9.9 / 10.1); with more tiles per wave both run at the rate of HBM (B16 H32
//    H_kv4 Nk16384 83.2 / 83).
//  * Up to 512 rows, in splits: a quarter of the splits, and of the partial results, fills the GPU, at the price of a tile fetched once per 32
//    rows, so that the tiles per wave are bounded.  B2 H8 Nq64 Nk4096 d128 17.1 / 14.2, B4 H4 Nq128 Nk4096 20.9 / 17.9, B1 H8 Nq128 Nk16384 29.3 / 26.4,
//    B1 H4 Nq512 Nk4096 20.7 / 15.3, B1 H8 H_kv4 Nq120 Nk6000 18.6 / 14.2, B1 H16 H_kv2 Nq40 Nk9000 (folded) 17.0 / 13.5, B1 H8 Nq128 Nk8192 d80 17.4 / 14.8, B1
//    H2 Nq128 Nk4096 d64 10.3 / 8.5; with more tiles than that: B4 H4 Nq130 Nk7000 d128 (10) 25.8 / 27.8, B2 H8 Nq100 Nk8000 d64 (8) 16.0 / 16.4, B1 H12
//    H_kv2 Nq100 Nk7000 d100 (6) 18.1 / 19.9, B1 H32 Nq128 Nk16384 d128 (32) 63 / 80.  Fewer than 96 work-groups
//    (0.92 ... 1.13) stay as they are.
//  * The other lines, 1260 random launches, old form at the estimate's count / this one.  At that count the form gains whatever the number of slices and work-groups: 96 to 191
//    of them above d = 64 1.05 ... 1.22 times as fast, one to three slices 1.05 ... 1.22, 33 to 64 splits 1.02 ... 1.17 in the mean; but such launches are rare, and most calls of few
//    slices come here with a count cut to 32: one to three slices, 32 to 96 work-groups, 0.80 ... 1.01 at whole buckets, 4 slices on 0.90 ... 0.94 above d = 64 up to 143 work-groups,
//    from 144 on 1.00 ... 1.03, up to d = 64 0.97 up to 95, 1.01 ... 1.07 beyond.  Whole, whole buckets: 64 to 95 slices 0.97 ... 1.02, 96 to 127 1.00 ... 1.04 (single ones 0.93), 128 to
//    159 1.05 ... 1.07, 160 to 256 1.09 ... 1.13.
inline bool rows_form_fits(long long slices, int rows, int d, int Nk, int splits, int keys_per_split)
{
    const int places = d <= 32 ? 2 * kNumCus : kNumCus;
    const long long groups = slices * ((rows + 31) / 32) * splits;
    if (rows > 512 || groups > places) return false;
    if (splits == 1) return rows <= 32 && groups >= 128 && groups <= kNumCus && Nk >= 512;
    const int per_wave = (keys_per_split + 255) / 256;
    if (splits > 32 || keys_per_split < 256) return false;
    if (rows > 32) return groups >= 96 && per_wave <= (d == 128 ? 8 : d % 32 == 0 ? 7 : 4);
    return groups >= (d <= 64 ? 48 : 192) && per_wave <= 8 && slices >= 4;
}
inline bool rows_form_serves(const FwdArgs& a, int variant)
{
    return (a.kv_group == 1 || a.Nq > kRowsLimit) && (variant & (kVarAlibi | kVarDropout)) == 0 && a.wl < 0 && a.wr < 0 && a.kernel_hint == 0;
}
inline bool fwd_uses_rows(const FwdArgs& a, int variant)
{
    return rows_form_serves(a, variant) && rows_form_fits((long long)a.B * a.H, a.Nq, a.d, a.Nk, a.num_splits, a.keys_per_split);
}
// Whether the last work-group of such a launch to arrive at a slice's counter merges its partial results.  A merge by a launch of its own takes 1.5-2 us,
// which the arrival (a store, an atomic and a load from memory in a row) and partial results written through and read past the L2 use up
// soon.  Its own launch / here, time over time, over 230 random launches of whole buckets, K and V from memory (called again with the same ones 1 % more):
// two to four rows, up to 4 / 5 to 8 splits d32 1.07 / 1.05, d64 1.05 / 1.05, d96 1.03 / 1.04, d128 1.03 / 1.03, none below 1.00; 9 to 12 0.98 ... 1.04, 13 to 16 0.89 ... 1.00, more,
// two batches of a wave, 0.79 ... 0.95; five to eight rows 0.98 ... 0.99 / 0.96 ... 0.98, more 0.5 ... 0.8; rows between the buckets, up to four, 0.85 ... 1.00.
inline bool rows_form_merges(const FwdArgs& a)
{
    return a.Nq <= 4 && a.d % 32 == 0 && a.num_splits <= 8;
}
// Split count with which such a launch fills the GPU, 0 if there is none that rows_form_fits.  Where the estimate splits: whole from 144 slices on (128 ... 143 0.96 ... 1.09
// times as fast as its count, 144 ... 168 1.00 ... 1.15); not up to 1280 keys of 16 slices or more, which come out in two to five splits of 256 keys and gain nothing (720 ... 1268
// keys d31 0.95 ... 1.01, d64 0.98 ... 1.02, d40 1.00 ... 1.05; 1407 ... 1520 d40, d32 1.05).  More than 32 rows with d < 32 take 256 work-groups, one per CU: 1.03 ... 1.16 there, 0.84 ... 1.00
// with two per CU (more than 1024 keys per split 0.54 ... 1.0 either way).
inline int rows_form_splits(long long slices, int rows, int d, int Nk)
{
    const int n_blocks = (Nk + 127) / 128;
    const long long groups = slices * ((rows + 31) / 32);
    if (rows > 512 || groups < 1) return 0;
    if (rows <= 32 && groups >= 144 && groups <= kNumCus && Nk >= 512) return 1;
    if (rows <= 32 && slices >= 16 && Nk <= 1280) return 0;
    long long s = (d == 32 || (d < 32 && rows <= kRowsLimit) ? 2 * kNumCus : kNumCus) / groups;
    if (s > (n_blocks + 1) / 2) s = (n_blocks + 1) / 2;
    if (s > 32) s = 32;
    if (s < 2) return 0;
    const int per = (int)((n_blocks + s - 1) / s), even = (n_blocks + per - 1) / per;  // all of them with keys
    return even >= 2 && rows_form_fits(slices, rows, d, Nk, even, 128 * per) ? even : 0;
}

// Whether it is the better one where the estimate for 128-row work-groups, whose count is never lower than this one, says `estimate`.  Time at the
// estimate's count / here over 760 random launches with such a count, K and V from memory:
//  * up to 32 rows, d = 64: 256 keys per split 0.93 ... 0.98 (1.00 ... 1.09 where the launch merges itself), more keys, one work-group per CU by the estimate, whose splits are
//    then more than 32, 0.98 ... 1.26, two per CU 0.93 ... 1.03, 0.985 in the mean; d = 96, two per CU, 0.97 ... 1.01; but d = 128 0.98 ... 1.07, d = 32 0.98 ... 1.22, rows between
//    the buckets 1.02 ... 1.25.  B8 H16 H_kv2 Nk1739 d64 7.2 us in 14 splits, 7.6 in 7, B8 H64 H_kv8 Nk5941 d64 19.8 in 8, 20.4 in 4, B13 H32 H_kv4 Nk5210 d96 21.1 in 9,
//    21.8 in 4; B6 H8 H_kv1 Nk31104 d64 16.0 in 41, 13.6 in 31.
//  * more rows, two row blocks, 256 keys per split, above d = 32, 96 ... 159 work-groups 0.90 ... 1.02 (33 to 50 rows; 56 to 59 rows up to 1.10), 160 on 1.02 ... 1.05 (B8 H4 H_kv1 Nq9 Nk1306
//    d128 9.4 in 11, 10.4 in 6; B17 H4 H_kv4 Nq57 Nk1700 d128 1.05 times as fast).
inline bool rows_form_lowers(long long slices, int rows, int d, int Nk, int splits, int estimate)
{
    const int n_blocks = (Nk + 127) / 128, keys_per_split = 128 * ((n_blocks + splits - 1) / splits);
    if (rows > kRowsLimit) return d <= 32 || rows > 64 || keys_per_split > 256 || 2 * slices * splits >= 160;
    if (splits == 1 || (d != 64 && d != 96)) return true;
    return (rows <= 4 && splits <= 8) || (slices * estimate <= kNumCus && keys_per_split >= 512);
}

template <int D, int VAR>
inline hipError_t launch_fwd_rows_instance(const FwdArgs& a, hipStream_t st)
{
    auto kern = fwd_kernel<D, 1, VAR | kVarNarrow | kVarRows>;
    static DeviceFlags attr_done;  // per instantiation and device
    constexpr int smem = narrow_lds<D, VAR>();
    if (hipError_t e = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), smem, attr_done); e != hipSuccess) return e;
    FwdArgs b = a;
    b.Tr = (a.Nq + 31) / 32;
    const long long slices = (long long)a.B * a.H;
    set_divisors(b, slices);
    return launch_kernel(kern, dim3((unsigned)(slices * a.num_splits * b.Tr)), dim3(256), smem, st, packed_rows(b));
}

// Paired work-groups (kPair in fwd_kernel): launches of at most one 128-row work-group per CU, whose SIMDs would have one
// wave each.  Measured against the unpaired instances on 60 random launches (unsplit / split):
//  * causal, 64-256 work-groups that the narrow instances leave: B2 H4 N1909 d100 36.3 -> 28.8 us, B1 H8 N1664 d100 32.0 ->
//    25.8, B1 H16 N768 d112 17.1 -> 15.0, B1 H16 N1244 d31 16.6 -> 14.3; split: B1 H64 Nq185 Nk3840 d112 46.8 -> 40.9, B1 H32
//    Nq128 Nk16384 d128 63.3 -> 60.6 (bound by HBM for half of it).
//  * causal with dropout: B2 H2 N2112 d100 59.9 -> 46.2 us, B2 H4 N1986 d96 50.1 -> 38.9, B1 H8 N3061 d64 65.2 -> 52.6, B4 H8
//    N683 d128 22.7 -> 20.1.
//  * eight tiles or more per work-group, a window's included (five where the last points say so): with fewer the merge costs what the shorter chain saves.
//    (Window of 500 keys B1 H16 N1500 d64 12.7 -> 10.7 us, of 1000 B2 H4 N2500 d96 21.5 -> 18.0.)
//  * with ALiBi and no visible key right of its row, whole: from 5 tiles on, 8 at d = 128, the chain of a tile being the longer one (110 random launches of
//    up to 512 work-groups, unpaired / paired): windows B1 H8 N3835 d40 of 1390 keys 21.3 / 17.4 us, B4 H2 N3551 d64 of 1858 26.8 / 21.8, B2 H8 N1533
//    d64 of 196 9.2 / 8.6, B1 H8 N1792 d96 of 1052 21.0 / 17.5, B1 H12 N1281 d100 of 1108 30.3 / 25.0, B2 H4 N1230 d128 of 941 22.1 / 19.5; causal N3502 d72
//    46.1 / 37.2, N848 d32 11.1 / 9.4; up to 512 of them under the lines without dropout (next but one) N2253 d100 48.6 / 38.5, N7577 d64 88.0 / 72.2, N875 d40 13.6 / 11.6;
//    from six on where no window cuts (290 to 320 keys, causal, unpaired / paired, time over time d64 0.97 ... 1.01, d72-96 0.96 ... 0.99; 337 on 1.01 ... 1.07: N320 d64 7.70 / 7.91 us);
//    left out: d128 windows of 159 ... 396 keys 11.0 / 11.1, of 257 to 512 work-groups 15.9 / 20.2.  Two-sided ALiBi, and with dropout, stay as they are.
//  * under a window that ends at the row, whole, without dropout: from 5 tiles on below d = 128, too (130 random launches, unpaired / paired, us): N4064 d32 of 219 keys 8.03 /
//    6.78, N904 d40 of 184 8.15 / 7.53, N3367 d64 of 212 9.48 / 8.80, N1554 d64 of 146 8.32 / 8.07, N1911 d72 of 208 10.51 / 9.58, N907 d100 of 231 12.50 / 11.69, N1126 d112 of
//    159 10.34 / 9.99 (five tiles at 96 < d < 128 up to 128 work-groups; 192 to 240 of them 0.95 ... 0.99, six tiles 1.00 ... 1.05: N1984 d112 of 192 12.23 / 12.82); but d128 of 202 12.74 / 13.77, of 293 14.44 / 14.85, and without a window N300 d96 7.94 / 8.42.  At 32 < d <= 64 up to 400 work-groups,
//    from 7 tiles on, without ALiBi: B1 H8 N4178 d64 of 480 12.02 / 10.58, B2 H32 N623 d64 of 346 11.27 / 10.21, B1 H12 N4037 d40 of 878 21.5 / 20.2, B4 H2 N6294 d64 of 1121 27.9 /
//    25.9; with 5 tiles N791 d40 8.93 / 9.06, d32 of 417 10.84 / 11.19, and above d = 64 0.7 ... 0.9 times as fast (d72 of 163 12.3 / 16.5).
//  * up to 32 rows only one wave of four has any, and a second one beside it gained 7-11 % at d = 32, but lost 4 % at
//    d = 112 (B2 H16 H_kv4 Nq2 Nk16960 18.2 -> 19.0).
//  * causal, unsplit and up to twice as many: two work-groups of a CU side by side last as long as the longer one, whose SIMDs
//    have one wave each once its light neighbour is done; as paired ones they follow each other, eight waves at a time.  The lines lie where 150
//    random launches cross over.  Up to 384 work-groups (unpaired / paired): N1238 d64 17.9 / 15.7 us, N1117 d80 19.2 / 16.0, N1184 d100 23.1 / 19.5, N1000
//    d40 14.7 / 13.7; with dropout N1267 d64 27.3 / 22.7, N640 d64 15.5 / 13.2, N1021 d128 28.7 / 24.0, N680 d128 20.8 / 18.3
//    (above d = 64 and 324 of them from 896 on: N704 d128 22.2 / 24.2, N822 d80 22.3 / 24.5, N842 d128 28.4 / 30.9, N749 d128 25.5 / 26.4, N921 d80 23.6 / 23.8; 1.00 ... 1.10 times as fast beyond); below the lines N675 d64
//    11.35 / 11.46, N926 d96 16.4 / 17.3, N660 d128 17.8 / 20.6, with dropout N668 d32 13.4 / 13.4, N556 d128 20.3 / 23.2.  More of them: B1 H16 N4096
//    d128 83.1 / 75.2, B4 H8 N2000 d96 36.1 / 34.2, N1645 d96 (390 of them) 28.5 / 25.9, N1672 d80 (448) 26.4 / 24.9, B4 H8 N2000 d80 with dropout 44.6 / 40.9, N1246 d64 (400 of them) 17.4 / 16.4;
//    below N1424 d80 24.7 / 26.8, N1785 d96 (504) 32.6 / 33.0, N1227 d64 with dropout 25.8 / 25.9.  Above 512 it loses (B5 H8 N1777 d100 42.5 / 47.8, 560 of them).
//    At 64 < d <= 96, 449 to 512 of them, d <= 80 has the instances for shorter rows and crosses over earlier: 220 launches of d = 72, 80 / 88, 96, unpaired / paired, time over
//    time, with K and V from memory and again with the same ones, N1650-1700 0.975, 0.998 / 0.956, 0.979, N1760-1855 0.991, 1.011 / 0.971, 0.994, N1880-1910 1.022, 1.048 / 1.006,
//    1.028; their number decides as much (450 to 480 of them up to 0.04 above, 490 to 510 below): N1700 d80 (490) 31.9 / 33.9, N1760 d72 (476) 31.7 / 31.2, N1825 d80 (480) 31.7 / 30.4;
//    N1760 d96 (490) 36.5 / 39.2, N1825 d88 (465) 35.3 / 36.2.
inline long long following_keys(int d, long long groups, bool dropout)
{
    const int bucket = (d + 31) / 32;
    constexpr int kPlain[4] = {704, 704, 960, 1104}, kDropout[4] = {960, 608, 608, 640};
    if (groups <= 384) return !dropout ? kPlain[bucket - 1] : groups > 324 && bucket > 2 ? 896 : kDropout[bucket - 1];
    if (dropout) return 1280;
    if (bucket == 3) return groups <= 448 ? 1600 : d <= 80 ? 1760 : 1856;
    return bucket <= 2 && groups <= 416 ? 1184 : 1856;
}
inline bool fwd_uses_pair(const FwdArgs& a, int bucket_d, int feat)
{
    const bool alibi = (feat & kVarAlibi) != 0, dropout = (feat & kVarDropout) != 0;
    if (alibi && (dropout || !a.alibi_left || a.num_splits != 1)) return false;
    if (a.kernel_hint != 0 || (a.Nq <= 32 && bucket_d > 32)) return false;
    const long long groups = (long long)a.Tr * a.B * a.H * a.num_splits;
    const long long left = a.wl >= 0 ? a.wl : a.Nk, right = a.causal ? 0 : a.wr >= 0 ? a.wr : a.Nk;
    if (a.causal && a.wl < 0 && a.num_splits == 1 && !a.fold_rows && 2 * (long long)a.Nq >= a.Nk && groups > kNumCus)
        return groups <= 2 * kNumCus && a.Nk >= following_keys(a.d, groups, dropout);
    const bool window = left + right + 128 < a.Nk && right == 0 && a.num_splits == 1 && !dropout;
    if (groups > kNumCus) return window && !alibi && bucket_d == 64 && groups <= 400 && left + 128 > 6 * 64;
    const bool six = alibi ? !window : a.d > 96 && groups > 128;  // tiles, where five are not enough
    const long long keys = a.d < 128 && (alibi || window) ? (six ? 5 * 64 + 1 : 4 * 64 + 1) : 8 * 64;
    return a.Nk >= keys * a.num_splits && left + right + 128 >= keys;
}

// 64 query rows per wave at d = 64 (NB = 2, 199 VGPRs, two work-groups of 256 rows per CU): a K or V fragment read from LDS
// feeds two MFMAs; the launch needs no fewer cycles than with 128 rows, but half the LDS instructions and 0.57 of the bytes
// fetched, and what those save in power comes back as clock.  Only without a mask -- causal it measured -9 %, with a window of
// 256 keys -21 %: wider diagonals --, where 256-row blocks add no more than 4 % of empty rows to what 128-row blocks have (N300
// -7 %) and no more than an eighth of the rows is empty, from two rounds of work-groups on, and from sixteen tiles on: shorter
// work-groups are better off four to a CU.  Tall / 128 rows: B32 H32 N512 96.6 / 91.1 us, B24 H16 N768 70.8 / 68.3, B16 H16 N768 46.5 /
// 46.9, B12 H16 N896 51.0 / 51.1, B16 H16 N1024 75.9 / 79.3, B8 H32 N2048 287 / 298, B4 H16 N4096 281 / 296; same bits.
inline bool fwd_uses_tall(const FwdArgs& a, int variant)
{
    if (variant != kVarVec || a.d != 64 || a.Nk < 1024 || a.num_splits != 1 || a.fold_rows || a.causal || a.wl >= 0 || a.wr >= 0 || a.kernel_hint != 0) return false;
    const long long blocks = (a.Nq + 255) / 256, added = 2 * blocks - (a.Nq + 127) / 128;  // in blocks of 128 rows
    return (long long)a.B * a.H * blocks >= 4 * kNumCus && 25 * added <= 2 * blocks && 8 * (256 * blocks - a.Nq) <= 256 * blocks;
}

// requests that only the instance which serves every request takes (kEvery in fwd_kernel)
inline bool fwd_needs_every_instance(const FwdArgs& a, int variant)
{
    return a.scale_log2 <= 0.0f || a.scores_out != nullptr || a.d < 8 || ((variant & kVarDropout) && a.drop_thr == 0);
}

// query rows per work-group of the launch that a takes (what the launchers below and launch_fwd_d128 do)
inline int fwd_rows_per_group(const FwdArgs& a, int variant)
{
    const bool every = fwd_needs_every_instance(a, variant);
    if (!a.fold_rows && fwd_uses_pingpong(a.d, !every, a.Nq, a.Nk, a.causal, a.wl, a.wr, (long long)a.B * a.H * a.num_splits, a.kernel_hint))
        return 256;
    if (fwd_uses_narrow(a, every) || (!every && fwd_uses_rows(a, variant))) return 32;
    return fwd_uses_tall(a, variant) ? 256 : 128;
}

template <int D, int NB, int ST>
inline int launch_fwd_bucket_st(const FwdArgs& a, int variant, hipStream_t st)
{
    hipError_t e;
    const int feat = variant & (kVarAlibi | kVarDropout);
    constexpr int AL = kVarAlibi | kVarAlibiLeft;  // ALiBi with no visible key right of its row
    // launch(kVarShort) where rows are at most D - 16 elements long, launch(0) otherwise
    auto by_length = [&](auto launch) {
        if constexpr (D >= 64) {
            if (a.d <= D - 16) return launch(std::integral_constant<int, kVarShort>{});
        }
        return launch(std::integral_constant<int, 0>{});
    };
    if (!fwd_needs_every_instance(a, variant) && fwd_uses_rows(a, variant)) {
        // By row length and alignment like the narrow ones; in the bucket of 32 columns rows at any alignment serve every shorter length.  When they served
        // all shorter lengths -> now, us, K and V from memory: B2 H4 Nq20 Nk6190 d80 in 25 splits 11.10 -> 9.85, B2 H16 H_kv2 Nq8 Nk9000 d112 in 24 14.01 -> 12.72, B2 H8
        // Nq11 Nk11200 d100 in 15 19.88 -> 19.25, whole B20 H64 H_kv8 Nk5263 d80 46.62 -> 46.62; rows of whole chunks give 4 % of it, short ones 1-2.
        auto rows = [&](auto var) {
            auto folded = [&](auto many) {
                constexpr int V = ST | decltype(var)::value | decltype(many)::value;
                if (a.fold_rows) return (int)launch_fwd_rows_instance<D, V | kVarFold>(a, st);
                if constexpr ((V & kVarFullD) != 0) return (int)launch_fwd_rows_instance<D, V>(a, st);
                else return (int)by_length([&](auto sh) { return launch_fwd_rows_instance<D, V | decltype(sh)::value>(a, st); });
            };
            // (rows of less than 64 bytes share lines, which neighbouring requests ask for: called again with K and V that the caches hold, ordinary requests take 0.66 ... 0.93 of
            // the time from 20 to 300 MiB on, from memory 1.03 ... 1.07: B21 H8 Nq3 Nk5952 d31 24.7 / 35.5 us and 38.4 / 37.0)
            constexpr bool kNarrowRows = D == 32 && (decltype(var)::value & kVarFullD) == 0;
            if constexpr (!kNarrowRows) {
                if (a.Nq <= kRowsLimit) return folded(std::integral_constant<int, 0>{});
            }
            return folded(std::integral_constant<int, kVarManyRows>{});
        };
        if (a.d == D) return rows(std::integral_constant<int, kVarVec | kVarFullD>{});
        if constexpr (D > 32) {
            if (variant & kVarVec) return rows(std::integral_constant<int, kVarVec>{});
        }
        return rows(std::integral_constant<int, 0>{});
    }
    if (fwd_uses_narrow(a, fwd_needs_every_instance(a, variant))) {
        // plain: by row length like the others; with ALiBi or dropout: the instances for rows at any alignment, which serve
        // every row length from eight elements on, and above 64 the ones for rows of the bucket's width
        auto with_features = [&](auto full_c) {
            constexpr int F = ST | (decltype(full_c)::value ? kVarVec | kVarFullD : 0);
            if (feat == kVarAlibi) return (int)launch_fwd_narrow_instance<D, F | kVarAlibi>(a, st);
            if (feat == kVarDropout) return (int)launch_fwd_narrow_instance<D, F | kVarDropout>(a, st);
            return (int)launch_fwd_narrow_instance<D, F | kVarAlibi | kVarDropout>(a, st);
        };
        if constexpr (D > 64) {
            if (feat != 0 && a.d == D) return with_features(std::true_type{});
        }
        if (feat != 0) return with_features(std::false_type{});
        if (a.fold_rows) {
            if (a.d == D) return (int)launch_fwd_narrow_instance<D, ST | kVarVec | kVarFullD | kVarFold>(a, st);
            if (variant & kVarVec) return (int)launch_fwd_narrow_instance<D, ST | kVarVec | kVarFold>(a, st);
            return (int)launch_fwd_narrow_instance<D, ST | kVarFold>(a, st);
        }
        if (a.d == D) return (int)launch_fwd_narrow_instance<D, ST | kVarVec | kVarFullD>(a, st);
        if (variant & kVarVec) return (int)by_length([&](auto sh) { return launch_fwd_narrow_instance<D, ST | kVarVec | decltype(sh)::value>(a, st); });
        return (int)by_length([&](auto sh) { return launch_fwd_narrow_instance<D, ST | decltype(sh)::value>(a, st); });
    }
    const bool pair = fwd_uses_pair(a, D, feat);
    auto halves = [&](auto var) {
        constexpr int V = decltype(var)::value;
        return pair ? launch_fwd_instance<D, NB, V | kVarPair>(a, st) : launch_fwd_instance<D, NB, V>(a, st);
    };
    // rows shorter than the bucket: V with paired work-groups where they fit, or alone
    auto shorter_rows = [&](auto var) {
        return by_length([&](auto sh) { return halves(std::integral_constant<int, decltype(var)::value | decltype(sh)::value>{}); });
    };
    auto shorter_rows_alone = [&](auto var) {
        return by_length([&](auto sh) { return launch_fwd_instance<D, NB, decltype(var)::value | decltype(sh)::value>(a, st); });
    };
    // (several row blocks per K/V head ask for the same tiles and have to find them in L2: folded launches of 129 rows or more,
    // non-temporal -> ordinary, 24 random shapes -1 ... +15 %, +4.4 % in the mean: B2 H32 H_kv8 Nq42 Nk3937 d128 23.5 -> 20.5 us, B16
    // H16 H_kv2 Nq50 Nk5711 d128 70.0 -> 62.9)
    const bool kv_once = a.Tr == 1 && a.kv_group == 1;
    if (a.fold_rows) {
        constexpr int F = ST | kVarFold;
        if (a.d == D && kv_once) return (int)halves(std::integral_constant<int, F | kVarVec | kVarFullD | kVarKvOnce>{});
        if (a.d == D) return (int)halves(std::integral_constant<int, F | kVarVec | kVarFullD>{});
        if (variant & kVarVec) return (int)halves(std::integral_constant<int, F | kVarVec>{});
        return (int)halves(std::integral_constant<int, F>{});
    }
    if (!(variant & kVarVec)) {
        // rows at any alignment: plain, ALiBi, dropout, both, and one more with both features compiled in (slope 0 /
        // threshold 0 make them identities) for every other request: a non-positive scale (its ALiBi step is where the
        // scores are scaled ahead of the row maximum), the score dump, rows of fewer than eight elements, a dropout
        // threshold of 0
        if (fwd_needs_every_instance(a, variant)) e = launch_fwd_instance<D, NB, ST | kVarAlibi | kVarDropout | kVarEvery>(a, st);
        else if (feat == 0) e = shorter_rows(std::integral_constant<int, ST>{});
        else if (feat == kVarAlibi) e = shorter_rows(std::integral_constant<int, ST | kVarAlibi>{});
        else if (feat == kVarDropout) e = shorter_rows(std::integral_constant<int, ST | kVarDropout>{});
        else e = shorter_rows_alone(std::integral_constant<int, ST | kVarAlibi | kVarDropout>{});
    } else if (a.d == D) {
        constexpr int V = ST | kVarVec | kVarFullD;
        if constexpr (D == 64) {
            if (fwd_uses_tall(a, variant)) {
                FwdArgs b = a;
                b.Tr = (a.Nq + 255) / 256;
                return (int)launch_fwd_instance<D, 2, V>(b, st);
            }
        }
        if (feat == 0) e = kv_once ? halves(std::integral_constant<int, V | kVarKvOnce>{}) : halves(std::integral_constant<int, V>{});
        else if (feat == kVarAlibi) e = a.alibi_left ? halves(std::integral_constant<int, V | AL>{}) : launch_fwd_instance<D, NB, V | kVarAlibi>(a, st);
        else if (feat == kVarDropout) e = halves(std::integral_constant<int, V | kVarDropout>{});
        else e = a.alibi_left ? launch_fwd_instance<D, NB, V | AL | kVarDropout>(a, st) : launch_fwd_instance<D, NB, V | kVarAlibi | kVarDropout>(a, st);
    } else {
        constexpr int V = ST | kVarVec;
        if (feat == 0) e = shorter_rows(std::integral_constant<int, V>{});
        else if (feat == kVarDropout) e = shorter_rows(std::integral_constant<int, V | kVarDropout>{});
        else if (feat == kVarAlibi) e = a.alibi_left ? shorter_rows(std::integral_constant<int, V | AL>{}) : shorter_rows_alone(std::integral_constant<int, V | kVarAlibi>{});
        else e = a.alibi_left ? shorter_rows_alone(std::integral_constant<int, V | AL | kVarDropout>{}) : shorter_rows_alone(std::integral_constant<int, V | kVarAlibi | kVarDropout>{});
    }
    return (int)e;
}

// every instance has an instrumented twin: the same launch, with time stamps
template <int D, int NB>
inline int launch_fwd_bucket(const FwdArgs& a, int variant, hipStream_t st)
{
    return a.stamps ? launch_fwd_bucket_st<D, NB, kVarStamp>(a, variant, st) : launch_fwd_bucket_st<D, NB, 0>(a, variant, st);
}

}  // namespace fa
