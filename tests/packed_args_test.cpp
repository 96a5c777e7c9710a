// What the tiled kernels unpack from their arguments (csrc/common.h: packed, unpacked) against what was packed, on the host, at the
// edges of every field's range; run by tests/test_packed_args.py.
#include "fwd_kernel.h"

#include <cstdio>
#include <cstring>
#include <random>

#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s (B %d H %d Hk %d Nq %d Nk %d d %d splits %d fold %d)\n", __LINE__, #x, a.B, a.H, a.Hk, a.Nq, a.Nk, a.d, a.num_splits, a.fold_rows); return 1; } } while (0)

template <bool kFold, typename P>
static int same(const fa::FwdArgs& a, const P& p, bool more)
{
    const fa::FwdArgs u = fa::unpacked<kFold>(p);
    const bool split = a.num_splits > 1;
    CHECK(u.Q == a.Q && u.K == a.K && u.V == a.V);
    CHECK(split ? u.O_partial == a.O_partial && u.LSE_partial == a.LSE_partial : u.O == a.O && u.LSE == a.LSE);
    CHECK(u.Nq == a.Nq && u.Nk == a.Nk && u.d == a.d && u.causal == a.causal && u.wl == a.wl && u.wr == a.wr);
    CHECK(u.scale_log2 == a.scale_log2 && u.num_splits == a.num_splits && u.keys_per_split == a.keys_per_split && u.Tr == a.Tr);
    CHECK(u.fold_rows == a.fold_rows && (!kFold || u.fold_group == a.fold_group));
    if (more) CHECK(u.H == a.H && u.alibi == a.alibi && u.keep_out == a.keep_out && u.scores_out == a.scores_out && u.stamps == a.stamps &&
                    u.drop_thr == a.drop_thr && u.drop_sub2 == a.drop_sub2 && u.drop_rscale == a.drop_rscale && u.seed_lo == a.seed_lo &&
                    u.seed_hi == a.seed_hi && u.off_lo == a.off_lo);
    std::mt19937 rng(3);
    const long long n = (long long)a.B * a.H * a.Tr * a.num_splits;
    for (int i = 0; i < 200; ++i) {
        const int block = (int)(i < 8 ? n - 1 - (i % n) : rng() % n), bh = (int)(rng() % ((long long)a.B * a.H)), row = (int)(rng() % a.Nq);
        const fa::WorkItem x = fa::work_item(a, block), y = fa::work_item(u, block);
        // (more query heads per K/V head than the field holds: the plain order, every slice once all the same)
        if (a.group_xcd < 65536) CHECK(x.bh == y.bh && x.split == y.split && x.m_block == y.m_block);
        CHECK(u.by_kv_group.quotient(bh) == bh / a.kv_group && (!kFold || u.by_fold.quotient(row) == row / a.fold_rows));
        if (more) CHECK(u.by_heads.quotient(bh) == bh / a.H);
    }
    return 0;
}

int main()
{
    std::mt19937_64 rng(1);
    auto below = [&](long long n) { return (long long)(rng() % (uint64_t)n); };
    for (int i = 0; i < 6000; ++i) {
        fa::FwdArgs a;
        std::memset(&a, 0, sizeof(a));
        const bool fold = i % 4 == 0, many = i % 50 == 1;
        const int group = fold ? 1 : many ? 65535 + (int)below(3) : 1 + (int)(below(4) * below(20));
        a.Hk = 1 + (int)below(many ? 3 : i % 3 ? 40 : 4000), a.kv_group = group, a.H = a.Hk * group, a.B = 1 + (int)below(many ? 2 : 9);
        a.Nq = 1 + (int)below(i % 2 ? 300 : 1 << 24), a.Nk = 1 + (int)below(i % 5 ? 5000 : (1 << 24) - 128), a.d = 1 + (int)below(128);
        a.num_splits = i % 3 ? 1 : 1 + (int)below(128), a.keys_per_split = 128 * (1 + (int)below(1 << 17)), a.causal = (int)below(2);
        a.wl = (int)below(a.Nk + 1) - 1, a.wr = (int)below(a.Nq + 1) - 1;
        a.scale_log2 = 0.01f * (float)i, a.alibi_left = (int)below(2);
        if (fold) {
            a.fold_rows = 2 + (int)below(63), a.fold_group = 2 + (int)below(1000);
            a.Nq = a.fold_rows * a.fold_group;
        }
        a.Tr = (a.Nq + 127) / 128;
        if ((long long)a.B * a.H * a.Tr * a.num_splits >= 0x7fffffffLL / 2) a.Tr = a.num_splits = 1;
        char* const base = reinterpret_cast<char*>(0x7f0012345000ull + (uint64_t)i * 16);
        a.Q = (fa::half_t*)base, a.K = (fa::half_t*)(base + 2), a.V = (fa::half_t*)(base + 4), a.O = (fa::half_t*)(base + 6);
        a.LSE = (float*)(base + 8), a.O_partial = (float*)(base + 16), a.LSE_partial = (float*)(base + 32), a.alibi = (float*)(base + 64);
        a.keep_out = (uint8_t*)(base + 65), a.scores_out = (float*)(base + 68), a.stamps = (uint64_t*)(base + 72);
        a.drop_thr = (uint32_t)below(65536), a.drop_sub2 = (uint32_t)rng(), a.drop_rscale = 1.25f;
        a.seed_lo = (uint32_t)rng(), a.seed_hi = (uint32_t)rng(), a.off_lo = (uint32_t)rng();
        fa::set_work_order<64, 1, fa::kVarVec>(a);
        const fa::PackedMore p = fa::packed(a);
        const fa::Packed core = p;
        if (fold ? same<true>(a, p, true) || same<true>(a, core, false) : same<false>(a, p, true) || same<false>(a, core, false)) return 1;
    }
    return 0;
}
