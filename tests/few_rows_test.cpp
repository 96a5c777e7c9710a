// Launches of few rows (csrc/common.h: packed_rows, unpacked_rows, rows_item), on the host, at the edges of every field's range; run by
// tests/test_few_rows.py.
#include "fwd_kernel.h"

#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s (slices %d rows %d d %d splits %d fold %d)\n", __LINE__, #x, a.B * a.H, a.Nq, a.d, a.num_splits, a.fold_rows); return 1; } } while (0)

// every slice, split and row block once, those of a split on one XCD but for the last few of the order
template <bool kOneBlock>
static int order(const fa::FwdArgs& a, const fa::FwdArgs& u)
{
    const int slices = a.B * a.H, pairs = slices * a.num_splits;
    std::vector<int> seen(pairs * a.Tr, -1);
    for (int i = 0; i < pairs * a.Tr; ++i) {
        const fa::WorkItem it = fa::rows_item<kOneBlock>(u, i);
        CHECK(it.bh >= 0 && it.bh < slices && it.split >= 0 && it.split < a.num_splits && it.m_block >= 0 && it.m_block < a.Tr);
        int& s = seen[(it.split * slices + it.bh) * a.Tr + it.m_block];
        CHECK(s < 0);
        s = i;
    }
    for (int p = 0; p < (pairs & ~7); ++p)
        for (int m = 1; m < a.Tr; ++m) CHECK(seen[p * a.Tr + m] % 8 == seen[p * a.Tr] % 8);
    return 0;
}

int main()
{
    std::mt19937_64 rng(1);
    auto below = [&](long long n) { return (long long)(rng() % (uint64_t)n); };
    for (int i = 0; i < 4000; ++i) {
        fa::FwdArgs a;
        std::memset(&a, 0, sizeof(a));
        a.B = 1 + (int)below(i % 2 ? 4 : 16), a.Hk = 1 + (int)below(16), a.kv_group = i % 3 ? 1 + (int)below(8) : 1, a.H = a.Hk * a.kv_group;
        a.Nq = 1 + (int)below(128);
        if (i % 3 == 0) {
            a.fold_rows = 1 + (int)below(64), a.fold_group = 1 + (int)below(128 / a.fold_rows);
            a.Nq = a.fold_rows * a.fold_group;
        }
        a.Nk = 1 + (int)below((1 << 24) - 128), a.d = 1 + (int)below(128), a.num_splits = 1 + (int)below(32), a.Tr = (a.Nq + 31) / 32;
        a.keys_per_split = 128 * (1 + (int)below(1 << 17)), a.causal = (int)below(2), a.combine_waves = below(2) ? 4 : 1;
        a.wl = (int)below(a.Nk + 1) - 1, a.wr = (int)below(a.Nq + 1) - 1, a.scale_log2 = 0.01f * (float)i;
        char* const base = reinterpret_cast<char*>(0x7f0012345000ull + (uint64_t)i * 16);
        a.Q = (fa::half_t*)base, a.K = (fa::half_t*)(base + 2), a.V = (fa::half_t*)(base + 4), a.O = (fa::half_t*)(base + 6);
        a.LSE = (float*)(base + 8), a.O_partial = (float*)(base + 16), a.LSE_partial = (float*)(base + 32);
        a.counters = (uint32_t*)(base + 36), a.stamps = (uint64_t*)(base + 72);
        fa::set_divisors(a, (long long)a.B * a.H);
        const fa::PackedRowsMore p = fa::packed_rows(a);
        const fa::PackedRows core = p;
        const fa::FwdArgs u = a.fold_rows ? fa::unpacked_rows<true>(core) : fa::unpacked_rows<false>(core);
        CHECK(u.Q == a.Q && u.K == a.K && u.V == a.V && u.O == a.O && u.LSE == a.LSE && u.O_partial == a.O_partial && u.LSE_partial == a.LSE_partial);
        CHECK(u.counters == a.counters && u.combine_waves == a.combine_waves && u.Nq == a.Nq && u.Nk == a.Nk && u.d == a.d && u.Tr == a.Tr);
        CHECK(u.causal == a.causal && u.wl == a.wl && u.wr == a.wr && u.scale_log2 == a.scale_log2 && u.num_splits == a.num_splits);
        CHECK(u.keys_per_split == a.keys_per_split && u.fold_rows == a.fold_rows && u.fold_group == a.fold_group);
        CHECK(fa::unpacked_rows<true>(p).stamps == a.stamps);
        for (int bh = 0; bh < a.B * a.H; ++bh) CHECK(u.by_kv_group.quotient(bh) == bh / a.kv_group);
        for (int r = 0; r < a.Nq && a.fold_rows; ++r) CHECK(u.by_fold.quotient(r) == r / a.fold_rows);
        if (a.Tr == 1 ? order<true>(a, u) : order<false>(a, u)) return 1;
        // a count that fills the GPU is one that the launch takes
        const int s = fa::rows_form_splits((long long)a.B * a.H, a.Nq, a.d, 1 + a.Nk % 60000), n = (a.Nk % 60000 + 128) / 128;
        if (s > 0) CHECK(s <= n && fa::rows_form_fits((long long)a.B * a.H, a.Nq, a.d, 1 + a.Nk % 60000, s, 128 * ((n + s - 1) / s)));
    }
    return 0;
}
