// The order in which the tiled kernel's launches deal out their work-groups (csrc/common.h: work_item, csrc/fwd_kernel.h:
// set_work_order), on the host; run by tests/test_work_order.py, which passes the name of a check.
#include "fwd_kernel.h"

#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s (B %d H %d G %d Tr %d splits %d chunk %d)\n", __LINE__, #x, a.B, a.H, a.kv_group, a.Tr, a.num_splits, a.slice_chunk); return 1; } } while (0)

static fa::FwdArgs args(int B, int H, int G, int Nq, int splits, int causal)
{
    fa::FwdArgs a;
    std::memset(&a, 0, sizeof(a));
    a.B = B, a.H = H, a.Hk = H / G, a.kv_group = G, a.Nq = Nq, a.Tr = (Nq + 127) / 128, a.num_splits = splits, a.causal = causal;
    a.wl = a.wr = -1;
    return a;
}

static constexpr int kPlain = fa::kVarVec | fa::kVarFullD;

// every head slice, split and row block once
template <int D, int VAR>
static int once(fa::FwdArgs a)
{
    fa::set_work_order<D, 1, VAR>(a);
    const int n = a.B * a.H * a.Tr * a.num_splits;
    std::vector<char> seen(n);
    for (int i = 0; i < n; ++i) {
        const fa::WorkItem it = fa::work_item(a, i);
        CHECK(it.bh >= 0 && it.bh < a.B * a.H && it.split >= 0 && it.split < a.num_splits && it.m_block >= 0 && it.m_block < a.Tr);
        char& s = seen[(it.bh * a.num_splits + it.split) * a.Tr + it.m_block];
        CHECK(!s);
        s = 1;
    }
    return 0;
}

static int bijection()
{
    std::mt19937 rng(1);
    auto below = [&](int n) { return (int)(rng() % n); };
    for (int i = 0; i < 4000; ++i) {
        const int G = 1 + below(3) * below(6), Hk = 1 + below(40), B = 1 + below(i % 4 ? 6 : 40);
        const fa::FwdArgs a = args(B, Hk * G, G, 1 + below(i % 2 ? 300 : 3000), i % 3 ? 1 : 1 + below(12), below(2));
        if (once<64, kPlain>(a) || once<96, kPlain | fa::kVarDropout>(a) || once<128, kPlain | fa::kVarPair>(a) || once<32, kPlain>(a)) return 1;
    }
    return 0;
}

// Four work-groups per CU, two row blocks per slice of which the second is nearly empty: a CU (work-group i goes to i % 256)
// holds as many of the one kind as of the other.
static int places()
{
    for (int B : {16, 32}) {
        fa::FwdArgs a = args(B, 512 / B, 1, 130, 1, 0);
        fa::set_work_order<64, 1, kPlain>(a);
        int full[256] = {};
        for (int i = 0; i < 1024; ++i) full[i % 256] += fa::work_item(a, i).m_block == 0;
        for (int n : full) CHECK(n == 2);
    }
    return 0;
}

// The query heads of a K/V head on one XCD (work-group i runs on i % 8), except for those of the last, incomplete round of eight
// K/V heads.
static int shared_heads()
{
    for (int G : {2, 3, 4, 7, 8})
        for (int Hk : {8, 11, 16, 75, 149})
            for (int Tr : {1, 3})
                for (int splits : {1, 3}) {
                    fa::FwdArgs a = args(1, Hk * G, G, 128 * Tr, splits, splits == 3);
                    fa::set_work_order<64, 1, kPlain>(a);
                    if (a.slice_chunk != a.H) continue;  // (chunks that are no multiple of G cannot)
                    std::vector<int> xcd(Hk * Tr * splits, -1), apart(Hk * Tr * splits);
                    for (int i = 0; i < a.H * Tr * splits; ++i) {
                        const fa::WorkItem it = fa::work_item(a, i);
                        const int k = (it.bh / G * splits + it.split) * Tr + it.m_block;
                        if (xcd[k] >= 0 && xcd[k] != i % 8) apart[k] = 1;
                        xcd[k] = i % 8;
                    }
                    int heads = 0;
                    for (int x : apart) heads += !x;
                    CHECK(heads >= Hk / 8 * 8 * Tr * splits);
                }
    return 0;
}

int main(int, char** argv)
{
    const char* what = argv[1];
    if (!std::strcmp(what, "bijection")) return bijection();
    if (!std::strcmp(what, "places")) return places();
    if (!std::strcmp(what, "shared_heads")) return shared_heads();
    return 2;
}
