// CPU check of the colouring within the batches (minisod2d_amd/csrc/msod_plan.h),
// built by tests/test_plan_colors.py with AddressSanitizer and UBSan.  The column
// kernels add a batch's elements of one colour to its node sums without atomics,
// in `rounds` rounds: elements of one colour must share no node, and every
// colour must have its round.
//
// Input file as for plan_check.cpp, with int32 q appended: nodes of a line.
// Prints "OK rounds=<r>" or the first violated invariant.
#include <cstdio>
#include <cstdlib>
#include <set>

#include "msod_plan.h"

static int die(const char *what, long long a = -1, long long b = -1)
{
    std::printf("FAIL %s (%lld, %lld)\n", what, a, b);
    return 1;
}

static int check(const msod::HostPlan &P, int64_t nelem, int nn)
{
    if ((int64_t)P.ecol.size() != nelem) return die("ecol size");
    int most = 0;
    for (int64_t b = 0; b < P.nbatch; ++b) {
        const int64_t e0 = b * P.B, e1 = std::min<int64_t>(nelem, e0 + P.B);
        std::vector<std::vector<int64_t>> last(P.uoff[b + 1] - P.uoff[b], std::vector<int64_t>(64, -1));
        for (int64_t e = e0; e < e1; ++e) {
            const int c = P.ecol[e];
            if (c >= P.rounds || c >= 64) return die("colour without a round", e, c);
            most = std::max(most, c + 1);
            for (int l = 0; l < nn; ++l) {
                int64_t &owner = last[P.lidx[e * nn + l]][c];
                if (owner != -1 && owner != e) return die("two elements of one colour share a node", owner, e);
                owner = e;
            }
        }
    }
    if (most != P.rounds) return die("rounds", most, P.rounds);
    return 0;
}

int main(int argc, char **argv)
{
    if (argc != 2) return die("usage");
    FILE *f = std::fopen(argv[1], "rb");
    if (!f) return die("open");
    int64_t nelem, npoin;
    int32_t nn, B, q;
    if (std::fread(&nelem, 8, 1, f) != 1 || std::fread(&npoin, 8, 1, f) != 1 || std::fread(&nn, 4, 1, f) != 1 ||
        std::fread(&B, 4, 1, f) != 1)
        return die("header");
    std::vector<int32_t> l2g(nn), raw(nelem * nn);
    if (std::fread(l2g.data(), 4, nn, f) != (size_t)nn || std::fread(raw.data(), 4, raw.size(), f) != raw.size() ||
        std::fread(&q, 4, 1, f) != 1)
        return die("body");
    std::fclose(f);

    msod::HostPlan P;
    std::string err;
    if (!msod::build_host_plan(raw.data(), nelem, npoin, l2g, B, P, &err)) return die(err.c_str());
    if (int st = check(P, nelem, nn)) return st;

    // the library colours from lists in the lane layout: entries of an element
    // lie in its batch, on lanes of its own, once each
    const int64_t lanes = (int64_t)B * q * q, per = q * lanes;
    std::vector<uint16_t> lane(P.nbatch * per, 0xffff);
    for (int64_t e = 0; e < nelem; ++e)
        for (int l = 0; l < nn; ++l) {
            const int64_t at = msod::lane_entry(q, B, e, l);
            if (at < e / B * per || at >= (e / B + 1) * per) return die("lane entry outside its batch", e, l);
            if (at % lanes / q % B != e % B) return die("lane of another element", e, l);
            if (lane[at] != 0xffff) return die("lane entry twice", e, l);
            lane[at] = P.lidx[e * nn + l];
        }
    msod::HostPlan L;
    L.B = P.B;
    L.nbatch = P.nbatch;
    L.uoff = P.uoff;
    msod::color_elements(L, nelem, nn, [&](int64_t e, int l) { return lane[msod::lane_entry(q, B, e, l)]; });
    if (L.ecol != P.ecol || L.rounds != P.rounds) return die("colours from the lane layout");
    std::printf("OK rounds=%d\n", P.rounds);
    return 0;
}
