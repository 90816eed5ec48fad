// Host check of which banded pairs the band kernel takes (no GPU needed):
// pairs on either side of what its int32 counts and H hold.
#include <stdio.h>

#include <vector>

#include "../../anchorwave_amd/csrc/ksw2_plan.h"

using namespace kswhip;

static int failures = 0;

static void expect(bool want, int qlen, int tlen, int w, int8_t q, int8_t e, int8_t q2, int8_t e2)
{
    static const std::vector<uint8_t> zeros(8 << 20);
    int8_t mat[25];
    for (int k = 0; k < 25; ++k) mat[k] = k % 6 == 0 ? 0 : -6;
    KswScore sc;
    ScoreClass cls;
    if (!normalise_scoring(5, mat, q, e, q2, e2, &sc, &cls)) {
        printf("scoring refused\n");
        ++failures;
        return;
    }
    ksw2_pair_t p;
    p.query = p.target = zeros.data(), p.qlen = qlen, p.tlen = tlen;
    p.w = w, p.zdrop = -1, p.end_bonus = 0, p.flag = 0;
    const bool got = takes_band(p, 5, cls);
    if (got == want) return;
    printf("qlen %d tlen %d w %d G1 %d: band kernel %d, expected %d\n", qlen, tlen, w, sc.G1, got, want);
    ++failures;
}

int main()
{
    // gap scores 8/2, 75/1 (G1 = 10): pairs of the lengths its counts hold
    for (int n : {1000, 300000, 515000, 516500, 520000, 523000})
        for (int w : {1, 64, 301, 512, 4096, 100000}) expect(w < n, n, n, w, 8, 2, 75, 1);
    expect(true, 800000, 400000, 700000, 8, 2, 75, 1);
    expect(true, 3000000, 100000, 2950000, 8, 2, 75, 1);
    // the largest gap scores (G1 = 64): H ends at 2.06 M anti-diagonals
    expect(true, 520000, 520000, 4096, 60, 4, 62, 2);
    expect(true, 1900000, 100000, 1899999, 60, 4, 62, 2);
    expect(false, 2100000, 100000, 2099999, 60, 4, 62, 2);
    // counts
    for (int w : {10, 4096}) expect(false, 526000, 526000, w, 8, 2, 75, 1);
    expect(false, 7000000, 7000000, 4096, 8, 2, 75, 1);
    if (failures) return 1;
    printf("route ok\n");
    return 0;
}
