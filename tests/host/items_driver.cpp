// Work items over ket segments (cut_items, cut_items_split, KetCursor), walked as the kernels walk them: for
// random segment lists, item sizes, lanes per ket and primitive splits, every (ket, bra primitive) pair of a bra
// is visited exactly once, and the cursor reads no segment outside the bra's.  Run by tests/test_host_items.py.
#include <cstdio>
#include <random>
#include <vector>

#include "../../iqcp_amd/csrc/eri_launch.h"

using namespace qcg;

int main() {
    std::mt19937 rng(11);
    auto pick = [&](int lo, int hi) { return (int)(lo + rng() % (unsigned)(hi - lo + 1)); };
    int bad_cover = 0, bad_segment = 0, bad_pack = 0;
    long kets = 0;
    for (int trial = 0; trial < 400; ++trial) {
        std::vector<int2> segs;
        const int before = pick(0, 3), n = pick(1, 12), npp = pick(0, 3) ? pick(1, 60) : pick(200, kItemMaxPrim);
        int next = 0;
        for (int i = 0; i < before + n + 2; ++i) {  // other bras' segments around the bra's own
            const int len = pick(1, pick(0, 4) ? 9 : 20000);
            next += pick(0, 5);
            segs.push_back(make_int2(next, len));
            next += len;
        }
        const int g0 = before, g1 = before + n, lg = pick(0, kItemMaxLg), block = 64 << pick(0, 2);
        const int ch = std::max(1, std::min(kItemMaxKets, block * pick(1, 64)) >> lg), split = pick(0, 2) ? pick(1, 80) : 0;
        std::vector<int4> items;
        cut_items_split(items, segs, g0, g1, 7, ch, npp, split, lg);
        std::vector<int> seen((size_t)next, 0);
        for (const int4& it : items) {
            bad_pack += it.x != 7 || item_lg(it) != lg || item_kets(it) < 1 || item_kets(it) > ch;
            std::vector<PairRec> bra(8);
            bra[7].npp = npp;
            bra[7].pp_off = 1000;
            const PairRec P = item_bra(bra.data(), it);
            bad_pack += P.npp < 1 || P.pp_off < 1000 || P.pp_off + P.npp > 1000 + npp;
            for (int tid = 0; tid < block; tid += 1 << lg) {  // the first lane of each group
                KetCursor cur{segs.data(), it.y, it.z + (tid >> lg)};
                for (int j = tid >> lg; j < item_kets(it); j += block >> lg, cur.r += block >> lg) {
                    const int q = cur.at();
                    bad_segment += cur.g < g0 || cur.g >= g1;
                    if (q < 0 || q >= next) ++bad_cover;
                    else seen[q] += P.npp;
                    ++kets;
                }
            }
        }
        std::vector<int> want((size_t)next, 0);
        for (int g = g0; g < g1; ++g)
            for (int i = 0; i < segs[g].y; ++i) want[segs[g].x + i] = npp;
        bad_cover += seen != want;
    }
    std::printf("kets %ld\nbad_cover %d\nbad_segment %d\nbad_pack %d\n", kets, bad_cover, bad_segment, bad_pack);
    return 0;
}
