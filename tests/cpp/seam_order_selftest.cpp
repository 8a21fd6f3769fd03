// The order of a periodic row's pairs among the wavefronts of the seam kernel:
// every pair once, pair 0 right before pair NP - 1 and in the same wavefront,
// no two seams in one.
#include <cstdio>
#include <set>

#include "exchange_plan.hpp"

int main() {
    for (int NP = 65; NP < 420; ++NP) {
        if (NP % 64 == 0) continue;  // such rows are split instead
        const int rows = 130;
        long long before = -1;  // wavefront of the last row's seam
        for (int row = 0; row < rows; ++row) {
            const int seam = lbm::seam_place(row, NP);
            std::set<int> seen;
            for (int place = 0; place < NP; ++place) seen.insert(lbm::seam_pair_at(place, seam, NP));
            const long long at = (long long)row * NP + seam;
            if ((int)seen.size() != NP || *seen.begin() != 0 || *seen.rbegin() != NP - 1 ||
                lbm::seam_pair_at(seam, seam, NP) != 0 || lbm::seam_pair_at(seam + 1, seam, NP) != NP - 1 ||
                at / 64 != (at + 1) / 64 || at / 64 == before) {
                std::printf("NP %d row %d\n", NP, row);
                return 1;
            }
            before = at / 64;
        }
    }
    std::printf("ok\n");
    return 0;
}
