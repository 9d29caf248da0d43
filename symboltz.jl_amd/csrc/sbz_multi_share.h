// How many modes of each family share an entry of a mixed-model launch.
#pragma once
#include <algorithm>

// per[f] for a family of n_inst[f] instances: 1 when they run in the one-mode body (rows[f] == 1), rows[f] in a
// row body, and with one hierarchy per lane (group[f] > 0 modes per wavefront) as few as let all the entries
// be resident at once: a step takes as long for one mode as for a full wavefront.  A family without
// instances has no entries and no say.
inline void sbz_multi_share(int n, const int* n_inst, const int* rows, const int* group, int resident, int* per) {
    int largest = 1;
    for (int f = 0; f < n; ++f)
        if (n_inst[f] > 0 && rows[f] > 1) largest = std::max(largest, group[f]);
    for (int share = 1; share <= largest; ++share) {
        long long entries = 0;
        for (int f = 0; f < n; ++f) {
            per[f] = (n_inst[f] <= 0 || rows[f] <= 1) ? 1 : group[f] ? std::min(share, group[f]) : rows[f];
            entries += ((long long)n_inst[f] + per[f] - 1) / per[f];
        }
        if (entries <= resident) break;
    }
}
