// SPDX-License-Identifier: Apache-2.0
#include "pcg_resident.hpp"

#include <algorithm>
#include <numeric>

namespace chysx_amd {

ResidentPlan plan_resident(const std::vector<ResidentInstance>& insts, const std::vector<int>& slice_ptr,
                           const std::vector<int>& cols, int bs, int max_wgs, int max_lds) {
    ResidentPlan none, P;
    int width = 0;
    for (size_t s = 0; s + 1 < slice_ptr.size(); ++s) width = std::max(width, slice_ptr[s + 1] - slice_ptr[s]);
    if (bs == 6 && width <= kResidentWidthA) P.variant = kResidentA;
    else if (bs == 6 && width <= kResidentWidthB) P.variant = kResidentB;
    else if (bs == 9 && width <= kResidentWidthC) P.variant = kResidentC;
    else return none;
    P.waves = P.variant == kResidentA ? kGroupSlices : kGroupSlices / 2;

    for (const ResidentInstance& I : insts)
        if ((I.nslices + P.waves - 1) / P.waves > max_wgs) return none;

    // Larger instances first: their workgroups iterate longest, and a batch
    // ends with the small ones.
    std::vector<int> order(insts.size());
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(),
                     [&](int a, int b) { return insts[size_t(a)].nslices > insts[size_t(b)].nslices; });

    P.loc.assign(cols.size(), 0);
    P.exported.assign((slice_ptr.size() - 1) * 64, 0);
    std::vector<int> halo;
    std::vector<int> place((slice_ptr.size() - 1) * 64, -1);  // of a halo row in the current workgroup's list
    for (int k : order) {
        const ResidentInstance& I = insts[size_t(k)];
        const int cluster = (I.nslices + P.waves - 1) / P.waves;
        P.max_cluster = std::max(P.max_cluster, cluster);
        const int first = int(P.wgs.size());
        for (int c = 0; c < cluster; ++c) {
            ResidentWg W{};
            W.inst = k;
            W.slice0 = I.slice0 + c * P.waves;
            W.nslices = std::min(P.waves, I.nslices - c * P.waves);
            W.group = c * P.waves / kGroupSlices;
            W.piece = (c * P.waves % kGroupSlices) / P.waves;
            W.cluster = cluster;
            W.first = first;
            const int r0 = W.slice0 * 64, nr = W.nslices * 64;
            halo.clear();
            const size_t e0 = size_t(slice_ptr[size_t(W.slice0)]) * 64;
            const size_t e1 = size_t(slice_ptr[size_t(W.slice0 + W.nslices)]) * 64;
            for (size_t q = e0; q < e1; ++q) {
                const int j = cols[q];
                if (j < 0 || (j >= r0 && j < r0 + nr) || place[size_t(j)] >= 0) continue;
                place[size_t(j)] = 0;
                halo.push_back(j);
            }
            std::sort(halo.begin(), halo.end());
            for (size_t q = 0; q < halo.size(); ++q) place[size_t(halo[q])] = int(q);
            const int rows = nr + int(halo.size()) + 1;
            // the offsets are 16 bits wide
            if (12 * rows > 65535) return none;
            P.lds_rows = std::max(P.lds_rows, rows);
            P.max_halo = std::max(P.max_halo, int(halo.size()));
            P.max_nslices = std::max(P.max_nslices, W.nslices);
            W.halo0 = int(P.halo.size());
            W.nhalo = int(halo.size());
            // LDS rows: own, halo, then the zero row that padding entries read
            for (size_t q = e0; q < e1; ++q) {
                const int j = cols[q];
                const int at = j < 0 ? nr + W.nhalo : (j >= r0 && j < r0 + nr) ? j - r0 : nr + place[size_t(j)];
                P.loc[q] = uint16_t(12 * at);
            }
            for (int r : halo) {
                P.exported[size_t(r)] = 1;
                place[size_t(r)] = -1;
            }
            P.halo.insert(P.halo.end(), halo.begin(), halo.end());
            P.wgs.push_back(W);
        }
    }
    if (resident_lds_bytes(P.lds_rows, P.max_halo, P.waves) > max_lds) return none;
    return P;
}

}  // namespace chysx_amd
