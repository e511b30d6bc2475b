// SPDX-License-Identifier: Apache-2.0
#include "pcg_resident.hpp"
#include "pcg_sweep.hpp"

#include <algorithm>
#include <numeric>

namespace chysx_amd {

ResidentPlan plan_resident(const std::vector<ResidentInstance>& insts, const std::vector<int>& slice_ptr,
                           const std::vector<int>& cols, int bs, int cus, int max_lds) {
    ResidentPlan none, P;
    const int max_wgs = std::min(cus, kResidentMaxWgs);
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
            W.pause = exchange_pause(cluster, P.waves < kGroupSlices);
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
    P.by_start = resident_by_start(int(P.wgs.size()), P.max_cluster, cus);
    std::vector<int> clusters;
    int groups = 0;
    for (const ResidentInstance& I : insts) {
        clusters.push_back((I.nslices + P.waves - 1) / P.waves);
        groups += (I.nslices + kGroupSlices - 1) / kGroupSlices;
    }
    P.min_iters = resident_min_iters(clusters, groups, P.variant == kResidentB, cus);
    for (ResidentWg& W : P.wgs) W.pause_z = exchange_pause_z(W.cluster, P.waves < kGroupSlices, P.max_halo > 64 * (P.waves - 1));
    return P;
}

SweepPlan plan_sweep(int nslices, const std::vector<int>& slice_ptr, const std::vector<int>& cols,
                     const std::vector<int>& mir, const std::vector<int>& nlower, int max_wgs, int max_lds) {
    SweepPlan none, P;
    const int ngroups = (nslices + kGroupSlices - 1) / kGroupSlices;
    P.groups = std::max(2, (ngroups + max_wgs - 1) / max_wgs);
    if (P.groups > kSweepMaxGroups) return none;
    for (int s = 0; s < nslices; ++s)
        if (slice_ptr[size_t(s) + 1] - slice_ptr[size_t(s)] > kSweepWidth || nlower[size_t(s)] > 3) return none;
    const int span = P.groups * kGroupSlices, all = int(slice_ptr.size()) - 1;
    P.packed.assign(size_t(all) * kSweepPacked * 64, 0u);
    P.exported.assign(size_t(all) * 64, 0);
    std::vector<int> halo, place(size_t(all) * 64, -1);
    for (int s0 = 0; s0 < nslices; s0 += span) {
        SweepWg W{};
        W.slice0 = s0;
        W.nslices = std::min(span, nslices - s0);
        W.group = s0 / kGroupSlices;
        const int r0 = s0 * 64, nr = W.nslices * 64;
        halo.clear();
        const size_t e0 = size_t(slice_ptr[size_t(s0)]) * 64, e1 = size_t(slice_ptr[size_t(s0 + W.nslices)]) * 64;
        for (size_t q = e0; q < e1; ++q) {
            const int j = cols[q];
            if (j < 0 || (j >= r0 && j < r0 + nr) || place[size_t(j)] >= 0) continue;
            place[size_t(j)] = 0;
            halo.push_back(j);
        }
        std::sort(halo.begin(), halo.end());
        for (size_t q = 0; q < halo.size(); ++q) place[size_t(halo[q])] = int(q);
        W.halo0 = int(P.halo.size());
        W.nhalo = int(halo.size());
        P.lds_rows = std::max(P.lds_rows, nr + W.nhalo + 1);
        P.max_halo = std::max(P.max_halo, W.nhalo);
        if (P.lds_rows > 65535 || sweep_lds_bytes(P.groups, P.lds_rows, P.max_halo) > max_lds) return none;
        auto row_of = [&](size_t e) {
            const int j = cols[e];
            return unsigned(j < 0 ? nr + W.nhalo : (j >= r0 && j < r0 + nr) ? j - r0 : nr + place[size_t(j)]);
        };
        for (int s = s0; s < s0 + W.nslices; ++s) {
            const int sb = slice_ptr[size_t(s)], w = slice_ptr[size_t(s) + 1] - sb;
            uint32_t* out = P.packed.data() + size_t(s) * kSweepPacked * 64;
            for (int lane = 0; lane < 64; ++lane) {
                auto at = [&](int k) { return size_t(sb + k) * 64 + size_t(lane); };
                uint32_t row[kSweepWidth], off[3];
                for (int t = 0; t < kSweepWidth; ++t)
                    row[t] = t < w ? row_of(at((t & 1) ? w - 1 - (t >> 1) : t >> 1)) : unsigned(nr + W.nhalo);
                for (int k = 0; k < 3; ++k) {
                    const int d = k < w && mir[at(k)] >= 0 ? mir[at(k)] - int(at(k)) : 0;
                    if (d < -32768 || d > 32767) return none;
                    off[k] = uint32_t(d) & 0xFFFFu;
                }
                for (int q = 0; q < 3; ++q) out[q * 64 + lane] = row[2 * q] | row[2 * q + 1] << 16;
                out[3 * 64 + lane] = off[0] | off[1] << 16;
                out[4 * 64 + lane] = uint32_t(int16_t(off[2]));
            }
        }
        for (int r : halo) {
            P.exported[size_t(r)] = 1;
            place[size_t(r)] = -1;
        }
        P.halo.insert(P.halo.end(), halo.begin(), halo.end());
        P.wgs.push_back(W);
    }
    return P;
}

}  // namespace chysx_amd
