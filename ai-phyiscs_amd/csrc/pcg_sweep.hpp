// SPDX-License-Identifier: Apache-2.0
//
// The iterations of one large cloth in one launch: the vectors stay on the
// chip, the matrix streams by.  Host plan and device view.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "cloth_kernels.hpp"
#include "pcg_resident.hpp"

namespace chysx_amd {

constexpr int kSweepWaves = 8;
constexpr int kSweepMaxGroups = 4;  // 16-slice groups of a workgroup: 8 rows a lane
constexpr int kSweepWidth = 6;      // entries of the widest row
constexpr int kSweepPacked = 5;     // words a row of packed indices
constexpr int kSweepKinds = 3;      // p . Ap; r . z, |r|^2

struct SweepWg {
    int slice0, nslices;  // slices holding rows
    int group;            // first 16-slice group
    int halo0, nhalo;     // rows of other workgroups that its rows couple to
};

struct SweepPlan {
    int groups = 0;  // groups of a workgroup (0: the problem does not fit)
    int lds_rows = 0, max_halo = 0;
    std::vector<SweepWg> wgs;
    // Per row: the LDS rows of its columns in the order they are visited (0,
    // w - 1, 1, w - 2, .., the zero row past the slice's width), two a word,
    // and the mirror offsets of its first three entries.
    std::vector<uint32_t> packed;
    std::vector<int> halo;
    std::vector<uint8_t> exported;
};

// Plan for one cloth of `nslices` row-holding slices with packed blocks; mir:
// entry index of an entry's mirror, -1 for none.  It takes rows of at most
// kSweepWidth entries, the lower ones among the first three, as a regularly
// triangulated grid has (every workgroup waits for the slowest each
// iteration: one with 2 of its 8 rows a lane on a loop for any width took half
// as long again); other meshes stay with the streaming kernels.
SweepPlan plan_sweep(int nslices, const std::vector<int>& slice_ptr, const std::vector<int>& cols,
                     const std::vector<int>& mir, const std::vector<int>& nlower, int max_wgs, int max_lds);

struct SweepView {
    int groups, nwg, ngroups, lds_rows, max_halo, rows;
    const SweepWg* wgs;
    const uint32_t* packed;
    const float* zeros;  // a block of an entry, all zero
    const int* halo;
    const uint8_t* exported;
    unsigned long long* zx;     // as ResidentView
    unsigned long long* slots;  // kinds x copies x 2 halves x groups words
    double* solo;               // 3 per slice, or null
    ResidentSync* sync;
    int meet_polls;
    int pause;  // before the look for p . Ap; the update's sums wait behind the iterate and need none
};
inline size_t sweep_slot_words(int ngroups) { return size_t(kSweepKinds) * kResidentCopies * 2 * size_t(ngroups); }
inline int sweep_lds_bytes(int groups, int lds_rows, int max_halo) {
    return 4 * 3 * (lds_rows + max_halo + groups * 16 * 64);
}
constexpr int kSweepStaticLds = 2048;

// Iterations from a started or restarted solve (r and z in v, p = z) until a
// true-residual check is due (the state says so and owes its advance) or the
// solve has stopped; x is complete then.  One instance.
void launch_pcg_sweep(const SweepView& R, const LaunchGeom& g, const DevMatrix& A, const DevVectors& v, InstState* st,
                      const InstParams* params, hipStream_t s);

}  // namespace chysx_amd
