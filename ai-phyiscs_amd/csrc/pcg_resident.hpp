// SPDX-License-Identifier: Apache-2.0
//
// The whole PCG solve of an instance as one launch: host plan and device view.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <functional>
#include <limits>
#include <vector>

#include "cloth_kernels.hpp"
#include "resident_gate.hpp"

namespace chysx_amd {

// One workgroup of the resident solve: up to `waves` consecutive slices of
// one instance.  A 16-wave workgroup owns one 16-slice group; 8-wave ones own
// half a group each (piece 0 or 1).  An instance's workgroups are consecutive.
struct ResidentWg {
    int inst;
    int slice0;   // first slice
    int nslices;  // slices holding rows
    int group;    // group within the instance
    int piece;
    int halo0;    // first entry of its halo list
    int nhalo;    // rows of other workgroups that its rows couple to
    int cluster;  // workgroups of the instance
    int first;    // the instance's first workgroup
    int pause;    // before it looks for a sum of one value, and for the
    int pause_z;  // neighbours' z with an update's sums: s_sleep units
};

// The three kernels, by what a lane's row takes of the registers: up to
// kResidentWidthA packed blocks (a grid's six, 36 registers) leave room for 16
// waves a compute unit at 128 registers; wider rows (96) and 9-float blocks
// (126) take 8 waves at 256.  One row a lane: what is left of a lane's
// registers would not hold a second row, and a problem that needs more
// workgroups than the device has compute units streams its matrix instead
// (512 x 512 is the largest square cloth here, 362 x 362 with bending).
enum ResidentVariant : int { kResidentNone = 0, kResidentA = 1, kResidentB = 2, kResidentC = 3 };
constexpr int kResidentWidthA = 6;   // packed
constexpr int kResidentWidthB = 16;  // packed
constexpr int kResidentWidthC = 14;  // 9 floats

constexpr int kResidentMaxWgs = 256;       // workgroups of an instance
constexpr int kResidentStaticLds = 36864;  // LDS of the kernels beside the dynamic part
constexpr int kResidentMeetPolls = 400000;  // about half a second

struct ResidentPlan {
    int variant = kResidentNone;
    int waves = 0;
    int max_nslices = 0;        // widest workgroup
    int max_cluster = 0;
    // Workgroups take their places in the order they start, not by their
    // number (resident_by_start).
    bool by_start = false;
    int min_iters = 0;          // iterations from which the solve is faster in one launch (resident_min_iters)
    int lds_rows = 0;           // own and halo rows of the largest workgroup, and the zero row
    int max_halo = 0;
    std::vector<ResidentWg> wgs;
    std::vector<uint16_t> loc;  // per matrix entry: byte offset of its column's vector in LDS
    std::vector<int> halo;      // row indices, ascending per workgroup
    std::vector<uint8_t> exported;  // per row: 1 when another workgroup needs it
};

// Which workgroup takes which place of a launch of `wgs` workgroups on `cus`
// compute units.  An XCD is given every 8th workgroup, in order, and no other,
// and a workgroup here has a compute unit to itself.
// In the order they start (true): at most one instance has only part of its
// workgroups running, and an XCD that is ahead takes more places than one that
// is behind (512 uneven cloths: 24.8 ms, and 26.1 ms by number).  But the
// waiting part of an instance must not be able to fill an XCD: the missing
// workgroups may be bound to that XCD, and then all wait until the start-up
// agreement gives up (two cloths of 198 workgroups: 164 ms a step on average,
// 0.8 ms by number).
// By number (false): an instance lies evenly over the XCDs, and the first one
// that has not met is next in line on each of them, so it always comes to run.
inline bool resident_by_start(int wgs, int max_cluster, int cus) {
    return max_cluster > 1 && (wgs <= cus || max_cluster <= cus / kXcds);
}

// How long a workgroup waits, in s_sleep units of 64 cycles, before it first
// looks for the sums of `wgs` workgroups.  The words need some 2600 cycles to
// arrive, and those of the slowest workgroup come the later the more there
// are; a look before that takes a round trip of 1500 cycles itself and,
// together with every other workgroup's, holds up the words looked for.  None
// up to 8 workgroups (12 units cost 2% at 4) or, of half groups, whose looks
// take nine words a group, up to 24 (12 units cost 1% at 20); then 12 (512
// cloths of up to 16 workgroups: 25.3 ms without and 24.8 with, 150 x 150: 5.5
// and 5.3 us an iteration), and 6 more with each doubling beyond 32: within 3%
// of the best of 0 to 32 units at 32 to 256 workgroups.  An iteration without
// and with it: 6.0 and 5.4 us at 64 workgroups, 9.0 and 6.4 at 157, 10.0 and
// 8.4 at 256; 12.3 and 10.3 us at 176 half-group workgroups.
inline int exchange_pause(int wgs, bool halves) {
    return wgs <= (halves ? 24 : 8) ? 0 : std::max(12, int(std::lround(6.0 * std::log2(wgs / 8.0))));
}
// The same before the neighbours' z, which is sent ahead of an update's sums:
// 6 units less.  `wide`: even the wave that waits for the sums has halo rows
// to receive, and their wait is most of the pause.  From 480 x 480 on 6 units
// are best (512 x 512: 8.5 us an iteration against 8.9 with 18), up to
// 430 x 430 the difference of 6 is (8.2 us with 18 units, 9.1 with 6).
inline int exchange_pause_z(int wgs, bool halves, bool wide) {
    const int p = exchange_pause(wgs, halves) - 6;
    return p <= 0 ? 0 : wide ? std::min(p, 6) : p;
}

// Iterations from which a batch is solved faster in one launch than by the
// streaming kernels; kResidentNever: at no count.  clusters: the instances'
// workgroups.  A batch whose workgroups all fit at once always is (1.2 to 3
// times at 1 to 50 iterations), and so is one of single workgroups.  Beyond
// that, whole groups lose at one iteration only (16 cloths of 256 x 256: 462
// and 429 us; at 10 iterations 1.2 to 1.7 times as fast, at 50 1.4 to 2.4).
// Half groups, on wide-row meshes, take twice the compute units for their
// rows, and cloths that leave many of them unused gain nothing or lose (16
// of 257 x 257, 130 workgroups each: 7.5 ms and 4.9 at 50 iterations).
// Microseconds an iteration of the two forms, fitted at 2 to 256 workgroups a
// cloth and 128 to 2048 groups (within 15%): 4.7 + 0.45 log2(workgroups) for
// each generation of cloths that fit side by side, and 0.082 a group, at
// least 20 to 24, or 33 from one group more than there are compute units on.
// Loading the blocks costs the solve in one launch 0.35 us a group.
constexpr int kResidentNever = std::numeric_limits<int>::max();
inline int resident_min_iters(const std::vector<int>& clusters, int groups, bool halves, int cus) {
    int wgs = 0, widest = 0;
    double one = 0.0;
    for (int c : clusters) {
        wgs += c;
        widest = std::max(widest, c);
        one += (4.7 + 0.45 * std::log2(double(c))) / double(std::max(1, cus / c));
    }
    if (wgs <= cus || widest <= 1) return 0;
    if (!halves) return 2;
    const double streamed = std::max(groups <= cus ? 20.0 + 0.015 * groups : 33.0, 0.082 * groups);
    return streamed <= one ? kResidentNever : int(std::ceil(0.35 * groups / (streamed - one)));
}

// One instance's rows for the plan.
struct ResidentInstance {
    int slice0, nslices;  // slices holding rows
};

// Plan for rows of `bs`-float blocks in the wave-sliced ELL layout (columns in
// row space, -1 for padding), on `cus` compute units.  variant kResidentNone:
// the problem stays with the kernels that stream the matrix (a row is too
// wide, an instance needs more than `cus` or kResidentMaxWgs workgroups, or a
// workgroup's own and halo rows do not fit in max_lds bytes).
ResidentPlan plan_resident(const std::vector<ResidentInstance>& insts, const std::vector<int>& slice_ptr,
                           const std::vector<int>& cols, int bs, int cus, int max_lds);

// What the host has to know of solves that it may not ask for their outcome,
// in pinned memory; stays until the host takes it back.
struct ResidentNotice {
    int lost;   // 1: a solve lost a workgroup, or was not started after one that did
    int alone;  // 1: an instance's workgroups did not meet in time, and one of them solved it
    int left;   // 1: the same of a launch that leaves the solve to the caller
};

// Steps on the streaming kernels after a solve whose workgroups did not meet
// in time: something else holds compute units (another process, a mask), and
// each try costs the start-up bound and, where the host does not wait for the
// solve, one by a single workgroup (up to a second or more).  1024 steps, then
// twice as many each time, until as many have met.
class ResidentHold {
public:
    static constexpr int kFirst = 1024, kLongest = 1 << 16;
    // Called once a step: whether it may be solved in one launch.
    bool may_run() {
        if (left_ > 0) {
            --left_;
            return false;
        }
        if (++met_ > next_) next_ = kFirst;
        return true;
    }
    void missed() {
        left_ = next_;
        next_ = std::min(2 * next_, kLongest);
        met_ = 0;
    }

private:
    int left_ = 0, next_ = kFirst, met_ = 0;
};

// Start-up agreement of an instance's workgroups, kept in device memory across
// launches (counts all zero at first).
struct ResidentSync {
    unsigned long long arrived;   // workgroups started, over all launches
    unsigned long long decision;  // 2 L: launch L (1, 2, ...) runs; 2 L + 1: its workgroups did not meet in time
    unsigned epoch;               // last tag used in the exchange words
    // 1: a wait of an exchange ran out.  Words with tags beyond the epoch may
    // be there or still come, so no solve starts until the host has cleared them.
    unsigned lost;
    ResidentNotice* notice;
};

struct ResidentView {
    int variant, waves, block_waves, nwg, lds_rows, lds_x, lds_bytes, max_cluster;
    const ResidentWg* wgs;
    const uint16_t* loc;
    const int* halo;
    const uint8_t* exported;
    unsigned long long* zx;     // 2 words a row (all first words, then all second ones): z of the exported rows
    int rows;                   // padded rows of the problem
    unsigned long long* slots;  // partial sums: kinds x pieces x copies x 2 halves x groups words
    double* solo;               // 3 per slice: partial sums of an instance solved by one workgroup;
                                // null: a launch whose workgroups do not meet leaves all as it was
    ResidentSync* sync;         // per instance
    unsigned long long* ticket; // workgroups started, over all launches; null: places by number
    int meet_polls;             // bound of the start-up wait, in polls of about a microsecond
};
constexpr int kResidentKinds = 6;   // 0: p . Ap; 1, 2: r . z, |r|^2; 3 .. 5: start, check and report sums
constexpr int kResidentPieces = 9;  // a group's sum, or its first half's and the waves of its second
// LDS of a workgroup, in floats: 3 a row for the own, halo and zero rows, 3 a
// halo row as received, then (8-byte aligned) 9 a lane for the iterate and a
// direction.
inline int resident_lds_x(int lds_rows, int max_halo) { return (3 * (lds_rows + max_halo) + 1) & ~1; }
inline int resident_lds_bytes(int lds_rows, int max_halo, int block_waves) {
    return 4 * (resident_lds_x(lds_rows, max_halo) + 9 * 64 * block_waves);
}
constexpr int kResidentCopies = 8;  // copies of the sums, for different readers
inline size_t resident_slot_words(int ngroups) {
    return size_t(kResidentKinds) * kResidentPieces * kResidentCopies * 2 * size_t(ngroups);
}

// Status of an instance whose solve lost a workgroup (a wait of the exchange
// ran out); the host reports an error.
constexpr int kResidentLost = 4;

// Start residual, iterations, true-residual checks, report residual and
// finalize of every instance, from the assembled system.  host_st: the solver
// states in pinned host memory.  start_given_r: the start residual is in v.r.
void launch_pcg_resident(const ResidentView& R, const LaunchGeom& g, const DevMatrix& A, const DevVectors& v,
                         const DevExt& e, const DevMesh& m, InstState* st, InstState* host_st,
                         const InstParams* params, float dt, int start_given_r, hipStream_t s);

// Runs `enqueue`, which puts a launch of `owner` on stream s, behind those of
// the device's launches in flight that it cannot run beside, and records
// `done` after it.  weight and room: gate_weight, gate_room.
struct GatedLaunch {
    const void* owner;
    hipEvent_t done;
    int device, weight, room;
};
void with_resident_gate(const GatedLaunch& L, hipStream_t s, const std::function<void()>& enqueue);
// The owner's launches have run, and its event goes away.
void leave_resident_gate(int device, const void* owner);

}  // namespace chysx_amd
