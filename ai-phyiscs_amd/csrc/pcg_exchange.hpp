// SPDX-License-Identifier: Apache-2.0
//
// What the one-launch solves share: sums over a wavefront, tagged words
// between workgroups, the start-up agreement and the solve by one workgroup.
#pragma once

#include <hip/hip_runtime.h>

#include "pcg_device.hpp"
#include "pcg_resident.hpp"

namespace chysx_amd {

namespace {

typedef unsigned long long u64;

constexpr int kKindSigma = 0, kKindUpdate = 1, kKindTrue = 3;
constexpr int kExchangePolls = 1 << 22;  // several seconds: a workgroup of the instance is lost

__device__ __forceinline__ u64 agent_load(const u64* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void agent_store(u64* p, u64 v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Keep a value from being known across the loop of the iterations: what is
// derived from it (addresses, unpacked offsets, masks) is then formed where it
// is used instead of being held in registers for the whole solve.
__device__ __forceinline__ int fresh(int x) {
    asm volatile("" : "+v"(x));
    return x;
}
__device__ __forceinline__ u64 tagged(unsigned tag, unsigned v) { return (u64(tag) << 32) | v; }

// Sum over the 64 lanes, in every lane: the exchanges of the xor butterfly
// 32, 16, .., 1 by register moves.  Below a row of 16 a rotation by n reaches
// a lane that holds the same sum as the lane n away by xor.
template <int CTRL>
__device__ __forceinline__ double add_rotated(double a) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(a), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(a), CTRL, 0xf, 0xf, false);
    return a + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_sum(double a) {
    const unsigned l0 = unsigned(__double2loint(a)), h0 = unsigned(__double2hiint(a));
    const auto l = __builtin_amdgcn_permlane32_swap(l0, l0, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(h0, h0, false, false);
    a = __hiloint2double(int(h[0]), int(l[0])) + __hiloint2double(int(h[1]), int(l[1]));
    const unsigned l1 = unsigned(__double2loint(a)), h1 = unsigned(__double2hiint(a));
    const auto m = __builtin_amdgcn_permlane16_swap(l1, l1, false, false);
    const auto n = __builtin_amdgcn_permlane16_swap(h1, h1, false, false);
    a = __hiloint2double(int(n[0]), int(m[0])) + __hiloint2double(int(n[1]), int(m[1]));
    a = add_rotated<0x128>(a);
    a = add_rotated<0x124>(a);
    a = add_rotated<0x122>(a);
    return add_rotated<0x121>(a);
}

// What the sums need to know of the instance.
struct Cluster {
    int size;      // workgroups
    int ngroups;   // groups that hold rows
    int nslices;   // slices that hold rows
    int group0;    // first group of the instance
    int total;     // groups of the problem
    int group, piece;
    int waves;     // of this workgroup that hold rows
    int copy;      // the copy of the sums that this workgroup reads
    u64* slots;
    int pause, pause_z;  // before the first look, see exchange_pause
};

__device__ __forceinline__ void pause(int n) {
#pragma nounroll
    for (; n > 0; --n) __builtin_amdgcn_s_sleep(1);
}

// A sum's words: the low halves of a copy's groups, then the high halves.
// Every workgroup reads all groups' words, so they are kept in several copies
// for different readers: in one copy, 256 workgroups wait at a few memory
// channels.
__device__ __forceinline__ u64* slot_of(const Cluster& C, int kind, int piece, int copy, int group) {
    return C.slots + ((kind * kResidentPieces + piece) * kResidentCopies + copy) * 2 * C.total + C.group0 + group;
}
__device__ __forceinline__ void slot_store(const Cluster& C, u64* w, unsigned tag, double d) {
    agent_store(w, tagged(tag, unsigned(__double2loint(d))));
    agent_store(w + C.total, tagged(tag, unsigned(__double2hiint(d))));
}
__device__ __forceinline__ double slot_wait(const Cluster& C, const u64* w, unsigned tag, int& failed) {
    u64 a, b;
    int n = 0;
#pragma nounroll
    do {
        a = agent_load(w);
        b = agent_load(w + C.total);
    } while ((unsigned(a >> 32) != tag || unsigned(b >> 32) != tag) && ++n < kExchangePolls);
    if (n >= kExchangePolls) failed = 1;
    return __hiloint2double(int(unsigned(b)), int(unsigned(a)));
}

// A wait of the exchange ran out, in this launch or an earlier one.
__device__ __forceinline__ void notify(int* word) {
    __hip_atomic_store(word, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ void lost_exchange(ResidentSync* S) {
    S->lost = 1;
    notify(&S->notice->lost);
}

// The instance's workgroups agree that they run: all of them have started, so
// every wait that follows ends.  If they have not met within R.meet_polls (the
// device's compute units are held by waiting workgroups of another process),
// one of them solves the instance alone and the others leave, or all leave
// where the caller goes on (`alone` false).  After a launch
// that lost a workgroup all leave (a loss in this launch comes after all have
// met, so they agree on that, too).
enum Meeting : int { kMeetRun = 0, kMeetLeave = 1, kMeetAlone = 2 };
__device__ int meet(ResidentSync* S, int cluster, int polls, bool alone) {
    if (S->lost != 0) {
        lost_exchange(S);
        return kMeetLeave;
    }
    const u64 a = __hip_atomic_fetch_add(&S->arrived, u64(1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const u64 run = 2 * (a / u64(cluster) + 1);
    if ((a + 1) % u64(cluster) == 0) {
        u64 old = agent_load(&S->decision);
        if (old < run)
            __hip_atomic_compare_exchange_strong(&S->decision, &old, run, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma nounroll
    for (int n = 0; n < polls; ++n) {
        const u64 d = agent_load(&S->decision);
        if (d >= run) return d == run ? kMeetRun : kMeetLeave;
        __builtin_amdgcn_s_sleep(2);
    }
    u64 old = agent_load(&S->decision);
    if (old < run && __hip_atomic_compare_exchange_strong(&S->decision, &old, run + 1, __ATOMIC_RELAXED,
                                                          __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
        notify(alone ? &S->notice->alone : &S->notice->left);
        return alone ? kMeetAlone : kMeetLeave;
    }
    return old == run ? kMeetRun : kMeetLeave;
}

// The solve of an instance by one workgroup, its vectors in global memory: the
// way out when the instance's workgroups cannot all run at once.
template <int NW>
struct Alone {
    const LaunchGeom& g;
    const DevMatrix& A;
    const DevVectors& v;
    const InstParams& pr;
    double* scratch;  // 3 per slice of the problem
    double* group;    // LDS, one per group of the instance
    int s0, ns;       // slices of the instance that hold rows
    int tid, wave, lane, ng;

    __device__ __forceinline__ Alone(const LaunchGeom& g_, const DevMatrix& A_, const DevVectors& v_,
                                     const InstParams& pr_, const InstState& S, double* scratch_, double* group_)
        : g(g_), A(A_), v(v_), pr(pr_), scratch(scratch_), group(group_), s0(S.slice0), ns(S.nslices) {
        tid = threadIdx.x;
        wave = uniform_int(tid >> 6);
        lane = tid & 63;
        ng = (ns + kGroupSlices - 1) / kGroupSlices;
    }

    // sums of the slices' values in scratch[slot * nslices + slice], in the streaming kernels' order
    __device__ __forceinline__ double total(int slot, bool wave_order) {
        double* part = scratch + size_t(slot) * g.nslices + s0;
        __syncthreads();
        for (int q = tid; q < ng; q += NW * 64) {
            double t = 0.0;
            for (int w = 0; w < kGroupSlices; ++w) t += 16 * q + w < ns ? part[16 * q + w] : 0.0;
            group[q] = t;
        }
        __syncthreads();
        double a = 0.0;
        for (int q0 = 0; q0 < ng; q0 += 64) {
            const double t = q0 + lane < ng ? group[q0 + lane] : 0.0;
            if (wave_order) a += t;
            else a += wave_sum(t);
        }
        const double out = wave_order ? wave_sum(a) : a;
        __syncthreads();
        return out;
    }
    __device__ __forceinline__ void put(int slot, int s, double val) {
        val = wave_sum(val);
        if (lane == 0) scratch[size_t(slot) * g.nslices + s] = val;
    }
    // true residual of every row; r, z = p = M^-1 r unless it is only reported
    __device__ __forceinline__ void residual(bool report, bool from_r) {
        for (int q = wave; q < ns; q += NW) {
            const int s = s0 + q, row = s * 64 + lane;
            const SliceDesc sd = g.slices[s];
            double a = 0.0, b = 0.0, c = 0.0;
            if (lane < sd.nvalid) {
                F3 rf, bf;
                if (from_r) {
                    rf = ld3(v.r, row);
                    bf = ld3(v.rhs, row);
                    a = fma3d(0.0, rf.x, rf.y, rf.z, rf.x, rf.y, rf.z);
                } else {
                    double r[3];
                    bf = true_residual<false>(A, v, s, lane, sd.nlower, r);
                    rf = f3(float(r[0]), float(r[1]), float(r[2]));
                    a = fma3d(0.0, r[0], r[1], r[2], r[0], r[1], r[2]);
                }
                b = fma3d(0.0, bf.x, bf.y, bf.z, bf.x, bf.y, bf.z);
                if (!report) {
                    const F3 zf = minv_mul(A, s, lane, rf);
                    st3(v.r, row, rf);
                    st3(v.z, row, zf);
                    st3(v.p0, row, zf);
                    c = fma3d(0.0, rf.x, rf.y, rf.z, zf.x, zf.y, zf.z);
                }
            }
            put(0, s, a);
            put(1, s, b);
            put(2, s, c);
        }
    }
    // Iterations until a check is due or the solve stops.  p0 holds the
    // direction (p = z at a start).
    __device__ __forceinline__ void iterate(InstState& S) {
        float* p = v.p0;
        while (S.status == kRunning && S.mode == kModeIter) {
            const float beta = float(S.beta);
            // the owed term of a deferred update needs the direction it belongs to
            for (int q = wave; q < ns; q += NW) {
                const int row = (s0 + q) * 64 + lane;
                if (lane < g.slices[s0 + q].nvalid) {
                    const F3 old = ld3(p, row);
                    st3(v.p1, row, old);
                    st3(p, row, dir3(ld3(v.z, row), old, beta));
                }
            }
            __syncthreads();
            for (int q = wave; q < ns; q += NW) {
                const int s = s0 + q, row = s * 64 + lane;
                double a = 0.0;
                if (lane < g.slices[s].nvalid) {
                    const int sb = A.slice_ptr[s], w = A.slice_ptr[s + 1] - sb;
                    float d[9];
                    load_diag(A, s, lane, d);
                    const F3 pi = ld3(p, row);
                    F3 y = f3(fma3(0.0f, d[0], d[1], d[2], pi), fma3(0.0f, d[3], d[4], d[5], pi),
                              fma3(0.0f, d[6], d[7], d[8], pi));
                    for (int k = 0; k < w; ++k) {
                        const int kk = A.sym ? sym_order(k, w) : k;
                        const size_t en = size_t(sb + kk) * 64 + lane;
                        const int c = A.col[en];
                        if (c < 0) continue;
                        load_block(A, A.val + size_t(sb + kk) * A.bs * 64 + lane, A.mir + en, c, row, d);
                        const F3 pj = ld3(p, c);
                        y = f3(fma3(y.x, d[0], d[1], d[2], pj), fma3(y.y, d[3], d[4], d[5], pj),
                               fma3(y.z, d[6], d[7], d[8], pj));
                    }
                    st3(v.ap, row, y);
                    a = fma3d(0.0, double(pi.x), double(pi.y), double(pi.z), y.x, y.y, y.z);
                }
                put(0, s, a);
            }
            const double sig = total(0, false);
            const double alpha = (sig > kGuard || sig < -kGuard) ? S.rho / sig : 0.0;
            for (int q = wave; q < ns; q += NW) {
                const int s = s0 + q, row = s * 64 + lane;
                double a = 0.0, b = 0.0;
                if (lane < g.slices[s].nvalid) {
                    const F3 pi = ld3(p, row), pp = ld3(v.p1, row);
                    double* x = v.x + 3 * row;
                    if (S.pend) {
                        x[0] = x_two(x[0], S.alpha_pend, pp.x, alpha, pi.x);
                        x[1] = x_two(x[1], S.alpha_pend, pp.y, alpha, pi.y);
                        x[2] = x_two(x[2], S.alpha_pend, pp.z, alpha, pi.z);
                    } else if (!S.defer) {
                        x[0] = fma(alpha, double(pi.x), x[0]);
                        x[1] = fma(alpha, double(pi.y), x[1]);
                        x[2] = fma(alpha, double(pi.z), x[2]);
                    }
                    const float* mv = A.minv + (size_t)s * 6 * 64 + lane;
                    const float mi[6] = {mv[0], mv[64], mv[128], mv[192], mv[256], mv[320]};
                    const F3 r = r_update(ld3(v.r, row), ld3(v.ap, row), float(alpha));
                    const F3 z = z_update(mi, r);
                    st3(v.r, row, r);
                    st3(v.z, row, z);
                    a = dot3d(r, z);
                    b = dot3d(r, r);
                }
                put(0, s, a);
                put(1, s, b);
            }
            const double rz = total(0, false), rr = total(1, false);
            S.sigma = sig;
            S.alpha = alpha;
            pcg_advance(S, pr, AdvanceSums{rz, rr});
            if (S.status == kRunning && S.mode == kModeFlush) {
                for (int q = wave; q < ns; q += NW) {
                    const int row = (s0 + q) * 64 + lane;
                    if (lane < g.slices[s0 + q].nvalid) {
                        const F3 pi = ld3(p, row);
                        double* x = v.x + 3 * row;
                        x[0] = fma(S.alpha_pend, double(pi.x), x[0]);
                        x[1] = fma(S.alpha_pend, double(pi.y), x[1]);
                        x[2] = fma(S.alpha_pend, double(pi.z), x[2]);
                    }
                }
                __syncthreads();
                pcg_advance(S, pr, AdvanceSums{0.0, 0.0});
            }
        }
    }
};

// Every field in scalar registers: all threads hold the same state.
__device__ __forceinline__ void uniform_state(InstState& S) {
    S.rho = uniform_double(S.rho);
    S.bb = uniform_double(S.bb);
    S.rr = uniform_double(S.rr);
    S.beta = uniform_double(S.beta);
    S.relres = uniform_double(S.relres);
    S.alpha = uniform_double(S.alpha);
    S.alpha_pend = uniform_double(S.alpha_pend);
    S.status = uniform_int(S.status);
    S.mode = uniform_int(S.mode);
    S.iters = uniform_int(S.iters);
    S.restarts = uniform_int(S.restarts);
    S.parity = uniform_int(S.parity);
    S.pend = uniform_int(S.pend);
    S.defer = uniform_int(S.defer);
}

// The outcome of a solve; what was set at build time stays.
__device__ __forceinline__ void store_state(const InstState& S, InstState& mem, InstState& host) {
    for (InstState* q : {&mem, &host}) {
        q->rho = S.rho;
        q->bb = S.bb;
        q->rr = S.rr;
        q->beta = S.beta;
        q->relres = S.relres;
        q->status = S.status;
        q->mode = S.mode;
        q->iters = S.iters;
        q->restarts = S.restarts;
        q->parity = S.parity;
        q->alpha_pend = S.alpha_pend;
        q->pend = S.pend;
        q->defer = S.defer;
        q->owed = 0;
    }
}

}  // namespace

}  // namespace chysx_amd
