// SPDX-License-Identifier: Apache-2.0
//
// The PCG solve of one instance in one launch.
//
// One lane owns one row for the whole solve: its blocks, its Jacobi inverse,
// r, z, p and the FP64 iterate stay in registers, and the directions that its
// neighbours gather stay in LDS.  Nothing of the matrix is read again between
// iterations.  What an iteration has to send through memory is z of the rows
// that other workgroups gather (24 bytes a row) and one partial sum per
// workgroup and inner product; both travel as 8-byte words that carry a tag
// beside their payload, so a reader knows a word has arrived from the word
// itself and no fence (a write-back of an XCD's whole L2) is needed.  An iteration is bound by the
// two dependent sums over the instance's workgroups, not by bandwidth.
//
// Measured on MI355X, a step of 50 iterations (the streaming kernels before):
// 21 x 21 drape 182 us (850), 64 x 64 294 us (953), 300 x 300 drape 615 us
// (1494); a 256 x 256 cloth converged in 97 iterations 595 us (1876); 512
// uneven cloths to convergence 12.4 ms (37.1).
//
// Sums, updates and the scalar step are those of the streaming kernels in the
// same order, so the results are the same bits.

#include <hip/hip_runtime.h>

#include <stdexcept>

#include "pcg_exchange.hpp"

namespace chysx_amd {

[[noreturn]] void throw_hip(hipError_t err, const char* what);

namespace {

constexpr int kMaxGroups = 256;

// Scratch of the sums.  wave: each wave's sums, in one set per kind of sum (a
// set is written again only after another sum's barrier); group: the group
// sums of a many-workgroup instance.
template <int NW>
struct SumShared {
    double wave[3][3][kGroupSlices];
    double top[3][3][kGroupSlices];
    double group[3 * (NW == 16 ? kMaxGroups : kResidentPieces * kMaxGroups / 2 + 128)];
    int failed;
};

// Sums v[0 .. N) over the instance's rows; every thread gets the totals.  The
// order is the streaming kernels': the lanes of a wave by a butterfly, the 16
// waves of a group in order, then the groups, either as a 1024-thread workgroup
// adds them (group t in thread t, butterfly, the waves in order) or, with
// wave_order, as one wavefront does (lane l adds groups l, l + 64, ..., butterfly).
// `meanwhile` runs between this workgroup's contribution and the wait for the
// others'.  SET: the kind's set of LDS scratch.
template <int NW, int N, int SET, class F>
__device__ __forceinline__ bool cluster_sum(const Cluster& C, SumShared<NW>& sh, double (&v)[N], int kind,
                                            unsigned tag, bool wave_order, double (&out)[N], F&& meanwhile) {
    const int tid = fresh(threadIdx.x), wave = tid >> 6, lane = tid & 63;
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] = wave_sum(v[j]);
    if (lane == 0) {
#pragma unroll
        for (int j = 0; j < N; ++j) sh.wave[SET][j][wave] = v[j];
    }
    __syncthreads();
    // the group's waves in order (absent ones add zero), 8 loads in flight
    auto in_order = [&](int j) {
        double t = 0.0;
#pragma unroll
        for (int w0 = 0; w0 < NW; w0 += 8) {
            if (w0 < C.waves) {
                double q[8];
#pragma unroll
                for (int w = 0; w < 8; ++w) q[w] = sh.wave[SET][j][w0 + w];
#pragma unroll
                for (int w = 0; w < 8; ++w) t += q[w];
            }
        }
        return t;
    };
    if (C.size == 1) {
#pragma unroll
        for (int j = 0; j < N; ++j) out[j] = uniform_double(in_order(j));
        meanwhile();
        return true;
    }
    if (NW == 16 || C.piece == 0) {
        const int j = tid / kResidentCopies;
        if (j < N)
            slot_store(C, slot_of(C, kind + j, 0, tid & (kResidentCopies - 1), C.group), tag, in_order(j));
    } else {
        const int w = tid / kResidentCopies, j = w >> 3;
        if (j < N)
            slot_store(C, slot_of(C, kind + j, 1 + (w & 7), tid & (kResidentCopies - 1), C.group), tag,
                       sh.wave[SET][j][w & 7]);
    }
    int failed = 0;
    pause(N == 1 ? C.pause : C.pause_z);
    if constexpr (NW == 16) {
        meanwhile();
        double t[N];
#pragma unroll
        for (int j = 0; j < N; ++j) t[j] = 0.0;
        if (tid < C.ngroups) {
#pragma unroll
            for (int j = 0; j < N; ++j) t[j] += slot_wait(C, slot_of(C, kind + j, 0, C.copy, tid), tag, failed);
        }
        if (wave_order) {
            if (tid < C.ngroups) {
#pragma unroll
                for (int j = 0; j < N; ++j) sh.group[j * kMaxGroups + tid] = t[j];
            }
        } else if (wave < kMaxGroups / 64) {
#pragma unroll
            for (int j = 0; j < N; ++j) t[j] = wave_sum(t[j]);
            if (lane == 0) {
#pragma unroll
                for (int j = 0; j < N; ++j) sh.top[SET][j][wave] = t[j];
            }
        }
        if (failed) sh.failed = 1;
        __syncthreads();
        if (wave_order) {
#pragma unroll
            for (int j = 0; j < N; ++j) {
                double a = 0.0;
#pragma nounroll
                for (int q = lane; q < C.ngroups; q += 64) a += sh.group[j * kMaxGroups + q];
                out[j] = wave_sum(a);
            }
        } else {
#pragma unroll
            for (int j = 0; j < N; ++j) {
                double a = 0.0;
#pragma unroll
                for (int w = 0; w < kMaxGroups / 64; ++w) a += sh.top[SET][j][w];
                out[j] = a;
            }
        }
    } else {
        // few workgroups: the sums come soon after z.  100 iterations of a
        // drape, sums first and z first: 20 workgroups 727 and 765 us, 64: 873
        // and 882, 104: 906 and 929, 130: 979 and 966, 176: 1055 and 1024, 256:
        // 1160 and 1066
        const bool z_first = C.size >= 120;
        if (z_first) meanwhile();
        // A group's first half is one value, its second half's waves are 8:
        // a few values a thread, all loaded before any is looked at.
        const int per = kResidentPieces * C.ngroups;
        constexpr int kBatch = N == 1 ? 3 : 5;
#pragma nounroll
        for (int q0 = tid; q0 < N * per; q0 += kBatch * NW * 64) {
            const u64* w[kBatch];
            bool there[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                const int q = q0 + u * NW * 64, j = q / per, pg = q - j * per, p = pg / C.ngroups, g = pg - p * C.ngroups;
                there[u] = q < N * per && (p == 0 || C.nslices > 16 * g + 8 + (p - 1));
                w[u] = there[u] ? slot_of(C, kind + j, p, C.copy, g) : slot_of(C, kind, 0, C.copy, 0);
            }
            u64 a[kBatch], b[kBatch];
            int n = 0;
            bool late;
#pragma nounroll
            do {
                late = false;
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    a[u] = agent_load(w[u]);
                    b[u] = agent_load(w[u] + C.total);
                }
#pragma unroll
                for (int u = 0; u < kBatch; ++u)
                    late = late || unsigned(a[u] >> 32) != tag || unsigned(b[u] >> 32) != tag;
            } while (late && ++n < kExchangePolls);
            if (late) failed = 1;
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                const int q = q0 + u * NW * 64;
                if (q < N * per)
                    sh.group[q] = there[u] ? __hiloint2double(int(unsigned(b[u])), int(unsigned(a[u]))) : 0.0;
            }
        }
        if (!z_first) meanwhile();
        if (failed) sh.failed = 1;
        __syncthreads();
        // wave (2 j + c) sums value j of the groups 64 c .. 64 c + 63
        if (wave < 2 * N) {
            const int j = wave >> 1, g = (wave & 1) * 64 + lane;
            double t = 0.0;
            if (g < C.ngroups) {
                double q[kResidentPieces];
#pragma unroll
                for (int p = 0; p < kResidentPieces; ++p) q[p] = sh.group[j * per + p * C.ngroups + g];
#pragma unroll
                for (int p = 0; p < kResidentPieces; ++p) t += q[p];
            }
            if (wave_order) sh.group[3 * kResidentPieces * (kMaxGroups / 2) + wave * 64 + lane] = t;
            else t = wave_sum(t);
            if (lane == 0) sh.top[SET][j][wave & 1] = t;
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < N; ++j) {
            if (wave_order) {
                const double* q = sh.group + 3 * kResidentPieces * (kMaxGroups / 2) + j * 128 + lane;
                out[j] = wave_sum((0.0 + q[0]) + q[64]);
            } else {
                out[j] = (0.0 + sh.top[SET][j][0]) + sh.top[SET][j][1];
            }
        }
        // the next sum writes sh.group again only after its own barrier
    }
#pragma unroll
    for (int j = 0; j < N; ++j) out[j] = uniform_double(out[j]);
    return uniform_int(sh.failed) == 0;
}

// Blocks of one row in the order the streaming kernel adds them, and where
// their columns' vectors lie in LDS.
template <bool PK, int MAXW>
struct Blocks {
    float m[MAXW][PK ? 6 : 9];
    unsigned at[(MAXW + 1) / 2];  // two 16-bit byte offsets each
};

template <bool PK, int MAXW>
__device__ __forceinline__ void load_blocks(const DevMatrix& A, const uint16_t* __restrict__ loc, int row, int sb,
                                            int w, unsigned zero, Blocks<PK, MAXW>& B) {
    const int lane = row & 63;
#pragma unroll
    for (int k = 0; k < (MAXW + 1) / 2; ++k) B.at[k] = zero * 0x10001u;
#pragma unroll
    for (int k = 0; k < MAXW; ++k) {
#pragma unroll
        for (int q = 0; q < (PK ? 6 : 9); ++q) B.m[k][q] = 0.0f;
        if (k < w) {  // wave-uniform
            const int kk = (PK || A.sym) ? sym_order(k, w) : k;
            const size_t e = size_t(sb + kk) * 64 + lane;
            const int c = A.col[e];
            if (c >= 0) {
                if (PK) {
                    const float* b = A.val + (c < row ? val_offset(A.mir[e], 6) : size_t(sb + kk) * 6 * 64 + lane);
#pragma unroll
                    for (int q = 0; q < 6; ++q) B.m[k][q] = b[q * 64];
                } else {
                    float m[9];
                    load_block(A, A.val + size_t(sb + kk) * 9 * 64 + lane, A.mir + e, c, row, m);
#pragma unroll
                    for (int q = 0; q < 9; ++q) B.m[k][PK ? 0 : q] = m[q];
                }
            }
            B.at[k >> 1] = (k & 1) ? (B.at[k >> 1] & 0xFFFFu) | (unsigned(loc[e]) << 16)
                                   : (B.at[k >> 1] & 0xFFFF0000u) | unsigned(loc[e]);
        }
        // one entry's loads at a time: issued together, those of every entry
        // would need more registers than the blocks themselves
        __builtin_amdgcn_sched_barrier(0);
    }
}

template <int NW>
__device__ __forceinline__ void solve_alone(const ResidentView& R, const LaunchGeom& g, const DevMatrix& A,
                                            const DevVectors& v, const DevExt& e, const DevMesh& m,
                                            const InstParams& pr, InstState& S, float dt, int given_r,
                                            SumShared<NW>& sh) {
    Alone<NW> a(g, A, v, pr, S, R.solo, sh.group);
    a.residual(false, given_r != 0);
    {
        const double rr = a.total(0, true), bb = a.total(1, true), rz = a.total(2, true);
        pcg_begin(S, pr, rr, bb, rz);
    }
    while (S.status == kRunning) {
        a.iterate(S);
        if (S.status != kRunning) break;
        a.residual(false, false);
        const double rr = a.total(0, false), rz = a.total(2, false);
        pcg_advance(S, pr, AdvanceSums{rz, rr});
    }
    if (S.status == kStopped) {
        a.residual(true, false);
        S.rr = a.total(0, true);
        S.relres = sqrt(S.rr / S.bb);
    }
    for (int q = a.wave; q < a.ns; q += NW) {
        const SliceDesc sd = g.slices[a.s0 + q];
        const int row = (a.s0 + q) * 64 + a.lane;
        if (a.lane < sd.nvalid)
            finalize_row(e, pr, dt, m.pin_inc_off, m.pin_inc, m.pin_tgt, row, sd.part0 + a.lane, v.x[3 * row],
                         v.x[3 * row + 1], v.x[3 * row + 2]);
    }
}

template <bool PK, int MAXW, int NW>
__global__ __launch_bounds__(64 * NW) void pcg_resident_kernel(ResidentView R, LaunchGeom g, DevMatrix A,
                                                               DevVectors v, DevExt e, DevMesh m,
                                                               InstState* __restrict__ st,
                                                               InstState* __restrict__ host_st,
                                                               const InstParams* __restrict__ params, float dt,
                                                               int given_r) {
    extern __shared__ __align__(16) float lds[];
    __shared__ SumShared<NW> sh;
    __shared__ int shared_int[2];
    const int tid = threadIdx.x, wave = uniform_int(tid >> 6), lane = tid & 63;
    const int threads = int(blockDim.x);
    int wgi = blockIdx.x;
    if (R.ticket != nullptr) {  // places in the order of starting (plan_resident says when)
        if (tid == 0)
            shared_int[0] = int(__hip_atomic_fetch_add(R.ticket, u64(1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) %
                                u64(R.nwg));
        __syncthreads();
        wgi = __builtin_amdgcn_readfirstlane(shared_int[0]);
    }
    const ResidentWg W = R.wgs[wgi];
    const InstParams& pr = params[W.inst];
    InstState& mem = st[W.inst];
    // absent waves add nothing
    for (int q = tid; q < 3 * 3 * kGroupSlices; q += threads) (&sh.wave[0][0][0])[q] = 0.0;
    if (tid == 0) sh.failed = 0;
    Cluster C;
    C.size = W.cluster;
    C.nslices = mem.nslices;
    C.ngroups = (C.nslices + kGroupSlices - 1) / kGroupSlices;
    C.group0 = mem.group0;
    C.total = g.ngroups;
    C.group = W.group;
    C.piece = W.piece;
    C.waves = W.nslices;
    C.copy = (wgi - W.first) & (kResidentCopies - 1);
    C.slots = R.slots;
    C.pause = W.pause;
    C.pause_z = W.pause_z;
    unsigned tag = 0;
    if (W.cluster > 1) {
        tag = R.sync[W.inst].epoch;
        if (tid == 0) shared_int[1] = meet(R.sync + W.inst, W.cluster, R.meet_polls, R.solo != nullptr);
    } else if (tid == 0) {
        shared_int[1] = kMeetRun;
    }
    __syncthreads();
    const int met = __builtin_amdgcn_readfirstlane(shared_int[1]);
    if (met == kMeetLeave) return;
    if (met == kMeetAlone) {
        InstState S = mem;
        solve_alone<NW>(R, g, A, v, e, m, pr, S, dt, given_r, sh);
        if (tid == 0) store_state(S, mem, host_st[W.inst]);
        return;
    }
    InstState S{};  // the fields that the solve works with
    S.parity = mem.parity;

    const int s = __builtin_amdgcn_readfirstlane(W.slice0 + wave);
    const bool live = wave < W.nslices;
    SliceDesc sd{};
    if (live) sd = g.slices[s];
    const bool valid = lane < sd.nvalid;
    const int row = s * 64 + lane;
    const int own = W.nslices * 64;  // LDS rows: own, halo, zero
    float* mine = lds + 3 * (wave * 64 + lane);
    float* zin = lds + 3 * R.lds_rows;  // z of the halo rows as received
    if (tid < 3) lds[3 * (own + W.nhalo) + tid] = 0.0f;
    const bool sends = valid && R.exported[row] != 0;
    auto nothing = [] {};
    // z of a row in two words, x with half of y and z with the other half, each
    // with the low 16 bits of the tag: a row's words are written once for every
    // tag that sends, so an old word never has the tag waited for.
    auto send_z = [&](F3 z, unsigned t) {
        if (sends) {
            u64* w = R.zx + fresh(row);
            const unsigned y = __float_as_uint(z.y);
            agent_store(w, tagged((t << 16) | (y & 0xFFFFu), __float_as_uint(z.x)));
            agent_store(w + R.rows, tagged((t << 16) | (y >> 16), __float_as_uint(z.z)));
        }
    };
    // The halo rows' z with tag t, into zin.  The last threads start, since
    // the first ones wait for the sums.
    auto receive_z = [&](unsigned t) {
#pragma nounroll
        for (int h = threads - 1 - fresh(tid); h < W.nhalo; h += threads) {
            const u64* w = R.zx + R.halo[W.halo0 + h];
            u64 a, b;
            int n = 0;
#pragma nounroll
            do {
                a = agent_load(w);
                b = agent_load(w + R.rows);
            } while ((((unsigned(a >> 32) ^ (t << 16)) | (unsigned(b >> 32) ^ (t << 16))) > 0xFFFFu) &&
                     ++n < kExchangePolls);
            if (n >= kExchangePolls) sh.failed = 1;
            zin[3 * h] = __uint_as_float(unsigned(a));
            zin[3 * h + 1] = __uint_as_float((unsigned(a >> 32) & 0xFFFFu) | (unsigned(b >> 32) << 16));
            zin[3 * h + 2] = __uint_as_float(unsigned(b));
        }
    };

    // The iterate and the direction that an owed term belongs to are touched
    // every other iteration: they lie in LDS, where they cost no registers.
    double* xl = reinterpret_cast<double*>(lds + R.lds_x) + 3 * tid;
    float* pl = lds + R.lds_x + 6 * threads + 3 * tid;
    F3 r = f3(0.0f, 0.0f, 0.0f), z = r, p = r;
    if (valid) {
        xl[0] = v.x[3 * row];
        xl[1] = v.x[3 * row + 1];
        xl[2] = v.x[3 * row + 2];
    }
    // The iterate goes to memory, for the residual's gathers and the next
    // step's guess.  Every wave's stores have arrived before its workgroup
    // contributes to the sum that all wait for.
    auto publish_x = [&] {
        if (valid) {
            double* xo = v.x + 3 * fresh(row);
#pragma unroll
            for (int c = 0; c < 3; ++c) __hip_atomic_store(xo + c, xl[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_waitcnt(0);
        double none[1] = {0.0}, got[1];
        ++tag;
        return cluster_sum<NW, 1, 0>(C, sh, none, kKindSigma, tag, false, got, nothing);
    };
    // Each round begins with a true residual: the start's, the check of a
    // solve whose recursive residual has passed the test, or the report of a
    // stopped one.
    enum Phase : int { kBegin, kCheck, kReport };
    int phase = kBegin;
    bool met_all = true;  // no wait ran out (left as a flag: a return from here would make the loops' exits divergent)
    for (;;) {
        {
            double part[3] = {0.0, 0.0, 0.0}, sum[3];
            if (valid) {
                const int ln = fresh(lane);
                if (phase == kBegin && given_r) {  // pcg_start_given_r_kernel
                    r = ld3(v.r, s * 64 + ln);
                    const F3 bf = ld3(v.rhs, s * 64 + ln);
                    part[0] = fma3d(0.0, r.x, r.y, r.z, r.x, r.y, r.z);
                    part[1] = fma3d(0.0, bf.x, bf.y, bf.z, bf.x, bf.y, bf.z);
                } else {
                    double rd[3];
                    const F3 bf = true_residual<true>(A, v, s, ln, sd.nlower, rd);
                    r = f3(float(rd[0]), float(rd[1]), float(rd[2]));
                    part[0] = fma3d(0.0, rd[0], rd[1], rd[2], rd[0], rd[1], rd[2]);
                    part[1] = fma3d(0.0, bf.x, bf.y, bf.z, bf.x, bf.y, bf.z);
                }
                z = minv_mul(A, s, ln, r);
                part[2] = fma3d(0.0, r.x, r.y, r.z, z.x, z.y, z.z);
            }
            ++tag;
            send_z(z, tag);
            met_all = cluster_sum<NW, 3, 2>(C, sh, part, kKindTrue, tag, phase != kCheck, sum, [&] { receive_z(tag); });
            if (!met_all) break;
            if (phase == kBegin) {
                pcg_begin(S, pr, sum[0], sum[1], sum[2]);
            } else if (phase == kCheck) {
                pcg_advance(S, pr, AdvanceSums{sum[2], sum[0]});
            } else {
                S.rr = sum[0];
                S.relres = sqrt(sum[0] / S.bb);
            }
            uniform_state(S);
            if (phase == kReport || S.status == kConverged) break;
            if (S.status == kStopped) {  // no iterations left after a failed check
                met_all = publish_x();
                if (!met_all) break;
                phase = kReport;
                continue;
            }
        }
        // Everything is set on every path, so that none of it stays live
        // through the next round's residual.
        Blocks<PK, MAXW> B;
        float dg[PK ? 6 : 9], mi[6];
#pragma unroll
        for (int q = 0; q < (PK ? 6 : 9); ++q) dg[q] = 0.0f;
#pragma unroll
        for (int q = 0; q < 6; ++q) mi[q] = 0.0f;
        const int sb = live ? A.slice_ptr[s] : 0;
        const int w = live ? A.slice_ptr[s + 1] - sb : 0;
        load_blocks<PK, MAXW>(A, R.loc, fresh(row), sb, w, 12u * unsigned(own + W.nhalo), B);
        if (live) {
            const float* dp = A.diag + (size_t)s * (PK ? 6 : 9) * 64 + fresh(lane);
#pragma unroll
            for (int q = 0; q < (PK ? 6 : 9); ++q) dg[q] = dp[q * 64];
            const float* mv = A.minv + (size_t)s * 6 * 64 + fresh(lane);
#pragma unroll
            for (int q = 0; q < 6; ++q) mi[q] = mv[q * 64];
        }
        // Where the iterations' code begins, modulo 32 bytes, is worth up to 3%:
        // 200 iterations of 10 x 10, 32 x 32 and 128 small cloths took 301 to
        // 314, 627 to 643 and 650 to 666 us at the 8 places; here 304, 627, 650.
        asm volatile(".p2align 6\n\ts_nop 0");
        bool first = true;  // a (re)start: p_prev = z, beta = 0
        while (S.status == kRunning && S.mode == kModeIter) {
            const float beta = float(S.beta);
            if (valid) {
                p = dir3(z, first ? z : p, beta);
                mine[0] = p.x;
                mine[1] = p.y;
                mine[2] = p.z;
            }
#pragma nounroll
            for (int h = threads - 1 - fresh(tid); h < W.nhalo; h += threads) {
                float* ph = lds + 3 * (own + h);
                const F3 zh = ld3(zin, h);
                const F3 d = dir3(zh, first ? zh : f3(ph[0], ph[1], ph[2]), beta);
                ph[0] = d.x;
                ph[1] = d.y;
                ph[2] = d.z;
            }
            first = false;
            __syncthreads();
            F3 ap = f3(0.0f, 0.0f, 0.0f);
            double sg[1] = {0.0}, sig[1];
            if (valid) {
                if (PK) {
                    ap.x = fma3(0.0f, dg[0], dg[1], dg[2], p);
                    ap.y = fma3(0.0f, dg[1], dg[3], dg[4], p);
                    ap.z = fma3(0.0f, dg[2], dg[4], dg[5], p);
                } else {
                    ap.x = fma3(0.0f, dg[0], dg[1], dg[2], p);
                    ap.y = fma3(0.0f, dg[3], dg[4], dg[5], p);
                    ap.z = fma3(0.0f, dg[PK ? 0 : 6], dg[PK ? 0 : 7], dg[PK ? 0 : 8], p);
                }
                // entries past the slice's width are zero blocks on the zero
                // row: no branch parts the gathers
#pragma unroll
                for (int k = 0; k < MAXW; ++k) {
                    const unsigned at = unsigned(fresh(int(B.at[k >> 1])));
                    const float* q = reinterpret_cast<const float*>(reinterpret_cast<const char*>(lds) +
                                                                    ((k & 1) ? at >> 16 : at & 0xFFFFu));
                    const F3 pj = f3(q[0], q[1], q[2]);
                    const float* b = B.m[k];
                    if (PK) {
                        ap.x = fma3(ap.x, b[0], b[1], b[2], pj);
                        ap.y = fma3(ap.y, b[1], b[3], b[4], pj);
                        ap.z = fma3(ap.z, b[2], b[4], b[5], pj);
                    } else {
                        ap.x = fma3(ap.x, b[0], b[1], b[2], pj);
                        ap.y = fma3(ap.y, b[3], b[4], b[5], pj);
                        ap.z = fma3(ap.z, b[PK ? 0 : 6], b[PK ? 0 : 7], b[PK ? 0 : 8], pj);
                    }
                }
                sg[0] = fma3d(0.0, double(p.x), double(p.y), double(p.z), ap.x, ap.y, ap.z);
            }
            ++tag;
            met_all = cluster_sum<NW, 1, 0>(C, sh, sg, kKindSigma, tag, false, sig, nothing);
            if (!met_all) break;
            const double alpha = (sig[0] > kGuard || sig[0] < -kGuard) ? S.rho / sig[0] : 0.0;
            double part[2] = {0.0, 0.0}, sum[2];
            ++tag;
            if (valid) {
                r = r_update(r, ap, float(alpha));
                z = z_update(mi, r);
                send_z(z, tag);
                part[0] = dot3d(r, z);
                part[1] = dot3d(r, r);
                if (S.pend) {  // the owed term and this one
                    xl[0] = x_two(xl[0], S.alpha_pend, pl[0], alpha, p.x);
                    xl[1] = x_two(xl[1], S.alpha_pend, pl[1], alpha, p.y);
                    xl[2] = x_two(xl[2], S.alpha_pend, pl[2], alpha, p.z);
                } else if (S.defer) {
                    pl[0] = p.x;
                    pl[1] = p.y;
                    pl[2] = p.z;
                } else {
                    xl[0] = fma(alpha, double(p.x), xl[0]);
                    xl[1] = fma(alpha, double(p.y), xl[1]);
                    xl[2] = fma(alpha, double(p.z), xl[2]);
                }
            }
            met_all = cluster_sum<NW, 2, 1>(C, sh, part, kKindUpdate, tag, false, sum, [&] { receive_z(tag); });
            if (!met_all) break;
            S.alpha = alpha;
            pcg_advance(S, pr, AdvanceSums{sum[0], sum[1]});
        }
        if (met_all && S.status == kRunning && S.mode == kModeFlush) {
            if (valid) {
                xl[0] = fma(S.alpha_pend, double(p.x), xl[0]);
                xl[1] = fma(S.alpha_pend, double(p.y), xl[1]);
                xl[2] = fma(S.alpha_pend, double(p.z), xl[2]);
            }
            pcg_advance(S, pr, AdvanceSums{0.0, 0.0});
            uniform_state(S);
        }
        if (!met_all) break;
        met_all = publish_x();
        if (!met_all) break;
        phase = S.status == kStopped ? kReport : kCheck;
    }
    if (!met_all) {
        if (tid == 0) {
            mem.status = kResidentLost;
            host_st[W.inst].status = kResidentLost;
            lost_exchange(R.sync + W.inst);
        }
        return;
    }
    if (valid) {
        const int own_row = fresh(row);  // this lane's own words of v.x
        finalize_row(e, pr, dt, m.pin_inc_off, m.pin_inc, m.pin_tgt, own_row, sd.part0 + lane, v.x[3 * own_row],
                     v.x[3 * own_row + 1], v.x[3 * own_row + 2]);
    }
    if (wgi == W.first && tid == 0) {
        store_state(S, mem, host_st[W.inst]);
        if (W.cluster > 1) R.sync[W.inst].epoch = tag;
    }
}

}  // namespace

void launch_pcg_resident(const ResidentView& R, const LaunchGeom& g, const DevMatrix& A, const DevVectors& v,
                         const DevExt& e, const DevMesh& m, InstState* st, InstState* host_st,
                         const InstParams* params, float dt, int start_given_r, hipStream_t s) {
    if (R.nwg <= 0) return;
    if (g.ngroups * kGroupSlices != g.nslices) throw std::invalid_argument("resident solve: whole 16-slice groups");
    if ((R.variant == kResidentC) != (A.bs == 9) || (R.max_cluster > 1 && R.block_waves != R.waves))
        throw std::invalid_argument("resident solve: the plan was made for another storage");
    const int block = 64 * R.block_waves;
#define CHYSX_RESIDENT(PK, MAXW, NW)                                                                             \
    pcg_resident_kernel<PK, MAXW, NW><<<R.nwg, block, R.lds_bytes, s>>>(R, g, A, v, e, m, st, host_st, params, dt, \
                                                                        start_given_r)
    if (R.variant == kResidentA) CHYSX_RESIDENT(true, kResidentWidthA, 16);
    else if (R.variant == kResidentB) CHYSX_RESIDENT(true, kResidentWidthB, 8);
    else if (R.variant == kResidentC) CHYSX_RESIDENT(false, kResidentWidthC, 8);
    else throw std::invalid_argument("resident solve: no plan");
#undef CHYSX_RESIDENT
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) throw_hip(err, "pcg_resident_kernel");
}

}  // namespace chysx_amd
