// SPDX-License-Identifier: Apache-2.0
//
// The iterations of one large cloth in one launch.
//
// A workgroup a compute unit owns up to 64 slices, 8 rows a lane.  r, A p, the
// Jacobi inverse and the diagonal blocks stay in registers, the directions of
// its rows and of its neighbours' boundary rows in LDS, so an iteration reads
// only the off-diagonal blocks and their packed indices (92 bytes a row and 18
// more for mirrors that have left the L2), every other time the iterate, and z
// of the boundary rows (16 bytes for up to half of the rows, both ways): 157
// bytes a row counted at 1024 x 1024 against 270 of the streaming kernels,
// which also pay two more launches.  The sums and z travel as in the resident
// solve.
//
// At 1024 x 1024 an iteration takes 31 us against 53 us (about 75 K cycles: 31
// to 36 K in the products, 15 to 22 K for p . Ap with 5 to 12 K of it waiting
// for the slowest workgroup, 17 K for the update's sums with the iterate under
// them), and three steps solved to 1e-6 take 10.9 ms where they took 18.7 ms.  It
// moves 164 MB beyond the L2, 5.4 TB/s; with 8 waves a compute unit more loads
// in flight would need registers that the vectors hold.  Fewer, larger pieces
// (2 groups at 512 x 512 on half the units) lose to the resident solve, and
// rows wider than 6 entries, which would have to take a generic loop, make
// their workgroup the one that all others wait for.
//
// Workgroups sweep their slices in alternating directions, so that two
// neighbours pass their common boundary at the same time and the lower entries
// there find their mirrors in the L2.

#include <hip/hip_runtime.h>

#include <stdexcept>
#include <type_traits>

#include "pcg_exchange.hpp"
#include "pcg_sweep.hpp"

namespace chysx_amd {

[[noreturn]] void throw_hip(hipError_t err, const char* what);

namespace {

constexpr int kThreads = 64 * kSweepWaves;

__device__ __forceinline__ double pack2(unsigned lo, unsigned hi) { return __hiloint2double(int(hi), int(lo)); }

__device__ __forceinline__ int fresh_uniform(int x) {  // as fresh(), for a wave-uniform value
    x = __builtin_amdgcn_readfirstlane(x);
    asm volatile("" : "+s"(x));
    return x;
}

// Two values of which the lanes with `bit` clear keep a, the others b, each
// added over the pair of lanes that differ in it: the butterfly's stage for
// both at once.
__device__ __forceinline__ double fold32(double a, double b) {
    const auto l = __builtin_amdgcn_permlane32_swap(unsigned(__double2loint(a)), unsigned(__double2loint(b)), false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(unsigned(__double2hiint(a)), unsigned(__double2hiint(b)), false, false);
    return pack2(l[0], h[0]) + pack2(l[1], h[1]);
}
__device__ __forceinline__ double fold16(double a, double b) {
    const auto l = __builtin_amdgcn_permlane16_swap(unsigned(__double2loint(a)), unsigned(__double2loint(b)), false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(unsigned(__double2hiint(a)), unsigned(__double2hiint(b)), false, false);
    return pack2(l[0], h[0]) + pack2(l[1], h[1]);
}
__device__ __forceinline__ double fold8(double a, double b, bool bit) {
    const double keep = bit ? b : a, give = bit ? a : b;
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(give), 0x128, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(give), 0x128, 0xf, 0xf, false);
    return keep + __hiloint2double(hi, lo);
}
// a of the lane 4, 2 or 1 away by xor, added
template <int XOR>
__device__ __forceinline__ int from_xor(int a) {
    if (XOR == 4) {  // lanes 0-3 and 8-11 of a row of 16 read 4 up, the others 4 down
        const int t = __builtin_amdgcn_update_dpp(0, a, 0x104, 0xf, 0x5, false);
        return __builtin_amdgcn_update_dpp(t, a, 0x114, 0xf, 0xa, false);
    }
    return __builtin_amdgcn_update_dpp(0, a, XOR == 2 ? 0x4E : 0xB1, 0xf, 0xf, false);  // quad_perm
}
template <int XOR>
__device__ __forceinline__ double add_xor(double a) {
    return a + __hiloint2double(from_xor<XOR>(__double2hiint(a)), from_xor<XOR>(__double2loint(a)));
}
// The sums over the 64 lanes of 8 values, value l >> 3 in lane l: the same
// additions as 8 butterflies, with a fifth of the instructions.
__device__ __forceinline__ double wave_sum8(const double (&v)[8], int lane) {
    double q[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = fold32(v[i], v[i + 4]);
    const double p0 = fold16(q[0], q[2]), p1 = fold16(q[1], q[3]);
    return add_xor<1>(add_xor<2>(add_xor<4>(fold8(p0, p1, (lane & 8) != 0))));
}

struct SweepShared {
    double slice[2][64];
    double top[2][16];
    int failed;
    int met;
};

// Sums of the rows' values v[j][i] (slice 8 i + wave of the workgroup) over
// the instance, in the streaming kernels' order; every thread gets them.
template <int GROUPS, int N, class F>
__device__ __forceinline__ bool sweep_sum(const SweepView& R, const SweepWg& W, SweepShared& sh,
                                          const double (&v)[N][8], int kind, unsigned tag, double (&out)[N],
                                          F&& meanwhile) {
    const int tid = fresh(threadIdx.x), wave = tid >> 6, lane = tid & 63;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const double t = wave_sum8(v[j], lane);
        if ((lane & 7) == 0) sh.slice[j][wave + lane] = t;  // slice wave + 8 (lane >> 3)
    }
    __syncthreads();
    auto slot = [&](int j, int copy, int group) {
        return R.slots + (size_t(kind + j) * kResidentCopies + copy) * 2 * R.ngroups + group;
    };
    {
        const int q = tid / kResidentCopies, j = q / GROUPS, i = q - j * GROUPS;
        if (j < N && W.group + i < R.ngroups) {
            double t = 0.0;
#pragma unroll
            for (int w0 = 0; w0 < kGroupSlices; w0 += 8) {
                double x[8];
#pragma unroll
                for (int w = 0; w < 8; ++w) x[w] = sh.slice[j][i * kGroupSlices + w0 + w];
#pragma unroll
                for (int w = 0; w < 8; ++w) t += x[w];
            }
            u64* w = const_cast<u64*>(slot(j, tid & (kResidentCopies - 1), W.group + i));
            agent_store(w, tagged(tag, unsigned(__double2loint(t))));
            agent_store(w + R.ngroups, tagged(tag, unsigned(__double2hiint(t))));
        }
    }
    if (N == 1) pause(R.pause);
    meanwhile();
    const int copy = int(blockIdx.x) & (kResidentCopies - 1);
    double t[N][2];
    {
        const bool two = tid + kThreads < R.ngroups;
        u64 a[N][2], b[N][2];
        bool late;
        int n = 0;
#pragma nounroll
        do {
            late = false;
            if (tid < R.ngroups) {
#pragma unroll
                for (int j = 0; j < N; ++j)
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const u64* w = slot(j, copy, u == 0 || two ? tid + u * kThreads : tid);
                        a[j][u] = agent_load(w);
                        b[j][u] = agent_load(w + R.ngroups);
                    }
#pragma unroll
                for (int j = 0; j < N; ++j)
#pragma unroll
                    for (int u = 0; u < 2; ++u)
                        late = late || unsigned(a[j][u] >> 32) != tag || unsigned(b[j][u] >> 32) != tag;
                if (late) __builtin_amdgcn_s_sleep(1);
            }
        } while (late && ++n < kExchangePolls);
        if (late) sh.failed = 1;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            t[j][0] = tid < R.ngroups ? 0.0 + pack2(unsigned(a[j][0]), unsigned(b[j][0])) : 0.0;
            t[j][1] = two ? 0.0 + pack2(unsigned(a[j][1]), unsigned(b[j][1])) : 0.0;
        }
    }
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            t[j][u] = wave_sum(t[j][u]);
            if (lane == 0) sh.top[j][wave + 8 * u] = t[j][u];
        }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < N; ++j) {
        double s = 0.0;
#pragma unroll
        for (int w0 = 0; w0 < 16; w0 += 8) {
            double x[8];
#pragma unroll
            for (int w = 0; w < 8; ++w) x[w] = sh.top[j][w0 + w];
#pragma unroll
            for (int w = 0; w < 8; ++w) s += x[w];
        }
        out[j] = uniform_double(s);
    }
    return uniform_int(sh.failed) == 0;
}

template <int GROUPS>
__global__ __launch_bounds__(kThreads) void pcg_sweep_kernel(SweepView R, LaunchGeom g, DevMatrix A, DevVectors v,
                                                             InstState* __restrict__ st,
                                                             const InstParams* __restrict__ params) {
    constexpr int RPL = 2 * GROUPS;  // rows a lane
    extern __shared__ __align__(16) float lds[];
    __shared__ SweepShared sh;
    const int tid = threadIdx.x, wave = uniform_int(tid >> 6), lane = tid & 63;
    // each XCD (workgroups go to them in turn) takes a contiguous eighth
    const int per = (R.nwg + 7) >> 3, wg = int(blockIdx.x & 7) * per + int(blockIdx.x >> 3);
    if (wg >= R.nwg) return;
    const SweepWg W = R.wgs[wg];
    InstState& mem = st[0];
    const InstParams& pr = params[0];
    unsigned tag = R.sync->epoch;
    if (tid == 0) {
        sh.failed = 0;
        sh.met = meet(R.sync, R.nwg, R.meet_polls, R.solo != nullptr);
    }
    __syncthreads();
    const int met = uniform_int(sh.met);
    if (met == kMeetLeave) return;
    // nobody writes the state before all have met, so all read the same
    if (mem.status != kRunning || mem.mode != kModeIter) return;
    InstState S{};
    S.status = kRunning;
    S.mode = kModeIter;
    S.rho = mem.rho;
    S.bb = mem.bb;
    S.rr = mem.rr;
    S.beta = mem.beta;
    S.iters = mem.iters;
    S.parity = mem.parity;
    S.defer = mem.defer;
    auto leave = [&](bool ok) {
        if (tid != 0) return;
        mem.rho = S.rho;
        mem.rr = S.rr;
        mem.beta = S.beta;
        mem.status = S.status;
        mem.mode = S.mode;
        mem.iters = S.iters;
        mem.parity = S.parity;
        mem.alpha_pend = S.alpha_pend;
        mem.pend = S.pend;
        mem.defer = S.defer;
        mem.owed = S.status == kRunning ? 1 : 0;  // the check pass that follows owes its advance
        if (!ok) lost_exchange(R.sync);
    };
    if (met == kMeetAlone) {
        S.slice0 = mem.slice0;
        S.nslices = mem.nslices;
        Alone<kSweepWaves> a(g, A, v, pr, S, R.solo, reinterpret_cast<double*>(lds));
        for (int q = a.wave; q < a.ns; q += kSweepWaves) {
            const int row = (a.s0 + q) * 64 + lane;
            st3(v.p0, row, ld3(v.z, row));
        }
        a.iterate(S);
        leave(true);
        return;
    }

    // rows: slice wave + 8 i of the workgroup's, for i < RPL
    const int own = W.nslices * 64;
    float* zin = lds + 3 * R.lds_rows;
    float* pl = zin + 3 * R.max_halo;
    unsigned vmask = 0, emask = 0;
    int first_w[RPL];  // the slices' first entries and widths, 8 first + width
    F3 r[RPL], ap[RPL];
    float dg[RPL][6], mi[RPL][6];
#pragma unroll
    for (int i = 0; i < RPL; ++i) {
        r[i] = ap[i] = f3(0.0f, 0.0f, 0.0f);
#pragma unroll
        for (int q = 0; q < 6; ++q) dg[i][q] = mi[i][q] = 0.0f;
        first_w[i] = 0;
        if (wave + 8 * i < W.nslices) {
            const int s = W.slice0 + wave + 8 * i, row = s * 64 + lane;
            const int sb = A.slice_ptr[s];
            first_w[i] = uniform_int(8 * sb + (A.slice_ptr[s + 1] - sb));
            if (lane < g.slices[s].nvalid) {
                vmask |= 1u << i;
                if (R.exported[row]) emask |= 1u << i;
                r[i] = ld3(v.r, row);
#pragma unroll
                for (int q = 0; q < 6; ++q) {
                    dg[i][q] = A.diag[(size_t(s) * 6 + q) * 64 + lane];
                    mi[i][q] = A.minv[(size_t(s) * 6 + q) * 64 + lane];
                }
            }
        }
    }
    if (tid < 3) lds[3 * (own + W.nhalo) + tid] = 0.0f;
    for (int h = tid; h < W.nhalo; h += kThreads) {  // the start's z, from the pass before
        const F3 z = ld3(v.z, R.halo[W.halo0 + h]);
        zin[3 * h] = z.x;
        zin[3 * h + 1] = z.y;
        zin[3 * h + 2] = z.z;
    }

    // A p, row by row, each row's blocks in the streaming kernel's entry order.
    // The blocks of the next row are loaded as this row's are used up, and the
    // packed indices a row before that, so loads are in flight throughout.
    unsigned c[3][kSweepPacked] = {};
    float b[kSweepWidth][6];
    auto indices = [&](int i, unsigned (&to)[kSweepPacked]) {
        const int sl = wave + 8 * i;
        // a row that does not exist has width 0 and loads zeros: its indices
        // have to be zero too, not another row's
#pragma unroll
        for (int k = 0; k < kSweepPacked; ++k) to[k] = 0;
        if (sl >= W.nslices) return;  // wave-uniform
        const uint32_t* q = R.packed + size_t(W.slice0 + sl) * kSweepPacked * 64 + fresh(lane);
#pragma unroll
        for (int k = 0; k < kSweepPacked; ++k) to[k] = q[k * 64];
    };
    // block t of row i: entry 0, w - 1, 1, w - 2, .. or its mirror; zeros past
    // the slice's width w
    auto load = [&](int i, int t, const unsigned (&from)[kSweepPacked]) {
        const int fw = fresh_uniform(first_w[i]), w = fw & 7;
        const int o1 = int(from[3]) >> 16, o2 = int(from[4]);
        // entries 0, 1 and 2 may be lower ones; in a narrow slice the last of
        // them is visited from the end
        const int off = t == 0 ? int(from[3] << 16) >> 16
                      : t == 2 ? o1
                      : t == 4 ? o2
                      : t == 1 ? (w == 3 ? o2 : w == 2 ? o1 : 0)
                      : t == 3 ? (w == 4 ? o2 : 0)
                               : 0;
        const float* base = t < w ? A.val + size_t(fw >> 3) * 384 : R.zeros;
        const int e = (t < w ? sym_order(t, w) * 64 + off : 0) + fresh(lane);
        const float* q = base + ((e >> 6) * 384 + (e & 63));
#pragma unroll
        for (int k = 0; k < 6; ++k) b[t][k] = q[k * 64];
    };
    auto times = [&](int i, int next, const unsigned (&at)[kSweepPacked], const unsigned (&after)[kSweepPacked]) {
        const int sl = wave + 8 * i, ln = fresh(lane);
        const F3 pi = sl < W.nslices ? ld3(lds, sl * 64 + ln) : f3(0.0f, 0.0f, 0.0f);  // wave-uniform
        float a0 = fma3(0.0f, dg[i][0], dg[i][1], dg[i][2], pi);
        float a1 = fma3(0.0f, dg[i][1], dg[i][3], dg[i][4], pi);
        float a2 = fma3(0.0f, dg[i][2], dg[i][4], dg[i][5], pi);
#pragma unroll
        for (int t = 0; t < kSweepWidth; ++t) {
            const F3 pj = ld3(lds, int((t & 1) ? at[t >> 1] >> 16 : at[t >> 1] & 0xFFFFu));
            a0 = fma3(a0, b[t][0], b[t][1], b[t][2], pj);
            a1 = fma3(a1, b[t][1], b[t][3], b[t][4], pj);
            a2 = fma3(a2, b[t][2], b[t][4], b[t][5], pj);
            // the products are formed before their block's registers are loaded
            // again: moved below the loads, all rows' blocks would be held at once
            asm volatile("" : "+v"(a0), "+v"(a1), "+v"(a2));
            if (next >= 0) load(next, t, after);
            __builtin_amdgcn_sched_barrier(0);
        }
        ap[i] = f3(a0, a1, a2);
    };
    auto sweep = [&](auto reversed) {
        constexpr bool kBack = decltype(reversed)::value;
        auto row = [](int step) { return step >= RPL ? -1 : kBack ? RPL - 1 - step : step; };
        indices(row(0), c[0]);
        indices(row(1), c[1]);
#pragma unroll
        for (int t = 0; t < kSweepWidth; ++t) load(row(0), t, c[0]);
#pragma unroll
        for (int k = 0; k < RPL; ++k) {
            if (k + 2 < RPL) indices(row(k + 2), c[(k + 2) % 3]);
            times(row(k), row(k + 1), c[k % 3], c[(k + 1) % 3]);
        }
    };
    // the halo rows' z with tag t, four of a thread's in flight
    auto receive_z = [&](unsigned t) {
        constexpr int U = 4;
#pragma nounroll
        for (int h0 = fresh(tid); h0 < W.nhalo; h0 += U * kThreads) {
            u64 a[U], b[U];
            bool late;
            int n = 0;
            const u64* w[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int h = h0 + u * kThreads;
                w[u] = R.zx + R.halo[W.halo0 + (h < W.nhalo ? h : h0)];
            }
#pragma nounroll
            do {
                late = false;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    a[u] = agent_load(w[u]);
                    b[u] = agent_load(w[u] + R.rows);
                }
#pragma unroll
                for (int u = 0; u < U; ++u)
                    late = late || ((unsigned(a[u] >> 32) ^ (t << 16)) | (unsigned(b[u] >> 32) ^ (t << 16))) > 0xFFFFu;
            } while (late && ++n < kExchangePolls);
            if (late) sh.failed = 1;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int h = h0 + u * kThreads;
                if (h < W.nhalo) {
                    zin[3 * h] = __uint_as_float(unsigned(a[u]));
                    zin[3 * h + 1] = __uint_as_float((unsigned(a[u] >> 32) & 0xFFFFu) | (unsigned(b[u] >> 32) << 16));
                    zin[3 * h + 2] = __uint_as_float(unsigned(b[u]));
                }
            }
        }
    };

    bool first = true, ok = true;
    while (S.status == kRunning && S.mode == kModeIter) {
        const float beta = float(S.beta);
#pragma unroll
        for (int i = 0; i < RPL; ++i) {
            if ((vmask >> i) & 1) {
                const int at = (wave + 8 * i) * 64 + fresh(lane);
                const F3 z = first ? ld3(v.z, W.slice0 * 64 + at) : z_update(mi[i], r[i]);
                st3(lds, at, dir3(z, first ? z : ld3(lds, at), beta));
            }
        }
#pragma nounroll
        for (int h = fresh(tid); h < W.nhalo; h += kThreads) {
            const F3 zh = ld3(zin, h);
            st3(lds, own + h, dir3(zh, first ? zh : ld3(lds, own + h), beta));
        }
        first = false;
        __syncthreads();
        if (wg & 1) sweep(std::true_type{});
        else sweep(std::false_type{});
        double sg[1][8], sig[1];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            sg[0][i] = 0.0;
            if (i < RPL && ((vmask >> i) & 1)) {
                const F3 pi = ld3(lds, (wave + 8 * i) * 64 + fresh(lane));
                const F3 y = ap[i < RPL ? i : 0];
                sg[0][i] = fma3d(0.0, double(pi.x), double(pi.y), double(pi.z), y.x, y.y, y.z);
            }
        }
        ++tag;
        ok = sweep_sum<GROUPS, 1>(R, W, sh, sg, 0, tag, sig, [] {});
        if (!ok) break;
        const double alpha = (sig[0] > kGuard || sig[0] < -kGuard) ? S.rho / sig[0] : 0.0;
        const float af = float(alpha);
        ++tag;
        double part[2][8], sum[2];
#pragma unroll
        for (int i = 0; i < 8; ++i) part[0][i] = part[1][i] = 0.0;
#pragma unroll
        for (int i = 0; i < RPL; ++i) {
            r[i] = r_update(r[i], ap[i], af);
            const F3 z = z_update(mi[i], r[i]);
            if ((emask >> i) & 1) {
                u64* w = R.zx + ((W.slice0 + wave + 8 * i) * 64 + fresh(lane));
                const unsigned y = __float_as_uint(z.y);
                agent_store(w, tagged((tag << 16) | (y & 0xFFFFu), __float_as_uint(z.x)));
                agent_store(w + R.rows, tagged((tag << 16) | (y >> 16), __float_as_uint(z.z)));
            }
            if ((vmask >> i) & 1) {
                part[0][i] = dot3d(r[i], z);
                part[1][i] = dot3d(r[i], r[i]);
            }
        }
        // the iterate, which the sums do not need, while they are under way
        auto meanwhile = [&] {
#pragma unroll
            for (int i = 0; i < RPL; ++i) {
                if ((vmask >> i) & 1) {
                    const int at = (wave + 8 * i) * 64 + fresh(lane);
                    const F3 p = ld3(lds, at);
                    double* x = v.x + 3 * (W.slice0 * 64 + at);
                    if (S.pend) {  // the owed term and this one
                        const F3 q = ld3(pl, at);
                        x[0] = x_two(x[0], S.alpha_pend, q.x, alpha, p.x);
                        x[1] = x_two(x[1], S.alpha_pend, q.y, alpha, p.y);
                        x[2] = x_two(x[2], S.alpha_pend, q.z, alpha, p.z);
                    } else if (S.defer) {
                        st3(pl, at, p);
                    } else {
                        x[0] = fma(alpha, double(p.x), x[0]);
                        x[1] = fma(alpha, double(p.y), x[1]);
                        x[2] = fma(alpha, double(p.z), x[2]);
                    }
                }
            }
            receive_z(tag);
        };
        ok = sweep_sum<GROUPS, 2>(R, W, sh, part, 1, tag, sum, meanwhile);
        if (!ok) break;
        S.alpha = alpha;
        pcg_advance(S, pr, AdvanceSums{sum[0], sum[1]});
    }
    if (ok && S.status == kRunning && S.mode == kModeFlush) {
#pragma unroll
        for (int i = 0; i < RPL; ++i) {
            if ((vmask >> i) & 1) {
                const int at = (wave + 8 * i) * 64 + fresh(lane);
                const F3 p = ld3(lds, at);
                double* x = v.x + 3 * (W.slice0 * 64 + at);
                x[0] = fma(S.alpha_pend, double(p.x), x[0]);
                x[1] = fma(S.alpha_pend, double(p.y), x[1]);
                x[2] = fma(S.alpha_pend, double(p.z), x[2]);
            }
        }
        pcg_advance(S, pr, AdvanceSums{0.0, 0.0});
    }
    if (wg == 0 || !ok) leave(ok);
    if (wg == 0 && tid == 0) R.sync->epoch = tag;
}

}  // namespace

void launch_pcg_sweep(const SweepView& R, const LaunchGeom& g, const DevMatrix& A, const DevVectors& v, InstState* st,
                      const InstParams* params, hipStream_t s) {
    if (R.nwg <= 0 || A.bs != 6) throw std::invalid_argument("sweep solve: packed blocks and a plan");
    if (g.ngroups * kGroupSlices != g.nslices || R.ngroups > g.ngroups || R.ngroups > R.nwg * R.groups)
        throw std::invalid_argument("sweep solve: the plan was made for another problem");
    const int grid = 8 * ((R.nwg + 7) / 8);
    const int bytes = sweep_lds_bytes(R.groups, R.lds_rows, R.max_halo);
    if (R.groups == 2) pcg_sweep_kernel<2><<<grid, kThreads, bytes, s>>>(R, g, A, v, st, params);
    else if (R.groups == 3) pcg_sweep_kernel<3><<<grid, kThreads, bytes, s>>>(R, g, A, v, st, params);
    else if (R.groups == 4) pcg_sweep_kernel<4><<<grid, kThreads, bytes, s>>>(R, g, A, v, st, params);
    else throw std::invalid_argument("sweep solve: 2 to 4 groups a workgroup");
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) throw_hip(err, "pcg_sweep_kernel");
}

}  // namespace chysx_amd
