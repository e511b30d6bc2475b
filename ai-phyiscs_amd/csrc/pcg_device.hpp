// SPDX-License-Identifier: Apache-2.0
//
// Device code shared by the kernels of the PCG solve: vector helpers, the
// true residual of a row, the row updates and the scalar step of the solver
// state.  Every expression whose rounding matters is written as explicit
// FMAs, so that all kernels that use it give the same bits.
#pragma once

#include <hip/hip_runtime.h>

#include "cloth_kernels.hpp"
#include "matrix_access.hpp"

namespace chysx_amd {

constexpr double kGuard = 1.0e-37;  // pcg_solver.cu:421-423,451

struct F3 {
    float x, y, z;
};
__device__ __forceinline__ F3 f3(float x, float y, float z) { return {x, y, z}; }
__device__ __forceinline__ F3 operator+(F3 a, F3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ F3 operator-(F3 a, F3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ F3 operator*(F3 a, float s) { return {a.x * s, a.y * s, a.z * s}; }
__device__ __forceinline__ float dot(F3 a, F3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ F3 ld3(const float* p, int i) { return {p[3 * i], p[3 * i + 1], p[3 * i + 2]}; }
__device__ __forceinline__ void st3(float* p, int i, F3 v) {
    p[3 * i] = v.x;
    p[3 * i + 1] = v.y;
    p[3 * i + 2] = v.z;
}

// a + (m0 p.x + m1 p.y + m2 p.z) as one fixed chain of FMAs.  Written out so
// that every kernel variant (unroll, padding mode, storage) rounds the same
// way whatever the compiler schedules.
__device__ __forceinline__ float fma3(float a, float m0, float m1, float m2, F3 p) {
    return fmaf(m2, p.z, fmaf(m1, p.y, fmaf(m0, p.x, a)));
}
__device__ __forceinline__ double fma3d(double a, double m0, double m1, double m2, double x0, double x1, double x2) {
    return fma(m2, x2, fma(m1, x1, fma(m0, x0, a)));
}
// z + beta p_prev, component-wise FMAs
__device__ __forceinline__ F3 dir3(F3 z, F3 pp, float beta) {
    return F3{fmaf(pp.x, beta, z.x), fmaf(pp.y, beta, z.y), fmaf(pp.z, beta, z.z)};
}

// x + (a0 p0 + a1 p1): the owed term of a deferred update and this one
__device__ __forceinline__ double x_two(double x, double a0, float p0, double a1, float p1) {
    return x + fma(a1, double(p1), a0 * double(p0));
}
// r - alpha Ap
__device__ __forceinline__ F3 r_update(F3 r, F3 ap, float alpha) {
    return F3{fmaf(-ap.x, alpha, r.x), fmaf(-ap.y, alpha, r.y), fmaf(-ap.z, alpha, r.z)};
}
// M^-1 r of an update pass, m = (xx, xy, xz, yy, yz, zz)
__device__ __forceinline__ F3 z_update(const float (&m)[6], F3 r) {
    return F3{fmaf(m[2], r.z, fmaf(m[0], r.x, m[1] * r.y)), fmaf(m[4], r.z, fmaf(m[1], r.x, m[3] * r.y)),
              fmaf(m[5], r.z, fmaf(m[2], r.x, m[4] * r.y))};
}
// a . b in FP64, as an update pass sums it
__device__ __forceinline__ double dot3d(F3 a, F3 b) {
    return fma(double(a.z), double(b.z), fma(double(a.x), double(b.x), double(a.y) * double(b.y)));
}

__device__ __forceinline__ F3 minv_mul(const DevMatrix& A, int s, int lane, F3 r) {
    const float* mv = A.minv + (size_t)s * 6 * 64 + lane;
    const float m0 = mv[0], m1 = mv[64], m2 = mv[128], m3 = mv[192], m4 = mv[256], m5 = mv[320];
    return f3(fma3(0.0f, m0, m1, m2, r), fma3(0.0f, m1, m3, m4, r), fma3(0.0f, m2, m4, m5, r));
}

// True residual of row (s, lane): b - A x with FP64 products and sums (x is FP64);
// returns b.  AGENT reads x with agent-scope loads, for an x that other
// workgroups of the same launch have written.
// Entries per load batch: two keeps both the residual kernel and the SpMV
// kernel (whose check mode runs it) at 64 VGPRs or fewer, 8 waves per SIMD.
constexpr int kResidualBatch = 2;

// nlow: the slice's nlower (entries at positions >= nlow hold no lower block
// in any lane, so their mirror index is not read).
template <bool AGENT>
__device__ __forceinline__ F3 true_residual(const DevMatrix& A, const DevVectors& v, int s, int lane, int nlow,
                                            double (&r)[3]) {
    const int row = s * 64 + lane;
    const double* x = v.x;
    auto ldx = [&](int i) { return AGENT ? __hip_atomic_load(x + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : x[i]; };
    float dm[9];
    load_diag(A, s, lane, dm);
    const double x0 = ldx(3 * row), x1 = ldx(3 * row + 1), x2 = ldx(3 * row + 2);
    double a0 = fma3d(0.0, dm[0], dm[1], dm[2], x0, x1, x2);
    double a1 = fma3d(0.0, dm[3], dm[4], dm[5], x0, x1, x2);
    double a2 = fma3d(0.0, dm[6], dm[7], dm[8], x0, x1, x2);
    const int sb = A.slice_ptr[s], w = A.slice_ptr[s + 1] - sb;
    const int* colp = A.col + (size_t)sb * 64 + lane;
    const int* mirp = A.mir + (size_t)sb * 64 + lane;
    const float* vp = A.val + (size_t)sb * A.bs * 64 + lane;
    // Batches of entries in three phases (the column and mirror indices, then
    // every block and x gather, then the FP64 FMAs in entry order, so the sums
    // are those of one entry at a time), so a batch costs two memory round
    // trips instead of three per entry.
    constexpr int RB = kResidualBatch;
    for (int k0 = 0; k0 < w; k0 += RB) {
        int c[RB], mi[RB];
#pragma unroll
        for (int u = 0; u < RB; ++u) {
            c[u] = -1;
            mi[u] = 0;
            if (k0 + u < w) {  // wave-uniform
                c[u] = colp[(k0 + u) * 64];
                if (A.sym && k0 + u < nlow) mi[u] = mirp[(k0 + u) * 64];  // wave-uniform
            }
        }
        float m[RB][9];
        double y[RB][3];
#pragma unroll
        for (int u = 0; u < RB; ++u) {
            if (c[u] >= 0) {
                load_block_at(A, vp + (k0 + u) * A.bs * 64, mi[u], c[u], row, m[u]);
                y[u][0] = ldx(3 * c[u]);
                y[u][1] = ldx(3 * c[u] + 1);
                y[u][2] = ldx(3 * c[u] + 2);
            }
        }
#pragma unroll
        for (int u = 0; u < RB; ++u) {
            if (c[u] >= 0) {
                a0 = fma3d(a0, m[u][0], m[u][1], m[u][2], y[u][0], y[u][1], y[u][2]);
                a1 = fma3d(a1, m[u][3], m[u][4], m[u][5], y[u][0], y[u][1], y[u][2]);
                a2 = fma3d(a2, m[u][6], m[u][7], m[u][8], y[u][0], y[u][1], y[u][2]);
            }
        }
    }
    const F3 bf = ld3(v.rhs, row);
    r[0] = double(bf.x) - a0;
    r[1] = double(bf.y) - a1;
    r[2] = double(bf.z) - a2;
    return bf;
}

// Entry order of the symmetric pass: 0, w-1, 1, w-2, ...  A row's columns
// ascend, so step t pairs its t-th lower entry with its t-th upper entry
// counted from the end.  On a grid, the mirror that step t reads for lower
// entry t (row i - W, i - W + 1 or i - 1) is the upper entry that its owner
// row, 16 slices earlier at W = 1024, streams at its own step t: both
// wavefronts touch the block at the same point of their lives, a fraction of
// a microsecond apart, while it is still in L2.  (In ascending order the
// mirror is read first and the owner reads it at the end of its loop, after
// the XCD has streamed several L2 capacities.)
__device__ __forceinline__ int sym_order(int k, int w) { return (k & 1) ? w - 1 - (k >> 1) : (k >> 1); }


// ---------------------------------------------------------------------------
// Advance of an instance's solver state by one SpMV/update pair, given the
// sums of the partials that pair wrote: r . z and |r|^2 of the update pass
// (Iter), or the true ones of the check pass (Check); none for a flush.  Scalar logic restates
// reduce_rho_beta_kernel (pcg_solver.cu:436-454) with its 1e-37 guard, plus
// the stopping rule: true relative residual sqrt(|b-Ax|^2 / max(|b|^2,1e-30))
// <= tol (pcg_solver.cu:595-641, 916-923), or exactly max_iter iterations
// when tol == 0 (pcg_solver.cu:542-592).  Runs in the next SpMV pass (every
// workgroup, identical inputs and order) or in pcg_advance_kernel.
// ---------------------------------------------------------------------------
struct AdvanceSums {
    double rz;  // r . z
    double rr;  // |r|^2
};
__device__ __forceinline__ void pcg_advance(InstState& S, const InstParams& pr, const AdvanceSums& t) {
    const double tol2 = pr.tol2;
    if (S.mode == kModeFlush) {  // x is whole again
        S.pend = 0;
        S.alpha_pend = 0.0;
        S.defer = 1;
        if (S.flush_to == kModeCheck) {
            S.mode = kModeCheck;
        } else {
            S.mode = kModeIter;
            S.status = kStopped;
        }
    } else if (S.mode == kModeCheck) {
        const double rr = t.rr;
        S.rr = rr;
        S.relres = sqrt(rr / S.bb);
        if (rr <= tol2 * S.bb) {
            S.status = kConverged;
        } else {  // residual replacement: restart the recursion from b - A x
            S.restarts += 1;
            S.rho = t.rz;
            S.beta = 0.0;
            S.mode = kModeIter;
            S.defer = 1;
            if (S.iters >= pr.max_iter) S.status = kStopped;
        }
    } else {
        const double rho = S.rho, rho_new = t.rz;
        if (S.pend) {  // this update pass added the owed term
            S.pend = 0;
        } else if (S.defer) {  // this update pass left x += alpha p to the next
            S.alpha_pend = S.alpha;  // the alpha that pass used
            S.pend = 1;
        }
        S.defer = S.pend ? 0 : 1;
        S.beta = (rho > kGuard || rho < -kGuard) ? rho_new / rho : 0.0;
        S.rho = rho_new;
        S.rr = t.rr;
        S.parity ^= 1;
        S.iters += 1;
        const bool check = tol2 > 0.0 && t.rr <= tol2 * S.bb;
        const bool stop = !check && S.iters >= pr.max_iter;
        if ((check || stop) && S.pend) {  // complete x first
            S.mode = kModeFlush;
            S.flush_to = check ? int(kModeCheck) : int(kStopped);
        } else if (check) {
            S.mode = kModeCheck;
        } else if (stop) {
            S.status = kStopped;
        }
    }
}

// A solve's state after the start pass: rr = |r|^2, bb = |b|^2, rz = r . z.
__device__ __forceinline__ void pcg_begin(InstState& S, const InstParams& pr, double rr, double bb, double rz) {
    S.bb = fmax(bb, 1.0e-30);
    S.rr = rr;
    S.relres = sqrt(rr / S.bb);
    S.iters = 0;
    S.restarts = 0;
    S.mode = kModeIter;
    S.beta = 0.0;
    S.rho = rz;
    S.pend = 0;
    S.alpha_pend = 0.0;
    S.defer = 1;
    S.owed = 0;
    S.status = (pr.tol2 > 0.0 && rr <= pr.tol2 * S.bb) ? kConverged : (pr.max_iter <= 0 ? kStopped : kRunning);
}

__device__ __forceinline__ int uniform_int(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ double uniform_double(double x) {
    const unsigned long long b = static_cast<unsigned long long>(__double_as_longlong(x));
    const unsigned lo = unsigned(__builtin_amdgcn_readfirstlane(int(unsigned(b))));
    const unsigned hi = unsigned(__builtin_amdgcn_readfirstlane(int(unsigned(b >> 32))));
    return __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
}
// One particle of the step's end: x = x_n + dx, v = dx / dt (times
// exp(-damping dt) when damping > 0) (finalize_step_kernel,
// cloth_simulator.cu:222-244).
__device__ __forceinline__ void finalize_row(const DevExt& e, const InstParams& pr, float dt,
                                             const int* __restrict__ pin_inc_off, const int* __restrict__ pin_inc,
                                             const float* __restrict__ pin_tgt, int row, int p, double x0, double x1,
                                             double x2) {
    F3 d = f3(float(x0), float(x1), float(x2));
    const F3 xn = ld3(e.pos, p);
    F3 xnew = xn + d;
    if (pr.pin_proj && pin_inc_off[row + 1] > pin_inc_off[row]) {  // a projected pin ends at its target
        xnew = ld3(pin_tgt, pin_inc[pin_inc_off[row]]);
        d = xnew - xn;
    }
    const float inv_dt = 1.0f / dt;
    F3 vn = d * inv_dt;
    if (pr.damping > 0.0f) vn = vn * expf(-pr.damping * dt);
    st3(e.pos, p, xnew);
    st3(e.vel, p, vn);
}

}  // namespace chysx_amd
