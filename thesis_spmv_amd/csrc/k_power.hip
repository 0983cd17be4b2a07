// Power method on a small matrix in one workgroup.
//
// A step of the general path is an SpMV launch and one or two launches that
// finish the norms.  On a matrix of a few thousand nonzeros each of them is
// only a chain of dependent memory latencies: 100 steps of CRS_Merge on a
// 37 x 29 Poisson grid (5 233 nonzeros) took 1 587 us, 15.9 us a step, of which
// the matrix needs none.  Here one 1024-thread workgroup runs the whole loop:
// the nonzeros stay in its registers (E per thread), both iterates and the
// step's products in LDS, and a step is
//   products   every thread multiplies its entries by x from LDS, products to
//              LDS;                                                 barrier
//   row sums   G lanes per row sum the row's products (row_sum, then the lanes'),
//              scale, write the new iterate to LDS and add up |y|^2, x.y, x.x;
//              wave sums to LDS;                                    barrier
// so nothing but LDS is touched between the first load and the last store:
// the step is bound by the latency of its LDS chains.  The norm of a step is
// needed only in the next step's row sums: wave 0 computes the scale (an FP64
// square root and division) while the others already multiply.
//
// The arithmetic is the general path's: products in the accumulator type, row
// sums (row_sum), out = sum / |y_previous| and the norms in FP64, every sum in a
// fixed order.  A step takes 1.1 us at 10 x 10, 1.7 us at 37 x 29 (15.9
// before) and 2.6 us at 52 x 51, FP64; 100 steps at 37 x 29 take 0.20 ms.
#include <algorithm>

#include "kernels.hpp"

namespace pwmk {

constexpr int kPsBS = 1024;
constexpr int kPsWaves = kPsBS / 64;
// LDS a workgroup may ask for beside the kernel's static arrays
constexpr int64_t kPsLds = 160 * 1024 - 2048;

template <typename VT, int E>
__global__ __launch_bounds__(kPsBS) void k_power_small(CrsDev A, int G, PowerArgs pw, int64_t k0, int64_t nsteps) {
    using X = typename Arith<VT>::X;
    using Acc = typename Arith<VT>::A;
    extern __shared__ __align__(16) unsigned char ps_smem[];
    __shared__ double red[2][3][kPsWaves];
    __shared__ double sc[2];
    if (k0 > 0 && pw.ctrl[1]) return;
    const int n = (int)A.nrows, nz = (int)A.nnz;
    const int np = (n + 1) & ~1;  // keeps the arrays behind it 8-byte aligned
    Acc* prod = (Acc*)ps_smem;    // one product per nonzero
    X* xs = (X*)(prod + ((nz + 1) & ~1));  // the two iterates
    int32_t* rs = (int32_t*)(xs + 2 * np);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

    int32_t c[E];
    Acc v[E];
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const int k = tid + j * kPsBS;
        c[j] = k < nz ? A.ci[k] : 0;
        v[j] = k < nz ? (Acc)widen(((const VT*)A.val)[k]) : (Acc)0;
    }
    for (int i = tid; i <= n; i += kPsBS) rs[i] = A.rs[i];
    const X* src = (const X*)((k0 & 1) ? pw.buf1 : pw.buf0);
    X* cur = xs + (k0 & 1) * np;
    for (int i = tid; i < n; i += kPsBS) cur[i] = src[i];
    double yy_prev = k0 > 0 ? pw.rec[4 * (k0 - 1)] : 0.0;
    double lam_prev = k0 > 0 ? pw.rec[4 * (k0 - 1) + 3] : 0.0;
    if (tid < 64) sc[k0 & 1] = k0 == 0 ? 1.0 : 1.0 / sqrt(yy_prev);
    __syncthreads();

    const int gl = tid & (G - 1), grp = tid / G, ngrp = kPsBS / G;
    int64_t k = k0;
    int done = 0;
    double scale = 1.0;
    for (;;) {
        const int par = (int)(k & 1);
        const X* __restrict__ x = xs + par * np;
        X* __restrict__ y = xs + (par ^ 1) * np;
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const int e = tid + j * kPsBS;
            if (e < nz) prod[e] = v[j] * (Acc)x[c[j]];
        }
        __syncthreads();
        scale = sc[par];
        double yy = 0.0, xy = 0.0, xx = 0.0;
        for (int r0 = 0; r0 < n; r0 += ngrp) {
            const int r = r0 + grp;
            double s = r < n ? row_sum(prod, rs[r] + gl, rs[r + 1], G) : 0.0;
            for (int off = 1; off < G; off <<= 1) s += __shfl_xor(s, off);
            if (gl == 0 && r < n) {
                const double xd = (double)x[r] * scale;
                const X out = (X)(s * scale);
                y[r] = out;
                const double yd = (double)out;
                yy += yd * yd;
                xy += xd * yd;
                xx += xd * xd;
            }
        }
        yy = group_sum<64>(yy);
        xy = group_sum<64>(xy);
        xx = group_sum<64>(xx);
        if (lane == 0) {
            red[par][0][wave] = yy;
            red[par][1][wave] = xy;
            red[par][2][wave] = xx;
        }
        __syncthreads();
        // the next step reads the other halves of red and sc: one barrier
        // (its products') separates their reuse
        const bool last = k + 1 >= pw.max_it || k + 1 >= k0 + nsteps;
        if (wave == 0 || pw.tol >= 0.0 || last) {
            yy = group_sum<16>(red[par][0][lane & (kPsWaves - 1)]);
            if (wave == 0) sc[par ^ 1] = 1.0 / sqrt(yy);
        }
        done = k + 1 >= pw.max_it;
        if (pw.tol >= 0.0 || last) {
            xy = group_sum<16>(red[par][1][lane & (kPsWaves - 1)]);
            xx = group_sum<16>(red[par][2][lane & (kPsWaves - 1)]);
            const double lam = xy / xx;
            if (pw.tol >= 0.0 && k >= 1 && fabs(lam - lam_prev) <= pw.tol * fabs(lam)) done = 1;
            if (done || last) {
                if (tid == 0) {
                    pw.rec[4 * k + 0] = yy;
                    pw.rec[4 * k + 1] = xy;
                    pw.rec[4 * k + 2] = xx;
                    pw.rec[4 * k + 3] = lam;
                    pw.ctrl[0] = (int)(k + 1);
                    pw.ctrl[1] = done;
                    double* result = (double*)(pw.ctrl + 4);
                    result[0] = lam;
                    result[1] = yy;
                }
                yy_prev = yy;
                break;
            }
            lam_prev = lam;
        }
        ++k;
    }
    // Step k read iterate `x` and wrote `y` (K = k + 1 steps so far).  Done:
    // both leave divided by their own norms, as k_power_finish does; the
    // caller's start vector (K == 1) stays as it is.  Not done (the launch's
    // share of the steps is over): as they are.
    const int par = (int)(k & 1);
    const X* __restrict__ x = xs + par * np;
    const X* __restrict__ y = xs + (par ^ 1) * np;
    X* gx = (X*)(par ? pw.buf1 : pw.buf0);
    X* gy = (X*)(par ? pw.buf0 : pw.buf1);
    const double s_last = 1.0 / sqrt(yy_prev);
    for (int i = tid; i < n; i += kPsBS) {
        gy[i] = done ? (X)((double)y[i] * s_last) : y[i];
        if (k > 0) gx[i] = done ? (X)((double)x[i] * scale) : x[i];
    }
}

// ---------------------------------------------------------------- norms of a step

constexpr int kFinBS = 1024;
constexpr int kSumBS = 256;
// Many slots: workgroup b leaves the sum of slots [b*per, (b+1)*per) in slot
// b*per.
__global__ __launch_bounds__(kSumBS) void k_power_sum(PowerArgs pw, int64_t n, int64_t per) {
    __shared__ double red[48];
    if (power_done(pw)) return;
    const int64_t i0 = (int64_t)blockIdx.x * per, i1 = i0 + per < n ? i0 + per : n;
    double yy = 0.0, xy = 0.0, xx = 0.0;
    slot_sum(pw.partials, i0 + threadIdx.x, kSumBS, i1, yy, xy, xx);
    block_sum3<kSumBS>(yy, xy, xx, red);
    if (threadIdx.x == 0) {
        pw.partials[3 * i0 + 0] = yy;
        pw.partials[3 * i0 + 1] = xy;
        pw.partials[3 * i0 + 2] = xx;
    }
}

// One workgroup: slots 0, step, 2*step, ... (n of them) into step k's record.
template <int BS>
__global__ __launch_bounds__(BS) void k_power_final(PowerArgs pw, const double* slots, int64_t n, int64_t step) {
    __shared__ double red[48];
    if (power_done(pw)) return;
    double yy = 0.0, xy = 0.0, xx = 0.0;
    slot_sum(slots, threadIdx.x * step, BS * step, n * step, yy, xy, xx);
    block_sum3<BS>(yy, xy, xx, red);
    if (threadIdx.x == 0) power_record(pw, pw.k, yy, xy, xx);
}

hipError_t launch_power_final(const PowerArgs& pw, const double* slots, int64_t n, int64_t step, hipStream_t s) {
    if (n <= kPsU * kSumBS)
        hipLaunchKernelGGL(k_power_final<kSumBS>, dim3(1), dim3(kSumBS), 0, s, pw, slots, n, step);
    else
        hipLaunchKernelGGL(k_power_final<kFinBS>, dim3(1), dim3(kFinBS), 0, s, pw, slots, n, step);
    return hipGetLastError();
}

// One workgroup reads kPsU slots per thread in one go; beyond two such rounds
// a launch that spreads the reading costs less than a third.
hipError_t launch_power_reduce(const PowerArgs& pw, int64_t n, hipStream_t s) {
    if (pw.defer) return hipSuccess;
    if (n <= 2 * kPsU * kFinBS) return launch_power_final(pw, pw.partials, n, 1, s);
    const int64_t per = std::max<int64_t>(kPsU * kSumBS, (n + kFinBS - 1) / kFinBS);
    const int64_t nb = (n + per - 1) / per;
    hipLaunchKernelGGL(k_power_sum, dim3((unsigned)nb), dim3(kSumBS), 0, s, pw, n, per);
    return launch_power_final(pw, pw.partials, nb, per, s);
}

// ---------------------------------------------------------------- the one-workgroup loop

// Entries per thread: the smallest instance that holds all nonzeros.  FP64
// entries take 3 registers each and FP32 ones 2, of the 128 a thread of a
// 1024-thread workgroup has.
static int ps_entries(int vtype, int64_t nnz) {
    const int64_t need = (nnz + kPsBS - 1) / kPsBS;
    for (int e : {2, 4, 8, 16, 24})
        if (need <= e && (vtype != VT_F64 || e <= 16)) return e;
    return 0;
}

static int64_t ps_lds(const CrsDev& A) {
    const int64_t b = A.vtype == VT_F64 ? 8 : 4;
    return b * ((A.nnz + 1) & ~(int64_t)1) + 2 * b * ((A.nrows + 1) & ~(int64_t)1) + 4 * (A.nrows + 1);
}

// Lanes per row of the row sums: a step's row sums cost about
// ceil(n G / 1024) rounds of ceil(longest row / G) dependent LDS reads (about
// 4 overlap) plus the norms' fixed part and log2(G) lane exchanges.
static int ps_lanes(int64_t n, int64_t row_max) {
    int best = 1;
    double cost = 1e300;
    for (int g = 1; g <= 64; g <<= 1) {
        const double rounds = (double)((n * g + kPsBS - 1) / kPsBS);
        const double c = rounds * ((double)((row_max + g - 1) / g) + 8.0 + 2.0 * __builtin_ctz(g));
        if (c < cost) {
            cost = c;
            best = g;
        }
    }
    return best;
}

// The matrix fits (registers, LDS) and its longest row does not leave one
// group of lanes summing alone: 64 lanes on the longest row stay within the
// 16 rounds the largest instance's products take.
bool power_small_fits(const CrsDev& A, int64_t row_max) {
    return A.nrows > 0 && A.nrows == A.ncols && ps_entries(A.vtype, A.nnz) > 0 && ps_lds(A) <= kPsLds &&
           row_max <= 16 * 64;
}

template <typename VT, int E>
static hipError_t launch_ps(const CrsDev& A, int G, const PowerArgs& pw, int64_t k0, int64_t nsteps, hipStream_t s) {
    hipLaunchKernelGGL((k_power_small<VT, E>), dim3(1), dim3(kPsBS), (size_t)ps_lds(A), s, A, G, pw, k0, nsteps);
    return hipGetLastError();
}

template <typename VT>
static hipError_t launch_ps_t(const CrsDev& A, int G, const PowerArgs& pw, int64_t k0, int64_t nsteps, hipStream_t s) {
    switch (ps_entries(A.vtype, A.nnz)) {
        case 2: return launch_ps<VT, 2>(A, G, pw, k0, nsteps, s);
        case 4: return launch_ps<VT, 4>(A, G, pw, k0, nsteps, s);
        case 8: return launch_ps<VT, 8>(A, G, pw, k0, nsteps, s);
        case 16: return launch_ps<VT, 16>(A, G, pw, k0, nsteps, s);
        case 24:
            if constexpr (sizeof(typename Arith<VT>::A) == 4) return launch_ps<VT, 24>(A, G, pw, k0, nsteps, s);
            return hipErrorInvalidValue;
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_power_small(const CrsDev& A, int64_t row_max, const PowerArgs& pw, int64_t k0, int64_t nsteps,
                              hipStream_t s) {
    const int G = ps_lanes(A.nrows, row_max);
    switch (A.vtype) {
        case VT_F64: return launch_ps_t<double>(A, G, pw, k0, nsteps, s);
        case VT_F32: return launch_ps_t<float>(A, G, pw, k0, nsteps, s);
        case VT_BF16: return launch_ps_t<bf16_t>(A, G, pw, k0, nsteps, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace pwmk
