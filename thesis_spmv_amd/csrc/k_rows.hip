// CRS SpMV over wave tiles (the CRS format's kernel for short rows).
//
// Tile t holds the rows [cut[t].x, cut[t+1].x): the cuts lie `step` entries
// apart, moved up to the next row start, so that a tile is at most 256 entries
// (one aligned group of 4 per lane of a wave) and 128 rows.  One wave a tile:
// it loads its group with 128-bit loads, gathers x, leaves the products in its
// own slice of LDS and sums the rows, a lane per row (row_sum).  No
// wave waits for another, the only chain is cut -> entries -> x, and the many
// short waves keep enough loads in flight to run at the rate a plain read of
// the arrays reaches.
//
// Blocks are renumbered (xcd_chunked) so that the chip as a whole reads one
// narrow front of the arrays while each XCD still gets stretches of
// consecutive rows, which share x lines in its L2.  With an eighth of the
// matrix per XCD (eight fronts a 2 GB array apart) HBM delivers a fifth less.
//
// Poisson 5000 x 5000, FP64 (2.0 GB): 441 us with the workgroup tiles of
// k_tiles, 406 with their blocks renumbered this way, 332 us here (6.0 TB/s; a
// plain read reaches 6.1).  1024 x 1024 over three copies: 16.0 -> 13.7 us.
// Two groups per lane (339 us), two or more tiles per wave with the next one's
// loads in flight (353 us) and resident waves (412 us) are slower.
#include "../../include/pwm_hip.h"
#include "kernels.hpp"
#include "merge_tile.hpp"

namespace pwmk {

constexpr int kRwSlots = 2;       // rows per lane
constexpr int kRwEntries = 256;   // entries per tile
constexpr int kRwMaxRow = 64;     // longest row: beyond, a lane's serial sum holds its wave up
constexpr int kRwChunk = 256;     // consecutive tiles per XCD in the block order (128 .. 256 within 1%)
constexpr int kRwBS = 64;         // threads per block of an SpMV

// Threads per block of a power step, one partial-sum slot a block: 256 (FP32
// 3000 x 3000: 92.7 us a step against 99.9 with 512, 100 x 100 4.2 against
// 4.7), but 512 where that brings the slots down to what the next step adds up
// itself (k_power.hip; FP64 600 x 600: 11.1 -> 8.5 us) or to 200 000, and 1024
// where 512 leave more slots than the fixed workspace of the no-allocation power
// method holds: 16 tiles a block are at least 3040 entries, more than the 2048
// merge items a slot of CRS_MERGE's merge kernels stands for, so it takes every
// matrix here that it takes there.
static int rows_power_bs(int64_t nt) {
    if ((nt + 7) / 8 > PWM_NOALLOC_MAX_SLOTS) return 1024;
    return (nt > 2048 && (nt + 7) / 8 <= kDeferSlots) || (nt + 3) / 4 > 200000 ? 512 : 256;
}

// First row whose entries start at or after p * step (n from the last cut on).
__device__ __forceinline__ int64_t rows_cut(const int32_t* __restrict__ rs, int64_t n, int64_t nt, int64_t step,
                                            int64_t p) {
    if (p >= nt) return n;
    const int64_t want = p * step;
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((int64_t)rs[mid] < want)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

__global__ void k_rows_plan(const int32_t* __restrict__ rs, int64_t n, int64_t step, int64_t nt, int2* __restrict__ cut,
                            int* __restrict__ too_many_rows) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t > nt) return;
    const int64_t a = rows_cut(rs, n, nt, step, t);
    cut[t] = make_int2((int)a, rs[a]);
    if (t < nt && rows_cut(rs, n, nt, step, t + 1) - a > 64 * kRwSlots) *too_many_rows = 1;
}

// POWER: 1 a power step, 2 one that adds up the last step's norms (deferred).
// NT: non-temporal entry loads (the entries, read once, leave the L2 to x).
template <typename VT, int BS, int POWER, bool NT>
__global__ __launch_bounds__(BS) void k_rows(CrsDev A, RowsPlan rp, const typename Arith<VT>::X* __restrict__ x_arg,
                                             typename Arith<VT>::X* __restrict__ y_arg, PowerArgs pw) {
    using X = typename Arith<VT>::X;
    using Acc = typename Arith<VT>::A;
    __shared__ __align__(16) Acc prods[BS / 64][kRwEntries];
    __shared__ double red[POWER ? 48 : 1];
    const X* __restrict__ x = x_arg;
    X* __restrict__ y = y_arg;
    double scale = 1.0;
    if constexpr (POWER) {
        if (power_done(pw)) return;
        const int64_t k = pw.k;
        x = (const X*)((k & 1) ? pw.buf1 : pw.buf0);
        y = (X*)((k & 1) ? pw.buf0 : pw.buf1);
        scale = POWER == 2 ? 1.0 / sqrt(last_norm<BS>(pw, red)) : recorded_scale(pw);
    }
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    Acc* prod = prods[wave];
    const int64_t t = xcd_chunked(blockIdx.x, gridDim.x, kRwChunk * 64 / BS) * (BS / 64) + wave;
    double yy = 0.0, xy = 0.0, xx = 0.0;
    if (t < rp.nt) {
        const int2 c0 = rp.cut[t], c1 = rp.cut[t + 1];
        const int a0 = c0.x, nr = c1.x - c0.x;
        const int off = c0.y & ~3;  // entry k of the tile has its product at k - off
        // lanes past the tile's last group reload that group
        const int g = 4 * min(lane, max(((c1.y - off + 3) >> 2) - 1, 0));
        const int32_t* __restrict__ ci = A.ci + off;
        const VT* __restrict__ val = (const VT*)A.val + off;
        vi4 jq;
        Quad<VT> vq;
        if constexpr (NT) {
            jq = __builtin_nontemporal_load(G((const vi4*)(ci + g)));
            vq.load_nt(val + g);
        } else {
            jq = *G((const vi4*)(ci + g));
            vq.load(val + g);
        }
        // an empty tile (a0 may be n) reads row 0's offsets and x
        const int64_t ra = nr > 0 ? a0 : 0;
        const int last = nr > 0 ? nr - 1 : 0;
        const int32_t* __restrict__ rs = A.rs + ra;
        int32_t beg[kRwSlots], end[kRwSlots];
        X xr[kRwSlots];
#pragma unroll
        for (int s = 0; s < kRwSlots; ++s) {
            if (s == 0 || nr > 64 * s) {
                const int r = min(lane + 64 * s, last);
                beg[s] = G(rs)[r];
                end[s] = G(rs)[r + 1];
                if constexpr (POWER) xr[s] = G(x)[ra + r];
            }
        }
        Acc pr[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) pr[e] = (Acc)G(x)[jq[e]];
#pragma unroll
        for (int e = 0; e < 4; ++e) pr[e] *= (Acc)vq.get(e);
        store4<Acc>(&prod[4 * lane], pr);
        // the wave's LDS accesses are in order; the fence keeps the compiler's
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int s = 0; s < kRwSlots; ++s) {
            const int r = lane + 64 * s;
            if (r < nr) {
                const double sum = row_sum(prod, beg[s] - off, end[s] - off, 1);
                if constexpr (POWER) {
                    const double xd = (double)xr[s] * scale;
                    const X out = (X)(sum * scale);
                    G(y)[a0 + r] = out;
                    const double yd = (double)out;
                    yy += yd * yd;
                    xy += xd * yd;
                    xx += xd * xd;
                } else {
                    G(y)[a0 + r] = (X)sum;
                }
            }
        }
    }
    if constexpr (POWER) {
        block_sum3<BS>(yy, xy, xx, red);
        if (threadIdx.x == 0) {
            pw.partials[3 * blockIdx.x + 0] = yy;
            pw.partials[3 * blockIdx.x + 1] = xy;
            pw.partials[3 * blockIdx.x + 2] = xx;
        }
    }
}

// Entries between cuts: a tile's last row may reach row_max - 1 entries past
// the next cut and its first group may start 3 entries early.  0: rows too
// long.
int64_t rows_step(int64_t row_max) {
    return row_max >= 1 && row_max <= kRwMaxRow ? kRwEntries - 3 - (row_max - 1) : 0;
}

int64_t rows_power_blocks(int64_t nt) {
    const int waves = rows_power_bs(nt) / 64;
    return (nt + waves - 1) / waves;
}

hipError_t launch_rows_plan(const CrsDev& A, int64_t step, int64_t nt, int2* cut, int* too_many_rows, hipStream_t s) {
    hipLaunchKernelGGL(k_rows_plan, dim3((unsigned)((nt + 256) / 256)), dim3(256), 0, s, A.rs, A.nrows, step, nt, cut,
                       too_many_rows);
    return hipGetLastError();
}

template <typename VT, int BS>
static void launch_rows_power(const CrsDev& A, const RowsPlan& rp, const PowerArgs& pw, hipStream_t s) {
    using X = typename Arith<VT>::X;
    auto k = pw.defer ? (A.nt ? k_rows<VT, BS, 2, true> : k_rows<VT, BS, 2, false>)
                      : (A.nt ? k_rows<VT, BS, 1, true> : k_rows<VT, BS, 1, false>);
    hipLaunchKernelGGL(k, dim3((unsigned)rows_power_blocks(rp.nt)), dim3(BS), 0, s, A, rp, (const X*)nullptr,
                       (X*)nullptr, pw);
}

template <typename VT>
static hipError_t launch_rows_t(const CrsDev& A, const RowsPlan& rp, const void* x, void* y, const PowerArgs* pw,
                                hipStream_t s) {
    using X = typename Arith<VT>::X;
    const int bs = pw ? rows_power_bs(rp.nt) : 0;
    if (bs == 256)
        launch_rows_power<VT, 256>(A, rp, *pw, s);
    else if (bs == 512)
        launch_rows_power<VT, 512>(A, rp, *pw, s);
    else if (bs == 1024)
        launch_rows_power<VT, 1024>(A, rp, *pw, s);
    else
        hipLaunchKernelGGL((A.nt ? k_rows<VT, kRwBS, 0, true> : k_rows<VT, kRwBS, 0, false>),
                           dim3((unsigned)((rp.nt + kRwBS / 64 - 1) / (kRwBS / 64))), dim3(kRwBS), 0, s, A, rp,
                           (const X*)x, (X*)y, PowerArgs{});
    return hipGetLastError();
}

hipError_t launch_rows(const CrsDev& A, const RowsPlan& rp, const void* x, void* y, const PowerArgs* pw, hipStream_t s) {
    switch (A.vtype) {
        case VT_F64: return launch_rows_t<double>(A, rp, x, y, pw, s);
        case VT_F32: return launch_rows_t<float>(A, rp, x, y, pw, s);
        case VT_BF16: return launch_rows_t<bf16_t>(A, rp, x, y, pw, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace pwmk
