// CSB and BlockCOH SpMV kernels for gfx950.
//
// Both formats are processed by workgroups that own a slab of rows and keep
// its y-slice in LDS (FP64 atomic adds, ds_add_f64, for every storage type:
// products are formed in the vectors' type and summed in FP64): every entry of a
// slab, wherever its block sits in the block row or band, adds into LDS and
// the slab is written to y once with coalesced stores.
//
// x locality: every workgroup walks its blocks in the same order (CSB: block
// columns ascending, CSB.hpp:354-363; BlockCOH: the Hilbert order of the
// blocks, which is the same sequence of block columns for every band whose
// rows fit one block row).  The workgroups resident on one XCD therefore
// gather from the same x-slice at about the same time, and that slice
// (beta * 8 bytes, 128-256 KB) stays in the XCD's 4 MB L2 instead of each
// gather missing to the Infinity Fabric as in a row-ordered CRS sweep over
// random columns.
//
// Swept slabs (k_csb_sweep) carry this to matrices whose x outgrows the L2:
// one persistent 1024-thread workgroup per CU owns an nnz-balanced row slab
// (y-slice in all of the CU's LDS) and walks x in windows of 1 MB, the slab's
// entries stored window by window.  The 32 slabs of an XCD start together and
// sweep at about the same rate, so the XCD fetches each window about once per
// SpMV and the gathers hit its L2; no partial sums are written.  Inside a
// window the entries are stored in column order, four to a lane and
// permuted so that the 64 lanes of one gather instruction read 64
// consecutive entries: with about one entry per x line per slab and window,
// a third of the gathers then share a line, and so an L2 request, with a
// neighbouring lane.
#include "blocked.hpp"
#include "kernels.hpp"
#include "merge_tile.hpp"

namespace blocked {

using pwmk::Arith;
using pwmk::bf16_t;
using pwmk::PowerArgs;
using pwmk::widen;

constexpr int kBS = kBlockedBS;
constexpr int kWaves = kBS / 64;
constexpr int kWin = 2 * kBS;  // CSB pieces staged per window

// Block-wide exclusive scan of one int per thread; returns the prefix and
// writes the total to *total.  `tmp` holds kWaves ints.
__device__ __forceinline__ int block_excl_scan(int v, int* tmp, int* total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int u = __shfl_up(incl, d);
        if (lane >= d) incl += u;
    }
    if (lane == 63) tmp[wave] = incl;
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        const int t = tmp[w];
        if (w < wave) before += t;
        all += t;
    }
    __syncthreads();
    *total = all;
    return before + incl - v;
}

// ---------------------------------------------------------------- CSB

// workgroup -> (slab task t, column group g).  With a multiple of 8 groups the
// launch runs in rounds of 8 groups so that XCD (b % 8) keeps one group per
// round: b = round * 8 * slabs_total + slab * 8 + xcd.
__device__ __forceinline__ void csb_task(const CsbArgs& a, int& g, int64_t& t) {
    if (a.groups % 8 == 0) {
        const int64_t per_round = (a.n_tasks / a.groups) * 8;
        const int64_t round = blockIdx.x / per_round, rem = blockIdx.x % per_round;
        t = rem / 8;
        g = (int)(round * 8 + rem % 8);
    } else {
        g = (int)(blockIdx.x % a.groups);
        t = blockIdx.x / a.groups;
    }
}

// Writes a slab's LDS sums: to ypart[g] with several column groups, else to
// y (POWER: scaled, with the slab's |y|^2, x.y, x.x in partial slot t).
template <typename X, typename Acc, int BS, bool POWER, bool NT = false>
__device__ __forceinline__ void csb_write_slab(const CsbArgs& a, const double* ylds, int h, int64_t row0, int g, int64_t t,
                                               const X* __restrict__ x, X* __restrict__ y, double scale,
                                               const PowerArgs& pw, double* red) {
    const int tid = threadIdx.x;
    if (a.groups > 1) {  // partial slab sums; k_csb_reduce finishes y
        Acc* yp = (Acc*)a.ypart + (int64_t)g * a.nor;
        for (int i = tid; i < h; i += BS) {
            const int64_t row = row0 + i;
            if (row >= a.nor) break;
            if constexpr (NT)
                __builtin_nontemporal_store((Acc)ylds[i], &yp[row]);
            else
                yp[row] = (Acc)ylds[i];
        }
        return;
    }
    double yy = 0.0, xy = 0.0, xx = 0.0;
    for (int i = tid; i < h; i += BS) {
        const int64_t row = row0 + i;
        if (row >= a.nor) break;
        if constexpr (POWER) {
            const X out = (X)(ylds[i] * scale);
            y[row] = out;
            const double yd = (double)out, xd = (double)x[row] * scale;
            yy += yd * yd;
            xy += xd * yd;
            xx += xd * xd;
        } else {
            y[row] = (X)ylds[i];
        }
    }
    if constexpr (POWER) {
        pwmk::block_sum3<BS>(yy, xy, xx, red);
        if (tid == 0) {
            pw.partials[3 * t + 0] = yy;
            pw.partials[3 * t + 1] = xy;
            pw.partials[3 * t + 2] = xx;
        }
    }
}

template <typename VT, bool POWER>
__global__ __launch_bounds__(kBS) void k_csb(CsbArgs a, const typename Arith<VT>::X* __restrict__ x_arg,
                                             typename Arith<VT>::X* __restrict__ y_arg, PowerArgs pw) {
    using X = typename Arith<VT>::X;
    using Acc = typename Arith<VT>::A;
    __shared__ double ylds[kCsbLdsRows];
    __shared__ int32_t p_start[kWin];
    __shared__ int32_t p_pre[kWin + 1];
    __shared__ int scan_tmp[kWaves];
    __shared__ double red[48];

    const X* __restrict__ x = x_arg;
    X* __restrict__ y = y_arg;
    double scale = 1.0;
    if constexpr (POWER) {
        if (pwmk::power_done(pw)) return;
        const int64_t k = pw.k;
        x = (const X*)((k & 1) ? pw.buf1 : pw.buf0);
        y = (X*)((k & 1) ? pw.buf0 : pw.buf1);
        scale = pwmk::recorded_scale(pw);
    }
    const VT* __restrict__ val = (const VT*)a.val;
    const uint32_t* __restrict__ ind = a.ind;
    const int tid = threadIdx.x;
    int g;
    int64_t t;
    csb_task(a, g, t);
    const int64_t br = t / a.slabs;
    const int s = (int)(t % a.slabs);
    const int64_t beta = (int64_t)1 << a.bits;
    const int h = (int)a.slab_rows;
    const int slab_base = s * h;
    for (int i = tid; i < h; i += kBS) ylds[i] = 0;

    const int64_t bc_lo = g * a.H / a.groups, bc_hi = (g + 1) * a.H / a.groups;
    const int64_t npieces = (bc_hi - bc_lo) * a.np;
    const Piece* __restrict__ P = a.pieces + t * a.H * a.np + bc_lo * a.np;
    for (int64_t w0 = 0; w0 < npieces; w0 += kWin) {
        const int nw = (int)(npieces - w0 < kWin ? npieces - w0 : kWin);
        __syncthreads();
        const int i0 = 2 * tid, i1 = 2 * tid + 1;
        int len0 = 0, len1 = 0;
        if (i0 < nw) {
            const Piece q = P[w0 + i0];
            p_start[i0] = q.start;
            len0 = q.end - q.start;
        }
        if (i1 < nw) {
            const Piece q = P[w0 + i1];
            p_start[i1] = q.start;
            len1 = q.end - q.start;
        }
        int total;
        const int base = block_excl_scan(len0 + len1, scan_tmp, &total);
        p_pre[i0] = base;
        p_pre[i1] = base + len0;
        if (tid == kBS - 1) p_pre[kWin] = total;
        __syncthreads();
        const int T = total;
        int cur = 0;
        for (int v = tid; v < T; v += 4 * kBS) {
            int kk[4], pc[4];
            bool ok[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int vv = v + u * kBS;
                ok[u] = vv < T;
                if (ok[u]) {
                    while (p_pre[cur + 1] <= vv) ++cur;
                    pc[u] = cur;
                    kk[u] = p_start[cur] + (vv - p_pre[cur]);
                } else {
                    pc[u] = 0;
                    kk[u] = 0;
                }
            }
            uint32_t w[4];
            Acc vv[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                w[u] = ok[u] ? ind[kk[u]] : 0u;
                vv[u] = ok[u] ? (Acc)widen(val[kk[u]]) : (Acc)0;
            }
            Acc xv[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int64_t bc = bc_lo + ((w0 + pc[u]) >> a.np_shift);
                xv[u] = ok[u] ? (Acc)x[bc * beta + (w[u] & 0xffffu)] : (Acc)0;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (ok[u]) atomicAdd(&ylds[(int)(w[u] >> 16) - slab_base], (double)(vv[u] * xv[u]));
        }
    }
    __syncthreads();
    csb_write_slab<X, Acc, kBS, POWER>(a, ylds, h, br * beta + slab_base, g, t, x, y, scale, pw, red);
}

// Slab-stream CSB: the workgroup's entries are one contiguous run
// [soff[t*H + bc_lo], soff[t*H + bc_hi]) read as aligned groups of 4 (128-bit
// index loads, 128-bit value loads); every entry adds val * x[col] into the
// slab's LDS rows.  Lanes past the run reload its last group and add nothing,
// so the loads carry no branch.
constexpr int kSBS = 256;

// POWER: 1 a power step, 2 one that adds up the last step's norms (deferred);
// kSU: groups of 4 entries per thread per step (2 or 4); NT: non-temporal
// entry loads and partial-slab stores; WIDE: ind holds the column and srows
// the row in the slab.
template <typename VT, int POWER, int kSU, bool NT, bool WIDE>
__global__ __launch_bounds__(kSBS) void k_csb_stream(CsbArgs a, const typename Arith<VT>::X* __restrict__ x_arg,
                                                     typename Arith<VT>::X* __restrict__ y_arg, PowerArgs pw) {
    using X = typename Arith<VT>::X;
    using Acc = typename Arith<VT>::A;
    extern __shared__ __align__(16) unsigned char csb_smem[];
    double* ylds = (double*)csb_smem;
    __shared__ double red[48];

    const X* __restrict__ x = x_arg;
    X* __restrict__ y = y_arg;
    double scale = 1.0;
    if constexpr (POWER) {
        if (pwmk::power_done(pw)) return;
        const int64_t k = pw.k;
        x = (const X*)((k & 1) ? pw.buf1 : pw.buf0);
        y = (X*)((k & 1) ? pw.buf0 : pw.buf1);
        scale = POWER == 2 ? 1.0 / sqrt(pwmk::last_norm<kSBS>(pw, red)) : pwmk::recorded_scale(pw);
    }
    const VT* __restrict__ val = (const VT*)a.val;
    const uint32_t* __restrict__ ind = a.ind;
    const int tid = threadIdx.x;
    int g;
    int64_t t;
    csb_task(a, g, t);
    const int h = (int)a.slab_rows;
    for (int i = tid; i < h; i += kSBS) ylds[i] = 0;
    const int64_t bc_lo = g * a.H / a.groups, bc_hi = (g + 1) * a.H / a.groups;
    // entry offsets fit 31 bits (int32 CRS row starts)
    const int32_t e0 = a.soff[t * a.H + bc_lo], e1 = a.soff[t * a.H + bc_hi];
    const int cb = a.col_bits;
    const uint32_t cmask = (uint32_t)((1ull << cb) - 1);
    __syncthreads();
    const int32_t q0 = e0 >> 2, q1 = (int32_t)(((int64_t)e1 + 3) >> 2);
    for (int32_t qb = q0; qb < q1; qb += kSBS * kSU) {
        pwmk::vi4 w[kSU];
        pwmk::vu2 r[kSU];
        pwmk::Quad<VT> v[kSU];
#pragma unroll
        for (int u = 0; u < kSU; ++u) {
            const int32_t q = qb + tid + u * kSBS;
            const int64_t qc = q < q1 ? q : q1 - 1;
            if constexpr (NT) {
                w[u] = __builtin_nontemporal_load(pwmk::G((const pwmk::vi4*)(ind + 4 * qc)));
                if constexpr (WIDE) r[u] = __builtin_nontemporal_load(pwmk::G((const pwmk::vu2*)(a.srows + 4 * qc)));
                v[u].load_nt(val + 4 * qc);
            } else {
                w[u] = *pwmk::G((const pwmk::vi4*)(ind + 4 * qc));
                if constexpr (WIDE) r[u] = *pwmk::G((const pwmk::vu2*)(a.srows + 4 * qc));
                v[u].load(val + 4 * qc);
            }
        }
        X xv[kSU][4];
#pragma unroll
        for (int u = 0; u < kSU; ++u)
#pragma unroll
            for (int j = 0; j < 4; ++j) xv[u][j] = x[WIDE ? (uint32_t)w[u][j] : ((uint32_t)w[u][j] & cmask)];
#pragma unroll
        for (int u = 0; u < kSU; ++u)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int64_t k = 4 * (int64_t)(qb + tid + u * kSBS) + j;
                uint32_t row;
                if constexpr (WIDE)
                    row = ((j < 2 ? r[u].x : r[u].y) >> (16 * (j & 1))) & 0xffffu;
                else
                    row = (uint32_t)w[u][j] >> cb;
                if (k >= e0 && k < e1) atomicAdd(&ylds[row], (double)((Acc)v[u].get(j) * (Acc)xv[u][j]));
            }
    }
    __syncthreads();
    const int64_t beta = (int64_t)1 << a.bits;
    const int64_t row0 = (t / a.slabs) * beta + (t % a.slabs) * (int64_t)h;
    csb_write_slab<X, Acc, kSBS, (POWER > 0), NT>(a, ylds, h, row0, g, t, x, y, scale, pw, red);
}

// y[r] = sum over the column groups of ypart[g][r], groups in order (and the
// power-method scale and partial sums).
template <typename VT, bool POWER>
__global__ __launch_bounds__(kBS) void k_csb_reduce(CsbArgs a, typename Arith<VT>::X* __restrict__ y_arg,
                                                    PowerArgs pw) {
    using X = typename Arith<VT>::X;
    using Acc = typename Arith<VT>::A;
    __shared__ double red[48];
    X* __restrict__ y = y_arg;
    const X* __restrict__ x = nullptr;
    double scale = 1.0;
    if constexpr (POWER) {
        if (pwmk::power_done(pw)) return;
        const int64_t k = pw.k;
        x = (const X*)((k & 1) ? pw.buf1 : pw.buf0);
        y = (X*)((k & 1) ? pw.buf0 : pw.buf1);
        scale = pwmk::recorded_scale(pw);
    }
    const Acc* __restrict__ yp = (const Acc*)a.ypart;
    double yy = 0.0, xy = 0.0, xx = 0.0;
    for (int64_t r = (int64_t)blockIdx.x * kBS + threadIdx.x; r < a.nor; r += (int64_t)gridDim.x * kBS) {
        Acc s = 0;
        for (int g = 0; g < a.groups; ++g) s += yp[(int64_t)g * a.nor + r];
        if constexpr (POWER) {
            const X out = (X)((double)s * scale);
            y[r] = out;
            const double yd = (double)out, xd = (double)x[r] * scale;
            yy += yd * yd;
            xy += xd * yd;
            xx += xd * xd;
        } else {
            y[r] = (X)s;
        }
    }
    if constexpr (POWER) {
        const double ra = pwmk::block_sum<kBS>(yy, red);
        const double rb = pwmk::block_sum<kBS>(xy, red);
        const double rc = pwmk::block_sum<kBS>(xx, red);
        if (threadIdx.x == 0) {
            pw.partials[3 * blockIdx.x + 0] = ra;
            pw.partials[3 * blockIdx.x + 1] = rb;
            pw.partials[3 * blockIdx.x + 2] = rc;
        }
    }
}

int csb_reduce_blocks(int64_t nor) {
    const int64_t b = (nor + kBS - 1) / kBS;
    return (int)(b < 2048 ? (b > 0 ? b : 1) : 2048);
}

// ---------------------------------------------------------------- CSB swept slabs

// Swept slabs: one persistent workgroup of kSwBS threads per CU, each
// owning an nnz-balanced row slab [sstart[t], sstart[t+1]) whose y-slice
// stays in LDS for the whole kernel.  The slab's entries are stored window
// by window: window p holds the columns [p ww, (p+1) ww) (ww <= 2^wb, 1 MB of x by
// default), and every workgroup walks the windows in the same order, adding
// val * x[col] into its LDS rows (ds_add).  In window p, wave w takes the
// chunks w, w + 16, ... of 64 x kSU groups of 4 entries of the slab's run;
// the first chunk of the next window's entries is loaded while the current
// one is gathered, and a workgroup barrier ends every window.  The barrier
// keeps a workgroup's 16 waves on one window, and the nnz-balanced
// workgroups, all started together, stay close enough that each XCD's L2
// holds the windows its workgroups gather from; no partial sums are written
// and read back.
constexpr int kSwBS = 1024;

template <typename VT, int kSU, bool NT>
struct SweepChunk {
    pwmk::vi4 w[kSU];
    pwmk::Quad<VT> v[kSU];
    // groups qb + lane + 64 u; a group past the run's last one (or of an
    // empty run) reloads a valid group and its entries are masked
    __device__ __forceinline__ void load(const uint32_t* __restrict__ ind, const VT* __restrict__ val, int32_t qb,
                                         int32_t q1, int lane) {
#pragma unroll
        for (int u = 0; u < kSU; ++u) {
            const int32_t q = qb + lane + u * 64;
            const int64_t qc = q < q1 ? q : (q1 > 0 ? q1 - 1 : 0);
            if constexpr (NT) {
                w[u] = __builtin_nontemporal_load(pwmk::G((const pwmk::vi4*)(ind + 4 * qc)));
                v[u].load_nt(val + 4 * qc);
            } else {
                w[u] = *pwmk::G((const pwmk::vi4*)(ind + 4 * qc));
                v[u].load(val + 4 * qc);
            }
        }
    }
};

// Turns of a workgroup's waves: chunk `ticket` of the sweep may add once the
// chunks before it have.  The waves of a workgroup are all resident and chunk
// 0 waits for nobody, so every wait ends.
__device__ __forceinline__ void turn_wait(const int* turn, int ticket) {
    // the next in line looks without a pause, the others sleep 64 clocks
    for (int d; (d = ticket - __hip_atomic_load(turn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) > 0;)
        if (d > 2) __builtin_amdgcn_s_sleep(1);
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ void turn_pass(int* turn, int ticket, int lane) {
    // the adds have been performed (lgkmcnt 0) before the next wave sees its
    // turn; a workgroup release fence would also wait for the entry loads in
    // flight (1.2 M power-law rows: 90.6 us with the fence, 77.2 without)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);
    asm volatile("" ::: "memory");
    if (lane == 0) __hip_atomic_store(turn, ticket + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// ORD: the chunk's products are formed first and added in the chunk's turn.
template <typename VT, int kSU, bool NT, bool ORD, typename X, typename LAcc>
__device__ __forceinline__ void sweep_add(const SweepChunk<VT, kSU, NT>& c, int32_t qb, int lane, int32_t e0, int32_t e1,
                                          const X* __restrict__ xw, uint32_t wmask, int wb, LAcc* ylds, int* turn,
                                          int ticket) {
    using Acc = typename Arith<VT>::A;
    // an entry outside [e0, e1) belongs to a neighbouring run (its column is
    // in another window), and an index 0xffffffff pads a column-ordered run:
    // such an entry gathers the window's first column, which exists, and
    // adds nothing
    bool ok[kSU][4];
    Acc pr[kSU][4];
#pragma unroll
    for (int u = 0; u < kSU; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t k = 4 * (int64_t)(qb + lane + u * 64) + j;
            ok[u][j] = k >= e0 && k < e1 && (uint32_t)c.w[u][j] != 0xffffffffu;
            pr[u][j] = (Acc)xw[ok[u][j] ? ((uint32_t)c.w[u][j] & wmask) : 0u];
        }
#pragma unroll
    for (int u = 0; u < kSU; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            pr[u][j] *= (Acc)c.v[u].get(j);
            // the product exists here, before the wait for the turn
            if constexpr (ORD) asm volatile("" : "+v"(pr[u][j]));
        }
    if constexpr (ORD) turn_wait(turn, ticket);
#pragma unroll
    for (int u = 0; u < kSU; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (ok[u][j]) atomicAdd(&ylds[(uint32_t)c.w[u][j] >> wb], (LAcc)pr[u][j]);
    if constexpr (ORD) turn_pass(turn, ticket, lane);
}

// LAcc: the LDS sums' type (float only for FP32 storage whose slabs have more
// rows than fit in FP64).
// ORD: the waves add their chunks in turn (window, chunk) instead of meeting
// at barriers, so that every row is summed in one fixed order: the CRS formats'
// sweep, whose results repeat bit for bit.  The gathers of up to 16 chunks run
// while one chunk's adds do; the turns cost FP64 sweeps nothing (1.2 M
// power-law rows 77.2 us against 77.8 at barriers, 3 M 228 against 227) and
// FP32 ones, whose gathers are shorter, a tenth to a third.
template <typename VT, bool POWER, bool NT, typename LAcc, int SU = 2, bool ORD = false>
__global__ __launch_bounds__(kSwBS) void k_csb_sweep(CsbArgs a, const typename Arith<VT>::X* __restrict__ x_arg,
                                                     typename Arith<VT>::X* __restrict__ y_arg, PowerArgs pw) {
    using X = typename Arith<VT>::X;
    constexpr int kSU = SU;  // groups of 4 entries per lane per chunk
    constexpr int kWv = kSwBS / 64;
    constexpr int kChunk = 64 * kSU;  // groups of 4 entries per wave per chunk
    extern __shared__ __align__(16) unsigned char csb_smem[];
    LAcc* ylds = (LAcc*)csb_smem;
    __shared__ double red[48];
    __shared__ int turn;  // ORD: the chunk whose turn it is
    if (ORD && threadIdx.x == 0) turn = 0;

    const X* __restrict__ x = x_arg;
    X* __restrict__ y = y_arg;
    double scale = 1.0;
    if constexpr (POWER) {
        if (pwmk::power_done(pw)) return;
        const int64_t k = pw.k;
        x = (const X*)((k & 1) ? pw.buf1 : pw.buf0);
        y = (X*)((k & 1) ? pw.buf0 : pw.buf1);
        scale = 1.0 / sqrt(pwmk::last_norm<kSwBS>(pw, red));
    }
    const VT* __restrict__ val = (const VT*)a.val;
    const uint32_t* __restrict__ ind = a.ind;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t t = blockIdx.x;
    const int32_t r0 = a.sstart[t];
    const int nrows = a.sstart[t + 1] - r0;
    for (int i = tid; i < nrows; i += kSwBS) ylds[i] = 0;
    const int wb = a.wb;
    const uint32_t wmask = (uint32_t)(((uint64_t)1 << wb) - 1);
    const int32_t* __restrict__ woff = a.soff + t * a.W;
    SweepChunk<VT, kSU, NT> cur, nxt;
    int32_t e0 = woff[0], e1 = woff[1];
    int32_t q0 = e0 >> 2, q1 = (int32_t)(((int64_t)e1 + 3) >> 2);
    cur.load(ind, val, q0 + wv * kChunk, q1, lane);
    int ticket = 0;  // ORD: the window's first chunk
    __syncthreads();
    for (int64_t p = 0; p < a.W; ++p) {
        const X* __restrict__ xw = x + p * a.ww;
        const int32_t pe0 = e0, pe1 = e1, pq0 = q0, pq1 = q1;
        if (p + 1 < a.W) {  // the next window's run and its first chunk, loaded ahead
            e0 = woff[p + 1];
            e1 = woff[p + 2];
            q0 = e0 >> 2;
            q1 = (int32_t)(((int64_t)e1 + 3) >> 2);
            nxt.load(ind, val, q0 + wv * kChunk, q1, lane);
        }
        // the wave's first chunk of this window, then the further ones, if its
        // share is larger
        if (!ORD || pq0 + wv * kChunk < pq1)
            sweep_add<VT, kSU, NT, ORD>(cur, pq0 + wv * kChunk, lane, pe0, pe1, xw, wmask, wb, ylds, &turn, ticket + wv);
        int c = wv + kWv;
        for (int32_t qb = pq0 + c * kChunk; qb < pq1; qb += kWv * kChunk, c += kWv) {
            SweepChunk<VT, kSU, NT> more;
            more.load(ind, val, qb, pq1, lane);
            sweep_add<VT, kSU, NT, ORD>(more, qb, lane, pe0, pe1, xw, wmask, wb, ylds, &turn, ticket + c);
        }
        if constexpr (ORD) ticket += (pq1 - pq0 + kChunk - 1) / kChunk;
        if (!ORD && ((p + 1) & (a.sync_every - 1)) == 0) __syncthreads();  // windows up to p done by every wave
        cur = nxt;
    }
    __syncthreads();
    double yy = 0.0, xy = 0.0, xx = 0.0;
    for (int i = tid; i < nrows; i += kSwBS) {
        const int64_t row = (int64_t)r0 + i;
        if constexpr (POWER) {
            const X out = (X)((double)ylds[i] * scale);
            y[row] = out;
            const double yd = (double)out, xd = (double)x[row] * scale;
            yy += yd * yd;
            xy += xd * yd;
            xx += xd * xd;
        } else {
            y[row] = (X)ylds[i];
        }
    }
    if constexpr (POWER) {
        pwmk::block_sum3<kSwBS>(yy, xy, xx, red);
        if (tid == 0) {
            pw.partials[3 * t + 0] = yy;
            pw.partials[3 * t + 1] = xy;
            pw.partials[3 * t + 2] = xx;
        }
    }
}

template <typename VT, typename LAcc>
static int sweep_blocks_t(int rows) {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_csb_sweep<VT, false, true, LAcc>, kSwBS,
                                                     (size_t)rows * sizeof(LAcc)) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return nb;
}

int csb_sweep_blocks_per_cu(int vtype, int rows, bool acc32) {
    switch (vtype) {
        case 0: return sweep_blocks_t<double, double>(rows);
        case 1: return acc32 ? sweep_blocks_t<float, float>(rows) : sweep_blocks_t<float, double>(rows);
        case 2: return acc32 ? sweep_blocks_t<bf16_t, float>(rows) : sweep_blocks_t<bf16_t, double>(rows);
    }
    return 0;
}

// ---------------------------------------------------------------- BlockCOH

// One workgroup per task (CohTask); its waves take the task's steps of
// kCohStep entries in turn, each on its own: no barrier between the first zero
// and the last sum.  A lane holds 4 consecutive entries and adds them up while
// the row stays the same (equal rows in many lanes would take turns: an LDS add
// of 64 lanes takes 16 clocks on random rows, 56 on runs of 5, 192 on one row);
// a step within one long row is added up by the wave.  The sums go to the
// band's y-slice in LDS (LDS tasks, which write it once) or to the band's rows
// of ysum with global atomics, FP64 both.  The block of an entry is the number
// of block starts before it: four ballots and a table of the blocks at the
// steps.
//
// BS: 512, or 64 where that times faster at load (blocked_host.hip): 8 waves
// that take a band's steps in turn are 2048 entries apart, on x far beyond an L2
// and scattered columns some 30 blocks, 4 MB of x; a wave per band keeps to a few
// blocks, the bands of an XCD walk x in the same order and meet in its L2.  Every
// workgroup reserves the LDS window of the largest band whatever its size, so
// waves on their own are as many per CU as their windows let in: 11 at 1542 rows,
// 6 at 3084, 3 at 6168.
//
// Bound by the gathers (FP64 9-point stencil with 2 random entries per row, 1 M
// rows: 215 G/s of the 213-233 G/s that the L2 serves) or, on a matrix of few
// blocks, by HBM.  Mean of back-to-back SpMVs on rotating copies, us, against
// workgroups that decode the stored jumps with two segmented scans per 2048
// entries: that stencil 88 -> 51, on 90 K rows 18.6 -> 8.2; Poisson 1024^2
// 39.8 -> 18, 3000^2 283 -> 145; power-law rows, 100 K 67 -> 18, 500 K 315 ->
// 64, 2 M 687 -> 261 (with 8 waves per band 278), 3 M 871 -> 411 (536).  Tried: 2
// or 4 steps at once (the same or slower), non-temporal entry loads (18 -> 22 on
// the Poisson matrix, 281 -> 275 on the 2 M rows), the step table read after the
// entries (278 -> 302).
template <typename VT, bool POWER, int BS>
__global__ __launch_bounds__(BS) void k_coh(CohArgs a, const typename Arith<VT>::X* __restrict__ x_arg,
                                            typename Arith<VT>::X* __restrict__ y_arg, PowerArgs pw) {
    using X = typename Arith<VT>::X;
    using Acc = typename Arith<VT>::A;
    // the LDS window holds the rows of the largest band accumulated in LDS
    // (at most coh_lds_rows), sized at launch
    extern __shared__ __align__(16) unsigned char coh_smem[];
    double* ylds = (double*)coh_smem;
    constexpr int kCohStage = 256;  // blocks of a band kept in LDS, where a band has no more
    __shared__ CohBlock bstage[kCohStage];
    __shared__ double red[48];

    const X* __restrict__ x = x_arg;
    X* __restrict__ y = y_arg;
    double scale = 1.0;
    if constexpr (POWER) {
        if (pwmk::power_done(pw)) return;
        const int64_t k = pw.k;
        x = (const X*)((k & 1) ? pw.buf1 : pw.buf0);
        y = (X*)((k & 1) ? pw.buf0 : pw.buf1);
        scale = 1.0 / sqrt(pwmk::last_norm<BS>(pw, red));
    }
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const CohTask task = a.tasks[blockIdx.x];
    const CohBand band = a.bands[task.band];
    const CohBlock* __restrict__ blocks = a.blocks + band.first_block;
    typedef const int32_t __attribute__((address_space(4))) * ScalarTable;
    const ScalarTable stab = (ScalarTable)(a.step_block + band.step_table);
    const bool lds = task.atomic == 0;
    double* __restrict__ ysum = a.ysum + band.sum;

    const bool staged = band.blocks <= kCohStage;
    if (lds)
        for (int i = tid; i < band.rows; i += BS) ylds[i] = 0;
    if (staged)
        for (int i = tid; i < band.blocks; i += BS) bstage[i] = blocks[i];
    __syncthreads();
    const int64_t first = band.entry, end = first + band.nnz, base = first & ~(int64_t)3;
    for (int s = task.step0 + wave; s < task.step0 + task.nsteps; s += (BS / 64)) {
        int b = stab[s];  // a scalar load, ahead of the entries
        const int64_t q = base + (int64_t)s * kCohStep + 4 * lane;
        // lanes beyond the band load its last quad (the arrays are padded)
        const int64_t qc = q < end ? q : (end - 1) & ~(int64_t)3;
        const pwmk::vi4 quad = *pwmk::G((const pwmk::vi4*)(a.ent + qc));
        const uint32_t en[4] = {(uint32_t)quad[0], (uint32_t)quad[1], (uint32_t)quad[2], (uint32_t)quad[3]};
        pwmk::Quad<VT> v;
        v.load((const VT*)a.val + qc);
        bool ok[4];
        uint64_t m[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            ok[j] = q + j >= first && q + j < end;
            m[j] = __ballot(ok[j] && (en[j] & kCohFirst));
        }
        CohBlock blk[4];
        if ((m[0] | m[1] | m[2] | m[3]) == 0) {  // the wave's entries lie in one block
            const CohBlock one = staged ? bstage[b] : blocks[b];
#pragma unroll
            for (int j = 0; j < 4; ++j) blk[j] = one;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                b = __builtin_amdgcn_mbcnt_hi((uint32_t)(m[j] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m[j], b));
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                b += (int)((m[j] >> lane) & 1);
                const int bi = b > 0 ? b : 0;  // -1 before the band's first entry
                blk[j] = staged ? bstage[bi] : blocks[bi];
            }
        }
        int row[4];
        Acc xv[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            row[j] = ok[j] ? blk[j].row + (int)(en[j] >> 15 & 0x7fff) : -1;
            xv[j] = (Acc)x[(int64_t)blk[j].col + (ok[j] ? en[j] & 0x7fff : 0)];
        }
        // (the products come after this test, which runs while the gathers are under way)
        double sum = 0.0;
        const int row0 = __builtin_amdgcn_readfirstlane(row[0]);
        if (row0 >= 0 && __ballot(row[1] != row0 || row[2] != row0 || row[3] != row0 || row[0] != row0) == 0) {
#pragma unroll
            for (int j = 0; j < 4; ++j) sum += (double)((Acc)v.get(j) * xv[j]);
            sum = pwmk::group_sum<64>(sum);
            if (lane == 0) {
                if (lds)
                    atomicAdd(&ylds[row0], sum);
                else
                    atomicAdd(&ysum[row0], sum);
            }
            continue;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const Acc p = (Acc)v.get(j) * xv[j];
            sum += (double)p;
            if (j < 3 && row[j + 1] == row[j]) continue;
            if (row[j] >= 0) {
                if (lds)
                    atomicAdd(&ylds[row[j]], sum);
                else
                    atomicAdd(&ysum[row[j]], sum);
            }
            sum = 0.0;
        }
    }
    if (!lds) {
        if constexpr (POWER)  // k_coh_finish sums these rows
            if (tid < 3) pw.partials[3 * blockIdx.x + tid] = 0.0;
        return;
    }
    __syncthreads();
    double yy = 0.0, xy = 0.0, xx = 0.0;
    for (int i = tid; i < band.rows; i += BS) {
        const int64_t row = (int64_t)band.start + i;
        if constexpr (POWER) {
            const X out = (X)(ylds[i] * scale);
            y[row] = out;
            const double yd = (double)out, xd = (double)x[row] * scale;
            yy += yd * yd;
            xy += xd * yd;
            xx += xd * xd;
        } else {
            y[row] = (X)ylds[i];
        }
    }
    if constexpr (POWER) {
        const double ra = pwmk::block_sum<BS>(yy, red);
        const double rb = pwmk::block_sum<BS>(xy, red);
        const double rc = pwmk::block_sum<BS>(xx, red);
        if (tid == 0) {
            pw.partials[3 * blockIdx.x + 0] = ra;
            pw.partials[3 * blockIdx.x + 1] = rb;
            pw.partials[3 * blockIdx.x + 2] = rc;
        }
    }
}

// The rows of atomic bands (one workgroup per piece): their sums to y, and back
// to zero for the next SpMV.  Power mode: also |y|^2, x^T y, x^T x, into the
// partial slots after the tasks' (slot n_tasks + i for piece i).
template <typename VT, bool POWER>
__global__ __launch_bounds__(kBS) void k_coh_finish(CohArgs a, typename Arith<VT>::X* __restrict__ y_arg, PowerArgs pw) {
    using X = typename Arith<VT>::X;
    __shared__ double red[48];
    const X* x = nullptr;
    X* y = y_arg;
    double scale = 1.0;
    if constexpr (POWER) {
        if (pwmk::power_done(pw)) return;
        const int64_t k = pw.k;
        x = (const X*)((k & 1) ? pw.buf1 : pw.buf0);
        y = (X*)((k & 1) ? pw.buf0 : pw.buf1);
        // with deferred norms k_coh, before this in the step, wrote the record: one
        // scale for all rows (its blocks may add the slots up in another order)
        scale = pwmk::recorded_scale(pw);
    }
    const CohRows piece = a.pieces[blockIdx.x];
    double yy = 0.0, xy = 0.0, xx = 0.0;
    for (int i = threadIdx.x; i < piece.rows; i += kBS) {
        const int64_t row = (int64_t)piece.start + i;
        const double sum = a.ysum[(int64_t)piece.sum + i];
        a.ysum[(int64_t)piece.sum + i] = 0.0;
        if constexpr (POWER) {
            const X out = (X)(sum * scale);
            y[row] = out;
            const double yd = (double)out, xd = (double)x[row] * scale;
            yy += yd * yd;
            xy += xd * yd;
            xx += xd * xd;
        } else {
            y[row] = (X)sum;
        }
    }
    if constexpr (POWER) {
        const double ra = pwmk::block_sum<kBS>(yy, red);
        const double rb = pwmk::block_sum<kBS>(xy, red);
        const double rc = pwmk::block_sum<kBS>(xx, red);
        if (threadIdx.x == 0) {
            const int64_t slot = a.n_tasks + blockIdx.x;
            pw.partials[3 * slot + 0] = ra;
            pw.partials[3 * slot + 1] = rb;
            pw.partials[3 * slot + 2] = rc;
        }
    }
}

// ---------------------------------------------------------------- launchers

template <typename VT>
static hipError_t csb_t(const CsbArgs& a, const void* x, void* y, const PowerArgs* pw, hipStream_t s, int part) {
    using X = typename Arith<VT>::X;
    using Acc = typename Arith<VT>::A;
    if (a.n_tasks <= 0) return hipSuccess;
    if (a.sweep) {
        if (part == 2) return hipSuccess;  // no column-group reduction
        const bool acc32 = sizeof(Acc) == 4 && a.acc32;
        const size_t lds = (size_t)a.max_rows * (acc32 ? sizeof(Acc) : sizeof(double));
        auto pick = [&](auto power, auto acc) {
            constexpr bool P = decltype(power)::value;
            using L = decltype(acc);
            if (a.unroll == 1) return a.nt ? k_csb_sweep<VT, P, true, L, 1> : k_csb_sweep<VT, P, false, L, 1>;
            if (a.unroll == 4) return a.nt ? k_csb_sweep<VT, P, true, L, 4> : k_csb_sweep<VT, P, false, L, 4>;
            return a.nt ? k_csb_sweep<VT, P, true, L, 2> : k_csb_sweep<VT, P, false, L, 2>;
        };
        auto pick_ord = [&](auto power) {
            constexpr bool P = decltype(power)::value;
            return a.nt ? k_csb_sweep<VT, P, true, double, 2, true> : k_csb_sweep<VT, P, false, double, 2, true>;
        };
        auto kp = a.ord     ? pick_ord(std::true_type{})
                  : acc32 ? pick(std::true_type{}, Acc{})
                          : pick(std::true_type{}, 0.0);
        auto kf = a.ord     ? pick_ord(std::false_type{})
                  : acc32 ? pick(std::false_type{}, Acc{})
                          : pick(std::false_type{}, 0.0);
        if (pw)
            hipLaunchKernelGGL(kp, dim3((unsigned)a.n_tasks), dim3(kSwBS), lds, s, a, (const X*)nullptr, (X*)nullptr,
                               *pw);
        else
            hipLaunchKernelGGL(kf, dim3((unsigned)a.n_tasks), dim3(kSwBS), lds, s, a, (const X*)x, (X*)y, PowerArgs{});
        return hipGetLastError();
    }
    if (part == 2) {
        // the column-group reduction only
    } else if (a.stream) {
        const size_t lds = (size_t)a.slab_rows * sizeof(double);
        const dim3 grid((unsigned)a.n_tasks);
        // kernel instance for (power step, width, unroll, non-temporal)
        auto pick = [&](auto power, auto wide) {
            constexpr int P = decltype(power)::value;
            constexpr bool W = decltype(wide)::value;
            if (a.unroll == 4) return a.nt ? k_csb_stream<VT, P, 4, true, W> : k_csb_stream<VT, P, 4, false, W>;
            return a.nt ? k_csb_stream<VT, P, 2, true, W> : k_csb_stream<VT, P, 2, false, W>;
        };
        auto pick_wide = [&](auto power) { return a.wide ? pick(power, std::true_type{}) : pick(power, std::false_type{}); };
        auto k = !pw         ? pick_wide(std::integral_constant<int, 0>{})
                 : pw->defer ? pick_wide(std::integral_constant<int, 2>{})
                             : pick_wide(std::integral_constant<int, 1>{});
        hipLaunchKernelGGL(k, grid, dim3(kSBS), lds, s, a, pw ? (const X*)nullptr : (const X*)x,
                           pw ? (X*)nullptr : (X*)y, pw ? *pw : PowerArgs{});
    } else if (pw) {
        hipLaunchKernelGGL((k_csb<VT, true>), dim3((unsigned)a.n_tasks), dim3(kBS), 0, s, a, (const X*)nullptr,
                           (X*)nullptr, *pw);
    } else {
        hipLaunchKernelGGL((k_csb<VT, false>), dim3((unsigned)a.n_tasks), dim3(kBS), 0, s, a, (const X*)x, (X*)y,
                           PowerArgs{});
    }
    if (a.groups > 1 && part != 1) {
        const unsigned rb = (unsigned)csb_reduce_blocks(a.nor);
        if (pw)
            hipLaunchKernelGGL((k_csb_reduce<VT, true>), dim3(rb), dim3(kBS), 0, s, a, (X*)nullptr, *pw);
        else
            hipLaunchKernelGGL((k_csb_reduce<VT, false>), dim3(rb), dim3(kBS), 0, s, a, (X*)y, PowerArgs{});
    }
    return hipGetLastError();
}

hipError_t launch_csb(const CsbArgs& a, const void* x, void* y, const PowerArgs* pw, hipStream_t s, int part) {
    switch (a.vtype) {
        case 0: return csb_t<double>(a, x, y, pw, s, part);
        case 1: return csb_t<float>(a, x, y, pw, s, part);
        case 2: return csb_t<bf16_t>(a, x, y, pw, s, part);
    }
    return hipErrorInvalidValue;
}

template <typename VT, bool POWER>
static hipError_t coh_t(const CohArgs& a, const void* x, void* y, const PowerArgs& pw, hipStream_t s) {
    using X = typename Arith<VT>::X;
    const size_t lds = (size_t)std::max<int32_t>(a.lds_rows, 1) * sizeof(double);
    auto k = a.one_wave ? k_coh<VT, POWER, 64> : k_coh<VT, POWER, kBS>;
    // no tasks: one band without entries, too tall for the LDS; its rows are pieces
    if (a.n_tasks > 0)
        hipLaunchKernelGGL(k, dim3((unsigned)a.n_tasks), dim3(a.one_wave ? 64 : kBS), lds, s, a, (const X*)x, (X*)y, pw);
    if (a.n_pieces > 0)
        hipLaunchKernelGGL((k_coh_finish<VT, POWER>), dim3((unsigned)a.n_pieces), dim3(kBS), 0, s, a, (X*)y, pw);
    return hipGetLastError();
}

hipError_t launch_coh(const CohArgs& a, const void* x, void* y, const PowerArgs* pw, hipStream_t s) {
    switch (a.vtype) {
        case 0: return pw ? coh_t<double, true>(a, x, y, *pw, s) : coh_t<double, false>(a, x, y, PowerArgs{}, s);
        case 1: return pw ? coh_t<float, true>(a, x, y, *pw, s) : coh_t<float, false>(a, x, y, PowerArgs{}, s);
        case 2: return pw ? coh_t<bf16_t, true>(a, x, y, *pw, s) : coh_t<bf16_t, false>(a, x, y, PowerArgs{}, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace blocked
