// Device-side helpers shared by the gfx950 kernels: storage/arithmetic types,
// wavefront reductions with DPP, and the XCD-aware block-to-work mapping.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pwmk {

// Storage type for BF16 matrix values (upper half of an IEEE float).
struct bf16_t {
    uint16_t u;
};

// Vector (x, y) and per-row accumulator types for each value storage type:
// FP64 values use FP64 vectors and FP64 accumulation; FP32 and BF16 values
// use FP32 vectors and FP32 accumulation.
template <typename VT> struct Arith;
template <> struct Arith<double> { using X = double; using A = double; };
template <> struct Arith<float> { using X = float; using A = float; };
template <> struct Arith<bf16_t> { using X = float; using A = float; };

__device__ __forceinline__ double widen(double v) { return v; }
__device__ __forceinline__ float widen(float v) { return v; }
__device__ __forceinline__ float widen(bf16_t v) { return __uint_as_float(((uint32_t)v.u) << 16); }

// ---- DPP lane exchange ---------------------------------------------------
// dpp_ctrl encodings (GCN3/CDNA): quad_perm = 0x00..0xFF,
// row_mirror = 0x140, row_half_mirror = 0x141.
template <int CTRL>
__device__ __forceinline__ int dpp_i32(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}
template <int CTRL>
__device__ __forceinline__ int dpp(int v) {
    return dpp_i32<CTRL>(v);
}
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(dpp_i32<CTRL>(__float_as_int(v)));
}
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
    long long b = __double_as_longlong(v);
    int lo = dpp_i32<CTRL>((int)(b & 0xffffffffll));
    int hi = dpp_i32<CTRL>((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// ds_swizzle in bit-mask mode: lane i reads lane (i ^ 16) inside each
// 32-lane half (and_mask 0x1f, or_mask 0, xor_mask 0x10).
__device__ __forceinline__ int swz16(int v) { return __builtin_amdgcn_ds_swizzle(v, 0x401F); }
__device__ __forceinline__ float swz16(float v) {
    return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x401F));
}
__device__ __forceinline__ double swz16(double v) {
    long long b = __double_as_longlong(v);
    int lo = __builtin_amdgcn_ds_swizzle((int)(b & 0xffffffffll), 0x401F);
    int hi = __builtin_amdgcn_ds_swizzle((int)(b >> 32), 0x401F);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Sum over aligned groups of G lanes (G = 1..64); every lane of a group ends
// with the group total.  Steps: xor 1 and xor 2 inside a quad (quad_perm),
// 4 via row_half_mirror, 8 via row_mirror (after the previous steps all lanes
// of a sub-group hold the same value, so a mirror is as good as an xor),
// 16 via ds_swizzle and 32 via ds_bpermute.  All 64 lanes must be active.
template <int G, typename T>
__device__ __forceinline__ T group_sum(T v) {
    if constexpr (G >= 2) v += dpp<0xB1>(v);   // quad_perm [1,0,3,2]
    if constexpr (G >= 4) v += dpp<0x4E>(v);   // quad_perm [2,3,0,1]
    if constexpr (G >= 8) v += dpp<0x141>(v);  // row_half_mirror
    if constexpr (G >= 16) v += dpp<0x140>(v); // row_mirror
    if constexpr (G >= 32) v += swz16(v);
    if constexpr (G >= 64) v += __shfl_xor(v, 32);
    return v;
}

// Block-wide FP64 sum of one value per thread in a fixed order (wave sums,
// then the waves' sums in wave order).  `scratch` holds >= 16 doubles.
// Result valid in every thread.
template <int BS>
__device__ __forceinline__ double block_sum(double v, double* scratch) {
    v = group_sum<64>(v);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) scratch[wave] = v;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < BS / 64; ++w) t += scratch[w];
    __syncthreads();
    return t;
}

// Global-address-space view of a device pointer.  Pointers read from memory
// (job descriptors) are otherwise generic, and generic (flat) accesses count
// against the LDS/scalar wait counter as well, so every LDS wait would also
// drain all outstanding global loads.
template <typename T>
using gptr = __attribute__((address_space(1))) T*;
template <typename T>
__device__ __forceinline__ gptr<T> G(T* p) {
    return (gptr<T>)p;
}

// Three block sums in one pass (same order as three block_sum calls).
// `scratch` holds >= 48 doubles.
template <int BS>
__device__ __forceinline__ void block_sum3(double& a, double& b, double& c, double* scratch) {
    a = group_sum<64>(a);
    b = group_sum<64>(b);
    c = group_sum<64>(c);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        scratch[wave] = a;
        scratch[16 + wave] = b;
        scratch[32 + wave] = c;
    }
    __syncthreads();
    double ta = 0.0, tb = 0.0, tc = 0.0;
#pragma unroll
    for (int w = 0; w < BS / 64; ++w) {
        ta += scratch[w];
        tb += scratch[16 + w];
        tc += scratch[32 + w];
    }
    __syncthreads();
    a = ta;
    b = tb;
    c = tc;
}

// Sum of the products prod[k], prod[k + stride], ... below e, in LDS, by one lane
// with four reads in flight.  FP64: left to right.  FP32 products are summed in
// FP64, but 16 at a time as four FP32 sums of four, since the conversions and FP64
// adds of a long row show (FP32 SpMV of rows of 64, us, all in FP64, so, and left
// to right in FP32: 20 000 rows 7.4 6.6 6.8, 300 000 rows 84.2 83.4 83.9; Poisson
// 3000 x 3000 84.9 86.7 84.8, 5000 x 5000 230 230 231; 100 power steps of one
// workgroup at 37 x 29 195 195 190).  A left-to-right FP32 sum is less exact than
// the lane trees of the vector and merge kernels: rms error over sum |a x| of a row
// of 8 / 16 / 64 3.1e-8 / 3.0e-8 / 2.9e-8, there 2.5e-8 / 2.1e-8 / 1.3e-8 and
// 2.9e-8 / 2.5e-8 / 1.5e-8; here 1.8e-8 / 2.0e-8 / 1.0e-8.
template <typename Acc>
__device__ __forceinline__ double row_sum(const Acc* prod, int k, int e, int stride) {
    double sum = 0.0;
    if constexpr (sizeof(Acc) == 4) {
        for (; k + 15 * stride < e; k += 16 * stride) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const Acc* p = prod + k + 4 * u * stride;
                sum += (double)((p[0] + p[stride]) + (p[2 * stride] + p[3 * stride]));
            }
        }
    }
    for (; k + 3 * stride < e; k += 4 * stride) {
        const Acc p0 = prod[k], p1 = prod[k + stride], p2 = prod[k + 2 * stride], p3 = prod[k + 3 * stride];
        if constexpr (sizeof(Acc) == 4) {
            sum += ((double)p0 + (double)p1) + ((double)p2 + (double)p3);
        } else {
            sum += p0;
            sum += p1;
            sum += p2;
            sum += p3;
        }
    }
    for (; k < e; k += stride) sum += (double)prod[k];
    return sum;
}

// MI355X dispatches consecutive workgroups round-robin over its 8 XCDs, each
// with its own 4 MB L2.  Renumber blocks so that XCD j works on the j-th
// contiguous eighth of the work items: neighbouring rows (which share x
// entries, e.g. the +-m neighbours of a stencil) then meet in the same L2.
__device__ __forceinline__ int64_t xcd_remap(int64_t b, int64_t nblocks) {
    constexpr int64_t kXcd = 8;
    if (nblocks < kXcd) return b;
    const int64_t per = nblocks / kXcd, extra = nblocks % kXcd;
    const int64_t xcd = b % kXcd, slot = b / kXcd;
    // XCD j owns per (+1 for the first `extra` XCDs) consecutive items
    return xcd * per + (xcd < extra ? xcd : extra) + slot;
}

// Renumbering in stretches of 8 C blocks: inside a stretch XCD j works on the
// j-th run of C consecutive items, so the chip reads one front of 8 C items
// while neighbouring items still meet in an L2.  The blocks beyond the last
// whole stretch are spread over the XCDs by xcd_remap.
__device__ __forceinline__ int64_t xcd_chunked(int64_t b, int64_t nblocks, int64_t C) {
    const int64_t stretch = 8 * C, s0 = b / stretch * stretch;
    if (s0 + stretch > nblocks) return s0 + xcd_remap(b - s0, nblocks - s0);
    const int64_t r = b - s0;
    return s0 + (r % 8) * C + r / 8;
}

// One step of the device-side power method.  The host issues the steps in
// order and passes each its number, so that a step's vectors are known without
// reading device memory; only a stop test (tol >= 0) can end the loop early.
struct PowerArgs {
    void* buf0;        // ping-pong vectors: step k reads buf[k&1], writes buf[(k+1)&1]
    void* buf1;
    int* ctrl;         // ctrl[0] = steps done, ctrl[1] = done flag, then (ctrl + 4) lambda and |y|^2 of the last step
    double* rec;       // rec[4k..4k+3] = |y|^2, x^T y, x^T x, lambda of step k
    double* partials;  // per-block FP64 partial sums (3 per block)
    int64_t max_it;
    double tol;        // < 0: never stop early
    int64_t k;         // this step
    // Deferred norms (tol < 0, few slots): a step leaves its partial sums, and
    // the blocks of the next step add up the previous step's prev_n slots
    // themselves (prev_n = 0: its record is complete).
    bool defer;
    const double* prev;
    int64_t prev_n;
};

// An earlier step met the stop test: this one does nothing.
__device__ __forceinline__ bool power_done(const PowerArgs& p) { return p.tol >= 0.0 && p.k > 0 && p.ctrl[1]; }

// Step k's record, stop test and step count, from its |y|^2, x^T y and x^T x
// (one thread).
__device__ __forceinline__ void power_record(const PowerArgs& pw, int64_t k, double yy, double xy, double xx) {
    const double lam = xy / xx;
    pw.rec[4 * k + 0] = yy;
    pw.rec[4 * k + 1] = xy;
    pw.rec[4 * k + 2] = xx;
    pw.rec[4 * k + 3] = lam;
    int done = (k + 1 >= pw.max_it);
    if (pw.tol >= 0.0 && k >= 1) {
        const double prev = pw.rec[4 * (k - 1) + 3];
        if (fabs(lam - prev) <= pw.tol * fabs(lam)) done = 1;
    }
    pw.ctrl[0] = (int)(k + 1);
    pw.ctrl[1] = done;
    double* result = (double*)(pw.ctrl + 4);
    result[0] = lam;
    result[1] = yy;
}

constexpr int kPsU = 4;  // slots a thread loads together

// Sum of the slots i0, i0 + stride, ... < end of this thread, in that order.
__device__ __forceinline__ void slot_sum(const double* slots, int64_t i0, int64_t stride, int64_t end, double& yy,
                                         double& xy, double& xx) {
    for (int64_t i = i0; i < end; i += kPsU * stride) {
        double a[kPsU], b[kPsU], c[kPsU];
#pragma unroll
        for (int u = 0; u < kPsU; ++u) {
            const int64_t j = i + u * stride;
            const bool ok = j < end;
            a[u] = ok ? slots[3 * j + 0] : 0.0;
            b[u] = ok ? slots[3 * j + 1] : 0.0;
            c[u] = ok ? slots[3 * j + 2] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < kPsU; ++u) {
            yy += a[u];
            xy += b[u];
            xx += c[u];
        }
    }
}

// |y_{k-1}|^2 (1 for the first step, which multiplies the caller's unnormalised
// start vector; the step's output is divided by the root of it): from the record
// of step k-1 or, deferred, from its slots, which every block of the kernel adds up
// in the same order (BS decides it: a step's other kernels take the record); block 0
// then writes the record.  All BS threads of the block call it; `scratch` holds >=
// 48 doubles.
template <int BS>
__device__ __forceinline__ double last_norm(const PowerArgs& p, double* scratch) {
    if (p.prev_n == 0) return p.k == 0 ? 1.0 : p.rec[4 * (p.k - 1)];
    double yy = 0.0, xy = 0.0, xx = 0.0;
    slot_sum(p.prev, threadIdx.x, BS, p.prev_n, yy, xy, xx);
    if (blockIdx.x == 0) {
        block_sum3<BS>(yy, xy, xx, scratch);
        if (threadIdx.x == 0) power_record(p, p.k - 1, yy, xy, xx);
    } else {
        yy = block_sum<BS>(yy, scratch);
    }
    return yy;
}

// The scale from the record, for steps that do not defer their norms.  (Kernels
// of many short workgroups have an instance of their own for deferred steps: the
// choice at run time, with its barrier, held up the first loads of every
// workgroup, FP64 Poisson 5000 x 5000 in CRS 358 -> 376 us a step.)
__device__ __forceinline__ double recorded_scale(const PowerArgs& p) {
    return p.k == 0 ? 1.0 : 1.0 / sqrt(p.rec[4 * (p.k - 1)]);
}

}  // namespace pwmk
