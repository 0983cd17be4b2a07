// Host-side launchers of the gfx950 kernels (defined in the k_*.hip files).
// Only plain pointers cross this header; the C ABI layer (api.cpp) owns all
// device buffers and streams.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "k_common.hpp"

namespace pwmk {

enum ValueType { VT_F64 = 0, VT_F32 = 1, VT_BF16 = 2 };

// Device CRS arrays (row_start[N+1], col_ind[Z], values[Z] of `vtype`).
struct CrsDev {
    int64_t nrows = 0, ncols = 0, nnz = 0;
    const int32_t* rs = nullptr;
    const int32_t* ci = nullptr;
    const void* val = nullptr;
    int vtype = VT_F64;
    int nt = 0;  // tiles kernels: non-temporal col_ind / value loads
};

// A slice of one long row handled by one workgroup: entries [k0, k1) of row
// `row`; `slot` is the long-row index the partial sums are gathered under.
struct LongChunk {
    int32_t row, slot;
    int32_t k0, k1;
};

struct LongRows {
    int32_t n_rows = 0;             // long rows
    int32_t n_chunks = 0;           // chunks over all long rows
    const LongChunk* chunks = nullptr;
    const int32_t* row_ids = nullptr;      // [n_rows]
    const int32_t* chunk_begin = nullptr;  // [n_rows+1] first chunk of each long row
    void* chunk_partial = nullptr;         // accumulator-typed [n_chunks]
    int32_t threshold = 1 << 30;           // rows longer than this are long
};

// ---- CRS vector kernel (k_crs.hip) ----------------------------------------
// Short rows: G lanes per row; long rows: chunked, finished by crs_finalize.
hipError_t launch_crs_vector(const CrsDev& A, int G, int n_vec_blocks, const LongRows& lr, const void* x,
                             void* y, const PowerArgs* pw, hipStream_t s);
// Finishes long rows (sum of chunk partials, in chunk order) and, for the
// power method, reduces the per-block partials into step k's record.
hipError_t launch_crs_finalize(const CrsDev& A, int n_partials, const LongRows& lr, void* y,
                               const PowerArgs* pw, hipStream_t s);

// ---- merge path (k_merge.hip) -----------------------------------------------
struct MergePlan {
    int64_t P = 0;                  // tiles (= logical threads of CRS_Merge::mv)
    int64_t items_per_tile = 0;     // ceil((N+Z)/P)
    int ipt = 8;                    // template items per thread (tile capacity 256*ipt)
    int64_t* split_a = nullptr;     // [P+1]
    int64_t* split_b = nullptr;     // [P+1]
    int32_t* carry_row = nullptr;   // [P]
    void* carry_val = nullptr;      // accumulator-typed [P]
};
hipError_t launch_merge_splits(const CrsDev& A, const MergePlan& mp, hipStream_t s);
hipError_t launch_merge_spmv(const CrsDev& A, const MergePlan& mp, const void* x, void* y, const PowerArgs* pw,
                             hipStream_t s);
hipError_t launch_merge_fixup(const CrsDev& A, const MergePlan& mp, void* y, const PowerArgs* pw, hipStream_t s);
// CRS over row-aligned tiles (k_tiles.hip): the tiles are the iteration
// engine's plan (struct ETile, engine.hpp) with tiles_items_per_thread()
// items per thread; carries go through launch_merge_fixup with mp.P = tiles.
struct ETile;
int tiles_items_per_thread();
hipError_t launch_tiles_spmv(const CrsDev& A, const ETile* tiles, const MergePlan& mp, const void* x, void* y,
                             const PowerArgs* pw, hipStream_t s);

// CRS over wave tiles (k_rows.hip), for matrices of short rows: tile t holds
// the rows [cut[t].x, cut[t+1].x) and entries [cut[t].y, cut[t+1].y).
struct RowsPlan {
    int64_t nt = 0;             // tiles (0: no plan)
    const int2* cut = nullptr;  // [nt + 1]
};
// Entries between cuts for this longest row, 0 when it is too long.
int64_t rows_step(int64_t row_max);
int64_t rows_power_blocks(int64_t nt);  // workgroups (partial-sum slots) of a power step
// Cuts of nt = ceil(nnz / step) tiles; sets *too_many_rows when one has more
// rows than the kernel takes.
hipError_t launch_rows_plan(const CrsDev& A, int64_t step, int64_t nt, int2* cut, int* too_many_rows, hipStream_t s);
hipError_t launch_rows(const CrsDev& A, const RowsPlan& rp, const void* x, void* y, const PowerArgs* pw, hipStream_t s);

// Power-mode carry fix-up runs in this many workgroups (each sums its share
// of the tile partials into a second-level slot after the P tile slots).
inline int merge_fix_blocks(int64_t P) {
    const int64_t b = (P + 255) / 256;
    return (int)(b < 1 ? 1 : (b > 256 ? 256 : b));
}

// ---- power method: norms of a step, and small matrices (k_power.hip) --------
// A step of at most kDeferSlots slots can leave its norms to the next one, whose
// blocks add the slots up before they scale.  A launch for it costs about 3 us of
// a step; n blocks that read n slots of 24 bytes each cost nothing that shows up
// to 500 slots and 2 us at 1200.  FP64 Poisson in CRS, us per step: 100 x 100 6.3
// -> 4.3, 300 x 300 7.4 -> 5.0, 600 x 600 11.3 -> 8.5, 700 x 700 (1229 slots)
// 13.0 -> 11.8.
constexpr int64_t kDeferSlots = 1280;
// The n partial-sum slots of step pw.k into its record (slots are overwritten);
// nothing for a step that defers its norms.
hipError_t launch_power_reduce(const PowerArgs& pw, int64_t n, hipStream_t s);
// The slots 0, step, 2 step, ... (n of them) of `slots`, by one workgroup.
hipError_t launch_power_final(const PowerArgs& pw, const double* slots, int64_t n, int64_t step, hipStream_t s);
// The whole loop of a small matrix in one workgroup:
// Steps [k0, min(k0 + nsteps, pw.max_it)) of the power loop; leaves the last
// one's record and step control.
bool power_small_fits(const CrsDev& A, int64_t row_max);
hipError_t launch_power_small(const CrsDev& A, int64_t row_max, const PowerArgs& pw, int64_t k0, int64_t nsteps,
                              hipStream_t s);

// ---- utilities (k_util.hip) -------------------------------------------------
// Util/Poisson.hpp:32-83 on the device, one thread per row.
hipError_t launch_fill_poisson(int64_t m, int64_t n, int32_t* rs, int32_t* ci, void* val, int vtype,
                               hipStream_t s);
// double -> storage type conversion of values.
hipError_t launch_convert_values(const double* src, void* dst, int64_t n, int vtype, hipStream_t s);
// storage type -> double widening of values (exports).
hipError_t launch_copy_values_f64(const void* src, int vtype, double* dst, int64_t n, hipStream_t s);
hipError_t launch_fill(void* p, int64_t n, int is_f64, double v, hipStream_t s);
hipError_t launch_copy_vec(const void* src_f64_or_f32, int src_f64, void* dst, int dst_f64, int64_t n,
                           hipStream_t s);
// Final normalisation of the power method (see api.cpp).
hipError_t launch_power_finish(const PowerArgs& pw, int64_t n, int is_f64, hipStream_t s);
// Rewrite a buffer (Infinity-Cache flush for the roofline timing).
hipError_t launch_flush(void* p, int64_t bytes, hipStream_t s);
// Plain streaming copy (profiler counter calibration).
hipError_t launch_stream_copy(void* dst, const void* src, int64_t bytes, hipStream_t s);
// Bytes between device and pinned host memory.
hipError_t launch_copy_bytes(void* dst, const void* src, size_t bytes, bool to_host, hipStream_t s);
// Distinct lines of 2^shift columns per group of 256 consecutive entries, over
// `groups` groups (nnz >= 256), added to *lines.
hipError_t launch_scatter(const int32_t* ci, int64_t nnz, int64_t groups, int shift, unsigned* lines, hipStream_t s);
// gather-rate probe: entries rounded down to whole workgroups; out holds
// (entries / 8192) * 256 doubles
int64_t gather_probe_entries(int64_t n);
hipError_t launch_gather_fill(uint32_t* idx, double* val, int64_t n, uint32_t window, hipStream_t s);
hipError_t launch_gather_probe(const uint32_t* idx, const double* val, const double* x, double* out, int64_t n,
                               int64_t window, int per_xcd, hipStream_t s);

}  // namespace pwmk
