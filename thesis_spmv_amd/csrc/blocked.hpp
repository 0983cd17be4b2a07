// Device-side descriptions of the CSB and BlockCOH layouts and the launchers
// of their kernels (k_blocked.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "k_common.hpp"

namespace blocked {

// Rows of y are summed in LDS in FP64 whatever the storage type: an LDS atomic
// add of 64 lanes takes 21 clocks in FP64 and 193 in FP32 (ds_add_f32 serves
// one lane after the other; both measured on random rows), which held every
// FP32 kernel here to 180 G entries/s.  Rows per workgroup: a CSB slab 32 KB,
// a BlockCOH band up to 32 KB (FP64 storage) or 64 KB.
constexpr int kCsbLdsRows = 4096;
inline int coh_lds_rows(int vtype) { return vtype == 0 ? 4096 : 8192; }

// A contiguous run [start, end) of CSB entries: the part of one block that
// falls into one workgroup's row slab.
struct Piece {
    int32_t start, end;
};

struct CsbArgs {
    int64_t nor = 0;
    int32_t bits = 0;        // beta = 2^bits
    int64_t H = 0;           // block columns
    int32_t slabs = 1;       // slabs per block row
    int64_t slab_rows = 0;   // beta / slabs
    int32_t np = 1;          // pieces per (block, slab), a power of two
    int32_t np_shift = 0;    // log2(np)
    const uint32_t* ind = nullptr;
    const void* val = nullptr;
    const Piece* pieces = nullptr;  // [slab task][bc][piece]
    int64_t n_tasks = 0;            // slab tasks x column groups
    // Column groups: task t works on slab t / groups and block columns
    // [g*H/groups, (g+1)*H/groups) with g = t % groups.  MI355X dispatches
    // workgroup t to XCD t % 8, so with 8 groups each XCD gathers only from
    // its own eighth of x.  With groups > 1 the slab sums go to
    // ypart[g * nor + row] and k_csb_reduce adds the groups in order.
    int32_t groups = 1;
    void* ypart = nullptr;          // accumulator type, groups * nor
    int vtype = 0;
    // Slab-stream layout: entries of slab task t in block columns [bc0, bc1)
    // are ind/val[soff[t*H + bc0] .. soff[t*H + bc1]), each index packed as
    // (row in slab << col_bits) | column; ind/val extend 4 zero entries past
    // the last one.  slabs/slab_rows describe these slabs; pieces is unused.
    int32_t stream = 0;
    int32_t nt = 0;          // slab streams: non-temporal entry loads and partial-slab stores
    int32_t col_bits = 0;
    const int32_t* soff = nullptr;
    int32_t unroll = 2;  // groups of 4 entries per thread per step: 2 or 4
    // Wide slab streams (wide = 1): ind holds the column itself and srows the
    // row in the slab (u16), for column indices too wide to pack.
    int32_t wide = 0;
    const uint16_t* srows = nullptr;
    // Swept slabs (sweep = 1): n_tasks slabs [sstart[t], sstart[t+1]), one
    // persistent workgroup each with max_rows LDS rows; entries of slab t in
    // column window p are ind/val[soff[t*W + p] .. soff[t*W + p + 1]),
    // packed (row in slab << wb) | column in window.
    int32_t sweep = 0;
    int32_t wb = 0;
    int64_t ww = 0;          // columns per window, at most 2^wb
    int64_t W = 0;
    int32_t max_rows = 0;
    int32_t ord = 0;         // 1: FP64 LDS sums in a fixed order (the CRS formats' sweep)
    int32_t acc32 = 0;       // 1: FP32 LDS sums (FP32 storage whose slabs do not fit in FP64)
    int32_t sync_every = 1;  // windows between workgroup barriers (a power of two)
    const int32_t* sstart = nullptr;
};

// Swept slabs: workgroups of the sweep kernel one CU holds at once with
// `rows` LDS rows, FP64 or (acc32) FP32 (0 if none fit).
int csb_sweep_blocks_per_cu(int vtype, int rows, bool acc32);


// Workgroup size of the blocked kernels.
constexpr int kBlockedBS = 512;

// BlockCOH entries, in the format's order (per band the blocks in Hilbert
// order, inside a block by rows): (first entry of its block) << 31 | row in the
// block << 15 | column in the block, both below beta <= 2^15.  The jumps of the
// format (ICRS inside a block) follow from two neighbours and are formed where
// they are asked for; stored, they cost the same 4 bytes and every SpMV two
// scans over the entries to undo them.
constexpr uint32_t kCohFirst = 0x80000000u;
inline uint32_t coh_pack(uint32_t row, uint32_t col, bool first) { return (first ? kCohFirst : 0u) | row << 15 | col; }

// A block: its first row (inside the band) and column.
struct CohBlock {
    int32_t row, col;
};

// A wave takes kCohStep consecutive entries of a band at a time, 4 per lane.
// The steps of a band begin at its first entry rounded down to a multiple of 4,
// so that a lane's 4 entries are aligned.
constexpr int kCohStep = 256;
__host__ __device__ inline int64_t coh_steps(int64_t entry, int64_t nnz) {
    return nnz > 0 ? (nnz + (entry & 3) + kCohStep - 1) / kCohStep : 0;
}

struct CohBand {
    int32_t start, rows, first_block, blocks, entry, nnz;
    int32_t step_table;  // offset of the band's step -> block table
    int32_t sum;         // atomic bands: the first row's place in CohArgs::ysum
};

// Unit of work of the BlockCOH kernel: steps [step0, step0+nsteps) of one
// band.  A band whose rows fit the LDS window and whose entries fit one task
// accumulates in LDS (atomic = 0); larger bands are cut into several tasks of
// two steps per wave that add into ysum with global atomics (atomic = 1).
constexpr int kCohTaskSteps = 128;
constexpr int kCohAtomicSteps = 16;
struct CohTask {
    int32_t band, step0, nsteps, atomic;
};

// Rows of atomic bands in pieces, one per workgroup of the kernel that finishes
// them; sum: the first row's place in CohArgs::ysum.
constexpr int kCohPieceRows = 2048;
struct CohRows {
    int32_t start, rows, sum;
};

struct CohArgs {
    int64_t nor = 0;
    int64_t n_tasks = 0;
    const CohTask* tasks = nullptr;
    const CohBand* bands = nullptr;
    const CohBlock* blocks = nullptr;
    const int32_t* step_block = nullptr;  // per band and step: the last block that starts before it (-1: none)
    const uint32_t* ent = nullptr;
    const void* val = nullptr;
    const CohRows* pieces = nullptr;
    int64_t n_pieces = 0;
    double* ysum = nullptr;  // rows of atomic bands, zero between two SpMVs
    int vtype = 0;
    int32_t lds_rows = 0;  // LDS window of the kernel: rows of the largest LDS-accumulated band
    int32_t one_wave = 0;  // 1: a task is one wave's, not a workgroup's of 8
};

// part: 0 = the whole SpMV, 1 = the slab kernel only, 2 = the column-group
// reduction only (nothing when groups = 1)
hipError_t launch_csb(const CsbArgs& a, const void* x, void* y, const pwmk::PowerArgs* pw, hipStream_t s,
                      int part = 0);
// workgroups of the CSB column-group reduction (= its power-method partials)
int csb_reduce_blocks(int64_t nor);
hipError_t launch_coh(const CohArgs& a, const void* x, void* y, const pwmk::PowerArgs* pw, hipStream_t s);

}  // namespace blocked
