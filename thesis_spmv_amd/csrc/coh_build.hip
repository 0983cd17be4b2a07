// BlockCOH layout built on the device (SOA_Implementations/BlockCOH.hpp:319-455,
// ICRS inside each block as in Util/TripletToCRS.hpp:402-452).
//
// The bands (a short sequential cut over the row lengths) and their block
// sizes come from the host; everything per entry runs here:
//  1. entry k of row r in band p gets the key  p << 2h | hilbert(r, c)  (the
//     block's Hilbert index on the band's grid, 2h bits enough for every
//     band) and the payload  k << 32 | lrow << 16 | lcol  (row and column
//     inside the block, both below beta <= 2^15);
//  2. a stable radix sort of (key, payload) puts each band's blocks in
//     Hilbert order with the entries of a block in CRS order -- the stable
//     counting sort of the host build;
//  3. per sorted entry, the packed position and the gathered value, and two
//     flags, block start and row start (new block, or another row than the entry
//     before it in the same block: the format's row jumps);
//  4. one inclusive scan of the packed flags numbers the row starts and the
//     blocks, so every block start writes its block in place;
//  5. per block, the block-level BICRS jumps (BlockCOH.hpp:433-439), a flag
//     for each block that starts a block row, and a second scan that places
//     row_jump_block;
//  6. per band, the step -> block table.
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "api_internal.hpp"
#include "blocked.hpp"
#include "kernels.hpp"

namespace pwmk {

// per band, what the build kernels need
struct CohBuildBand {
    int32_t start, rows, beta_bits, hs;  // hs = Hilbert grid side (hsize >> beta_bits, 0 when hsize < beta)
    int32_t H, pad;
    int64_t off_nz;
};

// BlockCOH.hpp:79-114 (Wikipedia xy2d with x = column, y = row; the flip uses
// the full grid side).
__device__ __forceinline__ uint64_t coh_hilbert(int64_t size, int64_t row, int64_t col) {
    uint64_t index = 0;
    for (int64_t s = size / 2; s > 0; s /= 2) {
        const int64_t rr = (row & s) > 0, cr = (col & s) > 0;
        index += (uint64_t)(s * s) * (uint64_t)((3 * cr) ^ rr);
        if (rr == 0) {
            if (cr == 1) {
                col = size - 1 - col;
                row = size - 1 - row;
            }
            const int64_t t = row;
            row = col;
            col = t;
        }
    }
    return index;
}

// the last row r with rs[r] <= k
__device__ __forceinline__ int64_t coh_row_of(const int32_t* __restrict__ rs, int64_t nor, int64_t k) {
    int64_t lo = 0, hi = nor - 1;
    while (lo < hi) {
        const int64_t mid = (lo + hi + 1) >> 1;
        if (rs[mid] <= k)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

struct CohKeyArgs {
    int64_t nor, nnz, n_bands;
    int hb2;  // 2h: bits of the Hilbert part of a key
};

__global__ void k_coh_keys(CohKeyArgs a, const CohBuildBand* __restrict__ bands, const int32_t* __restrict__ rs,
                           const int32_t* __restrict__ ci, uint64_t* __restrict__ keys, uint64_t* __restrict__ pay) {
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < a.nnz; k += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = coh_row_of(rs, a.nor, k);
        // the last band starting at or before r (an empty band shares its
        // start with the next one, which is the one holding the row)
        int64_t lo = 0, hi = a.n_bands - 1;
        while (lo < hi) {
            const int64_t mid = (lo + hi + 1) >> 1;
            if (bands[mid].start <= r)
                lo = mid;
            else
                hi = mid - 1;
        }
        const CohBuildBand b = bands[lo];
        const int64_t lrow = r - b.start, c = ci[k];
        const int64_t mask = ((int64_t)1 << b.beta_bits) - 1;
        const uint64_t h = coh_hilbert(b.hs, lrow >> b.beta_bits, c >> b.beta_bits);
        keys[k] = ((uint64_t)lo << a.hb2) | h;
        pay[k] = ((uint64_t)k << 32) | ((uint64_t)(lrow & mask) << 16) | (uint64_t)(c & mask);
    }
}

__device__ __forceinline__ uint32_t pay_row(uint64_t p) { return (uint32_t)(p >> 16) & 0xffffu; }
__device__ __forceinline__ uint32_t pay_col(uint64_t p) { return (uint32_t)p & 0xffffu; }

// step 3: flags (row start << 32 | block start), the packed position and the value
template <typename E>
__global__ void k_coh_entries(CohKeyArgs a, const uint64_t* __restrict__ keys, const uint64_t* __restrict__ pay,
                              const E* __restrict__ val, uint64_t* __restrict__ flags, uint32_t* __restrict__ ent,
                              E* __restrict__ data) {
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < a.nnz; q += (int64_t)gridDim.x * blockDim.x) {
        const uint64_t key = keys[q], p = pay[q];
        const bool bs = q == 0 || keys[q - 1] != key;
        const bool rsf = bs || pay_row(pay[q - 1]) != pay_row(p);
        ent[q] = (bs ? blocked::kCohFirst : 0u) | pay_row(p) << 15 | pay_col(p);
        data[q] = val[p >> 32];
        flags[q] = ((uint64_t)rsf << 32) | (uint64_t)bs;
    }
}

// step 4: blocks.  With s = inclusive scan of the flags, the block of entry q
// is number (s[q] & 0xffffffff) - 1.
__global__ void k_coh_scatter(CohKeyArgs a, const CohBuildBand* __restrict__ bands, const int32_t* __restrict__ rs,
                              const int32_t* __restrict__ ci, const uint64_t* __restrict__ keys,
                              const uint64_t* __restrict__ pay, const uint64_t* __restrict__ flags,
                              const uint64_t* __restrict__ scan, blocked::CohBlock* __restrict__ blocks,
                              int32_t* __restrict__ block_q, int32_t* __restrict__ block_band) {
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < a.nnz; q += (int64_t)gridDim.x * blockDim.x) {
        if (!(flags[q] & 1)) continue;
        const int64_t band = (int64_t)(keys[q] >> a.hb2);
        const CohBuildBand b = bands[band];
        const int64_t e = (int64_t)(pay[q] >> 32);
        const int64_t r = coh_row_of(rs, a.nor, e);
        const int64_t blk = (int64_t)(scan[q] & 0xffffffffu) - 1;
        blocks[blk] = blocked::CohBlock{(int32_t)((r - b.start) >> b.beta_bits << b.beta_bits),
                                        (int32_t)(ci[e] >> b.beta_bits << b.beta_bits)};
        block_q[blk] = (int32_t)q;
        block_band[blk] = (int32_t)band;
    }
}

// step 5: block-level BICRS jumps, block sizes and the block-row-start flags
__global__ void k_coh_blocks(int64_t total, int64_t nnz, const CohBuildBand* __restrict__ bands,
                             const uint64_t* __restrict__ scan, const blocked::CohBlock* __restrict__ blocks,
                             const int32_t* __restrict__ block_q, const int32_t* __restrict__ block_band,
                             int16_t* __restrict__ col_jump_block, int16_t* __restrict__ rjb_val,
                             uint32_t* __restrict__ row_flag, int32_t* __restrict__ block_nnz) {
    for (int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; b < total; b += (int64_t)gridDim.x * blockDim.x) {
        const CohBuildBand bd = bands[block_band[b]];
        const int64_t first = (int64_t)(scan[bd.off_nz] & 0xffffffffu) - 1;
        const int64_t brow = blocks[b].row >> bd.beta_bits, bcol = blocks[b].col >> bd.beta_bits;
        int64_t cj, rj = 0;
        uint32_t fl = 1;
        if (b == first) {
            rj = brow;
            cj = bcol;
        } else {
            const int64_t prow = blocks[b - 1].row >> bd.beta_bits, pcol = blocks[b - 1].col >> bd.beta_bits;
            if (brow == prow) {
                fl = 0;
                cj = bcol - pcol;
            } else {
                rj = brow - prow;
                cj = bcol - pcol + bd.H;
            }
        }
        col_jump_block[b] = (int16_t)cj;
        rjb_val[b] = (int16_t)rj;
        row_flag[b] = fl;
        block_nnz[b] = (b + 1 < total ? block_q[b + 1] : (int32_t)nnz) - block_q[b];
    }
}

__global__ void k_coh_rjb(int64_t total, const uint32_t* __restrict__ row_flag, const uint32_t* __restrict__ row_scan,
                          const int16_t* __restrict__ rjb_val, int16_t* __restrict__ row_jump_block) {
    for (int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; b < total; b += (int64_t)gridDim.x * blockDim.x)
        if (row_flag[b]) row_jump_block[row_scan[b] - 1] = rjb_val[b];
}

// per band: blocks, row jumps and block-row jumps (zero for an empty band)
__global__ void k_coh_band_counts(int64_t n_bands, const CohBuildBand* __restrict__ bands,
                                  const int64_t* __restrict__ band_nnz, const uint64_t* __restrict__ scan,
                                  const uint32_t* __restrict__ row_scan, int32_t* __restrict__ out) {
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n_bands; p += (int64_t)gridDim.x * blockDim.x) {
        const int64_t n = band_nnz[p];
        int32_t nb = 0, nrj = 0, nrjb = 0;
        if (n > 0) {
            const uint64_t s0 = scan[bands[p].off_nz], s1 = scan[bands[p].off_nz + n - 1];
            const int64_t b0 = (int64_t)(s0 & 0xffffffffu) - 1, b1 = (int64_t)(s1 & 0xffffffffu) - 1;
            nb = (int32_t)(b1 - b0 + 1);
            nrj = (int32_t)((s1 >> 32) - (s0 >> 32) + 1);
            nrjb = (int32_t)(row_scan[b1] - row_scan[b0] + 1);
        }
        out[3 * p] = nb;
        out[3 * p + 1] = nrj;
        out[3 * p + 2] = nrjb;
    }
}

// step 6: the last block of band p that starts before step i of the band (-1:
// none)
__global__ void k_coh_steps(int64_t n_bands, const blocked::CohBand* __restrict__ table,
                            const int32_t* __restrict__ block_q, int32_t* __restrict__ stab) {
    for (int64_t p = blockIdx.x; p < n_bands; p += gridDim.x) {
        const blocked::CohBand bd = table[p];
        const int64_t steps = blocked::coh_steps(bd.entry, bd.nnz);
        const int32_t* __restrict__ bq = block_q + bd.first_block;
        for (int64_t i = threadIdx.x; i < steps; i += blockDim.x) {
            const int64_t q = (bd.entry & ~3) + i * blocked::kCohStep;
            int64_t lo = 0, hi = bd.blocks;  // blocks starting before q: in [lo, hi]
            while (lo < hi) {
                const int64_t mid = (lo + hi) >> 1;
                if (bq[mid] < q)
                    lo = mid + 1;
                else
                    hi = mid;
            }
            stab[bd.step_table + i] = (int32_t)lo - 1;
        }
    }
}

static unsigned grid_of(int64_t n) {
    const int64_t b = (n + 255) / 256;
    return (unsigned)(b < 8192 ? (b > 0 ? b : 1) : 8192);
}

}  // namespace pwmk

namespace pwm_impl {

int coh_layout_device(pwm_matrix* h, int64_t lds_rows) {
    CohDev& c = h->coh;
    std::vector<CohBandMeta>& B = c.bands;
    const int64_t P = (int64_t)B.size(), nnz = h->nnz, nor = h->nor, noc = h->noc;
    const size_t vs = value_size(h->vtype);
    hipError_t e;
    // host side of step 1: the band table and the width of the Hilbert part
    std::vector<pwmk::CohBuildBand> bb(P);
    std::vector<int64_t> band_nnz(P);
    int hbits = 0;
    for (int64_t p = 0; p < P; ++p) {
        const CohBandMeta& m = B[p];
        int lg = 0;
        while (((int64_t)1 << lg) < std::max(m.rows, noc)) ++lg;  // hsize = 2^lg (BlockCOH.hpp:401)
        const int hs_bits = lg >= m.beta_bits ? lg - m.beta_bits : -1;
        bb[p] = pwmk::CohBuildBand{(int32_t)m.start, (int32_t)m.rows, m.beta_bits, hs_bits >= 0 ? (1 << hs_bits) : 0,
                                   m.H, 0, m.off_nz};
        band_nnz[p] = m.nnz;
        hbits = std::max(hbits, hs_bits);
    }
    int pbits = 0;
    while (((int64_t)1 << pbits) < P) ++pbits;
    pwmk::CohKeyArgs ka{nor, nnz, P, 2 * hbits};

    const int64_t zpad = std::max<int64_t>(nnz, 1) + 64;
    if ((e = c.ent.alloc(zpad * 4)) != hipSuccess || (e = c.data.alloc(zpad * vs)) != hipSuccess)
        return hip_fail(h, e, "BlockCOH allocation");
    if ((e = hipMemsetAsync(c.ent.p, 0, zpad * 4, h->stream)) != hipSuccess ||
        (e = hipMemsetAsync(c.data.p, 0, zpad * vs, h->stream)) != hipSuccess)
        return hip_fail(h, e, "BlockCOH allocation");

    DevBuf d_bands, d_bnnz, keys, keys_out, pay, pay_out, tmp, block_q, block_band, rjb_val, row_flag, row_scan,
        d_counts;
    std::vector<int32_t> counts(3 * std::max<int64_t>(P, 1), 0);
    int64_t total = 0;
    if ((e = d_bands.alloc(P * sizeof(pwmk::CohBuildBand))) != hipSuccess ||
        (e = hipMemcpy(d_bands.p, bb.data(), P * sizeof(pwmk::CohBuildBand), hipMemcpyHostToDevice)) != hipSuccess)
        return hip_fail(h, e, "BlockCOH band table");
    if (nnz > 0) {
        if ((e = keys.alloc(nnz * 8)) != hipSuccess || (e = keys_out.alloc(nnz * 8)) != hipSuccess ||
            (e = pay.alloc(nnz * 8)) != hipSuccess || (e = pay_out.alloc(nnz * 8)) != hipSuccess)
            return hip_fail(h, e, "BlockCOH build allocation");
        const dim3 g(pwmk::grid_of(nnz)), t(256);
        hipLaunchKernelGGL(pwmk::k_coh_keys, g, t, 0, h->stream, ka, d_bands.as<pwmk::CohBuildBand>(),
                           h->rs.as<int32_t>(), h->ci.as<int32_t>(), keys.as<uint64_t>(), pay.as<uint64_t>());
        if ((e = hipGetLastError()) != hipSuccess) return hip_fail(h, e, "BlockCOH keys");
        const unsigned end_bit = (unsigned)std::max(pbits + 2 * hbits, 1);
        size_t tb = 0;
        e = rocprim::radix_sort_pairs(nullptr, tb, keys.as<uint64_t>(), keys_out.as<uint64_t>(), pay.as<uint64_t>(),
                                      pay_out.as<uint64_t>(), (size_t)nnz, 0u, end_bit, h->stream);
        if (e == hipSuccess) e = tmp.alloc(std::max<size_t>(tb, 4));
        if (e == hipSuccess)
            e = rocprim::radix_sort_pairs(tmp.p, tb, keys.as<uint64_t>(), keys_out.as<uint64_t>(), pay.as<uint64_t>(),
                                          pay_out.as<uint64_t>(), (size_t)nnz, 0u, end_bit, h->stream);
        if (e != hipSuccess) return hip_fail(h, e, "BlockCOH sort");
        // keys / pay now hold the flags and their scan
        uint64_t* flags = keys.as<uint64_t>();
        uint64_t* scan = pay.as<uint64_t>();
        if (vs == 8)
            hipLaunchKernelGGL(pwmk::k_coh_entries<uint64_t>, g, t, 0, h->stream, ka, keys_out.as<uint64_t>(),
                               pay_out.as<uint64_t>(), h->val.as<uint64_t>(), flags, c.ent.as<uint32_t>(),
                               c.data.as<uint64_t>());
        else if (vs == 4)
            hipLaunchKernelGGL(pwmk::k_coh_entries<uint32_t>, g, t, 0, h->stream, ka, keys_out.as<uint64_t>(),
                               pay_out.as<uint64_t>(), h->val.as<uint32_t>(), flags, c.ent.as<uint32_t>(),
                               c.data.as<uint32_t>());
        else
            hipLaunchKernelGGL(pwmk::k_coh_entries<uint16_t>, g, t, 0, h->stream, ka, keys_out.as<uint64_t>(),
                               pay_out.as<uint64_t>(), h->val.as<uint16_t>(), flags, c.ent.as<uint32_t>(),
                               c.data.as<uint16_t>());
        if ((e = hipGetLastError()) != hipSuccess) return hip_fail(h, e, "BlockCOH entries");
        tb = 0;
        e = rocprim::inclusive_scan(nullptr, tb, flags, scan, (size_t)nnz, rocprim::plus<uint64_t>(), h->stream);
        if (e == hipSuccess && tb > tmp.bytes) {
            tmp.release();
            e = tmp.alloc(tb);
        }
        if (e == hipSuccess)
            e = rocprim::inclusive_scan(tmp.p, tb, flags, scan, (size_t)nnz, rocprim::plus<uint64_t>(), h->stream);
        uint64_t last = 0;
        if (e == hipSuccess) e = hipMemcpyAsync(&last, scan + nnz - 1, 8, hipMemcpyDeviceToHost, h->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
        if (e != hipSuccess) return hip_fail(h, e, "BlockCOH scan");
        total = (int64_t)(last & 0xffffffffu);
        c.total_blocks = total;
        if ((e = c.block_coords.alloc(total * sizeof(blocked::CohBlock))) != hipSuccess ||
            (e = c.block_nnz.alloc(total * 4)) != hipSuccess || (e = c.col_jump_block.alloc(total * 2)) != hipSuccess ||
            (e = c.row_jump_block.alloc(total * 2)) != hipSuccess || (e = block_q.alloc(total * 4)) != hipSuccess ||
            (e = block_band.alloc(total * 4)) != hipSuccess || (e = rjb_val.alloc(total * 2)) != hipSuccess ||
            (e = row_flag.alloc(total * 4)) != hipSuccess || (e = row_scan.alloc(total * 4)) != hipSuccess ||
            (e = d_bnnz.alloc(P * 8)) != hipSuccess || (e = d_counts.alloc(3 * P * 4)) != hipSuccess)
            return hip_fail(h, e, "BlockCOH block allocation");
        hipLaunchKernelGGL(pwmk::k_coh_scatter, g, t, 0, h->stream, ka, d_bands.as<pwmk::CohBuildBand>(),
                           h->rs.as<int32_t>(), h->ci.as<int32_t>(), keys_out.as<uint64_t>(), pay_out.as<uint64_t>(),
                           flags, scan, c.block_coords.as<blocked::CohBlock>(),
                           block_q.as<int32_t>(), block_band.as<int32_t>());
        const dim3 gb(pwmk::grid_of(total));
        hipLaunchKernelGGL(pwmk::k_coh_blocks, gb, t, 0, h->stream, total, nnz, d_bands.as<pwmk::CohBuildBand>(),
                           scan, c.block_coords.as<blocked::CohBlock>(), block_q.as<int32_t>(),
                           block_band.as<int32_t>(), c.col_jump_block.as<int16_t>(), rjb_val.as<int16_t>(),
                           row_flag.as<uint32_t>(), c.block_nnz.as<int32_t>());
        if ((e = hipGetLastError()) != hipSuccess) return hip_fail(h, e, "BlockCOH blocks");
        tb = 0;
        e = rocprim::inclusive_scan(nullptr, tb, row_flag.as<uint32_t>(), row_scan.as<uint32_t>(), (size_t)total,
                                    rocprim::plus<uint32_t>(), h->stream);
        if (e == hipSuccess && tb > tmp.bytes) {
            tmp.release();
            e = tmp.alloc(tb);
        }
        if (e == hipSuccess)
            e = rocprim::inclusive_scan(tmp.p, tb, row_flag.as<uint32_t>(), row_scan.as<uint32_t>(), (size_t)total,
                                        rocprim::plus<uint32_t>(), h->stream);
        if (e != hipSuccess) return hip_fail(h, e, "BlockCOH block scan");
        hipLaunchKernelGGL(pwmk::k_coh_rjb, gb, t, 0, h->stream, total, row_flag.as<uint32_t>(),
                           row_scan.as<uint32_t>(), rjb_val.as<int16_t>(), c.row_jump_block.as<int16_t>());
        if ((e = hipMemcpyAsync(d_bnnz.p, band_nnz.data(), P * 8, hipMemcpyHostToDevice, h->stream)) != hipSuccess)
            return hip_fail(h, e, "BlockCOH band counts");
        hipLaunchKernelGGL(pwmk::k_coh_band_counts, dim3(pwmk::grid_of(P)), t, 0, h->stream, P,
                           d_bands.as<pwmk::CohBuildBand>(), d_bnnz.as<int64_t>(), scan, row_scan.as<uint32_t>(),
                           d_counts.as<int32_t>());
        if ((e = hipGetLastError()) == hipSuccess)
            e = hipMemcpyAsync(counts.data(), d_counts.p, 3 * P * 4, hipMemcpyDeviceToHost, h->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
        if (e != hipSuccess) return hip_fail(h, e, "BlockCOH band counts");
    }
    // band metadata, the kernel's band table and the step-table offsets
    std::vector<blocked::CohBand> table(P);
    int64_t off_blk = 0, off_rjb = 0, off_stab = 0;
    for (int64_t p = 0; p < P; ++p) {
        CohBandMeta& m = B[p];
        m.blocks = counts[3 * p];
        m.row_jumps = counts[3 * p + 1];
        m.block_row_jumps = counts[3 * p + 2];
        m.off_blk = off_blk;
        m.off_rjb = off_rjb;
        off_blk += m.blocks;
        off_rjb += m.block_row_jumps;
        blocked::CohBand& t = table[p];
        t.start = (int32_t)m.start;
        t.rows = (int32_t)m.rows;
        t.first_block = (int32_t)m.off_blk;
        t.blocks = (int32_t)m.blocks;
        t.entry = (int32_t)m.off_nz;
        t.nnz = (int32_t)m.nnz;
        t.step_table = (int32_t)off_stab;
        off_stab += blocked::coh_steps(m.off_nz, m.nnz);
    }
    if (off_blk != total) return fail(h, PWM_ERR_HIP, "BlockCOH build: band block counts disagree");
    std::vector<blocked::CohTask> tasks;
    std::vector<blocked::CohRows> pieces;
    coh_plan_tasks(B, lds_rows, tasks, pieces, table, &c.lds_rows);
    c.n_tasks = (int64_t)tasks.size();
    if ((e = c.band_table.alloc(P * sizeof(blocked::CohBand))) != hipSuccess ||
        (e = hipMemcpy(c.band_table.p, table.data(), P * sizeof(blocked::CohBand), hipMemcpyHostToDevice)) !=
            hipSuccess ||
        (e = c.tasks.alloc(off_stab * 4)) != hipSuccess ||
        (e = c.task_list.alloc(tasks.size() * sizeof(blocked::CohTask))) != hipSuccess ||
        (!tasks.empty() && (e = hipMemcpy(c.task_list.p, tasks.data(), tasks.size() * sizeof(blocked::CohTask),
                                          hipMemcpyHostToDevice)) != hipSuccess) ||
        (e = c.row_pieces.alloc(pieces.size() * sizeof(blocked::CohRows))) != hipSuccess ||
        (!pieces.empty() && (e = hipMemcpy(c.row_pieces.p, pieces.data(), pieces.size() * sizeof(blocked::CohRows),
                                           hipMemcpyHostToDevice)) != hipSuccess) ||
        (e = coh_clear_sums(h, pieces)) != hipSuccess)
        return hip_fail(h, e, "BlockCOH tables");
    if (nnz > 0)
        hipLaunchKernelGGL(pwmk::k_coh_steps, dim3((unsigned)std::min<int64_t>(std::max<int64_t>(P, 1), 8192)), dim3(256),
                           0, h->stream, P, c.band_table.as<blocked::CohBand>(), block_q.as<int32_t>(),
                           c.tasks.as<int32_t>());
    if ((e = hipGetLastError()) == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) return hip_fail(h, e, "BlockCOH step tables");
    drop_crs(h);
    return PWM_OK;
}

}  // namespace pwm_impl
