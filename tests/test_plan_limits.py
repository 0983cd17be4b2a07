"""Plan sizes of matrices too large to load in a test, from the library's own
planning functions (no GPU)."""
import ctypes as C

import pytest

pw = pytest.importorskip("thesis_spmv_amd")
F64, F32, BF16 = 0, 1, 2
MAX_SLOTS = 262133  # PWM_NOALLOC_MAX_SLOTS


def _fn(name, *args):
    f = getattr(pw.lib(), name)
    f.restype, f.argtypes = C.c_int, args
    return f


@pytest.mark.parametrize("vtype", [F32, BF16])
@pytest.mark.parametrize("n", [1 << 28, 1 << 29, 1 << 30, (1 << 30) + 1, 1500000001])
def test_csb_fp32_slab_streams_of_the_tallest_matrices(n, vtype):
    """Square CSB matrices of FP32 vectors keep the slab streams (a 64-bit sort key)
    and the no-allocation power method (a slot per slab)."""
    lds_bits = _fn("_ZN8pwm_impl12csb_lds_bitsEil", C.c_int, C.c_int64)(vtype, n)
    key_bits = _fn("_ZN8pwm_impl12csb_key_bitsEli", C.c_int64, C.c_int)
    bits = 16 if n > 1 << 30 else 15  # the reference's block size
    beta = 1 << bits
    blocks = -(-n // beta)
    slabs = blocks * (beta >> lds_bits)
    assert key_bits(blocks * slabs, bits) <= 64 and slabs <= MAX_SLOTS


@pytest.mark.parametrize("row_max", [1, 5, 33, 60, 64])
def test_wave_tiles_need_no_more_slots_than_merge_tiles(row_max):
    step = _fn("_ZN4pwmk9rows_stepEl", C.c_int64)(row_max)
    blocks = _fn("_ZN4pwmk17rows_power_blocksEl", C.c_int64)
    assert step == 253 - (row_max - 1)
    # the most entries that CRS_MERGE's merge tiles (2048 items, 256 more slots) take
    nnz = min((MAX_SLOTS - 256) * 2048 * row_max // (row_max + 1), 2 ** 31 - 65536)
    for z in (nnz, nnz * 3 // 4, nnz // 2, 1000):
        assert blocks(-(-z // step)) <= MAX_SLOTS
