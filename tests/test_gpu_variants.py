"""Kernel variants at the sizes where they can go wrong (edges of tiles, remainders, the smallest
and largest of their range), against the CPU oracle or a plain FP64 reference."""
import ctypes

import numpy as np
import pytest

import oracle as orc
import utopia_amd as ua

pytestmark = pytest.mark.gpu


def P(d):
    return ctypes.c_void_p(d.ptr)


def _rows_of_lengths(lengths, ncols, seed):
    rng = np.random.default_rng(seed)
    rp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(ncols, k, replace=False)) for k in lengths]).astype(np.int32)
    return ua.Csr(rp, col, rng.standard_normal(col.size), (len(lengths), ncols))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("block_nnz", [1024, 2048])
def test_row_block_sums_in_column_order_at_every_length_and_alignment(ctx, dtype, block_nnz):
    # every length up to five 16-entry steps (one row after the other, so each LDS alignment
    # occurs), and the longest rows that one lane sums alone
    lengths = list(range(0, 83)) + [block_nnz + block_nnz // 4 - k for k in range(4)] + [1, 0, 35]
    A = _rows_of_lengths(lengths, 6000, 5)
    x = ua.gen_uniform(6, A.shape[1]).astype(dtype)
    D = ua.DeviceCsr(ctx, A, dtype, block_nnz)
    xd, yd = ua.DeviceArray.from_numpy(ctx, x), ua.DeviceArray(ctx, A.shape[0], dtype)
    D.spmv(xd, yd)
    ref = orc.spmv(A, x) if dtype == np.float64 else orc.spmv_f32(A, x)
    assert np.array_equal(yd.numpy(), ref)
