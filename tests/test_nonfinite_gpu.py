"""Infinities and NaNs in B: the entry kernels give what the sum over a row's stored entries is."""
import os

import numpy as np
import pytest

from test_spmm_gpu import convert, gpu_spmm, torch_cuda  # noqa: F401
from util import decode, encode

pytestmark = pytest.mark.gpu

# kernel mode, environment
FAMILIES = {"entries": (0, {"HSPMM_ENTRIES": "1", "HSPMM_TILE": "0"})}


def _plan(hs, A, family):
    mode, env = FAMILIES[family]
    os.environ.update(env)
    hs.set_kernel_mode(mode)
    try:
        return hs.Plan(convert(hs, A))
    finally:
        hs.set_kernel_mode(0)
        for name in env:
            os.environ.pop(name, None)


def _csr(D, dtype):
    row_ptr = np.concatenate([[0], np.cumsum((D != 0).sum(1))]).astype(np.uint32)
    return dict(rows=D.shape[0], cols=D.shape[1], nnzs=int(row_ptr[-1]), dtype=dtype, row_ptr=row_ptr,
                col_idx=np.nonzero(D)[1].astype(np.uint32), values=encode(D[D != 0].astype(np.float32), dtype))


def _rounded(x, dtype):
    """Exact sums (whole numbers) as the one rounding to the element type leaves them."""
    return decode(encode(x.astype(np.float32), dtype), dtype)


def _stored_sum(D, B):
    """The sum over the stored entries alone, in fp64 (a zero that is not stored meets no infinity)."""
    with np.errstate(invalid="ignore"):
        return np.array([(D[r, D[r] != 0][:, None] * B[D[r] != 0]).sum(0) for r in range(D.shape[0])])


@pytest.mark.parametrize("dtype", [0, 1, 2])
def test_an_infinity_under_a_rows_last_entry_is_multiplied_once(torch_cuda, hs, dtype):
    """Rows of the entry kernels are units of four entries: what fills the last unit up takes no part in the sum."""
    rng = np.random.default_rng(31 + dtype)
    rows, cols = 500, 900
    lengths = [1, 2, 3, 4, 5, 6, 7, 8, 30, 31, 33, 64, 65, 127, 600, 897] + [int(n) for n in rng.integers(1, 20, rows - 16)]
    D = np.zeros((rows, cols))
    for r, n in enumerate(lengths):
        D[r, np.sort(rng.choice(cols - 1, n - 1, replace=False))] = rng.integers(1, 4, n - 1)
        D[r, cols - 1] = -2
    plan = _plan(hs, _csr(D, dtype), "entries")
    for N in (1, 2, 3, 8, 16, 40, 64, 130):
        Bm = rng.integers(-4, 5, (cols, N)).astype(np.float64)
        Bm[cols - 1, 0] = np.inf
        Bm[cols - 1, N // 2] = -np.inf
        Bm[cols - 1, N - 1] = np.inf if N > 1 else -np.inf
        got = decode(gpu_spmm(torch_cuda, hs, dict(dtype=dtype, rows=rows), encode(Bm.astype(np.float32), dtype), N, plan=plan), dtype)
        assert np.array_equal(got, _rounded(_stored_sum(D, Bm), dtype), equal_nan=True), "N=%d" % N
    plan.close()
