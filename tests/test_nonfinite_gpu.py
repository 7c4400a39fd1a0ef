"""An infinity or a NaN in row k of B reaches, in every kernel family, only outputs whose unit of windows names column k;
where the kernels multiply stored entries only - entry and full-tile kernels - only rows with an entry in column k, and
those get what the sum over their stored entries is.  Everything else is the product without it."""
import os

import numpy as np
import pytest

from test_spmm_gpu import convert, gpu_spmm, torch_cuda  # noqa: F401
from util import decode, encode

pytestmark = pytest.mark.gpu

# kernel mode, environment, feature dimensions, main kernel
FAMILIES = {
    "all-shapes": (1, {}, (9, 33), "spmm_scalar_kernel"),
    "gather": (3, {}, (16, 33, 64, 136), "spmm_mfma_kernel"),
    "panel": (4, {}, (128, 200), "spmm_panel_kernel"),
    "panel, fp32 products": (5, {}, (128, 200), "spmm_panel_kernel"),
    "entries": (0, {"HSPMM_ENTRIES": "1", "HSPMM_TILE": "0"}, (9, 16, 33, 64, 130), "spmm_entries_kernel"),
    "tile": (0, {"HSPMM_TILE": "1"}, (9, 16, 24, 33, 64, 100, 127), "spmm_tile_kernel"),
}


def _plan(hs, A, family):
    mode, env = FAMILIES[family][:2]
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


def _near(D, k):
    """Rows of a window that names column k and of the three effective windows on both sides (units of up to four)."""
    rows = D.shape[0]
    windows = -(-rows // 8)
    padded = np.zeros((windows * 8, D.shape[1]))
    padded[:rows] = D
    effective = [w for w in range(windows) if (padded[8 * w:8 * w + 8] != 0).any()]
    out = np.zeros(windows * 8, bool)
    for i, w in enumerate(effective):
        if (padded[8 * w:8 * w + 8, k] != 0).any():
            for j in effective[max(0, i - 3):i + 4]:
                out[8 * j:8 * j + 8] = True
    return out[:rows]


# (700 columns: C tiles of the full-tile kernels cut between workgroups; 130: several whole ones per workgroup)
@pytest.mark.parametrize("family", list(FAMILIES))
@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("rows,cols", [(600, 700), (1100, 130)])
def test_infinities_and_nans_stay_with_the_rows_that_name_them(torch_cuda, hs, family, dtype, rows, cols):
    rng = np.random.default_rng(rows + dtype)
    D = rng.integers(1, 4, (rows, cols)) * rng.choice([-1, 1], (rows, cols)) * (rng.random((rows, cols)) < 0.05)
    D[40:75] = 0                                        # rows and windows without entries
    D[256:384] = 0                                      # a whole block of 128 rows
    unnamed = (50, cols - 3)
    D[:, unnamed] = 0
    named = (5, 63, 64, cols - 1)
    for k in named:
        D[:, k] = 0
        D[rng.choice(np.r_[0:40, 80:200, 400:rows], 12, replace=False), k] = 2
    plan = _plan(hs, _csr(D, dtype), family)
    strict = family in ("entries", "tile")
    for N in FAMILIES[family][2]:
        Bm = rng.integers(-4, 5, (cols, N)).astype(np.float64)
        clean = _rounded(D @ Bm, dtype)
        bad, pairs = {}, {}                             # feature -> rows of B
        for f, (k, v) in enumerate([(unnamed[0], np.inf), (unnamed[1], np.nan), (named[0], np.inf), (named[1], -np.inf),
                                    (named[2], np.nan), (named[3], np.inf)]):
            Bm[k, f] = v
            bad.setdefault(f, []).append(k)
        Bm[named[0], N - 1], Bm[named[1], N - 1] = np.inf, -np.inf
        bad.setdefault(N - 1, []).extend([named[0], named[1]])
        if family == "gather" and dtype != 1:           # (two adjacent features of a 16-bit type are one operand word)
            for f in list(bad):
                for pair in (f - 1, f + 1):
                    if 0 <= pair < N:
                        pairs.setdefault(pair, []).extend(bad[f])
        got = decode(gpu_spmm(torch_cuda, hs, dict(dtype=dtype, rows=rows), encode(Bm.astype(np.float32), dtype), N, plan=plan), dtype)
        assert plan.last_kernel() == FAMILIES[family][3]
        want = _rounded(_stored_sum(D, Bm), dtype)
        what = "%s, dtype %d, N=%d" % (family, dtype, N)
        fine = [f for f in range(N) if f not in bad and f not in pairs]
        assert np.array_equal(got[:, fine], clean[:, fine]), what
        for f in set(pairs) - set(bad):
            reach = np.any([_near(D, k) for k in pairs[f]], axis=0)
            assert np.array_equal(got[~reach, f], clean[~reach, f]), what + ": feature %d beside one that is not finite" % f
        for f, ks in bad.items():
            ks = ks + pairs.get(f, [])
            names = (D[:, bad[f]] != 0).any(1)
            reach = names if strict else np.any([_near(D, k) for k in ks], axis=0)
            # (the features of an unnamed row have no reach at all; the row of B that is not finite counts for nothing elsewhere)
            assert np.array_equal(got[~reach, f], clean[~reach, f]), what + ": feature %d beyond the rows that name it" % f
            assert not np.isfinite(got[names, f]).any(), what + ": feature %d lost" % f
            if strict:
                assert np.array_equal(got[names, f], want[names, f], equal_nan=True), what + ": feature %d" % f
    plan.close()


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
