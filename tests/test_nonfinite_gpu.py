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
        bad = {}                                        # feature -> rows of B
        for f, (k, v) in enumerate([(unnamed[0], np.inf), (unnamed[1], np.nan), (named[0], np.inf), (named[1], -np.inf),
                                    (named[2], np.nan), (named[3], np.inf)]):
            Bm[k, f] = v
            bad.setdefault(f, []).append(k)
        Bm[named[0], N - 1], Bm[named[1], N - 1] = np.inf, -np.inf
        bad.setdefault(N - 1, []).extend([named[0], named[1]])
        got = decode(gpu_spmm(torch_cuda, hs, dict(dtype=dtype, rows=rows), encode(Bm.astype(np.float32), dtype), N, plan=plan), dtype)
        assert plan.last_kernel() == FAMILIES[family][3]
        want = _rounded(_stored_sum(D, Bm), dtype)
        what = "%s, dtype %d, N=%d" % (family, dtype, N)
        fine = [f for f in range(N) if f not in bad]
        assert np.array_equal(got[:, fine], clean[:, fine]), what
        for f, ks in bad.items():
            names = (D[:, ks] != 0).any(1)
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


# environment, ranges per SIMD, paired windows
FORMS = {
    "whole units": ({}, 0, False),
    "cut units, second launch": ({"HSPMM_FUSED_FIXUP": "0"}, 16, False),
    "cut units, added where the last part ends": ({"HSPMM_FUSED_FIXUP": "1"}, 16, False),
    "a workgroup per unit": ({"HSPMM_ALIGNED_SMALL": "4"}, 0, False),
    "bitmap tiles": ({"HSPMM_GATHER_BITMAP": "1"}, 16, False),
    "pairs of windows": ({}, 0, True),
    "pairs of windows, cut": ({"HSPMM_FUSED_FIXUP": "1"}, 16, True),
}


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("dtype", [0, 2])
def test_adjacent_features_of_the_gather_kernels_do_not_mix(torch_cuda, hs, form, dtype):
    """Their 16-bit operand words are two adjacent features: one that is not finite leaves the other alone."""
    torch = torch_cuda
    env, ranges, paired = FORMS[form]
    rng = np.random.default_rng(70 + dtype)
    rows, cols = 328, 6000
    D = rng.integers(1, 4, (rows, cols)) * (rng.random((rows, cols)) < 0.02)
    if paired:                                          # 16 rows with one list of columns
        lists = rng.random((-(-rows // 16), cols)) < 0.05
        lists[10] = rng.random(cols) < 0.9              # (long enough to be cut)
        D = np.repeat(lists, 16, axis=0)[:rows] * rng.integers(1, 4, (rows, cols))
    D[40:56] = 0
    D[:, 77] = 0
    D[(3, 100, 101, 250), 77] = 2
    A = _csr(D, dtype)
    hs.set_kernel_mode(3)
    hs.set_window_pairing(2 if paired else 0)
    hs.configure(producer_warp_group_num=ranges)
    os.environ.update(env)
    try:
        plan = hs.Plan(convert(hs, A))
    finally:
        hs.set_kernel_mode(0)
        hs.set_window_pairing(0)
        hs.configure()
        for name in env:
            os.environ.pop(name, None)
    info = plan.info()
    assert (info["n_paired_units"] > 0) == paired and (info["n_split_windows"] > 0 or "cut" not in form)
    assert info["gather_bitmap"] == ("HSPMM_GATHER_BITMAP" in env)
    stream = torch.cuda.current_stream().cuda_stream
    for N in (1, 2, 16, 31, 64, 100, 128, 136, 256):
        Bm = rng.integers(-4, 5, (cols, N)).astype(np.float64)
        clean = _rounded(D @ Bm, dtype)
        bad = sorted({0, N // 2, max(0, N - 2)})
        for f, v in zip(bad, (np.inf, np.nan, -np.inf)):
            Bm[77, f] = v
        dB = torch.from_numpy(encode(Bm.astype(np.float32), dtype).view(np.int16)).cuda()
        dC = torch.empty((rows, N), dtype=torch.int16, device="cuda")
        plan.prepare(N)
        for launch in (plan.run, plan.run_static):
            dC.fill_(0x7E01)
            launch(dB.data_ptr(), dC.data_ptr(), N, stream)
            torch.cuda.synchronize()
            assert plan.last_kernel() == "spmm_mfma_kernel"
            got = decode(dC.cpu().numpy().view(np.uint16), dtype)
            fine = [f for f in range(N) if f not in bad]
            assert np.array_equal(got[:, fine], clean[:, fine]), "N=%d" % N
            reach = _near(D, 77)
            assert np.array_equal(got[~reach][:, bad], clean[~reach][:, bad]), "N=%d" % N
            assert not np.isfinite(got[(3, 100, 101, 250), :][:, bad]).any(), "N=%d" % N
    plan.close()
