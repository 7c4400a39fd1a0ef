"""The gather kernels on windows dealt out by a schedule where they can go wrong: windows cut into many parts and a window alone, rows without
entries in front, between and behind, both feature splits, the sums of parts in one kernel and in two, infinities and NaNs."""
import os

import numpy as np
import pytest

from test_block_gpu import _csr, _device, _host
from test_spmm_gpu import convert, torch_cuda  # noqa: F401
from util import decode, encode

pytestmark = pytest.mark.gpu


def _plan(hs, A, **env):
    env = {**dict(HSPMM_SCHEDULE="16", HSPMM_GATHER_BITMAP="1", HSPMM_XCD_SPLIT="1"), **env}
    os.environ.update(env)
    hs.set_kernel_mode(3)
    try:
        return hs.Plan(convert(hs, A))
    finally:
        hs.set_kernel_mode(0)
        for name in env:
            os.environ.pop(name)


def _mask(rng, rows, cols, heavy, empty):
    """Rows of 0 to 30 entries, every tenth window's first row `heavy` of the columns; windows whose number `empty` says are without."""
    counts = rng.integers(0, 31, rows)
    counts[::80] = int(heavy * cols)
    mask = np.argsort(rng.random((rows, cols)), 1) < counts[:, None]
    for w in empty:
        mask[8 * w:8 * w + 8] = False
    return mask


@pytest.mark.parametrize("dtype", [0, 2])
@pytest.mark.parametrize("fused", ["0", "1"])
@pytest.mark.parametrize("rows,cols,heavy,empty", [(8, 9000, 0.9, ()), (8, 1, 1.0, ()), (163, 7000, 0.8, (0, 1, 7, 8, 20)), (3001, 2500, 0.7, (0, 2, 374, 375)),
                                                   (700, 400, 0.0, (87,))])
def test_exact_sums(torch_cuda, hs, dtype, fused, rows, cols, heavy, empty):
    torch = torch_cuda
    rng = np.random.default_rng(rows)
    mask = _mask(rng, rows, cols, heavy, empty)
    values = rng.choice([-2, -1, 1, 2], int(mask.sum()))
    D = np.zeros((rows, cols), np.float32)              # (whole numbers below 2^24: exact in any order)
    D[mask] = values
    A = _csr(mask, values, dtype)
    tiles = convert(hs, A)
    plan = _plan(hs, A, HSPMM_FUSED_FIXUP=fused)
    stream = torch.cuda.current_stream().cuda_stream
    for N in (64, 128, 192, 256, 320, 512):
        Bm = rng.integers(-1, 2, (cols, N)).astype(np.float32)
        want = _device(torch, D @ Bm, dtype)
        dB = _device(torch, Bm, dtype)
        plan.prepare(N)
        for launch in (plan.run, plan.run_static, plan.run):
            dC = torch.full_like(want, 0x7E01)
            launch(dB.data_ptr(), dC.data_ptr(), N, stream)
            torch.cuda.synchronize()
            assert torch.equal(dC, want), "N=%d" % N
            assert plan.last_kernel() == "spmm_mfma_kernel" and plan.last_walk()["scheduled"]
        # (16 waves of 24 tiles and more; cut are the windows that are longer than a wave's share)
        waves = min(16, -(-tiles["total_tiles"] // 24))
        cut = int((np.diff(tiles["rowOffset"].astype(np.int64)) > -(-tiles["total_tiles"] // waves)).sum())
        assert plan.last_walk()["split_windows"] == cut and plan.last_walk()["ranges"] <= waves
    plan.close()


@pytest.mark.parametrize("fused", ["0", "1"])
def test_features_behind_the_last_block_take_a_launch_of_their_own(torch_cuda, hs, fused):
    """128 features of rows of 130: the sums are those of rows of 128, bit for bit, and not those in the order of the rows."""
    torch = torch_cuda
    rng = np.random.default_rng(9)
    rows, cols = 1003, 2500
    mask = _mask(rng, rows, cols, 0.7, (0, 2, 60))
    A = _csr(mask, rng.normal(size=int(mask.sum())), 0)
    stream = torch.cuda.current_stream().cuda_stream
    wide = _device(torch, rng.normal(size=(cols, 130)), 0)
    got = {}
    for schedule in ("16", "0"):
        plan = _plan(hs, A, HSPMM_FUSED_FIXUP=fused, HSPMM_SCHEDULE=schedule)
        for N in (130, 128):
            B = wide[:, :N].contiguous()
            C = torch.full((rows, N), 0x7E01, dtype=torch.int16, device="cuda")
            plan.run(B.data_ptr(), C.data_ptr(), N, stream)
            torch.cuda.synchronize()
            got[schedule, N] = C[:, :128]
        assert plan.last_walk()["scheduled"] == (schedule == "16")
        plan.close()
    assert torch.equal(got["16", 130], got["16", 128]) and torch.equal(got["0", 130], got["0", 128])
    assert not torch.equal(got["16", 130], got["0", 130])


@pytest.mark.parametrize("fused", ["0", "1"])
def test_two_streams_on_one_plan(torch_cuda, hs, fused):
    torch = torch_cuda
    rng = np.random.default_rng(10)
    rows, cols, N = 163, 7000, 128
    mask = _mask(rng, rows, cols, 0.8, (0, 7))
    values = rng.choice([-2, -1, 1, 2], int(mask.sum()))
    D = np.zeros((rows, cols), np.float32)
    D[mask] = values
    plan = _plan(hs, _csr(mask, values, 0), HSPMM_FUSED_FIXUP=fused)
    streams = [torch.cuda.Stream() for _ in range(2)]
    Bs = [rng.integers(-1, 2, (cols, N)).astype(np.float32) for _ in streams]
    want, dB = [_device(torch, D @ B, 0) for B in Bs], [_device(torch, B, 0) for B in Bs]
    dC = [[torch.full_like(w, 0x7E01) for _ in range(20)] for w in want]
    torch.cuda.synchronize()
    for i in range(20):
        for s, b, c in zip(streams, dB, dC):
            plan.run(b.data_ptr(), c[i].data_ptr(), N, s.cuda_stream)
    torch.cuda.synchronize()
    assert plan.last_walk()["scheduled"] and plan.last_walk()["split_windows"] > 0
    assert all(torch.equal(x, w) for c, w in zip(dC, want) for x in c)
    plan.close()


def test_infinities_and_nans_stay_with_the_windows_that_name_them(torch_cuda, hs):
    torch = torch_cuda
    rng = np.random.default_rng(11)
    rows, cols = 330, 3000
    mask = _mask(rng, rows, cols, 0.6, (3,))
    A = _csr(mask, rng.normal(size=int(mask.sum())), 0)
    D = np.zeros(mask.shape)
    D[mask] = decode(A["values"], 0)
    windows = np.kron(np.logical_or.reduceat(mask, np.arange(0, rows, 8)), np.ones((8, 1), bool))[:rows]
    for fused in ("0", "1"):
        plan = _plan(hs, A, HSPMM_FUSED_FIXUP=fused)
        for N in (64, 128):
            B = decode(encode(rng.normal(size=(cols, N)).astype(np.float32), 0), 0)
            finite = D @ B
            B[17, 5], B[2900, 6] = np.inf, np.nan
            dB = _device(torch, B, 0)
            dC = torch.empty((rows, N), dtype=dB.dtype, device="cuda")
            plan.run(dB.data_ptr(), dC.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
            assert plan.last_walk()["scheduled"]
            got = decode(_host(dC, 0), 0)
            hit, near = np.zeros(got.shape, bool), np.zeros(got.shape, bool)
            hit[mask[:, 17], 5] = hit[mask[:, 2900], 6] = True
            near[windows[:, 17], 5] = near[windows[:, 2900], 6] = True
            assert not np.isfinite(got[hit]).any() and np.isfinite(got[~near]).all()
            # (sums of up to 1800 products, each within 2^-24 of its size, and one rounding to fp16)
            assert (abs(got - finite)[~near] <= 1801 * 2.0**-24 * (abs(D) @ abs(np.where(np.isfinite(B), B, 0)))[~near] + 2.0**-11 * abs(finite)[~near] + 1e-7).all()
        plan.close()


def _hot(rng, rows, cols, power):
    """A graph of uneven rows over hot columns: CSR of whole numbers, the row of every entry."""
    counts = np.minimum(rng.zipf(2.0, rows), 2000)
    keys = np.unique(np.repeat(np.arange(rows), counts) * cols + (cols * rng.random(int(counts.sum())) ** power).astype(np.int64))
    r, c = keys // cols, keys % cols
    values = rng.choice([-2.0, -1.0, 1.0, 2.0], len(keys)).astype(np.float32)
    A = dict(rows=rows, cols=cols, nnzs=len(keys), dtype=0, row_ptr=np.concatenate([[0], np.cumsum(np.bincount(r, minlength=rows))]).astype(np.uint32),
             col_idx=c.astype(np.uint32), values=encode(values, 0))
    return A, r, values


def _sums(torch, A, r, values, B):
    """(whole numbers below 2^24: exact in any order, and rounded once)"""
    out = torch.zeros((A["rows"], B.shape[1]), dtype=torch.float32, device="cuda")
    r, c, v = (torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in (r, A["col_idx"].astype(np.int64), values))
    for at in range(0, len(values), 1 << 18):
        out.index_add_(0, r[at:at + (1 << 18)], B[c[at:at + (1 << 18)]].float() * v[at:at + (1 << 18), None])
    return out.half()


def _graph_plans(hs, A, *schedules):
    tiles = convert(hs, A)
    assert A["nnzs"] > 1.01 * (tiles["tcA2B"] != 0xFFFFFFFF).sum()
    os.environ["HSPMM_GATHER_BITMAP"] = "1"             # (tiles of 8 MB and more have them by themselves)
    plans = []
    try:
        for schedule in schedules:
            os.environ["HSPMM_SCHEDULE"] = schedule
            plans.append(hs.Plan(tiles))
    finally:
        os.environ.pop("HSPMM_GATHER_BITMAP")
        os.environ.pop("HSPMM_SCHEDULE", None)
    return plans


def test_graphs_of_many_columns_have_one(torch_cuda, hs):
    """Words of B and C at 128 features are walked by it, also where nothing may be built; between two words the launch is another kernel's."""
    torch = torch_cuda
    rng = np.random.default_rng(5)
    rows, cols, N = 1 << 18, 1 << 18, 128
    A, r, values = _hot(rng, rows, cols, 6)
    plan, without = _graph_plans(hs, A, "-1", "0")
    assert plan.info()["device_bytes"] > without.info()["device_bytes"]
    B = torch.randint(-1, 2, (cols, N), dtype=torch.int8, device="cuda").half()
    want = _sums(torch, A, r, values, B)
    stream = torch.cuda.current_stream().cuda_stream
    between = torch.cat([B.reshape(-1)[:1], B.reshape(-1)])
    # the static entry point does not change kernels with what ran before: B between two words is the entry kernels' launch
    dC = torch.full_like(want, float("nan"))
    for _ in range(2):
        plan.run(B.data_ptr(), dC.data_ptr(), N, stream)
    with pytest.raises(hs.HspmmError, match="hspmm_prepare"):
        plan.run_static(between.data_ptr() + 2, dC.data_ptr(), N, stream)
    for p, walked in ((plan, True), (without, False)):
        p.prepare(N)
        for at in (B.data_ptr(), between.data_ptr() + 2, B.data_ptr()):
            for launch in (p.run_static, p.run, p.run_static):
                dC.fill_(float("nan"))
                launch(at, dC.data_ptr(), N, stream)
                torch.cuda.synchronize()
                assert torch.equal(dC, want)
                scheduled = walked and at == B.data_ptr()
                assert p.last_walk()["scheduled"] == scheduled and p.last_kernel() == ("spmm_mfma_kernel" if scheduled else "spmm_entries_kernel")
        # (C of 32 MB: too short a launch)
        p.run(B.data_ptr(), dC.data_ptr(), 64, stream)
        torch.cuda.synchronize()
        assert not p.last_walk()["scheduled"]
        p.close()


def test_more_columns_than_a_schedule_reaches(torch_cuda, hs):
    """2^24 columns: offsets into B do not fit 32 bits and the launch is the entry kernels'."""
    torch = torch_cuda
    rng = np.random.default_rng(6)
    rows, cols, N = 1 << 19, (1 << 24) + 40, 64
    A, r, values = _hot(rng, rows, cols, 8)
    (plan,) = _graph_plans(hs, A, "-1")
    B = torch.randint(-1, 2, (cols, N), dtype=torch.int8, device="cuda").half()
    C = torch.full((rows, N), float("nan"), dtype=torch.float16, device="cuda")
    plan.run(B.data_ptr(), C.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert plan.last_kernel() == "spmm_entries_kernel" and not plan.last_walk()["scheduled"]
    assert torch.equal(C, _sums(torch, A, r, values, B))
    plan.close()
