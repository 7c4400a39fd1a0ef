"""The full-tile kernels (blocks of 128 rows put together in LDS from stored entries) at the sizes where they can go wrong:
rows and columns on both sides of a block, blocks without entries and blocks over a quarter full, feature dimensions on
both sides of a tile's width, C tiles cut between workgroups, the entry point that allocates nothing."""
import os

import numpy as np
import pytest

from test_spmm_gpu import convert, torch_cuda  # noqa: F401
from util import encode

pytestmark = pytest.mark.gpu


def _matrix(rng, rows, cols, density, dtype):
    D = rng.integers(-3, 4, (rows, cols)) * (rng.random((rows, cols)) < density)
    if rows > 40:
        D[8:24] = 0                                     # windows without entries
    if cols > 400:
        D[:, 130:330] = 0                               # whole blocks without entries
        D[-5:, :64] = rng.integers(1, 4, (5, 64))       # and a denser corner
    counts = (D != 0).sum(1)
    row_ptr = np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32)
    A = dict(rows=rows, cols=cols, nnzs=int(row_ptr[-1]), dtype=dtype, row_ptr=row_ptr, col_idx=np.nonzero(D)[1].astype(np.uint32),
             values=encode(D[D != 0].astype(np.float32), dtype))
    return D, A


def _plan(hs, A):
    os.environ["HSPMM_TILE"] = "1"
    try:
        return hs.Plan(convert(hs, A))
    finally:
        os.environ.pop("HSPMM_TILE", None)


# (4200 rows: more C tiles than a workgroup per compute unit has whole ones; 0.6: more units of entries than threads hold)
@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("rows,cols,density", [(128, 64, 0.3), (129, 65, 0.3), (127, 129, 0.6), (1000, 517, 0.1), (4200, 1030, 0.05)])
def test_exact_sums_on_both_sides_of_every_block(torch_cuda, hs, dtype, rows, cols, density):
    torch = torch_cuda
    rng = np.random.default_rng(rows + dtype)
    D, A = _matrix(rng, rows, cols, density, dtype)
    plan = _plan(hs, A)
    stream = torch.cuda.current_stream().cuda_stream
    tt = torch.float32 if dtype == 1 else torch.int16
    guard = 64
    for N in (4 if dtype == 1 else 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 100, 127, 130):
        Bm = rng.integers(-4, 5, (cols, N))
        B, want = encode(Bm.astype(np.float32), dtype), encode((D @ Bm).astype(np.float32), dtype)
        dB = torch.from_numpy(B if dtype == 1 else B.view(np.int16)).cuda()
        buf = torch.full((rows * N + 2 * guard,), 7, dtype=tt, device="cuda")
        dC = buf[guard:guard + rows * N]
        plan.prepare(N)
        for launch in (plan.run, plan.run_static, plan.run):        # (counters of cut tiles are zero again after a launch)
            dC.fill_(0x7E01 if dtype != 1 else float("nan"))
            launch(dB.data_ptr(), dC.data_ptr(), N, stream)
            torch.cuda.synchronize()
            out = buf.cpu().numpy()
            assert (out[:guard] == 7).all() and (out[-guard:] == 7).all(), "N=%d: wrote outside C" % N
            assert np.array_equal(out[guard:-guard].view(np.uint8), want.reshape(-1).view(np.uint8)), "N=%d" % N
        assert plan.info()["last_kernel_family"] == 3
    plan.close()


@pytest.mark.parametrize("dtype,N", [(0, 24), (1, 16), (2, 64)])
def test_chosen_for_wide_enough_launches_of_dense_enough_matrices(torch_cuda, hs, dtype, N):
    torch = torch_cuda
    rng = np.random.default_rng(7 + dtype)
    D, A = _matrix(rng, 4096, 4096, 0.35, dtype)
    plan = hs.Plan(convert(hs, A))
    Bm = rng.integers(-1, 2, (4096, N))
    B, want = encode(Bm.astype(np.float32), dtype), encode((D @ Bm).astype(np.float32), dtype)
    dB = torch.from_numpy(B if dtype == 1 else B.view(np.int16)).cuda()
    dC = torch.full((4096, N), 7, dtype=torch.float32 if dtype == 1 else torch.int16, device="cuda")
    plan.run(dB.data_ptr(), dC.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert np.array_equal(dC.cpu().numpy().view(np.uint8), want.view(np.uint8))
    assert plan.info()["last_kernel_family"] == 3
    plan.close()


def _sampled_csr(rng, rows, cols, per_row, dtype, values):
    """per_row entries in every row, at columns without any order to them; values(n) gives them."""
    step = cols // per_row
    col_idx = (np.arange(per_row, dtype=np.int64)[None, :] * step + rng.integers(0, step, (rows, per_row))).astype(np.uint32)
    return dict(rows=rows, cols=cols, nnzs=rows * per_row, dtype=dtype, row_ptr=(np.arange(rows + 1, dtype=np.int64) * per_row).astype(np.uint32),
                col_idx=col_idx.reshape(-1), values=encode(values(rows * per_row).astype(np.float32), dtype))


def _random_operand(torch, rng, cols, N, dtype):
    B = encode(rng.normal(size=(cols, N)).astype(np.float32), dtype)
    return B, torch.from_numpy(B if dtype == 1 else B.view(np.int16)).cuda()


# (17000 rows at N = 96: three workgroups per compute unit leave more sums than the fixed array holds; 70000: more C tiles
# than workgroups)
@pytest.mark.parametrize("dtype,rows,cols,per_row,N", [(2, 17000, 4096, 200, 96), (0, 70000, 1024, 60, 64), (1, 9000, 4096, 455, 20)])
def test_entry_point_that_allocates_nothing_runs_what_hspmm_run_does(torch_cuda, hs, dtype, rows, cols, per_row, N):
    torch = torch_cuda
    rng = np.random.default_rng(90 + dtype)
    A = _sampled_csr(rng, rows, cols, per_row, dtype, lambda n: rng.normal(size=n))
    plan = hs.Plan(convert(hs, A))
    _, dB = _random_operand(torch, rng, cols, N, dtype)
    outs = [torch.full((rows, N), 7, dtype=dB.dtype, device="cuda") for _ in range(3)]
    stream = torch.cuda.current_stream().cuda_stream
    plan.prepare(N)
    plan.run_static(dB.data_ptr(), outs[0].data_ptr(), N, stream)
    assert plan.info()["last_kernel_family"] == 3
    plan.run(dB.data_ptr(), outs[1].data_ptr(), N, stream)
    assert plan.info()["last_kernel_family"] == 3
    plan.run_static(dB.data_ptr(), outs[2].data_ptr(), N, stream)
    torch.cuda.synchronize()
    bits = [o.view(torch.int32 if dtype == 1 else torch.int16) for o in outs]
    assert torch.equal(bits[0], bits[1]) and torch.equal(bits[0], bits[2])
    plan.close()
