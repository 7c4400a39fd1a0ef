"""The wide-tile kernels (16-bit types, A as operands of 16 rows x 64 columns) at the sizes where they can go wrong, in each of their
shapes: rows and columns on both sides of a workgroup's and a chunk's, the last feature tile moved back, infinities and NaNs."""
import os

import numpy as np
import pytest

import test_nonfinite_gpu as nonfinite
from test_spmm_gpu import convert, torch_cuda  # noqa: F401
from test_tile_gpu import _matrix, _random_operand, _sampled_csr
from util import decode, encode

pytestmark = pytest.mark.gpu

FEWEST = [32, 32, 64, 32, 64, 64, 64, 128, 128]         # features of a tile, by shape


def _plan(hs, A, **env):
    env = {"HSPMM_" + name: str(value) for name, value in env.items()}
    os.environ.update(env)
    try:
        return hs.Plan(convert(hs, A))
    finally:
        for name in env:
            os.environ.pop(name, None)


@pytest.mark.parametrize("shape", range(9))
@pytest.mark.parametrize("dtype,rows,cols,cuts", [(0, 193, 257, 1), (2, 191, 64, 1), (2, 417, 575, 1), (0, 17, 65, 1), (2, 7, 3, 1), (2, 193, 575, 3), (0, 400, 2050, 5),
                                                  (2, 33, 2100, 16)])
def test_exact_sums_in_every_shape(torch_cuda, hs, shape, dtype, rows, cols, cuts):
    torch = torch_cuda
    rng = np.random.default_rng(100 * rows + shape)
    D, A = _matrix(rng, rows, cols, 0.1 if cols > 3 else 0.5, dtype)
    plan = _plan(hs, A, WIDE=1, WIDE_SHAPE=shape, WIDE_CUTS=cuts)
    stream = torch.cuda.current_stream().cuda_stream
    guard, nt = 64, FEWEST[shape]
    for N in (nt, nt + 1, 2 * nt - 1, 2 * nt, 2 * nt + 8):
        Bm = rng.integers(-4, 5, (cols, N))
        want = encode((D @ Bm).astype(np.float32), dtype)
        dB = torch.from_numpy(encode(Bm.astype(np.float32), dtype).view(np.int16)).cuda()
        buf = torch.full((rows * N + 2 * guard,), 7, dtype=torch.int16, device="cuda")
        dC = buf[guard:guard + rows * N]
        for launch in (plan.run, plan.run_static):
            dC.fill_(0x7E01)
            launch(dB.data_ptr(), dC.data_ptr(), N, stream)
            torch.cuda.synchronize()
            out = buf.cpu().numpy()
            assert (out[:guard] == 7).all() and (out[-guard:] == 7).all(), "N=%d: wrote outside C" % N
            assert np.array_equal(out[guard:-guard].view(np.uint8), want.reshape(-1).view(np.uint8)), "N=%d" % N
        assert plan.last_kernel() == "spmm_wide_kernel"
    plan.close()


@pytest.mark.parametrize("cuts", [1, 4])
def test_the_kernel_that_adds_cut_tiles_has_a_time_of_its_own(torch_cuda, hs, cuts):
    """hspmm_profile: 0 ms where no C tile is cut."""
    torch = torch_cuda
    D, A = _matrix(np.random.default_rng(cuts), 400, 2050, 0.1, 2)
    plan = _plan(hs, A, WIDE=1, WIDE_SHAPE=2, WIDE_CUTS=cuts)
    dB = torch.zeros((2050, 64), dtype=torch.int16, device="cuda")
    dC = torch.full((400, 64), 7, dtype=torch.int16, device="cuda")
    main_ms, sum_ms = plan.profile(dB.data_ptr(), dC.data_ptr(), 64, runs=3)
    assert plan.last_kernel() == "spmm_wide_kernel"
    assert main_ms > 0 and (sum_ms > 0) == (cuts > 1), (main_ms, sum_ms)
    assert not dC.any()
    plan.close()


@pytest.mark.parametrize("shape,cuts", [(0, 1), (6, 1), (7, 1), (4, 2)])
@pytest.mark.parametrize("dtype", [0, 2])
@pytest.mark.parametrize("rows,cols", [(600, 700), (1100, 130)])
def test_infinities_and_nans_stay_with_the_rows_that_name_them(torch_cuda, hs, monkeypatch, shape, cuts, dtype, rows, cols):
    """By the rule of the kernels that multiply stored entries only, whose check this is."""
    monkeypatch.setitem(nonfinite.FAMILIES, "tile", (0, {"HSPMM_WIDE": "1", "HSPMM_WIDE_SHAPE": str(shape), "HSPMM_WIDE_CUTS": str(cuts)}, (128, 130, 200), "spmm_wide_kernel"))
    nonfinite.test_infinities_and_nans_stay_with_the_rows_that_name_them(torch_cuda, hs, "tile", dtype, rows, cols)


# Against fp64: a product of two 16-bit numbers is exact in fp32 and every addition rounds once, so the sum of n of them is off by no more
# than n 2^-24 of the sum of their sizes, and the result's own rounding adds 2^-11 (fp16) or 2^-8 (bf16) of it.
@pytest.mark.parametrize("dtype,rows,cols,per_row,N,kernel", [
    (2, 5003, 3001, 600, 333, "wide"), (0, 4096, 4096, 409, 256, "wide"), (2, 3840, 1155, 340, 58, "wide"), (0, 4096, 4096, 82, 256, "panel"),
    (0, 512, 1024, 100, 512, "wide"), (0, 512, 11008, 1100, 64, "wide"), (2, 5120, 2007, 200, 24, "tile"), (1, 4096, 4096, 409, 256, "panel")])
def test_chosen_where_they_are_faster(torch_cuda, hs, dtype, rows, cols, per_row, N, kernel):
    torch = torch_cuda
    rng = np.random.default_rng(N + dtype)
    A = _sampled_csr(rng, rows, cols, per_row, dtype, lambda n: rng.normal(size=n))
    plan = hs.Plan(convert(hs, A))
    B, dB = _random_operand(torch, rng, cols, N, dtype)
    dC = torch.full((rows, N), 7, dtype=dB.dtype, device="cuda")
    plan.run(dB.data_ptr(), dC.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert (plan.last_kernel() == "spmm_wide_kernel") == (kernel == "wide")
    if kernel == "wide":
        D = np.zeros((rows, cols))
        D[np.repeat(np.arange(rows), per_row), A["col_idx"]] = decode(A["values"], dtype)
        Bm = decode(B, dtype).astype(np.float64)
        bound = per_row * 2.0**-24 * (abs(D) @ abs(Bm))
        want = D @ Bm
        off = abs(decode(dC.cpu().numpy().view(np.uint16), dtype).astype(np.float64) - want)
        assert (off <= bound + (2.0**-11 if dtype == 0 else 2.0**-8) * (abs(want) + bound)).all()
    plan.close()


def test_chosen_for_blocks_where_they_are_faster(torch_cuda, hs):
    torch = torch_cuda
    rng = np.random.default_rng(5)
    D = np.kron(rng.random((128, 128)) < 0.4, np.ones((16, 16), int)) * rng.integers(-2, 3, (2048, 2048))
    counts = (D != 0).sum(1)
    A = dict(rows=2048, cols=2048, nnzs=int(counts.sum()), dtype=2, row_ptr=np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32),
             col_idx=np.nonzero(D)[1].astype(np.uint32), values=encode(D[D != 0].astype(np.float32), 2))
    plan = hs.Plan(convert(hs, A))
    for N, wide in ((32, False), (63, True), (95, True), (130, None)):
        Bm = rng.integers(-2, 3, (2048, N))
        dB = torch.from_numpy(encode(Bm.astype(np.float32), 2).view(np.int16)).cuda()
        dC = torch.empty((2048, N), dtype=torch.int16, device="cuda")
        plan.run(dB.data_ptr(), dC.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert wide is None or (plan.last_kernel() == "spmm_wide_kernel") == wide, N
        assert np.array_equal(dC.cpu().numpy().view(np.uint16), encode((D @ Bm).astype(np.float32), 2)), N
    plan.close()
