"""The entry kernels on rows of B of 513 to 1024 fp32 features, in up to eight and more blocks, and which launches are theirs: those rows, and
power-law graphs that are dense in their hot columns."""
import numpy as np
import pytest

from test_block_gpu import _csr, _device
from test_entries_gpu import _check_guarded, _plan, _rows_of_lengths
from test_spmm_gpu import convert, make_b, oracle_spmm, torch_cuda  # noqa: F401
from util import encode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [513, 516, 640, 767, 1000, 1023, 1024])
def test_wide_rows_of_fp32(torch_cuda, hs, oracle, N):
    rng = np.random.default_rng(N)
    A = _rows_of_lengths(rng, [0, 1, 2, 5, 16, 33, 129, 700, 0, 2049] + [9] * 90 + [0] * 3 + [60], 2500, 1)
    B = make_b(rng, A["cols"], N, 1)
    ref, mag = oracle_spmm(oracle, A, B, N)
    plan = _plan(hs, A)
    _check_guarded(torch_cuda, plan, A, B, N, 1, ref, mag, "N=%d" % N)
    assert plan.last_kernel() == "spmm_entries_kernel"
    plan.close()


def _graph(rng, vertices, edges):
    """Rows and columns with weights that fall like a power law."""
    weight = 1.0 / np.arange(4, vertices + 4) ** 0.9
    weight /= weight.sum()
    mask = np.zeros((vertices, vertices), bool)
    mask[rng.choice(vertices, vertices * edges, p=weight), rng.choice(vertices, vertices * edges, p=weight)] = True
    return mask


@pytest.mark.parametrize("dtype,N,taken", [(0, 45, True), (2, 64, True), (0, 133, True), (0, 512, True), (0, 800, False), (1, 94, True), (1, 640, True)])
def test_graphs_with_dense_columns(torch_cuda, hs, dtype, N, taken):
    torch = torch_cuda
    rng = np.random.default_rng(8)
    mask = _graph(rng, 4096, 20)
    tiles = convert(hs, _csr(mask, rng.choice([-2, -1, 1, 2], int(mask.sum())), dtype))
    per_column = mask.sum() / float((tiles["tcA2B"] != 0xFFFFFFFF).sum())
    assert 1.25 < per_column < 1.4
    D = np.zeros(mask.shape, np.float32)
    values = rng.choice([-2, -1, 1, 2], int(mask.sum()))
    D[mask] = values
    plan = hs.Plan(convert(hs, _csr(mask, values, dtype)))
    Bm = rng.integers(-1, 2, (4096, N)).astype(np.float32)
    want = _device(torch, D @ Bm, dtype)                # (whole numbers below 2^24: exact in any order)
    dB = _device(torch, Bm, dtype)
    for _ in range(2):
        dC = torch.full_like(want, 0x7E01)
        plan.run(dB.data_ptr(), dC.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(dC, want) if dtype != 1 else torch.equal(dC.view(torch.float32), want.view(torch.float32))
    assert (plan.last_kernel() == "spmm_entries_kernel") == taken
    plan.close()


# few rows, all long: 4, 8 and 16 units of four entries to a subgroup
@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("rows,cols,keep", [(33, 1100, 0.9), (1274, 2000, 0.15), (3000, 1024, 0.3), (1000, 2100, 0.55)])
def test_rows_all_long(torch_cuda, hs, dtype, rows, cols, keep):
    torch = torch_cuda
    rng = np.random.default_rng(rows)
    mask = rng.random((rows, cols)) < keep
    values = rng.choice([-2, -1, 1, 2], int(mask.sum()))
    D = np.zeros(mask.shape, np.float32)                # (whole numbers below 2^24: exact in any order)
    D[mask] = values
    plan = _plan(hs, _csr(mask, values, dtype))
    for N in (1, 2, 5, 8, 16, 33, 64):
        Bm = rng.integers(-1, 2, (cols, N)).astype(np.float32)
        want, dB = _device(torch, D @ Bm, dtype), _device(torch, Bm, dtype)
        plan.prepare(N)
        for launch in (plan.run, plan.run_static):
            dC = torch.full_like(want, 0x7E01)
            launch(dB.data_ptr(), dC.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
            assert torch.equal(dC, want) if dtype != 1 else torch.equal(dC.view(torch.float32), want.view(torch.float32)), "N=%d" % N
        assert plan.last_kernel() == "spmm_entries_kernel"
    plan.close()
