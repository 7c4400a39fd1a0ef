"""The kernels for few features of weights in 16 x 16 blocks where they can go wrong: every number of features, blocks that end
inside the matrix, a window alone, rows without blocks, an odd number of blocks, B and C between two words, infinities and NaNs."""
import os

import numpy as np
import pytest

from test_spmm_gpu import convert, torch_cuda  # noqa: F401
from util import decode, encode

pytestmark = pytest.mark.gpu


def _blocks(rng, rows, cols, keep, without=0.0, half=False):
    """Which elements are stored; without: rows of blocks that are empty; half: the lower window of the second row of blocks is."""
    kept = rng.random((-(-rows // 16), -(-cols // 16))) < keep
    kept[rng.random(len(kept)) < without] = False
    kept[0, 0] = True
    mask = np.kron(kept, np.ones((16, 16), bool))[:rows, :cols]
    if half:
        mask[24:32] = False
    return mask


def _csr(mask, values, dtype):
    counts = mask.sum(1)
    return dict(rows=mask.shape[0], cols=mask.shape[1], nnzs=int(counts.sum()), dtype=dtype, row_ptr=np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32),
                col_idx=np.nonzero(mask)[1].astype(np.uint32), values=encode(values.astype(np.float32), dtype))


def _device(torch, x, dtype):
    """Storage as a tensor on the GPU: whole numbers of the same size."""
    return torch.from_numpy(encode(np.asarray(x, np.float32), dtype).view(np.int32 if dtype == 1 else np.int16)).cuda()


def _host(t, dtype):
    return t.cpu().numpy().view(np.float32 if dtype == 1 else np.uint16)


def _plan(hs, A, block):
    os.environ["HSPMM_BLOCK"] = str(block)
    try:
        return hs.Plan(convert(hs, A))
    finally:
        os.environ.pop("HSPMM_BLOCK")


@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("rows,cols,keep,without,half", [(16, 16, 1.0, 0, False), (40, 24, 1.0, 0.3, False), (250, 333, 0.5, 0.2, True), (9, 100, 1.0, 0, False),
                                                         (1000, 2000, 0.3, 0.05, True), (130, 16500, 0.9, 0, False),
                                                         (34, 17400, 1.0, 0, False)])           # (over 1024 steps: a wave's second 64 pairs)
def test_exact_sums_at_every_edge(torch_cuda, hs, dtype, rows, cols, keep, without, half):
    torch = torch_cuda
    rng = np.random.default_rng(rows + cols)
    mask = _blocks(rng, rows, cols, keep, without, half)
    values = rng.choice([-2, -1, 1, 2], int(mask.sum()))
    D = np.zeros((rows, cols), np.float32)              # (whole numbers below 2^24: exact in any order)
    D[mask] = values
    plan = _plan(hs, _csr(mask, values, dtype), 1)
    stream = torch.cuda.current_stream().cuda_stream
    guard = 65
    for N in (1, 2, 3, 7, 8, 9, 15, 16, 17, 25, 31, 32, 34, 40, 48, 62, 64):
        Bm = rng.integers(-1, 2, (cols, N)).astype(np.float32)
        want = _device(torch, (D @ Bm).reshape(-1), dtype)
        filled = torch.full_like(want, 0x7FC07E01 if dtype == 1 else 0x7E01)
        for shift in (0, 1):                            # (16-bit types: B and C on a word, or between two)
            b_buf = torch.cat([filled[:shift], _device(torch, Bm.reshape(-1), dtype)])
            c_buf = torch.full((rows * N + 2 * guard + shift,), 7, dtype=want.dtype, device="cuda")
            inside = c_buf[guard + shift:guard + shift + rows * N]
            for launch in (plan.run, plan.run_static):
                inside.copy_(filled)
                launch(b_buf.data_ptr() + b_buf.element_size() * shift, inside.data_ptr(), N, stream)
                torch.cuda.synchronize()
                assert (c_buf[:guard + shift] == 7).all() and (c_buf[guard + shift + rows * N:] == 7).all(), "N=%d: wrote outside C" % N
                assert torch.equal(inside + 0, want) if dtype != 1 else torch.equal(inside.view(torch.float32), want.view(torch.float32)), "N=%d shift=%d" % (N, shift)
            assert plan.last_kernel() == "spmm_block_kernel"
    plan.close()


@pytest.mark.parametrize("dtype", [0, 1, 2])
def test_infinities_and_nans_stay_with_the_rows_that_name_them(torch_cuda, hs, dtype):
    """A column of the matrix loses half of its entries first, so that blocks hold zeros beside them; rows of blocks without any, windows alone.
    Every other sum, those of the same features among them, is what it is without (bound: see below)."""
    torch = torch_cuda
    rng = np.random.default_rng(3 + dtype)
    mask = _blocks(rng, 300, 400, 0.5, 0.1, True)
    mask[::3, ::5] = False
    mask[24:32] = False
    mask[8:16] = False
    A = _csr(mask, rng.normal(size=int(mask.sum())), dtype)
    D = np.zeros(mask.shape)
    D[mask] = decode(A["values"], dtype)
    plan = _plan(hs, A, 1)
    assert plan.info()["n_units"] > plan.info()["n_paired_units"] > 0
    for N in (5, 16, 31, 64):
        B = decode(encode(rng.normal(size=(400, N)).astype(np.float32), dtype), dtype)
        finite, sizes = D @ B, abs(D) @ abs(B)
        bad = B.copy()
        bad[17, N - 1], bad[240, 0] = np.inf, np.nan
        dB = _device(torch, bad, dtype)
        dC = torch.empty((300, N), dtype=dB.dtype, device="cuda")
        plan.run(dB.data_ptr(), dC.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        got = decode(_host(dC, dtype), dtype)
        hit = np.zeros(finite.shape, bool)
        hit[mask[:, 17], N - 1] = True
        hit[mask[:, 240], 0] = True
        assert not np.isfinite(got[hit]).any() and np.isfinite(got[~hit]).all()
        assert (np.isinf(got[:, N - 1]) == mask[:, 17])[~mask[:, 240] | (N > 1)].all()
        off = abs(got - finite)
        assert (off <= (mask.sum(1).max() + 1) * 2.0**-24 * sizes + 2.0**{0: -11, 1: -24, 2: -8}[dtype] * abs(finite) + 1e-7)[~hit].all()
    assert plan.last_kernel() == "spmm_block_kernel"
    plan.close()


# Against fp64: a product of two 16-bit numbers is exact in fp32 and every addition rounds once, so the sum of n of them is off by no more
# than n 2^-24 of the sum of their sizes, and the result's own rounding adds 2^-11 (fp16) or 2^-8 (bf16) of it; of fp32 numbers the product rounds once more.
@pytest.mark.parametrize("dtype,rows,cols,keep,N,taken", [(0, 4096, 14336, 0.5, 16, True), (2, 2048, 3000, 0.3, 31, True), (0, 4096, 4096, 0.5, 64, True),
                                                          (2, 2048, 3000, 0.3, 33, False), (0, 4096, 4096, 0.5, 128, False),
                                                          (1, 4096, 4096, 0.5, 16, True), (1, 2048, 3000, 0.3, 47, True), (1, 4096, 4096, 0.5, 64, False)])
def test_chosen_where_they_are_faster(torch_cuda, hs, dtype, rows, cols, keep, N, taken):
    torch = torch_cuda
    rng = np.random.default_rng(N + dtype)
    mask = _blocks(rng, rows, cols, keep)
    A = _csr(mask, rng.normal(size=int(mask.sum())), dtype)
    plan = hs.Plan(convert(hs, A))
    B = encode(rng.normal(size=(cols, N)).astype(np.float32), dtype)
    dB = _device(torch, decode(B, dtype), dtype)
    dC = torch.empty((rows, N), dtype=dB.dtype, device="cuda")
    plan.run(dB.data_ptr(), dC.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert (plan.last_kernel() == "spmm_block_kernel") == taken
    if taken:
        D = np.zeros((rows, cols))
        D[mask] = decode(A["values"], dtype)
        Bm = decode(B, dtype)
        want, sizes = D @ Bm, abs(D) @ abs(Bm)
        off = abs(decode(_host(dC, dtype), dtype) - want)
        assert (off <= (mask.sum(1).max() + 1) * 2.0**-24 * sizes + 2.0**{0: -11, 1: -24, 2: -8}[dtype] * abs(want) + 1e-7).all()
    plan.close()
