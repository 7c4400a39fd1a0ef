"""The entry kernels' rows of an odd number of 16-bit elements: both parities of a row, the first and the last row of B, one block and
several, rows cut between subgroups, B that does not begin on a word, infinities and NaNs."""
import numpy as np
import pytest

import test_nonfinite_gpu as nonfinite
from test_spmm_gpu import convert, torch_cuda  # noqa: F401
from test_tile_gpu import _matrix
from test_wide_gpu import _plan
from util import encode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [0, 2])
@pytest.mark.parametrize("rows,cols,density", [(40, 2, 0.6), (300, 63, 0.2), (33, 700, 0.4), (1000, 901, 0.02), (9, 9000, 0.3)])
def test_exact_sums(torch_cuda, hs, dtype, rows, cols, density):
    torch = torch_cuda
    rng = np.random.default_rng(rows + cols)
    D, A = _matrix(rng, rows, cols, density, dtype)
    plan = _plan(hs, A, ENTRIES=1, TILE=0)
    stream = torch.cuda.current_stream().cuda_stream
    guard, nan = 64, 0x7E01 if dtype == 0 else 0x7FC0
    for N in (9, 11, 15, 17, 31, 33, 63, 65, 127, 129, 255, 257, 379, 511, 1023):
        Bm = rng.integers(-4, 5, (cols, N))
        want = encode((D @ Bm).astype(np.float32), dtype)
        for off in (64, 65):                            # (B on a word, and not)
            room = torch.full((cols * N + 128,), nan, dtype=torch.int16, device="cuda")
            dB = room[off:off + cols * N]
            dB.copy_(torch.from_numpy(encode(Bm.astype(np.float32), dtype).view(np.int16)).reshape(-1))
            buf = torch.full((rows * N + 2 * guard,), 7, dtype=torch.int16, device="cuda")
            dC = buf[guard:guard + rows * N]
            dC.fill_(nan)
            plan.run(dB.data_ptr(), dC.data_ptr(), N, stream)
            torch.cuda.synchronize()
            out = buf.cpu().numpy()
            assert plan.last_kernel() == "spmm_entries_kernel"
            assert (out[:guard] == 7).all() and (out[-guard:] == 7).all(), "N=%d: wrote outside C" % N
            assert np.array_equal(out[guard:-guard].view(np.uint8), want.reshape(-1).view(np.uint8)), "N=%d" % N
    plan.close()


@pytest.mark.parametrize("dtype", [0, 2])
@pytest.mark.parametrize("rows,cols", [(600, 700), (1100, 131)])
def test_infinities_and_nans_stay_with_the_rows_that_name_them(torch_cuda, hs, monkeypatch, dtype, rows, cols):
    monkeypatch.setitem(nonfinite.FAMILIES, "entries", nonfinite.FAMILIES["entries"][:2] + ((15, 17, 63, 129, 301), "spmm_entries_kernel"))
    nonfinite.test_infinities_and_nans_stay_with_the_rows_that_name_them(torch_cuda, hs, "entries", dtype, rows, cols)
