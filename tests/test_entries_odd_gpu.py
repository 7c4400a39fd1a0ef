"""The entry kernels' rows of an odd number of 16-bit elements: both parities of a row, the first and the last row of B, one block and
several, rows cut between subgroups, B that does not begin on a word, infinities and NaNs."""
import numpy as np
import pytest

import test_nonfinite_gpu as nonfinite
from test_entries_gpu import _rows_of_lengths
from test_spmm_gpu import convert, torch_cuda  # noqa: F401
from test_tile_gpu import _matrix, _random_operand
from test_wide_gpu import _plan
from util import decode, encode

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


# Against fp64, with real numbers, whose sums show a feature in another's place by its size and not only by a whole number: a product of
# two 16-bit numbers is exact in fp32 and every one of the n additions rounds once (n 2^-24 of the sum of sizes), the result once more
# (2^-11 or 2^-8 of it).  Rows cut into parts (1500 entries), rows in pieces (2600), every row with an entry in B's last row.
@pytest.mark.parametrize("dtype,N", [(0, 9), (2, 17), (0, 33), (2, 65), (0, 77), (2, 131), (0, 257), (2, 301), (0, 511)])
def test_rows_cut_into_parts_and_the_last_row_of_b(torch_cuda, hs, dtype, N):
    torch = torch_cuda
    rng = np.random.default_rng(N)
    rows, cols = 3000, 6001
    lengths = rng.integers(1, 12, rows)
    lengths[[3, 700, 2100]], lengths[2900] = 1500, 2600
    A = _rows_of_lengths(rng, [int(n) for n in lengths], cols, dtype)
    A["col_idx"][A["row_ptr"][1:].astype(np.int64) - 1] = cols - 1
    plan = _plan(hs, A, ENTRIES=1, TILE=0)
    B, dB = _random_operand(torch, rng, cols, N, dtype)
    dC = torch.full((rows, N), 0x7E01 if dtype == 0 else 0x7FC0, dtype=torch.int16, device="cuda")
    plan.run(dB.data_ptr(), dC.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert plan.last_kernel() == "spmm_entries_kernel"
    D = np.zeros((rows, cols))
    D[np.repeat(np.arange(rows), lengths), A["col_idx"]] = decode(A["values"], dtype)
    Bm = decode(B, dtype).astype(np.float64)
    want, bound = D @ Bm, lengths[:, None] * 2.0**-24 * (abs(D) @ abs(Bm))
    off = abs(decode(dC.cpu().numpy().view(np.uint16), dtype).astype(np.float64) - want)
    assert (off <= bound + (2.0**-11 if dtype == 0 else 2.0**-8) * (abs(want) + bound) + (2.0**-25 if dtype == 0 else 0.0)).all()
    plan.close()
