"""The narrow kernels (16-bit types, up to 32 features, a wave per 16 rows x 128 columns) at the sizes where they can go wrong: rows and
columns on both sides of a block's and an operand's, odd features, blocks with more entries than are asked for ahead and with none,
infinities and NaNs."""
import numpy as np
import pytest

import test_nonfinite_gpu as nonfinite
from test_spmm_gpu import convert, torch_cuda  # noqa: F401
from test_tile_gpu import _matrix, _random_operand, _sampled_csr
from test_wide_gpu import _plan
from util import decode, encode

pytestmark = pytest.mark.gpu


# (2100: several blocks a wave; 0.7: more entries than are asked for ahead, twice over)
@pytest.mark.parametrize("waves", [4, 8, 16])
@pytest.mark.parametrize("dtype,rows,cols,density", [(0, 16, 2, 0.9), (2, 1, 31, 0.5), (2, 33, 32, 0.3), (0, 17, 33, 0.3), (2, 48, 127, 0.7), (0, 100, 129, 0.1),
                                                     (2, 95, 2100, 0.7), (0, 200, 8321, 0.05)])
def test_exact_sums_on_both_sides_of_every_block(torch_cuda, hs, waves, dtype, rows, cols, density):
    torch = torch_cuda
    rng = np.random.default_rng(10 * rows + cols)
    D, A = _matrix(rng, rows, cols, density, dtype)
    plan = _plan(hs, A, NARROW=1, NARROW_WAVES=waves)
    stream = torch.cuda.current_stream().cuda_stream
    guard = 64
    for N in (1, 2, 3, 8, 14, 15, 16, 17, 18, 28, 29, 30, 32):
        Bm = rng.integers(-4, 5, (cols, N))
        want = encode((D @ Bm).astype(np.float32), dtype)
        for off in (0, 1):                              # (B that begins between two words)
            room = torch.full((cols * N + off,), 0x7E01 if dtype == 0 else 0x7FC0, dtype=torch.int16, device="cuda")
            dB = room[off:]
            dB.copy_(torch.from_numpy(encode(Bm.astype(np.float32), dtype).view(np.int16)).reshape(-1))
            buf = torch.full((rows * N + 2 * guard,), 7, dtype=torch.int16, device="cuda")
            dC = buf[guard:guard + rows * N]
            for launch in (plan.run, plan.run_static):
                dC.fill_(0x7E01)
                launch(dB.data_ptr(), dC.data_ptr(), N, stream)
                torch.cuda.synchronize()
                out = buf.cpu().numpy()
                assert (out[:guard] == 7).all() and (out[-guard:] == 7).all(), "N=%d: wrote outside C" % N
                assert np.array_equal(out[guard:-guard].view(np.uint8), want.reshape(-1).view(np.uint8)), "N=%d" % N
            assert plan.last_kernel() == "spmm_narrow_kernel"
    plan.close()


@pytest.mark.parametrize("dtype", [0, 2])
@pytest.mark.parametrize("rows,cols", [(600, 700), (1100, 130)])
def test_infinities_and_nans_stay_with_the_rows_that_name_them(torch_cuda, hs, monkeypatch, dtype, rows, cols):
    """By the rule of the kernels that multiply stored entries only, whose check this is."""
    monkeypatch.setitem(nonfinite.FAMILIES, "tile", (0, {"HSPMM_NARROW": "1"}, (9, 16, 24, 29, 32), "spmm_narrow_kernel"))
    nonfinite.test_infinities_and_nans_stay_with_the_rows_that_name_them(torch_cuda, hs, "tile", dtype, rows, cols)


def test_plans_that_keep_the_callers_cuts_leave_launches_to_the_kernels_that_honour_them(torch_cuda, hs):
    torch = torch_cuda
    rng = np.random.default_rng(8)
    A = _sampled_csr(rng, 4096, 4096, 600, 2, lambda n: rng.integers(1, 3, n))
    grouped = hs.bitmap_to_grouped(hs.csr_to_bitmap(4096, 4096, A["row_ptr"], A["col_idx"], A["values"], 2), min_len=40)
    hs.set_group_cuts(1)
    try:
        kept = hs.Plan(grouped)
    finally:
        hs.set_group_cuts(0)
    free = hs.Plan(grouped)
    assert kept.info()["group_cuts_kept"] == 1 and free.info()["group_cuts_kept"] == 0
    stream = torch.cuda.current_stream().cuda_stream
    for N, chosen, left in ((4, "spmm_narrow_kernel", "spmm_mfma_kernel"), (16, "spmm_narrow_kernel", "spmm_mfma_kernel"), (256, "spmm_wide_kernel", "spmm_panel_kernel")):
        dB = torch.from_numpy(encode(rng.integers(-1, 2, (4096, N)).astype(np.float32), 2).view(np.int16)).cuda()     # (exact sums)
        outs = [torch.full((4096, N), 7, dtype=torch.int16, device="cuda") for _ in range(2)]
        for plan, out, kernel in ((free, outs[0], chosen), (kept, outs[1], left)):
            plan.run(dB.data_ptr(), out.data_ptr(), N, stream)
            assert plan.last_kernel() == kernel, N
        assert torch.equal(outs[0], outs[1])
    kept.close()
    free.close()


@pytest.mark.parametrize("dtype", [0, 2])
def test_sums_beside_an_infinity_do_not_depend_on_what_c_held(torch_cuda, hs, dtype):
    """Two tiles of an odd N share a feature: a wave that sums again reads its own features of C alone.  Sums of real numbers, whose bits
    show the order of the additions; finite features are those of the product without the infinity."""
    torch = torch_cuda
    rng = np.random.default_rng(dtype)
    A = _sampled_csr(rng, 1000, 1500, 200, dtype, lambda n: rng.normal(size=n))
    plan = _plan(hs, A, NARROW=1)
    stream = torch.cuda.current_stream().cuda_stream
    nan = 0x7E01 if dtype == 0 else 0x7FC0
    for N in range(17, 30, 2):
        _, dB = _random_operand(torch, rng, 1500, N, dtype)
        clean = torch.full((1000, N), nan, dtype=torch.int16, device="cuda")
        plan.run(dB.data_ptr(), clean.data_ptr(), N, stream)
        for bad in (0, 13, 14, 15, N - 1):
            worse = dB.clone()
            worse[700, bad] = 0x7C00 if dtype == 0 else 0x7F80
            outs = []
            for held in (nan, 7, nan):
                dC = torch.full((1000, N), held, dtype=torch.int16, device="cuda")
                plan.run(worse.data_ptr(), dC.data_ptr(), N, stream)
                outs.append(dC)
            assert plan.last_kernel() == "spmm_narrow_kernel"
            assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2]), (N, bad)
            fine = [f for f in range(N) if f != bad]
            assert torch.equal(outs[0][:, fine], clean[:, fine]), (N, bad)
    plan.close()


# Against fp64, as for the wide-tile kernels: n additions of exact products, and the result's own rounding.
@pytest.mark.parametrize("dtype,rows,cols,per_row,N,narrow", [
    (2, 4096, 11008, 1100, 16, True), (0, 4096, 4096, 1200, 15, True), (2, 1500, 9001, 2000, 29, True), (0, 4096, 11008, 1100, 1, True),
    (0, 4096, 4096, 40, 16, False), (2, 2048, 2048, 200, 33, False), (1, 4096, 4096, 800, 16, False)])
def test_chosen_where_they_are_faster(torch_cuda, hs, dtype, rows, cols, per_row, N, narrow):
    torch = torch_cuda
    rng = np.random.default_rng(N + dtype)
    A = _sampled_csr(rng, rows, cols, per_row, dtype, lambda n: rng.normal(size=n))
    plan = hs.Plan(convert(hs, A))
    B, dB = _random_operand(torch, rng, cols, N, dtype)
    dC = torch.full((rows, N), 7, dtype=dB.dtype, device="cuda")
    plan.run(dB.data_ptr(), dC.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert (plan.last_kernel() == "spmm_narrow_kernel") == narrow
    if narrow:
        D = np.zeros((rows, cols))
        D[np.repeat(np.arange(rows), per_row), A["col_idx"]] = decode(A["values"], dtype)
        Bm = decode(B, dtype).astype(np.float64)
        bound = per_row * 2.0**-24 * (abs(D) @ abs(Bm))
        want = D @ Bm
        off = abs(decode(dC.cpu().numpy().view(np.uint16), dtype).astype(np.float64) - want)
        assert (off <= bound + (2.0**-11 if dtype == 0 else 2.0**-8) * (abs(want) + bound)).all()
    plan.close()
