"""The entry kernels (narrow feature dimensions: stored entries in units of four, rows sorted by length) at the sizes
where they can go wrong: lane widths and blocks that end inside a row, rows on both sides of every class of lengths,
rows cut into pieces, rows without entries, plans whose windows were paired."""
import os

import numpy as np
import pytest

from test_spmm_gpu import assert_parity, convert, gpu_spmm, make_b, oracle_spmm, torch_cuda  # noqa: F401
from util import decode, encode

pytestmark = pytest.mark.gpu


def _rows_of_lengths(rng, lengths, cols, dtype):
    lists = [np.sort(rng.choice(cols, size=n, replace=False)) for n in lengths]
    row_ptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint32)
    col_idx = np.concatenate(lists).astype(np.uint32)
    return dict(rows=len(lengths), cols=cols, nnzs=int(col_idx.size), dtype=dtype, row_ptr=row_ptr, col_idx=col_idx,
                values=encode(rng.uniform(-1, 1, col_idx.size), dtype))


def _plan(hs, A, always=True):
    if always:
        os.environ["HSPMM_ENTRIES"] = "1"
    try:
        return hs.Plan(convert(hs, A))
    finally:
        os.environ.pop("HSPMM_ENTRIES", None)


def _check_guarded(torch, plan, A, B, N, dtype, ref, mag, what):
    es, guard = (4, 32) if dtype == 1 else (2, 64)
    tt = torch.float32 if dtype == 1 else torch.int16
    buf = torch.full((A["rows"] * N + 2 * guard,), 7, dtype=tt, device="cuda")
    dB = torch.from_numpy(B if dtype == 1 else np.ascontiguousarray(B).view(np.int16)).cuda()
    dC = buf[guard:guard + A["rows"] * N]
    for _ in range(2):                                              # (counters of cut rows are zero again after a launch)
        dC.fill_(0x7E01 if dtype != 1 else float("nan"))
        plan.run(dB.data_ptr(), dC.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        info = plan.info()
        assert info["last_kernel_family"] == 2 and info["last_mfma_kind"] == 0, what
        out = buf.cpu().numpy()
        assert (out[:guard] == 7).all() and (out[-guard:] == 7).all(), what + ": wrote outside C"
        got = out[guard:-guard].reshape(A["rows"], N)
        assert_parity(got if dtype == 1 else got.view(np.uint16), ref, mag, dtype, what, tight=False)


@pytest.mark.parametrize("dtype", [0, 1, 2])
def test_every_width_and_class_of_lengths(torch_cuda, hs, oracle, dtype):
    torch = torch_cuda
    rng = np.random.default_rng(400 + dtype)
    # units of four: 1 .. 4, then both sides of 4, 8, 16 .. 512 units, above which rows are cut into pieces
    lengths = [0, 1, 2, 3, 4, 5, 8, 9, 12, 13, 16, 17, 20, 0, 0, 32, 33, 63, 64, 65, 128, 129, 255, 256, 257, 0, 512, 513, 1024,
               1025, 2047, 2048, 2049, 4096, 4097, 5001] + [0] * 9 + [7] * 70 + [41]
    A = _rows_of_lengths(rng, lengths, 6000, dtype)
    plan = _plan(hs, A)
    for N in (1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 31, 33, 48, 64, 65, 100, 128) + (() if dtype == 1 else (129, 200, 255, 256)):
        B = make_b(rng, A["cols"], N, dtype)
        ref, mag = oracle_spmm(oracle, A, B, N)
        _check_guarded(torch, plan, A, B, N, dtype, ref, mag, "N=%d" % N)
    plan.close()


@pytest.mark.parametrize("dtype", [0, 1, 2])
def test_rows_cut_into_parts_and_wide_rows_in_blocks(torch_cuda, hs, oracle, dtype):
    torch = torch_cuda
    rng = np.random.default_rng(405 + dtype)
    # mostly short rows; the others on both sides of the lengths at which one, two, four ... parts are taken, and of a piece
    lengths = [2] * 1500 + [0, 32, 33, 64, 65, 128, 129, 257, 511, 513, 1025, 2048, 2049, 2500]
    A = _rows_of_lengths(rng, lengths, 2600, dtype)
    plan = _plan(hs, A)
    for N in (130, 135, 257, 260, 376, 512) + (() if dtype == 1 else (513, 720, 1023, 1024)):
        B = make_b(rng, A["cols"], N, dtype)
        ref, mag = oracle_spmm(oracle, A, B, N)
        _check_guarded(torch, plan, A, B, N, dtype, ref, mag, "N=%d" % N)
    plan.close()


@pytest.mark.parametrize("dtype,cols,N", [(0, 40000, 128), (1, 40000, 64), (1, 20000, 128)])
def test_blocks_on_xcds_of_their_own(torch_cuda, hs, oracle, dtype, cols, N):
    torch = torch_cuda
    rng = np.random.default_rng(410 + dtype)
    A = _rows_of_lengths(rng, list(rng.integers(0, 40, 3001)), cols, dtype)
    plan = _plan(hs, A, always=False)
    B = make_b(rng, cols, N, dtype)
    ref, mag = oracle_spmm(oracle, A, B, N)
    _check_guarded(torch, plan, A, B, N, dtype, ref, mag, "xcd blocks")
    plan.close()


@pytest.mark.parametrize("dtype", [0, 1])
def test_paired_windows_static_entry_point_and_capture(torch_cuda, hs, oracle, dtype):
    torch = torch_cuda
    rng = np.random.default_rng(420 + dtype)
    # rows of one 16-row block share their columns (paired windows); two rows longer than a piece
    lists = [np.sort(rng.choice(9000, 5000 if b == 1 else 40, replace=False)) for b in range(3) for _ in (0,)]
    per_row = [lists[r // 16] for r in range(48)]
    row_ptr = np.concatenate([[0], np.cumsum([len(x) for x in per_row])]).astype(np.uint32)
    A = dict(rows=48, cols=9000, dtype=dtype, row_ptr=row_ptr, col_idx=np.concatenate(per_row).astype(np.uint32),
             values=encode(rng.integers(-3, 4, int(row_ptr[-1])).astype(np.float32), dtype))
    A["nnzs"] = int(row_ptr[-1])
    plan = _plan(hs, A)
    assert plan.info()["n_paired_units"] > 0
    N = 8
    B = encode(rng.integers(-4, 5, (9000, N)).astype(np.float32), dtype)      # exact: one rounding of the exact sum
    tt = torch.float32 if dtype == 1 else torch.int16
    dB = torch.from_numpy(B if dtype == 1 else B.view(np.int16)).cuda()
    dC = torch.full((48, N), 7, dtype=tt, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    with pytest.raises(hs.HspmmError) as e:
        plan.run_static(dB.data_ptr(), dC.data_ptr(), N, stream)
    assert "hspmm_prepare" in str(e.value)
    plan.prepare(N)
    held = plan.info()["device_bytes"]
    want = oracle_spmm(oracle, A, B, N)[0]
    for _ in range(2):
        dC.fill_(7)
        plan.run_static(dB.data_ptr(), dC.data_ptr(), N, stream)
        torch.cuda.synchronize()
        assert np.array_equal(dC.cpu().numpy().view(np.uint8), np.ascontiguousarray(want).view(np.uint8))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        plan.run(dB.data_ptr(), dC.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
    assert plan.info()["device_bytes"] == held
    for _ in range(3):
        dC.fill_(7)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(dC.cpu().numpy().view(np.uint8), np.ascontiguousarray(want).view(np.uint8))
    del graph
    plan.close()


@pytest.mark.parametrize("N,lengths,cols,family", [
    (1024, [2001] * 1150 + [1] * 10500, 4001, 2),       # parts of cut rows: 36 MiB of sums; uncut rows leave none
    (1024, [2100] * 5400, 2200, 3),                     # pieces of rows above 2048 entries: 42 MiB in any case
])
def test_sums_that_do_not_fit_the_fixed_array_choose_another_shape(torch_cuda, hs, N, lengths, cols, family):
    """hspmm_run_static serves what hspmm_prepare has prepared, and its results are those of hspmm_run."""
    torch = torch_cuda
    rng = np.random.default_rng(95)
    n = np.asarray(lengths)
    start = np.concatenate([[0], np.cumsum(n)]).astype(np.int64)
    place = np.arange(start[-1]) - np.repeat(start[:-1], n)
    col_idx = (place * (cols // np.repeat(n, n)) + np.repeat(rng.integers(0, 2, n.size) * (cols % 2), n)) % cols
    A = dict(rows=n.size, cols=cols, nnzs=int(start[-1]), dtype=0, row_ptr=start.astype(np.uint32), col_idx=col_idx.astype(np.uint32),
             values=encode(rng.integers(1, 4, int(start[-1])).astype(np.float32), 0))
    plan = _plan(hs, A)
    B = rng.integers(-1, 2, (cols, N)).astype(np.float32)
    dB = torch.from_numpy(encode(B, 0).view(np.int16)).cuda()
    outs = [torch.full((n.size, N), 7, dtype=torch.int16, device="cuda") for _ in range(2)]
    stream = torch.cuda.current_stream().cuda_stream
    plan.prepare(N)
    plan.run_static(dB.data_ptr(), outs[0].data_ptr(), N, stream)
    plan.run(dB.data_ptr(), outs[1].data_ptr(), N, stream)
    torch.cuda.synchronize()
    assert plan.info()["last_kernel_family"] == family
    assert torch.equal(outs[0], outs[1])
    rows = np.concatenate([np.arange(4), rng.integers(0, n.size, 20), [n.size - 1]])
    got = outs[0].cpu().numpy().view(np.float16)
    for r in rows:
        s = slice(start[r], start[r + 1])
        want = (decode(A["values"][s], 0)[:, None] * B[col_idx[s]]).sum(0)
        assert np.array_equal(got[r].astype(np.float64), want.astype(np.float16).astype(np.float64)), "row %d" % r
    plan.close()


def test_without_memory_for_the_stream_the_other_kernels_serve(torch_cuda, hs, oracle):
    """The stream of stored entries is a second copy of the matrix, made by the first launch that wants it: when the device
    has no room for it, that launch and all that follow go to the kernels that need none."""
    torch = torch_cuda
    rng = np.random.default_rng(97)
    rows, per_row, N = 1 << 17, 64, 16
    col_idx = (np.arange(per_row, dtype=np.int64)[None, :] * (rows // per_row) + rng.integers(0, rows // per_row, (rows, per_row)))
    A = dict(rows=rows, cols=rows, nnzs=rows * per_row, dtype=1, row_ptr=(np.arange(rows + 1, dtype=np.int64) * per_row).astype(np.uint32),
             col_idx=col_idx.astype(np.uint32).reshape(-1), values=rng.integers(1, 4, rows * per_row).astype(np.float32))
    B = rng.integers(-4, 5, (rows, N)).astype(np.float32)
    dB = torch.from_numpy(B).cuda()
    outs = [torch.full((rows, N), float("nan"), device="cuda") for _ in range(3)]
    stream = torch.cuda.current_stream().cuda_stream
    plan = hs.Plan(convert(hs, A))
    torch.cuda.empty_cache()
    rest = [torch.empty(torch.cuda.mem_get_info()[0] - (1 << 30), dtype=torch.uint8, device="cuda")]
    for _ in range(512):                                # what is left, down to one block: the stream takes 67 MB
        try:
            rest.append(torch.empty(24 << 20, dtype=torch.uint8, device="cuda"))
        except torch.OutOfMemoryError:
            break
    rest.pop()
    torch.cuda.empty_cache()
    try:
        plan.run(dB.data_ptr(), outs[0].data_ptr(), N, stream)
        assert plan.info()["last_kernel_family"] == 2 and plan.info()["last_mfma_kind"] != 0
    finally:
        torch.cuda.synchronize()
        del rest
        torch.cuda.empty_cache()
    plan.run(dB.data_ptr(), outs[1].data_ptr(), N, stream)          # (room again: the plan's results do not change)
    assert plan.info()["last_mfma_kind"] != 0
    other = hs.Plan(convert(hs, A))
    other.run(dB.data_ptr(), outs[2].data_ptr(), N, stream)
    assert other.info()["last_mfma_kind"] == 0
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])      # (small whole numbers: every order gives the same)
    want = oracle_spmm(oracle, A, B, N)[0]
    assert np.array_equal(outs[0].cpu().numpy(), want)
    plan.close()
    other.close()


# (rows of B of 1 to 9 blocks: whole lines in blocks of one, two and four lines, and rows that begin anywhere)
@pytest.mark.parametrize("dtype,widths", [(0, (72, 150, 192, 320, 448, 543, 576, 640, 700, 896, 1000)), (2, (66, 171, 384, 529, 832)),
                                          (1, (35, 75, 96, 160, 192, 224, 288, 300, 448, 500))])
def test_every_number_of_blocks_a_row_is_cut_into(torch_cuda, hs, oracle, dtype, widths):
    torch = torch_cuda
    rng = np.random.default_rng(430 + dtype)
    for cols, lengths in ((9000, list(rng.integers(0, 30, 900))), (700, [3] * 600 + [0, 257, 600])):
        A = _rows_of_lengths(rng, lengths, cols, dtype)
        plan = _plan(hs, A)
        for N in widths:
            B = make_b(rng, cols, N, dtype)
            ref, mag = oracle_spmm(oracle, A, B, N)
            _check_guarded(torch, plan, A, B, N, dtype, ref, mag, "cols=%d N=%d" % (cols, N))
        plan.close()
