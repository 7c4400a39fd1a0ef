"""One plan launched on several streams, first launched by several threads, and recorded in a graph, where its kernels leave sums of parts
in memory and are chosen automatically - cut rows of the entry kernels, cut C tiles of the full-tile and the wide-tile kernels, cut windows
of the gather kernels' schedule -, and the narrow and the block kernels, which leave none."""
import threading

import numpy as np
import pytest

from test_block_gpu import _blocks, _csr
from test_entries_gpu import _rows_of_lengths
from test_schedule_gpu import _hot
from test_spmm_gpu import convert, torch_cuda  # noqa: F401
from test_tile_gpu import _random_operand, _sampled_csr

pytestmark = pytest.mark.gpu


def _entry_rows(rng, dtype):
    lengths = [int(n) for n in rng.integers(0, 12, 6000)]
    for r in (3, 700, 2100, 4444):
        lengths[r] = 1500                               # longer than a launch this short leaves whole
    lengths[5000] = 2600                                # a row in pieces
    return _rows_of_lengths(rng, lengths, 60000, dtype)


# (entries, N = 65 and 301: rows of an odd number of elements, one block and several)
CASES = [("entries", 0, 88), ("entries", 1, 24), ("entries", 2, 65), ("entries", 0, 301), ("tile", 2, 64), ("tile", 0, 24), ("tile", 1, 16),
         ("wide", 2, 64), ("wide", 0, 333), ("narrow", 0, 16), ("narrow", 2, 29),
         ("block", 0, 16), ("block", 2, 31), ("block", 1, 47), ("mfma", 0, 128)]


def _case(hs, which, dtype):
    rng = np.random.default_rng(60 + dtype)
    if which == "entries":
        A = _entry_rows(rng, dtype)
    elif which == "block":
        mask = _blocks(rng, 1024, 2000, 0.4)
        A = _csr(mask, rng.normal(size=int(mask.sum())), dtype)
    elif which == "mfma":
        A = _hot(rng, 1 << 18, 1 << 18, 6)[0]
    else:
        rows, cols, per_row = {"tile": (4096, 4096, 1300), "wide": (512, 11008, 1100), "narrow": (4096, 4096, 600)}[which]
        A = _sampled_csr(rng, rows, cols, per_row, dtype, lambda n: rng.normal(size=n))
    return rng, A, convert(hs, A)


def _check_kernel(plan, which):
    assert plan.last_kernel() == "spmm_%s_kernel" % which
    assert plan.last_walk()["scheduled"] == (which == "mfma") and (which != "mfma" or plan.last_walk()["split_windows"])


def _lane(torch, rng, A, N, dtype):
    _, dB = _random_operand(torch, rng, A["cols"], N, dtype)
    return dB, torch.full((A["rows"], N), 7, dtype=dB.dtype, device="cuda"), torch.cuda.Stream()


@pytest.mark.parametrize("which,dtype,N", CASES)
def test_launches_on_three_streams_leave_each_others_sums_alone(torch_cuda, hs, which, dtype, N):
    torch = torch_cuda
    rng, A, b = _case(hs, which, dtype)
    plan = hs.Plan(b)
    lanes, alone = [_lane(torch, rng, A, N, dtype) for _ in range(3)], []
    for dB, dC, _ in lanes:
        plan.run(dB.data_ptr(), dC.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
        _check_kernel(plan, which)
        torch.cuda.synchronize()
        alone.append(dC.clone())
        dC.fill_(7)
    torch.cuda.synchronize()
    one_stream = plan.info()["device_bytes"]
    for _ in range(30):
        for dB, dC, stream in lanes:
            plan.run(dB.data_ptr(), dC.data_ptr(), N, stream.cuda_stream)
    torch.cuda.synchronize()
    assert (plan.info()["device_bytes"] > one_stream) == (which not in ("narrow", "block"))      # (a set of sums and counters each)
    for (_, dC, _), want in zip(lanes, alone):
        assert torch.equal(dC.view(torch.uint8), want.view(torch.uint8))
    plan.close()


@pytest.mark.parametrize("which,dtype,N", CASES)
def test_first_launches_of_a_plan_by_several_threads(torch_cuda, hs, which, dtype, N):
    torch = torch_cuda
    rng, A, b = _case(hs, which, dtype)
    dB, want, _ = _lane(torch, rng, A, N, dtype)
    plan = hs.Plan(b)
    plan.run(dB.data_ptr(), want.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    plan.close()
    for _ in range(4):
        plan = hs.Plan(b)
        outs, streams = [torch.full_like(want, 7) for _ in range(4)], [torch.cuda.Stream() for _ in range(4)]
        torch.cuda.synchronize()
        start, errors = threading.Barrier(4), []

        def first(k):
            try:
                start.wait()
                for _ in range(3):
                    plan.run(dB.data_ptr(), outs[k].data_ptr(), N, streams[k].cuda_stream)
            except Exception as e:                      # noqa: BLE001 (reported below)
                errors.append(e)

        threads = [threading.Thread(target=first, args=(k,)) for k in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        torch.cuda.synchronize()
        assert not errors, errors
        for out in outs:
            assert torch.equal(out.view(torch.uint8), want.view(torch.uint8))
        plan.close()


@pytest.mark.parametrize("which,dtype,N", [c for c in CASES if c[0] != "tile"])
def test_launches_recorded_on_a_stream_the_plan_has_not_seen(torch_cuda, hs, which, dtype, N):
    """What hspmm_prepare has made is enough to record a launch; every replay, between eager launches with other numbers, gives the bits
    of an eager launch."""
    torch = torch_cuda
    rng, A, b = _case(hs, which, dtype)
    plan = hs.Plan(b)
    dB, dC, side = _lane(torch, rng, A, N, dtype)
    other, _, _ = _lane(torch, rng, A, N, dtype)
    eager = torch.full_like(dC, 7)
    plan.prepare(N)
    before = plan.info()["device_bytes"]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        plan.run(dB.data_ptr(), dC.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
    assert plan.info()["device_bytes"] == before
    _check_kernel(plan, which)
    first, second = dB.clone(), other.clone()
    for replay in range(5):
        dB.copy_(second if replay % 2 else first)
        dC.fill_(7)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        eager.fill_(7)
        plan.run(dB.data_ptr(), eager.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(dC.view(torch.uint8), eager.view(torch.uint8)), "replay %d" % replay
    del graph
    plan.close()


def test_threads_that_ask_for_other_feature_dimensions_in_turn(torch_cuda, hs):
    """The kernel and the shape of a launch are kept by feature dimension, in words that all threads share."""
    torch = torch_cuda
    rng, A, b = _case(hs, "wide", 2)
    plan = hs.Plan(b)
    widths = [16, 29, 32, 33, 64, 96, 128, 130, 256, 333, 512, 1024]
    work = []
    for N in widths:
        dB, want, _ = _lane(torch, rng, A, N, 2)
        plan.run(dB.data_ptr(), want.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
        work.append((N, dB, want))
    torch.cuda.synchronize()
    outs = [[torch.full_like(want, 7) for _, _, want in work] for _ in range(4)]
    streams, errors = [torch.cuda.Stream() for _ in range(4)], []
    torch.cuda.synchronize()

    def launch(k):
        try:
            for i in range(3 * len(work)):
                j = (i * 5 + k) % len(work)
                N, dB, _ = work[j]
                plan.run(dB.data_ptr(), outs[k][j].data_ptr(), N, streams[k].cuda_stream)
        except Exception as e:                          # noqa: BLE001 (reported below)
            errors.append(e)

    threads = [threading.Thread(target=launch, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for k in range(4):
        for j, (N, _, want) in enumerate(work):
            assert torch.equal(outs[k][j].view(torch.uint8), want.view(torch.uint8)), (k, N)
    plan.close()
