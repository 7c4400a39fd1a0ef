"""One plan launched on several streams, and first launched by several threads, where its kernels leave sums of parts in memory
and are chosen automatically: cut rows of the entry kernels, cut C tiles of the full-tile kernels."""
import threading

import numpy as np
import pytest

from test_entries_gpu import _rows_of_lengths
from test_spmm_gpu import convert, torch_cuda  # noqa: F401
from test_tile_gpu import _random_operand, _sampled_csr

pytestmark = pytest.mark.gpu


def _entry_rows(rng, dtype):
    lengths = [int(n) for n in rng.integers(0, 12, 6000)]
    for r in (3, 700, 2100, 4444):
        lengths[r] = 1500                               # longer than a launch this short leaves whole
    lengths[5000] = 2600                                # a row in pieces
    return _rows_of_lengths(rng, lengths, 60000, dtype)


CASES = [("entries", 0, 88), ("entries", 1, 24), ("tile", 2, 64), ("tile", 0, 24), ("tile", 1, 16)]


def _case(hs, which, dtype):
    rng = np.random.default_rng(60 + dtype)
    A = _entry_rows(rng, dtype) if which == "entries" else _sampled_csr(rng, 4096, 4096, 1300, dtype, lambda n: rng.normal(size=n))
    return rng, A, convert(hs, A)


def _check_kernel(plan, which):
    assert plan.last_kernel() == {"entries": "spmm_entries_kernel", "tile": "spmm_tile_kernel"}[which]


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
    assert plan.info()["device_bytes"] > one_stream     # (a set of sums and counters each)
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
