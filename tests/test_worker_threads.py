"""The converters share a pool of waiting worker threads: callers on several threads at once, and a process forked from one
whose threads are waiting, get what a caller alone gets."""
import multiprocessing
import threading

import numpy as np

from util import random_csr


def _convert(hs, A):
    b = hs.csr_to_btcf(A["rows"], A["cols"], A["row_ptr"], A["col_idx"], A["values"], A["dtype"])
    m = hs.csr_to_bitmap(A["rows"], A["cols"], A["row_ptr"], A["col_idx"], A["values"], A["dtype"])
    return [b[k] for k in ("rowOffset", "tcA2B", "data", "rowIdx")] + [m[k] for k in ("nnzOffset", "tcBit", "data")]


def _matrices():
    rng = np.random.default_rng(5)
    return [random_csr(rng, 9000, 3000, density, dtype, 0.1) for density, dtype in ((0.01, 0), (0.02, 1), (0.004, 2))]


def _same(got, want):
    return all(a.tobytes() == b.tobytes() for a, b in zip(got, want))


def test_conversions_on_several_threads_at_once(hs):
    matrices = _matrices()
    alone = [_convert(hs, A) for A in matrices]
    wrong = []

    def work(k):
        for i in range(4):
            which = (k + i) % len(matrices)
            if not _same(_convert(hs, matrices[which]), alone[which]):
                wrong.append((k, i))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    assert not any(t.is_alive() for t in threads) and not wrong


def _child(conn, A, want):
    import hopper_spmm_amd as hs
    conn.send(_same(_convert(hs, A), want))
    conn.close()


def test_conversions_in_processes_forked_while_the_threads_wait(hs):
    matrices = _matrices()
    alone = [_convert(hs, A) for A in matrices]                    # (the pool's threads wait for a second from here on)
    fork = multiprocessing.get_context("fork")
    children = []
    for A, want in zip(matrices, alone):
        here, there = fork.Pipe(duplex=False)
        p = fork.Process(target=_child, args=(there, A, want))
        p.start()
        children.append((p, here))
    for p, here in children:
        assert here.poll(60), "a forked process did not answer"
        assert here.recv()
        p.join(timeout=60)
        assert p.exitcode == 0
    assert all(_same(_convert(hs, A), want) for A, want in zip(matrices, alone))
