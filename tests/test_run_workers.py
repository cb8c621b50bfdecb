"""run_workers: every worker on a thread of its own that Python's threading knows, results and exceptions in order."""
import threading

import pytest

from drone_amd.pagerank import run_workers


def test_every_worker_has_its_own_thread():
    caller, here, together = threading.current_thread(), threading.local(), threading.Barrier(3)
    here.device = "the caller's"
    traced = []

    def work(i):
        me = threading.current_thread()
        assert me is not caller and me in threading.enumerate() and not me.daemon
        assert not hasattr(here, "device")  # what belongs to a thread (the current GPU, say) is not the caller's
        here.device = i
        together.wait(20)                   # all of them run at once
        return i, me.ident

    threading.settrace(lambda *a: traced.append(threading.get_ident()))
    try:
        got = run_workers([lambda i=i: work(i) for i in range(3)])
    finally:
        threading.settrace(None)
    assert [g[0] for g in got] == [0, 1, 2] and len({g[1] for g in got}) == 3
    assert {g[1] for g in got} <= set(traced)
    assert here.device == "the caller's"


def test_exceptions_and_no_workers():
    def fail(i):
        raise (KeyError if i == 1 else ValueError)(i)

    with pytest.raises(KeyError, match="1"):
        run_workers([lambda: 0, lambda: fail(1), lambda: fail(2)])
    assert run_workers([]) == []
