"""The re-integration queue's count of working waves (work_queue.hpp, built for
the host): over every interleaving of the atomic operations of a wave with work
and one that asks whether the queue has drained, the answer is never "drained"
while anything is left to do or can still be queued, and it is given once
nothing is."""
import ctypes
import os
import subprocess

import pytest

EMUL = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emul")


@pytest.mark.parametrize("kind", [0, 1, 2], ids=["queue", "trace_ahead", "last_chunk"])
def test_drained_only_when_nothing_is_left(kind):
    subprocess.run(["make", "-s", "-C", EMUL, "libqueue_emul.so"], check=True)
    h = ctypes.CDLL(os.path.join(EMUL, "libqueue_emul.so"))
    h.emul_queue.restype = ctypes.c_longlong
    h.emul_queue.argtypes = [ctypes.c_int, ctypes.c_void_p]
    runs = (ctypes.c_longlong * 2)()
    wrong = h.emul_queue(kind, runs)
    print(kind, list(runs), wrong)
    assert wrong == 0 and runs[0] > 100 and runs[1] > 0
