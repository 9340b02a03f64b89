"""The native binding of the layer, lookup and rotation calls (csrc/host.cpp) as far as it needs no GPU."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

FIRST_USE = """
import sys, threading
sys.path.insert(0, {root!r})
from uniql_amd import _capi
_capi.load()
sys.setswitchinterval(1e-6)
for _ in range(60):
    # as in a process that has not used the binding yet
    _capi._host = None
    sys.modules.pop("uniql_amd._host", None)
    start, seen, errors = threading.Barrier(16), [], []
    def use():
        start.wait()
        try:
            seen.append((_capi.host(), _capi.host().Linear, _capi.host().embedding))
        except BaseException as e:
            errors.append(repr(e))
    threads = [threading.Thread(target=use) for _ in range(16)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not errors, errors
    assert len(seen) == 16
"""


def test_first_use_by_several_threads():
    """every thread gets the whole module, bound, however the first calls fall together"""
    done = subprocess.run([sys.executable, "-c", FIRST_USE.format(root=ROOT)], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stderr[-2000:]

OTHER_THREADS = """
import sys, threading, time
sys.path.insert(0, {root!r})
import torch
from uniql_amd import _capi, ops
torch.set_num_threads(1)
n = k = 256
handle = _capi.host().Linear(torch.zeros(k // 16, 2 * n, dtype=torch.int32), torch.zeros(k // 128, n, dtype=torch.half),
                             torch.zeros(64, dtype=torch.int32), None, n, k, n, 0, 1.0, False)
x = torch.zeros(1, k, 300000, dtype=torch.half).transpose(1, 2)   # rows that have to be copied first
ticks, stop = [], False
def tick():
    while not stop:
        ticks.append(time.perf_counter())
        time.sleep(0)
other = threading.Thread(target=tick)
other.start()
time.sleep(0.05)
began = time.perf_counter()
try:
    handle.forward(x, None, False, 0, ops._accumulator)
    raise SystemExit("a CPU tensor was taken")
except RuntimeError as e:
    assert "must be a GPU tensor" in str(e), e
ended = time.perf_counter()
stop = True
other.join()
inside = [began] + [t for t in ticks if began < t < ended] + [ended]
longest = max(b - a for a, b in zip(inside, inside[1:]))
assert ended - began > 0.02, ended - began
assert longest < 0.5 * (ended - began), (longest, ended - began)
"""


def test_other_threads_run_while_a_call_waits():
    """the interpreter lock is given up for a call's own copies too, not only for its launch"""
    done = subprocess.run([sys.executable, "-c", OTHER_THREADS.format(root=ROOT)], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stderr[-2000:]
