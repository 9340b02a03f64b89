"""The native binding of the layer, lookup and rotation calls (csrc/host.cpp) as far as it needs no GPU."""
import os
import pickle
import subprocess
import sys

import pytest
import torch

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


class _SlotsState:
    """pickles like a PreparedLinear whose fields were slots of its own"""

    def __init__(self, **fields):
        self.fields = fields

    def __reduce_ex__(self, protocol):
        from uniql_amd.ops import PreparedLinear
        return object.__new__, (PreparedLinear,), (None, self.fields)


def test_earlier_pickles_of_a_handle_load():
    """the tensors come back whatever device they are mapped to; validation waits for the first use"""
    import copy
    n = k = 256
    fields = dict(B=torch.arange(k // 16 * 2 * n, dtype=torch.int32).reshape(k // 16, 2 * n), s=torch.ones(k // 128, n).half(),
                  workspace=torch.zeros(64, dtype=torch.int32), bias=None, b_ptr=1, s_ptr=2, ws_ptr=3, ws_len=64, bias_ptr=None,
                  size_n=n, size_k=k, n_out=200, groups=2, had_block=128, had_scale=0.25, silu_mul=False, needs={})
    handle = pickle.loads(pickle.dumps(_SlotsState(**fields)))
    for again in (handle, copy.copy(handle), copy.deepcopy(handle), pickle.loads(pickle.dumps(handle))):
        state = again.__getstate__()
        assert torch.equal(state["B"], fields["B"]) and state["n_out"] == 200 and state["had_scale"] == 0.25
        assert "b_ptr" not in state


@pytest.mark.parametrize("missing", ["compiler", "torch"])
def test_the_library_is_installed_without_the_binding(tmp_path, monkeypatch, missing):
    """a build where only the binding fails leaves the new library, says so, and leaves no binding of another build"""
    from uniql_amd import build as B
    lib, host = tmp_path / "libuniql_amd.so", tmp_path / "_host.so"
    lib.write_text("old")
    host.write_text("old")

    def run(cmd, verbose):
        if cmd[0] == "g++":
            raise RuntimeError("g++: not found")
        open(cmd[cmd.index("-o") + 1], "w").write("new")

    def no_torch(dst):
        raise ImportError("No module named 'torch'")

    monkeypatch.setattr(B, "LIB_DIR", str(tmp_path))
    monkeypatch.setattr(B, "LIB_PATH", str(lib))
    monkeypatch.setattr(B, "HOST_PATH", str(host))
    monkeypatch.setattr(B, "_run", run)
    if missing == "torch":
        monkeypatch.setattr(B, "_host_command", no_torch)
    with pytest.raises(RuntimeError, match="_host.so"):
        B.build(verbose=False)
    assert lib.read_text() == "new" and sorted(os.listdir(tmp_path)) == ["libuniql_amd.so"]
