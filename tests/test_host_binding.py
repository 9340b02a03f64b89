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
