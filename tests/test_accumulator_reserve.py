"""The words that captures find zeroed (uniql_amd.ops), as far as they are plain bookkeeping: host tensors in the place of
device memory."""
import types

import pytest
import torch

from uniql_amd import ops

DEVICE = torch.device("cuda", 0)


@pytest.fixture
def host_memory(monkeypatch):
    """torch.zeros on the CPU, no streams; `fail` names the step that raises"""
    state = types.SimpleNamespace(fail=None)
    zeros = torch.zeros

    def host_zeros(words, dtype, device):
        if state.fail == "zeros" and words == ops._RESERVE_WORDS:
            raise RuntimeError("operation not permitted when stream is capturing")
        return zeros(words, dtype=dtype)

    def wait():
        if state.fail == "wait":
            raise RuntimeError("operation not permitted when stream is capturing")

    for name in ("_accum_cache", "_accum_in_capture", "_accum_reserve"):
        monkeypatch.setattr(ops, name, {})
    monkeypatch.setattr(ops, "_accum_retired", [])
    monkeypatch.setattr(ops, "_RESERVE_WORDS", 1 << 12)
    monkeypatch.setattr(ops, "_RESERVE_SHARE", 1 << 9)
    monkeypatch.setattr(ops, "_capture_id", lambda stream: 0)
    monkeypatch.setattr(ops.torch, "zeros", host_zeros)
    monkeypatch.setattr(ops.torch.cuda, "current_stream", lambda device: types.SimpleNamespace(synchronize=wait))
    return state


@pytest.mark.parametrize("step", ["zeros", "wait"])
def test_a_call_does_not_fail_for_words_it_does_not_need(host_memory, step):
    host_memory.fail = step
    assert ops._accumulator(DEVICE, 1 << 10, stream=7).numel() * 8 >= 1 << 10
    assert not ops._accum_reserve and ops._from_reserve(DEVICE, 256) is None
    host_memory.fail = None
    ops._accumulator(DEVICE, 1 << 10, stream=8)      # the next new buffer
    assert ops._from_reserve(DEVICE, 256) is not None
