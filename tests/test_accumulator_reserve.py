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

    for name in ("_accum_cache", "_accum_in_capture", "_accum_reserve", "_accum_reserve_old"):
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


def test_shares_outlive_a_reset_and_are_not_handed_out_again(host_memory):
    """a graph that was captured before reset_accumulators() may be replayed by mistake: its words stay allocated, and no
    later capture gets them"""
    import gc
    import weakref
    spans, roots = [], []

    def take(words):
        share = ops._from_reserve(DEVICE, 8 * words)
        assert share is not None and int(share.count_nonzero()) == 0
        spans.append((share.data_ptr(), share.data_ptr() + 8 * share.numel()))

    for words in (512, 64, 512, 512, 512, 512):     # more than half of the first reserve: the last ones come from a second
        ops._accumulator(DEVICE, 1 << 10, stream=7)
        roots.append(weakref.ref(ops._accum_reserve[0][0]))
        take(words)
        take(32)
        ops.reset_accumulators()
        assert not ops._accum_reserve and not ops._accum_cache
        gc.collect()
        assert all(root() is not None for root in roots)
    spans.sort()
    assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:]))
    assert len({w.untyped_storage().data_ptr() for w, _ in ops._accum_reserve_old[0]}) == 2
