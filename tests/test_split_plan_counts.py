"""A split plan's counts, read from their pinned copy by several threads at once (no GPU: a stand-in for the event)."""
import threading
import time

import pytest
import torch

from budgetformer_amd.hip_ops import DEVICE_PLAN_MAX_ITEMS, AttentionIndex, SplitPlan


class _Event:
    """Landed from the start; synchronising takes long enough for the other threads to come."""

    def query(self):
        return True

    def synchronize(self):
        time.sleep(0.01)


def test_counts_are_read_once_by_one_of_many_threads(monkeypatch):
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    given, seen, errors = [], [], []
    empty = torch.empty(0, dtype=torch.int32)
    host = torch.tensor([7, 3], dtype=torch.int32)
    plan = SplitPlan(-1, -1, empty, empty, empty, empty, empty, 100, 50)
    plan.host_counts, plan.ready = host, _Event()

    def give():
        given.append(1)
        host.fill_(99)             # the slot is another plan's from here on

    plan._slot = give
    start = threading.Barrier(8)

    def layer(i):
        try:
            start.wait()
            seen.append((plan.pending, plan.items, plan.heavy) if i % 2 else (False, plan.items, plan.heavy))
        except Exception as e:     # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=layer, args=(i,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors and given == [1] and seen == [(False, 7, 3)] * 8


class _CapturedEvent:
    """An event of a copy that has not landed, under a capture that refuses to be asked or waited on."""

    def query(self):
        raise RuntimeError("operation not permitted when stream is capturing")

    synchronize = query


@pytest.mark.parametrize("item_cap", [100, 10 * DEVICE_PLAN_MAX_ITEMS])
def test_a_capturing_stream_neither_waits_nor_asks(monkeypatch, item_cap):
    """An index whose counts are still on their way when a capture starts: its layer launches for the capacities."""
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    empty = torch.empty(0, dtype=torch.int32)
    known = SplitPlan(0, 0, empty, empty, empty, empty)
    plan = SplitPlan(-1, -1, empty, empty, empty, empty, empty, item_cap, 50)
    plan.host_counts, plan.ready = torch.tensor([7, 3], dtype=torch.int32), _CapturedEvent()
    x = torch.zeros(5, dtype=torch.int64)
    idx = AttentionIndex(n_q=4, n_kv=4, qptr=x, kv_all=x, qplan=known, kplan=plan, kptr=x, kq_all=x, korder=x)
    idx._counts = empty
    tensors, ints = idx.op_args(backward=True, per_edge=False)
    assert ints[AttentionIndex._INT_FIELDS.index("k_items")] == item_cap
    assert tensors[AttentionIndex._TENSOR_FIELDS.index("plan_counts")] is empty
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    plan.ready.__class__ = _Event                  # the capture is over and the copy has landed
    plan._slot = lambda: None
    tensors, ints = idx.op_args(backward=True, per_edge=False)
    assert ints[AttentionIndex._INT_FIELDS.index("k_items")] == 7
    assert tensors[AttentionIndex._TENSOR_FIELDS.index("plan_counts")] is None
