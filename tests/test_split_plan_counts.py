"""A split plan's counts, read from their pinned copy by several threads at once (no GPU: a stand-in for the event)."""
import threading
import time

import torch

from budgetformer_amd.hip_ops import SplitPlan


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
