"""An index's sort keys, dropped by the first backward, when that runs on another stream than the index's build."""
import numpy as np
import pytest
import torch

from budgetformer_amd import hip_ops
from budgetformer_amd.hip_ops import AttentionIndex, ReverseKeys


class _Keys:
    """Stands in for a device tensor: notes the streams it is recorded on."""
    device = torch.device("cuda", 0)

    def __init__(self):
        self.recorded = []

    def record_stream(self, stream):
        self.recorded.append(stream)


@pytest.mark.parametrize("built_on,used_on", [(7, 7), (7, 8)])
@pytest.mark.parametrize("kind", ["list", "table", "slots"])
def test_keys_are_recorded_on_the_stream_that_spends_them(monkeypatch, kind, built_on, used_on):
    monkeypatch.setattr(hip_ops, "_raw_stream", lambda device: used_on, raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: used_on)
    some = torch.zeros(4, dtype=torch.int64)
    keys = _Keys()
    rk = ReverseKeys(keys, 3, 2, False, -1)
    later = ReverseKeys(_Keys(), 3, 2, False, -1)
    idx = AttentionIndex(n_q=3, n_kv=3, qptr=some, kv_all=some, qplan=object(), kplan=object(), korder=some)
    idx._key_stream = built_on
    monkeypatch.setattr(hip_ops, "coo_reverse", lambda *a: (some, some))
    monkeypatch.setattr(hip_ops, "reverse_index_packed", lambda *a, **k: (some, some, None, later))
    monkeypatch.setattr(hip_ops, "reverse_slots", lambda *a: some)
    if kind == "list":
        idx._coo_keys = (keys, False)
    elif kind == "table":
        idx._rkeys = rk
    else:
        idx.kptr, idx._sorted = some, rk
    if kind == "slots":
        idx.ensure_entries()
    else:
        idx.ensure_backward()
    assert idx._coo_keys is None and idx._rkeys is None
    assert keys.recorded == ([] if built_on == used_on else [used_on])
    if kind == "table":          # the sorted keys are the using stream's own, until a third one needs the slots
        monkeypatch.setattr(hip_ops, "_raw_stream", lambda device: 9)
        monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: 9)
        idx.ensure_entries()
        assert later.keys.recorded == [9]


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["list", "table"])
def test_first_backward_on_another_stream(hip_device, how):
    """Built on one stream, sorted late on another (behind a long wait), while the first allocates and fills blocks of
    the keys' size: the reverse index is numpy's."""
    n, width = 20_000, 8
    rng = np.random.default_rng(3)
    ids = np.sort(np.minimum((n * rng.random((n, width)) ** 3).astype(np.int64), n - 1), axis=1)
    kv, q = ids.ravel(), np.repeat(np.arange(n), width)
    table = torch.from_numpy(ids.astype(np.int32)).to(hip_device)
    row_len = torch.full((n,), width, dtype=torch.int32, device=hip_device)
    coo = torch.from_numpy(np.stack([kv, q])).to(hip_device)
    build, use = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(build):
        idx = AttentionIndex.from_table(table, row_len, n_kv=n, check=False) if how == "table" else \
            AttentionIndex.from_coo(coo, n)
    use.wait_stream(build)
    with torch.cuda.stream(use):
        torch.cuda._sleep(20_000_000)
        idx.ensure_backward()
    with torch.cuda.stream(build):
        taken = [torch.full((n * width,), -1, dtype=torch.int64, device=hip_device) for _ in range(8)]
    torch.cuda.synchronize()
    del taken
    order = np.argsort(kv, kind="stable")
    assert np.array_equal(idx.kptr.cpu().numpy(), np.searchsorted(kv[order], np.arange(n + 1)))
    assert np.array_equal(idx.kq.cpu().numpy(), q[order])
