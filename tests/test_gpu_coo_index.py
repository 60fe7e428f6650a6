"""An edge list's index (coo_rows_to_csr, coo_reverse, coo_reverse_slots) and its coalesced form against numpy, for
every order a list can come in: none, column order, coalesced (column-major), row-major, with repeated entries,
typed or not, and the two lists the sorts never see (empty, one entry). Integer work: bit-exact."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

N_Q, N_KV = 70, 4000


def _list(order, nnz, typed, seed):
    rng = np.random.default_rng(seed)
    kv = np.minimum((N_KV * rng.random(nnz) ** 3).astype(np.int64), N_KV - 3)     # skewed, the last ids unused
    q = rng.integers(0, N_Q - 2, nnz)
    t = rng.integers(0, 2, nnz) if typed else np.zeros(nnz, dtype=np.int64)
    if nnz > 20:
        kv[10:14], q[10:14], t[10:14] = kv[10], q[10], t[10]                       # a pair four times over
    keys = {"none": None, "by_col": (kv, t), "col_major": (q, kv, t), "row_major": (kv, t, q)}[order]
    if keys is not None:
        o = np.lexsort(keys)
        kv, q, t = kv[o], q[o], t[o]
    return kv, q, t


@pytest.mark.parametrize("typed", [False, True])
@pytest.mark.parametrize("order", ["none", "by_col", "col_major", "row_major"])
@pytest.mark.parametrize("nnz", [1, 1023, 1024, 70_001])
def test_list_index_in_every_order(hip_device, order, nnz, typed):
    from budgetformer_amd import hip_ops
    kv, q, t = _list(order, nnz, typed, nnz)
    dev = [torch.from_numpy(x).to(hip_device) for x in (q, kv, t)]
    qptr, ids, keys = hip_ops.coo_rows_to_csr(dev[0], dev[1], N_Q, N_KV, dev[2] if typed else None, with_keys=True)
    kptr, kq = hip_ops.coo_reverse(keys, N_Q, N_KV, typed)
    ks = hip_ops.coo_reverse_slots(qptr, ids, kptr, kq)
    o = np.lexsort((kv, t, q))                       # rows ascend by (type, kv)
    kv, q, t = kv[o], q[o], t[o]
    slot = np.arange(nnz) - np.searchsorted(q, q)
    assert np.array_equal(qptr.cpu().numpy(), np.searchsorted(q, np.arange(N_Q + 1)))
    assert np.array_equal(ids.cpu().numpy().view(np.uint32), (kv | (t << 31)).astype(np.uint32))
    r = np.argsort(kv, kind="stable")
    assert np.array_equal(kptr.cpu().numpy(), np.searchsorted(kv[r], np.arange(N_KV + 1)))
    assert np.array_equal(kq.cpu().numpy().view(np.uint32), (q[r] | (t[r] << 31)).astype(np.uint32))
    assert np.array_equal(ks.cpu().numpy(), slot[r])
    if not typed:
        ref = hip_ops.reverse_index(qptr, ids, N_KV)
        assert all(torch.equal(a, b) for a, b in zip((kptr, kq, ks), ref))


def test_typed_index_takes_an_id_and_its_type_as_one_number(hip_device):
    """(n_kv + i, type 0) is (i, type 1); what no pair gives is refused."""
    from budgetformer_amd.hip_ops import AttentionIndex
    ei = torch.tensor([[3, 5, 1], [0, 1, 1], [0, 1, 0]], device=hip_device)
    same = torch.tensor([[3, 15, 1], [0, 1, 1], [0, 0, 0]], device=hip_device)
    a, b = AttentionIndex.from_typed_coo(ei, 2, 10), AttentionIndex.from_typed_coo(same, 2, 10)
    assert torch.equal(a.kv, b.kv) and torch.equal(a.kq, b.kq) and torch.equal(a.ks, b.ks)
    for bad, what in (([[20], [0], [0]], "ids outside"), ([[3], [2], [0]], "ids outside"), ([[3], [0], [2]], "types")):
        with pytest.raises(ValueError, match=what):
            AttentionIndex.from_typed_coo(torch.tensor(bad, device=hip_device), 2, 10)
    for bad in ([[10], [0]], [[-1], [0]], [[0], [2]], [[0], [-1]]):
        with pytest.raises(ValueError, match="ids outside"):
            AttentionIndex.from_coo(torch.tensor(bad, device=hip_device), 2, 10)


def test_slots_of_a_list_index_come_on_first_use(hip_device):
    from budgetformer_amd.hip_ops import AttentionIndex
    kv, q, _ = _list("none", 3000, False, 5)
    ei = torch.from_numpy(np.stack([kv, q])).to(hip_device)
    a = AttentionIndex.from_coo(ei, N_Q, N_KV).ensure_backward()
    assert a.ks_all is None
    b = AttentionIndex.from_coo(ei, N_Q, N_KV).ensure_backward(entries=True)
    assert b.ks_all is not None and torch.equal(a.ks, b.ks) and torch.equal(a.to_coo(), b.to_coo())
    empty = AttentionIndex.from_coo(ei[:, :0], N_Q, N_KV).ensure_backward()
    assert empty.nnz == 0 and int(empty.qptr[-1]) == 0 and int(empty.kptr[-1]) == 0


@pytest.mark.parametrize("nnz", [0, 1, 4096, 4097, 100_003])
@pytest.mark.parametrize("n", [50, 3001])
def test_coalesce_and_bidirected(hip_device, nnz, n):
    """Many duplicates (50 nodes) and few; a coalesced list comes back equal, in memory of its own."""
    from budgetformer_amd import hip_ops
    from budgetformer_amd.graph import to_bidirected
    rng = np.random.default_rng(nnz + n)
    ei = rng.integers(0, n, (2, nnz))

    def ref(x):
        return np.stack(np.divmod(np.unique(x[0] * n + x[1]), n)) if x.size else x

    dev = torch.from_numpy(ei).to(hip_device)
    got = hip_ops.coalesce(dev, n)
    assert np.array_equal(got.cpu().numpy(), ref(ei))
    assert np.array_equal(to_bidirected(dev, n).cpu().numpy(), ref(np.concatenate([ei, ei[::-1]], axis=1)))
    again = hip_ops.coalesce(got, n)
    assert torch.equal(again, got) and (nnz == 0 or again.data_ptr() != got.data_ptr())
    # both CSRs of the list as it comes, of its coalesced form, and of the coalesced list itself
    for x, flag in ((dev, False), (dev, True), (again, True), (again.flip(0), False)):
        e = ref(ei) if flag else x.cpu().numpy()
        out = hip_ops.graph_csrs(x, n, coalesced=flag)
        for ptr, ids, r, c in ((out[0], out[1], e[0], e[1]), (out[2], out[3], e[1], e[0])):
            o = np.lexsort((c, r))
            assert np.array_equal(ptr.cpu().numpy(), np.searchsorted(r[o], np.arange(n + 1)))
            assert np.array_equal(ids.cpu().numpy(), c[o])
    if nnz:
        for bad in (n, -1):
            dev[0, 0] = bad
            with pytest.raises(ValueError, match="ids outside"):
                hip_ops.graph_csrs(dev, n)


@pytest.mark.parametrize("token", [False, True])
@pytest.mark.parametrize("how", ["full", "shard", "ids"])
@pytest.mark.parametrize("n_rows,width", [(1, 1), (511, 3), (513, 8), (5000, 33), (530_000, 2)])
def test_table_to_list_equals_the_index_route(hip_device, n_rows, width, how, token):
    """A table's list against its CSR's reverse index (the route it replaces) and fix_edge_index's order; rows empty,
    full and past a block of rows, one row with the multiset's repeated id; bad tables refused."""
    from budgetformer_amd.edges import EdgeTable
    from budgetformer_amd.hip_ops import AttentionIndex
    rng = np.random.default_rng(n_rows + width)
    n = max(6000, n_rows + 800)
    ids = np.sort(np.minimum((n * rng.random((n_rows, width)) ** 3).astype(np.int32), n - 1), axis=1)
    ids[0, -1] = n - 1
    if width > 2:
        ids[0, 1] = ids[0, 0]
    row_len = rng.integers(0, width + 1, n_rows).astype(np.int32)
    row_len[0] = width
    ids[np.arange(width)[None, :] >= row_len[:, None]] = -1
    table, lens = torch.from_numpy(ids).to(hip_device), torch.from_numpy(row_len).to(hip_device)
    q_lo = 700 if how == "shard" else 0
    qids = torch.arange(3, 3 + n_rows, dtype=torch.int32, device=hip_device) if how == "ids" else None
    tab = EdgeTable(table, lens, n, q_lo=q_lo, global_token=token, query_ids=qids)
    got = tab.to_edge_index()
    coo = AttentionIndex.from_table(table, lens, False, n_kv=n).to_coo()
    ref = torch.stack([coo[0], coo[1] + (3 if how == "ids" else q_lo)])
    if token:
        ar = torch.arange(1, n + 1, device=hip_device)
        rows = ar if how == "ids" else torch.arange(q_lo + 1, q_lo + n_rows + 1, device=hip_device)
        parts = [ref + 1] + ([torch.stack([ar, torch.zeros_like(ar)])] if how != "shard" else [])
        ref = torch.cat(parts + [torch.stack([torch.zeros_like(rows), rows])], dim=1)
    assert torch.equal(got, ref)
    table[-1, 0], lens[-1] = n, 1
    with pytest.raises(ValueError, match="table ids outside"):
        EdgeTable(table, lens, n).to_edge_index()
    lens[-1] = width + 1
    with pytest.raises(ValueError, match="row lengths outside"):
        EdgeTable(table, lens, n).to_edge_index()


def test_table_of_two_to_the_32_entries_is_refused(hip_device):
    """1024 blocks of rows whose lengths add up to 2^32 exactly (0 in 32 bits): refused for its size, and for its ids
    where those are bad as well. 17 GB of table, no list is written."""
    from budgetformer_amd.edges import EdgeTable
    if torch.cuda.mem_get_info(hip_device)[0] < 40 * 2 ** 30:
        pytest.skip("needs 17 GB for the table")
    n_rows, width = 1024 * 512, 8192
    table = torch.zeros(n_rows, width, dtype=torch.int32, device=hip_device)
    lens = torch.full((n_rows,), width, dtype=torch.int32, device=hip_device)
    with pytest.raises(ValueError, match=f"{n_rows * width} entries"):
        EdgeTable(table, lens, 5).to_edge_index()
    table.fill_(-1)
    with pytest.raises(ValueError, match=f"{n_rows * width} table ids outside"):
        EdgeTable(table, lens, 5).to_edge_index()
    del table
    torch.cuda.empty_cache()


@pytest.mark.parametrize("n_rows", [1, 63, 4095, 4096, 4097, 70_000])
@pytest.mark.parametrize("threshold,item,share", [(8, 3, 0.01), (1, 1, 1.0), (1000, 768, 0.0)])
def test_split_plan_at_block_edges(hip_device, n_rows, threshold, item, share):
    """Few rows to split, every row, none; one row of more items than a wave has lanes, at the end of a block."""
    from budgetformer_amd import hip_ops
    rng = np.random.default_rng(n_rows + threshold)
    lens = rng.integers(0, threshold + 1, n_rows)
    lens[rng.random(n_rows) < share] += threshold + 5
    lens[min(n_rows - 1, 4095)] += 150 * item if share else 0
    ptr = np.concatenate([[0], np.cumsum(lens)])
    plan = hip_ops.split_plan(torch.from_numpy(ptr).to(hip_device), int(ptr[-1]), threshold, item)
    n = np.array([hip_ops.split_row_items(int(x), item) if x > threshold else 0 for x in lens])
    off = np.concatenate([[0], np.cumsum(n)])[:-1]
    assert (plan.items, plan.heavy) == (n.sum(), (n > 0).sum())
    assert np.array_equal(plan.nitems.cpu().numpy()[:n_rows], n)
    assert np.array_equal(plan.item_off.cpu().numpy()[:n_rows], off)
    assert np.array_equal(plan.item_row.cpu().numpy()[:plan.items], np.repeat(np.arange(n_rows), n))
    assert np.array_equal(plan.heavy_rows.cpu().numpy()[:plan.heavy], np.flatnonzero(n))


def test_list_calls_refuse_and_take_what_they_did(hip_device):
    """Empty graphs and lists without columns are refused; a coalesced list of any shape comes back [2, E]; a table
    list takes query ids past its rows."""
    from budgetformer_amd import hip_ops
    from budgetformer_amd.edges import EdgeTable
    from budgetformer_amd.graph import CSRGraph
    from budgetformer_amd.hip_ops import AttentionIndex
    none = torch.zeros(2, 0, dtype=torch.int64, device=hip_device)
    for call in (lambda: CSRGraph.from_edge_index(none, 0), lambda: hip_ops.graph_csrs(none, 0, coalesced=True),
                 lambda: hip_ops.coo_to_csr(none, 3, 0), lambda: AttentionIndex.from_coo(none, 0),
                 lambda: AttentionIndex.from_typed_coo(torch.cat([none, none[:1]]), 3, 0),
                 lambda: hip_ops.coalesce(none, 0)):
        with pytest.raises(ValueError):
            call()
    ei = torch.tensor([[0, 1, 1, 4], [2, 0, 3, 4]], device=hip_device)
    assert torch.equal(hip_ops.coalesce(ei.view(2, 2, 2), 5), ei)
    assert torch.equal(hip_ops.graph_csrs(ei.view(2, 2, 2), 5, coalesced=True)[1].long(), ei[1])
    table = torch.tensor([[0, 2], [1, -1]], dtype=torch.int32, device=hip_device)
    lens = torch.tensor([2, 1], dtype=torch.int32, device=hip_device)
    ids = torch.tensor([3, 4, 0], dtype=torch.int32, device=hip_device)
    got = EdgeTable(table, lens, 5, query_ids=ids).to_edge_index()
    assert got.tolist() == [[0, 1, 2], [3, 4, 3]]
    with pytest.raises(ValueError, match="query_ids"):
        EdgeTable(table, lens, 5, query_ids=ids[:1]).to_edge_index()


@pytest.mark.parametrize("n_rows", [255, 256, 257, 5000, 1_048_576, 1_048_577, 4_194_304, 4_194_305])
def test_split_plan_of_rows_in_order_of_length(hip_device, n_rows):
    """Long rows next to each other, as in a graph numbered by degree: rows of no item, of fewer items than their lane
    writes, of more, and of more than a wave has lanes; at the edges of the plan's three forms."""
    from budgetformer_amd import hip_ops
    lens = np.minimum(40_000.0 / (1.0 + np.arange(n_rows)) ** 0.9, 9000.0).astype(np.int64)
    ptr = np.concatenate([[0], np.cumsum(lens)])
    for threshold, item in ((32, 32), (3, 50)):
        plan = hip_ops.split_plan(torch.from_numpy(ptr).to(hip_device), int(ptr[-1]), threshold, item)
        split = lens > threshold
        n = np.zeros(n_rows, dtype=np.int64)
        n[split] = [hip_ops.split_row_items(int(x), item) for x in lens[split]]
        assert (plan.items, plan.heavy) == (n.sum(), split.sum())
        assert np.array_equal(plan.nitems.cpu().numpy()[:n_rows], n)
        assert np.array_equal(plan.item_off.cpu().numpy()[:n_rows], np.cumsum(n) - n)
        assert np.array_equal(plan.item_row.cpu().numpy()[:plan.items], np.repeat(np.arange(n_rows), n))
        assert np.array_equal(plan.heavy_rows.cpu().numpy()[:plan.heavy], np.flatnonzero(split))


@pytest.mark.parametrize("n_rows", [0, 1, 257, 1_100_000])
def test_rows_longer_than(hip_device, n_rows):
    """The hub lists of a graph: several thresholds at once, one that no row passes, an empty CSR."""
    from budgetformer_amd import hip_ops
    lens = np.minimum((3.0 / np.maximum(np.random.default_rng(n_rows).random(n_rows), 1e-4)).astype(np.int64), 20_000)
    ptr = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)])).to(hip_device)
    got = hip_ops.rows_longer_than(ptr, int(lens.sum()), (32, 1, 1024, 30_000))
    for t, ids in zip((32, 1, 1024, 30_000), got):
        assert ids.dtype == torch.int32 and np.array_equal(ids.cpu().numpy(), np.flatnonzero(lens > t))
    with pytest.raises(ValueError):
        hip_ops.rows_longer_than(ptr, int(lens.sum()), (32, 0))
