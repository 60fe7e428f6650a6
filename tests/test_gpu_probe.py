"""GPU parity of the Adaptive-Budget probe build (budgetformer_amd.probe) against the oracle."""
import numpy as np
import pytest
import torch

from oracle import edge_table as et
from oracle import philox

pytestmark = pytest.mark.gpu


def _setup(n, e, seed, dev):
    from budgetformer_amd.graph import CSRGraph, chung_lu_csr
    rowptr, col = chung_lu_csr(n, e, exponent=2.1, seed=seed)
    g = CSRGraph.from_csr(rowptr, col, n, device=dev)
    src = np.repeat(np.arange(n), np.diff(rowptr))
    return g, np.stack([src, col.astype(np.int64)])


def _pairs(ei):
    return sorted(zip(ei[0].tolist(), ei[1].tolist()))


@pytest.mark.parametrize("layers", [1, 2, 3])
def test_reception_cone_matches_oracle(hip_device, layers):
    from budgetformer_amd.probe import reception_cone
    g, ei = _setup(3000, 12000, 21, hip_device)
    probe = torch.tensor([5, 17, 2999, 1200, 64], dtype=torch.int64)
    got = reception_cone(g, probe.to(hip_device), layers)
    ref = et.reception_cone(ei, probe.numpy(), layers)
    assert np.array_equal(got.cpu().numpy(), np.asarray(ref))


@pytest.mark.parametrize("P,L,thr", [(2, 4, 1024), (4, 4, 16), (3, 5, 8)])
def test_probe_candidates_bit_exact(hip_device, P, L, thr):
    from budgetformer_amd.probe import build_probe, reception_cone
    n, seed = 2500, 42
    g, ei = _setup(n, 20000, P * 7 + L, hip_device)
    rng = np.random.default_rng(P + L)
    u_full = rng.random((n * P, L), dtype=np.float32)
    probe = torch.from_numpy(rng.choice(n, 40, replace=False))
    F = reception_cone(g, probe.to(hip_device), 2)
    Fn = F.cpu().numpy()
    u_F = torch.from_numpy(u_full.reshape(n, P, L)[Fn].reshape(-1, L)).to(hip_device)
    pb = build_probe(g, F, max_real=6, max_rw=6, walk_length=L, walks_per_node=P, edge_seed=seed, u=u_F,
                     hub_threshold=thr)
    pools = et.probe_edge_pools(ei, n, Fn, L, P, u_full)
    for b_r, b_w in [(4, 4), (6, 4), (4, 6), (0, 5), (3, 0), (1, 1)]:
        got = pb.table(b_r, b_w).to_edge_index().cpu().numpy()
        ref = et.assemble_edges_from_pools(pools, n, b_r, b_w, seed)
        if b_r > 0 and b_w > 0:
            assert np.array_equal(got, ref)                 # merged: coalesce order
        else:
            assert _pairs(got) == _pairs(ref)               # one part: the sampled multiset
    typed = pb.typed_edge_index(3, 4).cpu().numpy()
    ref_t = et.assemble_edges_from_pools(pools, n, 3, 4, seed, exphormer=True)
    for t in (0, 1):
        assert _pairs(typed[:2, typed[2] == t]) == _pairs(ref_t[:2, ref_t[2] == t])


def test_probe_token_form_and_attention_index(hip_device):
    from budgetformer_amd.probe import build_probe
    n, P, L, seed = 1500, 2, 4, 7
    g, ei = _setup(n, 9000, 5, hip_device)
    rng = np.random.default_rng(1)
    u_full = rng.random((n * P, L), dtype=np.float32)
    Fn = np.sort(rng.choice(n, 300, replace=False))
    u_F = torch.from_numpy(u_full.reshape(n, P, L)[Fn].reshape(-1, L)).to(hip_device)
    pb = build_probe(g, torch.from_numpy(Fn).to(hip_device), max_real=4, max_rw=4, walk_length=L,
                     walks_per_node=P, edge_seed=seed, u=u_F, global_token=True)
    tab = pb.table(4, 4)
    ref = et.assemble_edges_from_pools(et.probe_edge_pools(ei, n, Fn, L, P, u_full), n, 4, 4, seed,
                                       graphormer_global_token=True)
    assert np.array_equal(tab.to_edge_index().cpu().numpy(), ref)
    idx = tab.attention_index()
    assert idx.n_q == n + 1 and idx.nnz == ref.shape[1]


def test_probe_rows_equal_training_rows_under_philox(hip_device):
    """Without the real pool (no subtraction) a probe row is the training build's row for that query."""
    from budgetformer_amd.edges import build_attention_edges
    from budgetformer_amd.probe import build_probe
    n, P, L, seed = 4000, 2, 4, 99
    g, _ = _setup(n, 30000, 12, hip_device)
    full = build_attention_edges(g, real_edges_per_query=0, rw_edges_per_query=5, walk_length=L,
                                 walks_per_node=P, edge_seed=seed)
    F = torch.arange(7, n, 13, device=hip_device)
    pb = build_probe(g, F, max_real=0, max_rw=5, walk_length=L, walks_per_node=P, edge_seed=seed, use_real=False)
    tab = pb.table(0, 5)
    assert torch.equal(tab.table, full.table[F]) and torch.equal(tab.row_len, full.row_len[F])
    # and the injected-uniform contract reproduces the Philox draw
    u_F = philox.walk_uniforms(0, n, P, L, seed).reshape(n, P, L)[F.cpu().numpy()].reshape(-1, L)
    pb2 = build_probe(g, F, max_real=0, max_rw=5, walk_length=L, walks_per_node=P, edge_seed=seed, use_real=False,
                      u=torch.from_numpy(u_F).to(hip_device))
    assert torch.equal(pb2.table(0, 5).table, tab.table)


def test_probe_wide_budgets_and_long_walks(hip_device):
    """The probe past the LDS staging: the real ranking at max_real = 800 (a workgroup per row, key
    order kept in the row's own slots), the RW ranking of P*L = 10,000 candidates with the real pool
    subtracted (streaming top-k), and candidates of up to 1,000 ids assembled in their table slots;
    bit-exact against the oracle's pools."""
    from budgetformer_amd.probe import build_probe
    n, P, L, seed = 1500, 100, 100, 11
    g, ei = _setup(n, 300_000, 29, hip_device)
    rng = np.random.default_rng(4)
    u_full = rng.random((n * P, L), dtype=np.float32)
    Fn = np.sort(rng.choice(n, 200, replace=False))
    u_F = torch.from_numpy(u_full.reshape(n, P, L)[Fn].reshape(-1, L)).to(hip_device)
    pb = build_probe(g, torch.from_numpy(Fn).to(hip_device), max_real=800, max_rw=500, walk_length=L,
                     walks_per_node=P, edge_seed=seed, u=u_F)
    pools = et.probe_edge_pools(ei, n, Fn, L, P, u_full)
    assert int(pb.real[1].max()) > 768
    for b_r, b_w in [(800, 200), (500, 500), (300, 300), (800, 0), (0, 500)]:
        got = pb.table(b_r, b_w).to_edge_index().cpu().numpy()
        ref = et.assemble_edges_from_pools(pools, n, b_r, b_w, seed)
        if b_r > 0 and b_w > 0:
            assert np.array_equal(got, ref)
        else:
            assert _pairs(got) == _pairs(ref)


@pytest.mark.parametrize("n", [15, 4096, 4097, 9001])
@pytest.mark.parametrize("layers", [2, 4])
def test_cone_and_query_list_at_the_edges_of_their_tiles(hip_device, n, layers):
    """Directed edges (nodes past the last edge id dropped, a hub row longer than a workgroup's share), probe ids out
    of range, repeated and in any order; the query list, its hubs and its flags against numpy."""
    from budgetformer_amd import hip_ops
    from budgetformer_amd.graph import CSRGraph
    from budgetformer_amd.probe import reception_cone
    rng = np.random.default_rng(n + layers)
    top = n - 3                                             # no edge at the last nodes
    ei = np.stack([rng.integers(0, top, 2 * n), rng.integers(0, top, 2 * n)])
    ei = np.concatenate([ei, np.stack([np.arange(top), np.full(top, top // 2)])], axis=1)    # a hub
    ei = et.coalesce(ei, n)
    g = CSRGraph.from_edge_index(torch.from_numpy(ei).to(hip_device), n)
    probe = torch.tensor([3, n - 1, top // 2, 3, -1, n + 5, n - 4], dtype=torch.int64)
    got = reception_cone(g, probe.to(hip_device), layers)
    assert np.array_equal(got.cpu().numpy(), np.asarray(et.reception_cone(ei, probe.numpy(), layers)))
    ids = torch.from_numpy(rng.integers(0, n, n // 2 + 1))
    deg = np.bincount(ei[1], minlength=n)
    hubs = np.flatnonzero(deg > 2).astype(np.int32)
    q, h, has = hip_ops.probe_queries(ids.to(hip_device), g.in_ptr, torch.from_numpy(hubs).to(hip_device))
    uniq = np.unique(ids.numpy())
    assert np.array_equal(q.cpu().numpy(), uniq) and np.array_equal(h.cpu().numpy(), np.intersect1d(hubs, uniq))
    assert has == bool((deg[uniq] > 0).any())
    assert hip_ops.probe_queries(torch.tensor([n - 1], device=hip_device), g.in_ptr)[2] is False
    assert hip_ops.probe_queries(torch.tensor([0, n], device=hip_device), g.in_ptr) is None


def test_probe_refuses_ids_outside_the_graph_and_takes_an_empty_filter(hip_device):
    from budgetformer_amd.probe import build_probe
    g, _ = _setup(500, 3000, 2, hip_device)
    for bad in ([0, 500], [-1, 4]):
        with pytest.raises(ValueError, match="query_ids"):
            build_probe(g, torch.tensor(bad, device=hip_device), max_real=4, max_rw=4)
    pb = build_probe(g, torch.zeros(0, dtype=torch.int64, device=hip_device), max_real=4, max_rw=4)
    assert pb.query_ids.numel() == 0 and not pb.real_nonempty and not pb.rw_nonempty
    assert pb.table(4, 4).to_edge_index().shape == (2, 0)


def test_probe_of_a_graph_of_no_nodes_is_empty(hip_device):
    from budgetformer_amd.graph import CSRGraph
    from budgetformer_amd.probe import build_probe
    ptr = torch.zeros(1, dtype=torch.int64, device=hip_device)
    ids = torch.zeros(0, dtype=torch.int32, device=hip_device)
    pb = build_probe(CSRGraph(ptr, ids, ptr, ids, 0), torch.zeros(0, dtype=torch.int64, device=hip_device), max_real=4,
                     max_rw=4)
    assert pb.query_ids.numel() == 0 and not pb.real_nonempty and not pb.rw_nonempty


@pytest.mark.parametrize("n", [0, 1, 255, 256, 1025, 300_000])
def test_any_nonzero(hip_device, n):
    """Nothing, and a single entry at either end: the read-back page is clean on every call."""
    from budgetformer_amd import hip_ops
    x = torch.zeros(n, dtype=torch.int32, device=hip_device)
    assert not hip_ops.any_nonzero(x)
    for at in {0, n - 1} if n else ():
        x[at] = -1
        assert hip_ops.any_nonzero(x)
        x[at] = 0
        assert not hip_ops.any_nonzero(x)


@pytest.mark.parametrize("dedup", [False, True])
@pytest.mark.parametrize("b_real,b_rw", [(1, 0), (0, 1), (8, 8), (9, 7), (16, 1), (17, 15), (20, 13), (31, 33), (40, 25)])
def test_assemble_rows_by_width(hip_device, b_real, b_rw, dedup):
    """Merged rows on both sides of 16, 32 and 64 entries (a row's lanes, then the LDS form), with repeats within and
    across the parts, empty and full rows, and a last block that is not full; whole numbers, so no tolerance."""
    from budgetformer_amd import hip_ops
    rng = np.random.default_rng(b_real * 100 + b_rw)
    n = 77
    sel = [rng.integers(0, 30, (n, b + 2)).astype(np.int32) for b in (b_real, b_rw)]
    cnt = [rng.integers(0, b + 3, n).astype(np.int32) for b in (b_real, b_rw)]
    for x, b in zip(cnt, (b_real, b_rw)):
        x[0], x[-1] = 0, b + 2
    sel[0][3, 0] = sel[1][3, 0] = 2 ** 31 - 1
    parts = [(torch.from_numpy(s).to(hip_device), torch.from_numpy(c).to(hip_device)) if b else None
             for s, c, b in zip(sel, cnt, (b_real, b_rw))]
    table, row_len = (t.cpu().numpy() for t in hip_ops.assemble_rows(*parts, b_real, b_rw, dedup=dedup))
    for r in range(n):
        row = np.concatenate([s[r, :min(c[r], b)] for s, c, b in zip(sel, cnt, (b_real, b_rw))])
        row = np.unique(row) if dedup else np.sort(row)
        assert row_len[r] == row.size and np.array_equal(table[r], np.pad(row, (0, table.shape[1] - row.size),
                                                                         constant_values=-1))


@pytest.mark.parametrize("layers", [2, 16, 17, 18, 33, 34, 300, 5000])
def test_deep_cones(hip_device, layers):
    """Cones past the hops between two looks (16) and past the levels a byte holds, on a long chain that still grows
    and on a short one that has ended (with another component that is never reached)."""
    from budgetformer_amd.graph import CSRGraph
    from budgetformer_amd.probe import reception_cone
    long, short = 1000, 20
    a = torch.arange(long - 1)
    b = torch.arange(short - 1)
    # every node reaches the next one: the cone of the last node is the nodes before it
    graph = CSRGraph.from_edge_index(torch.stack([a, a + 1]), long, device=hip_device)
    got = reception_cone(graph, torch.tensor([long - 1], device=hip_device), layers)
    assert got.tolist() == list(range(max(long - layers, 0), long))
    both = torch.cat([torch.stack([b, b + 1]), torch.stack([b, b + 1]) + 50], dim=1)
    graph = CSRGraph.from_edge_index(both, 70, device=hip_device)
    got = reception_cone(graph, torch.tensor([short - 1], device=hip_device), layers)
    assert got.tolist() == list(range(max(short - layers, 0), short))


def test_mark_in_neighbors(hip_device):
    """The single hop of the C interface: every source of an edge into the frontier, and nothing unmarked."""
    from budgetformer_amd import hip_ops
    rng = np.random.default_rng(8)
    n = 1003
    src, dst = rng.integers(0, n, 5000), np.sort(rng.integers(0, n, 5000))
    frontier, reached = rng.random(n) < 0.05, rng.random(n) < 0.1
    want = reached.copy()
    want[src[frontier[dst]]] = True
    marks = torch.from_numpy(reached.astype(np.uint8)).to(hip_device)
    hip_ops.mark_in_neighbors(torch.from_numpy(np.searchsorted(dst, np.arange(n + 1))).to(hip_device),
                              torch.from_numpy(src.astype(np.int32)).to(hip_device),
                              torch.from_numpy(frontier.astype(np.uint8)).to(hip_device), marks)
    assert np.array_equal(marks.cpu().numpy().astype(bool), want)
