"""The reference module's selection, noise, backup and subtree operators on the GPU (through
torch_ops, the accelerator class and the C ABI) against the numpy restatements and the C
oracle, bit for bit: random dense tables with negative and out-of-range entries, coarse values
(exact ties), per-simulation priors and legal masks; Dirichlet rows against the oracle's gamma
stream; random trees and graphs with repeated children and cycles, with levels beyond one
1024-thread chunk."""
import numpy as np
import pytest
import torch

from omoknuni_quantum_amd import _lib, torch_ops
from omoknuni_quantum_amd.mcts_gpu_accelerator import get_mcts_gpu_accelerator
from oracle import ref_np

from test_reference_ops_more import (EDGE_EXPECT, PSVL_EXPECT, UCBD_EXPECT, _csr, _edge_case,
                                     _psvl_case, _ucbd_case, dirichlet_rows)

pytestmark = pytest.mark.gpu
F = np.float32


def _t(a, device):
    return torch.from_numpy(np.ascontiguousarray(a)).to(device)


def _np(x):
    torch.cuda.synchronize()
    return x.cpu().numpy()


# ---- parallel_select_with_virtual_loss -------------------------------------------------------
def test_psvl_known_answer_on_gpu(device):
    parents, children, N, VL, W, P, acts, masks = _psvl_case()
    vl = _t(VL, device)
    sel = torch_ops.parallel_select_with_virtual_loss(
        _t(parents, device), _t(children, device), _t(N, device), vl, _t(W, device),
        _t(P, device), None, _t(masks, device), _t(acts, device), 1.0, -1.0, 0.0, True)
    assert _np(sel).tolist() == PSVL_EXPECT
    _, vl_want = ref_np.parallel_select_with_virtual_loss(parents, children, N, VL, W, P, acts,
                                                          1.0, -1.0, masks)
    assert _np(vl).tolist() == vl_want.tolist()


@pytest.mark.parametrize("seed,mc,per_sim,masked", [(0, 8, False, False), (1, 64, False, True),
                                                    (2, 65, True, False), (3, 300, True, True),
                                                    (4, 1000, True, True)])
def test_psvl_random(device, seed, mc, per_sim, masked):
    rng = np.random.default_rng(40 + seed)
    nn, S, A = 1500, 2100, 50
    ch = rng.integers(-2, nn + 3, (nn, mc)).astype(np.int32)  # negatives and ids past the nodes
    N = rng.integers(0, 6, nn).astype(np.int32)
    VL = rng.integers(0, 3, nn).astype(np.int32)
    W = (np.round(rng.random(nn) * 16 - 8) / 8).astype(F)
    acts = rng.integers(-1, A + 2, nn).astype(np.int32)
    parents = rng.integers(-2, nn + 2, S).astype(np.int32)
    parents[:50] = 0  # the root, which ignores the masks
    if per_sim:
        P = (np.round(rng.random((S, nn - 7)) * 8) / 8).astype(F)  # children past it skipped
    else:
        P = (np.round(rng.random(nn) * 8) / 8).astype(F)
    masks = rng.random((S, A)) < 0.7 if masked else None
    exp, vl_exp = ref_np.parallel_select_with_virtual_loss(parents, ch, N, VL, W, P, acts, 1.4,
                                                           1.0, masks)
    vl = _t(VL, device)
    got = torch_ops.parallel_select_with_virtual_loss(
        _t(parents, device), _t(ch, device), _t(N, device), vl, _t(W, device), _t(P, device),
        None, _t(masks, device) if masked else None, _t(acts, device), 1.4, 1.0, 0.0, masked)
    assert np.array_equal(_np(got), exp)
    assert np.array_equal(_np(vl), vl_exp)


def test_psvl_accelerator_method(device):
    """MCTSGPUAccelerator.parallel_select_with_virtual_loss (mcts_gpu_accelerator.py:289-297):
    nine arguments, no masks."""
    parents, children, N, VL, W, P, acts, masks = _psvl_case()
    acc = get_mcts_gpu_accelerator(device)
    got = acc.parallel_select_with_virtual_loss(
        _t(parents, device), _t(children, device), _t(N, device), _t(VL, device),
        _t(W, device), _t(P, device), _t(acts, device), 1.0, -1.0)
    exp, _ = ref_np.parallel_select_with_virtual_loss(parents, children, N, VL, W, P, acts, 1.0,
                                                      -1.0, None)
    assert np.array_equal(_np(got), exp)


# ---- fused_ucb_with_noise ----------------------------------------------------------------------
@pytest.mark.parametrize("C", [1, 64, 65, 362, 4672])
def test_fused_ucb_with_noise_random(device, C):
    rng = np.random.default_rng(C)
    S = 700
    q = (np.round(rng.random(C) * 8 - 4) / 8).astype(F)
    n = rng.integers(0, 5, C).astype(np.int32)
    p = (np.round(rng.random(C) * 8) / 8).astype(F)
    noise = (np.round(rng.random((S, C)) * 4) / 4).astype(F)
    noise[:3] = 0.0  # identical rows: exact ties settle on the lowest position
    exp = ref_np.fused_ucb_with_noise(q, n, p, noise, 3.0, 1.4, 0.25)
    got = torch_ops.fused_ucb_with_noise(_t(q, device), _t(n, device), _t(p, device),
                                         _t(noise, device), 3.0, 1.4, 0.25)
    assert np.array_equal(_np(got), exp)
    acc = get_mcts_gpu_accelerator(device)
    got2 = acc.fused_ucb_with_noise(_t(q, device), _t(n, device), _t(p, device),
                                    _t(noise, device), 3.0, 1.4, 0.25)
    assert np.array_equal(_np(got2), exp)
    low = np.full(C, -1e11, F)  # nothing above -1e10: position 0
    got3 = torch_ops.fused_ucb_with_noise(_t(low, device), _t(n, device), _t(p, device),
                                          _t(noise, device), 3.0, 1.4, 0.25)
    assert not _np(got3).any()


# ---- batched_ucb_selection_dense -------------------------------------------------------------
def test_ucb_dense_known_answer_on_gpu(device):
    args = [_t(a, device) for a in _ucbd_case()]
    assert _np(torch_ops.batched_ucb_selection_dense(*args, 1.0)).tolist() == UCBD_EXPECT


@pytest.mark.parametrize("M", [3, 64, 65, 200, 1000])
def test_ucb_dense_random(device, M):
    rng = np.random.default_rng(100 + M)
    B, NV = 1300, 400
    bc = rng.integers(-2, NV + 3, (B, M)).astype(np.int32)
    bp = (np.round(rng.random((B, M)) * 8) / 8).astype(F)
    valid = rng.random((B, M)) < 0.8
    pv = rng.integers(0, 30, B).astype(np.int32)
    cn = rng.integers(0, 4, NV).astype(np.int32)
    cv = (np.round(rng.random(NV) * 8 - 4) / 8).astype(F)
    exp = ref_np.batched_ucb_selection_dense(bc, bp, pv, cn, cv, valid, 1.4)
    got = torch_ops.batched_ucb_selection_dense(_t(bc, device), _t(bp, device), _t(pv, device),
                                                _t(cn, device), _t(cv, device),
                                                _t(valid, device), 1.4)
    assert np.array_equal(_np(got), exp)


# ---- batched_dirichlet_noise -------------------------------------------------------------------
@pytest.mark.parametrize("S,A,alpha", [(5, 362, 0.03), (40, 225, 0.3), (3, 1, 1.5),
                                       (7, 70, 2.5), (2, 4672, 0.3)])
def test_dirichlet_rows_match_oracle(device, S, A, alpha):
    torch_ops.set_noise_seed(1234)
    got = torch_ops.batched_dirichlet_noise(S, A, alpha, 0.25, device)
    got2 = torch_ops.batched_dirichlet_noise(S, A, alpha, 0.25, device)  # counter 1
    assert np.array_equal(_np(got), dirichlet_rows(S, A, alpha, 1234, 0))
    assert np.array_equal(_np(got2), dirichlet_rows(S, A, alpha, 1234, 1))
    acc = get_mcts_gpu_accelerator(device)
    got3 = acc.batched_dirichlet_noise(S, A, alpha, 0.25, device)  # counter 2
    assert np.array_equal(_np(got3), dirichlet_rows(S, A, alpha, 1234, 2))


# ---- optimized_backup_scatter -------------------------------------------------------------------
def test_optimized_backup_scatter_equals_vectorized_backup(device):
    rng = np.random.default_rng(9)
    B, D, nn = 300, 7, 80
    paths = rng.integers(-1, nn + 2, (B, D)).astype(np.int32)
    plen = rng.integers(0, D + 2, B).astype(np.int32)
    vals = (rng.integers(-4, 5, B) / 4).astype(F)  # exact sums in any order
    # expected: per path, d < min(len, D), node in range: N += 1, W += v (-1)^(len-1-d)
    n_exp = np.zeros(nn, np.int32)
    w_exp = np.zeros(nn, np.float64)
    for b in range(B):
        L = int(plen[b])
        for d in range(min(L, D)):
            x = int(paths[b, d])
            if 0 <= x < nn:
                n_exp[x] += 1
                w_exp[x] += vals[b] * (-1) ** (L - 1 - d)
    n1, w1 = torch.zeros(nn, dtype=torch.int32, device=device), torch.zeros(nn, device=device)
    torch_ops.optimized_backup_scatter(_t(paths, device), _t(plen, device), _t(vals, device),
                                       n1, w1)
    acc = get_mcts_gpu_accelerator(device)
    n2, w2 = torch.zeros_like(n1), torch.zeros_like(w1)
    acc.optimized_backup_scatter(_t(paths, device), _t(plen, device), _t(vals, device), n2, w2)
    n3, w3 = torch.zeros_like(n1), torch.zeros_like(w1)
    torch_ops.vectorized_backup(_t(paths, device), _t(plen, device), _t(vals, device), n3, w3)
    assert np.array_equal(_np(n1), n_exp) and np.array_equal(_np(w1), w_exp.astype(F))
    assert torch.equal(n1, n2) and torch.equal(w1, w2)
    assert torch.equal(n1, n3) and torch.equal(w1, w3)


@pytest.mark.parametrize("B,D,nn", [(1, 1, 1), (256, 9, 4000), (257, 8, 40), (700, 20, 5000)])
def test_backup_and_virtual_loss_node_tables(device, B, D, nn):
    """Paths whose workgroup meets more distinct nodes than its table holds, fewer, and entries
    past the levels that go through it; the same nodes as a virtual-loss list of several
    workgroups."""
    rng = np.random.default_rng(B)
    paths = rng.integers(-1, nn + 1, (B, D)).astype(np.int32)
    paths[:, 0] = 0
    plen = np.full(B, D, np.int32)
    vals = (rng.integers(-4, 5, B) / 4).astype(F)  # exact sums in any order
    n_exp, w_exp = np.zeros(nn, np.int64), np.zeros(nn, np.float64)
    on = (paths >= 0) & (paths < nn)
    sign = np.where((D - 1 - np.arange(D)) % 2 == 0, 1.0, -1.0)
    np.add.at(n_exp, paths[on], 1)
    np.add.at(w_exp, paths[on], (vals[:, None] * sign)[on])
    n, w = torch.zeros(nn, dtype=torch.int32, device=device), torch.zeros(nn, device=device)
    torch_ops.vectorized_backup(_t(paths, device), _t(plen, device), _t(vals, device), n, w)
    assert np.array_equal(_np(n), n_exp) and np.array_equal(_np(w), w_exp.astype(F))
    vl = torch.zeros(nn, dtype=torch.int32, device=device)
    torch_ops.batch_apply_virtual_loss(_t(paths.reshape(-1), device), vl)
    assert np.array_equal(_np(vl), n_exp)
    torch_ops.batch_remove_virtual_loss(_t(paths.reshape(-1), device), vl)
    assert not _np(vl).any()


@pytest.mark.parametrize("n", [1, 255, 257, 16384, 16385, 40_000])
@pytest.mark.parametrize("kind", ["one node", "in order", "shuffled", "few", "runs"])
def test_virtual_loss_lists(device, n, kind):
    """Lists around the sizes where the work per thread changes: one node throughout, distinct
    nodes in and out of order, a few nodes often, and runs of consecutive nodes that repeat, with
    entries outside the array."""
    rng = np.random.default_rng(n)
    nn = 50_000
    idx = {"one node": np.full(n, 77), "in order": 3 + np.arange(n),
           "shuffled": rng.permutation(nn)[:n], "few": rng.integers(0, 9, n) ** 4,
           "runs": (np.arange(n) % 640) + np.where(np.arange(n) % 1000 < 700, 0, nn - 300),
           }[kind].astype(np.int32)
    want = np.zeros(nn, np.int64)
    np.add.at(want, idx[idx < nn], 1)
    vl = torch.zeros(nn, dtype=torch.int32, device=device)
    torch_ops.batch_apply_virtual_loss(_t(idx, device), vl)
    assert np.array_equal(_np(vl), want)
    torch_ops.batch_remove_virtual_loss(_t(idx, device), vl)
    assert not _np(vl).any()


@pytest.mark.parametrize("trees,paths", [(1, 2000), (64, 64), (300, 300)])
def test_backup_of_tree_paths(device, trees, paths):
    """Root-to-leaf paths of one and of many trees (one path each): workgroups whose nodes are
    nearly all shared, and not at all."""
    rng = np.random.default_rng(trees)
    D, per, fan = 20, 3000, 3
    P = np.full((paths, D), -1, np.int32)
    plen = np.zeros(paths, np.int32)
    for b in range(paths):
        node, up = int(rng.integers(0, per)), []
        while node > 0:
            up.append(node)
            node = (node - 1) // fan
        up = [0] + up[::-1]
        plen[b] = len(up)
        P[b, :len(up)] = np.array(up) + (b % trees) * per
    nn = per * trees
    vals = (rng.integers(-4, 5, paths) / 4).astype(F)  # exact sums in any order
    n_exp, w_exp = np.zeros(nn, np.int64), np.zeros(nn, np.float64)
    for b in range(paths):
        for d in range(plen[b]):
            n_exp[P[b, d]] += 1
            w_exp[P[b, d]] += vals[b] * (1.0 if (plen[b] - 1 - d) % 2 == 0 else -1.0)
    n, w = torch.zeros(nn, dtype=torch.int32, device=device), torch.zeros(nn, device=device)
    torch_ops.vectorized_backup(_t(P, device), _t(plen, device), _t(vals, device), n, w)
    assert np.array_equal(_np(n), n_exp) and np.array_equal(_np(w), w_exp.astype(F))


@pytest.mark.parametrize("paths", [1, 63, 64, 65, 129, 8192, 8193])
@pytest.mark.parametrize("shared", [3, 13, 30])
def test_backup_of_batches_around_the_workgroup_sizes(device, paths, shared):
    """Paths that follow one line for their first levels (past the levels that meet in LDS, and to
    the end), of several lengths, with padding and entries outside the array on the way."""
    rng = np.random.default_rng(paths + shared)
    D, nn = 30, 30 * paths + 40
    P = np.where(np.arange(D) < shared, np.arange(D), 40 + np.arange(paths * D).reshape(paths, D))
    plen = np.where(rng.random(paths) < 0.7, D, rng.integers(0, D + 5, paths)).astype(np.int32)
    odd = rng.random((paths, D)) < 0.02
    P = np.where(odd, rng.choice([-1, nn, nn + 7], (paths, D)), P).astype(np.int32)
    vals = (rng.integers(-4, 5, paths) / 4).astype(F)  # exact sums in any order
    d = np.arange(D)
    on = (d < plen[:, None]) & (P >= 0) & (P < nn)
    sign = np.where((plen[:, None] - 1 - d) % 2 == 0, 1.0, -1.0)
    n_exp, w_exp = np.zeros(nn, np.int64), np.zeros(nn, np.float64)
    np.add.at(n_exp, P[on], 1)
    np.add.at(w_exp, P[on], (vals[:, None] * sign)[on])
    n, w = torch.zeros(nn, dtype=torch.int32, device=device), torch.zeros(nn, device=device)
    torch_ops.vectorized_backup(_t(P, device), _t(plen, device), _t(vals, device), n, w)
    assert np.array_equal(_np(n), n_exp) and np.array_equal(_np(w), w_exp.astype(F))


# ---- parallel_bfs_subtree / extract_subtree_edges --------------------------------------------
def _check_subtree(device, rows, root, n, actions=True):
    ptr, col = _csr(rows)
    ins_e, remap_e, k_e = ref_np.parallel_bfs_subtree(ptr, col, root, n)
    ins, remap, cnt = torch_ops.parallel_bfs_subtree(_t(ptr, device), _t(col, device), root, n)
    assert int(_np(cnt)[0]) == k_e
    assert np.array_equal(_np(ins), ins_e) and np.array_equal(_np(remap), remap_e)
    act = np.arange(len(col)).astype(np.int16) if actions else None
    pe, ce, ae = ref_np.extract_subtree_edges(ptr, col, act, ins_e, remap_e)
    p, c, a = torch_ops.extract_subtree_edges(_t(ptr, device), _t(col, device),
                                              _t(act, device) if actions else None, ins, remap,
                                              max(len(col), 1))
    assert np.array_equal(_np(p), pe) and np.array_equal(_np(c), ce)
    assert np.array_equal(_np(a), ae)


def test_subtree_known_answers_on_gpu(device):
    from test_reference_ops_more import G_DAG, G_TREE
    _check_subtree(device, G_TREE, 0, 8)
    _check_subtree(device, G_TREE, 1, 8, actions=False)
    _check_subtree(device, G_DAG, 0, 5)
    _check_subtree(device, G_DAG, 1, 5)
    ptr, col, act, ins, remap = _edge_case()
    p, c, a = torch_ops.extract_subtree_edges(_t(ptr, device), _t(col, device), _t(act, device),
                                              _t(ins, device), _t(remap, device), 20)
    assert (_np(p).tolist(), _np(c).tolist(), _np(a).tolist()) == EDGE_EXPECT
    with pytest.raises(RuntimeError, match="max_edges"):
        torch_ops.extract_subtree_edges(_t(ptr, device), _t(col, device), _t(act, device),
                                        _t(ins, device), _t(remap, device), 6)


@pytest.mark.parametrize("seed", range(4))
def test_subtree_random_trees(device, seed):
    """Random trees (levels beyond one 1024-thread chunk in the wide ones) and the subtree of
    a random node."""
    rng = np.random.default_rng(60 + seed)
    n = [3000, 20000, 60000, 5][seed]
    fan = [2, 40, 300, 3][seed]
    parent = [-1] + [max(0, i - 1 - int(rng.integers(0, fan))) for i in range(1, n)]
    rows = [[] for _ in range(n)]
    for i in range(1, n):
        rows[parent[i]].append(i)
    for r in rows:
        rng.shuffle(r)
    for root in (0, int(rng.integers(0, n))):
        _check_subtree(device, rows, root, n)


@pytest.mark.parametrize("seed", range(3))
def test_subtree_random_graphs(device, seed):
    """Graphs with repeated children, cycles and ids past max_nodes: the first occurrence in
    breadth-first order numbers a node."""
    rng = np.random.default_rng(80 + seed)
    n = [50, 3000, 20000][seed]
    rows = [list(rng.integers(0, n + 3, int(rng.integers(0, 6)))) for _ in range(n)]
    rows = [[int(c) for c in r] for r in rows]
    _check_subtree(device, rows, int(rng.integers(0, n)), n)


@pytest.mark.parametrize("repeat", [0, 1])
def test_subtree_wide_levels(device, repeat):
    """Levels of 16000 nodes and 48000 edges, several chunks of rows and of candidates; with
    every row listed again behind itself, a level has more candidates than the queue has room
    for."""
    rng = np.random.default_rng(7 + repeat)
    sizes = [1, 40, 1600, 16000, 48000]
    base = np.concatenate([[0], np.cumsum(sizes)])
    n = int(base[-1])
    rows = [[] for _ in range(n)]
    for d in range(4):
        kids = rng.permutation(np.arange(base[d + 1], base[d + 2]))
        for c, p in zip(kids, rng.integers(base[d], base[d + 1], len(kids))):
            rows[int(p)].append(int(c))
    rows = [r + (r[::-1] if repeat else []) for r in rows]
    _check_subtree(device, rows, 0, n)
    _check_subtree(device, rows, int(np.argmax([len(r) for r in rows[1:41]])) + 1, n)


@pytest.mark.parametrize("seed", range(10))
def test_subtree_narrow_levels(device, seed):
    """Levels of 1 to 300 nodes with short rows (among them 64 and 65 nodes, and about 64 and 256
    candidates), children repeated within and across rows, edges back to earlier levels and out of
    the graph, in graphs of node counts on both sides of 8192."""
    rng = np.random.default_rng(500 + seed)
    sizes = [1] + [int(rng.choice([1, 2, 16, 63, 64, 65, 128, 300])) for _ in range(25)]
    base = np.concatenate([[0], np.cumsum(sizes)])
    used = int(base[-1])
    n = [used, 8192, 8193][seed % 3]
    ids = rng.permutation(n)[:used]  # (levels are not runs of consecutive nodes)
    rows = [[] for _ in range(n)]
    for d in range(len(sizes) - 1):
        most = int(rng.choice([2, 4, 9, 300 // sizes[d] + 2]))
        for i in range(sizes[d]):
            kids = [int(c) for c in ids[rng.integers(base[d + 1], base[d + 2],
                                                     int(rng.integers(0, most)))]]
            if rng.random() < 0.3:
                kids += kids[:2] + [int(ids[rng.integers(0, base[d + 1])]), n + 3, -1]
            rows[int(ids[base[d] + i])] += kids
        rows[int(ids[base[d]])].append(int(ids[base[d + 1]]))  # (the next level is reached)
    _check_subtree(device, rows, int(ids[0]), n)
    _check_subtree(device, rows, int(ids[base[3]]), n)


@pytest.mark.parametrize("width", [523, 525])
def test_subtree_around_32_bit_scans(device, width):
    """About 2^31 / 4096 edges, from where a chunk's scan takes 64 bits, in rows that repeat their
    children."""
    rng = np.random.default_rng(width)
    n = 3001
    rows = [list(range(1, 1001))] + [[int(c) for c in rng.integers(0, n, width)]
                                     for _ in range(1000)] + [[] for _ in range(2000)]
    assert (sum(map(len, rows)) > 0x7FFFFFFF // 4096) == (width == 525)
    _check_subtree(device, rows, 0, n)


def test_subtree_of_the_largest_node_count(device):
    """max_nodes = 2^31 - 1 (the most an int32 holds): the subtree of the last node, with children
    at both ends."""
    n = 2**31 - 1
    if torch.cuda.mem_get_info()[0] < 80 * 2**30:
        pytest.skip("needs 42 GiB of device memory for the graph and the workspace")
    ptr = torch.zeros(n + 1, dtype=torch.int32, device=device)
    ptr[n] = 3
    col = _t(np.array([5, n - 2, 5], np.int32), device)
    ins, remap, cnt = torch_ops.parallel_bfs_subtree(ptr, col, n - 1, n)
    assert int(_np(cnt)[0]) == 3
    assert [int(remap[i]) for i in (n - 1, 5, n - 2)] == [0, 1, 2]
    assert int(ins.sum()) == 3 and int((remap != -1).sum()) == 3
    assert bool(ins[n - 1]) and bool(ins[5]) and bool(ins[n - 2])
    del ptr, ins, remap
    torch.cuda.empty_cache()


@pytest.mark.parametrize("n", [1, 17, 255, 256, 257, 1023, 1024, 1025, 1300, 70_000])
@pytest.mark.parametrize("kind", ["tree", "front", "back", "overlap"])
def test_edges_of_spread_groups(device, n, kind):
    """The extraction at the edges of its chunks: rows all over the nodes, only in the first or the
    last of them (long rows), and rows that overlap, of a random half of the nodes."""
    rng = np.random.default_rng(n)
    if kind == "tree":
        lens = rng.integers(0, 3, n)
    elif kind == "overlap":
        lens = rng.integers(0, 10 if n < 2000 else 2, n)
    else:
        lens = np.zeros(n, np.int64)
        few = max(1, min(n, 20))
        lens[:few] = rng.integers(0, 700, few)
        lens = lens if kind == "front" else lens[::-1]
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ne = int(ptr[-1])
    if kind == "overlap":  # (rows that start anywhere and end past the next one's start)
        ptr = np.sort(rng.integers(0, max(ne, 1), n + 1)).astype(np.int32)
        ptr[::3] = 0
        ptr[-1] = min(ne, 500)
    col = rng.integers(-2, n + 3, ne).astype(np.int32)
    act = rng.integers(-9, 9, ne).astype(np.int16)
    ins = rng.random(n) < (0.5 if n < 2000 or kind != "overlap" else 0.002)
    remap = rng.permutation(n).astype(np.int32)
    pe, ce, ae = ref_np.extract_subtree_edges(ptr, col, act, ins, remap)
    p, c, a = torch_ops.extract_subtree_edges(_t(ptr, device), _t(col, device), _t(act, device),
                                              _t(ins, device), _t(remap, device), max(len(pe), 1))
    assert np.array_equal(_np(p), pe) and np.array_equal(_np(c), ce) and np.array_equal(_np(a), ae)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 256, 257, 4097, 9000])
def test_subtree_workspaces_hold_what_is_used(device, n):
    """The search and the extraction on workspaces of just the declared sizes, whose neighbours
    keep their contents, against the reference."""
    rng = np.random.default_rng(n)
    rows = [[] for _ in range(n)]
    for i in range(1, n):
        rows[int(rng.integers(max(0, i - 40), i))].append(i)
    ptr, col = _csr(rows)
    ins_e, remap_e, k_e = ref_np.parallel_bfs_subtree(ptr, col, 0, n)
    pe, ce, _ = ref_np.extract_subtree_edges(ptr, col, None, ins_e, remap_e)
    lib = _lib.load()
    ne = len(col)
    tp, tc = _t(ptr, device), _t(np.append(col, 0).astype(np.int32), device)
    ins = torch.empty(n, dtype=torch.uint8, device=device)
    remap, out = [torch.empty(n, dtype=torch.int32, device=device) for _ in range(2)]
    child = torch.empty_like(out)
    acts = torch.empty(n, dtype=torch.int16, device=device)
    count = torch.empty(1, dtype=torch.int32, device=device)
    stream = torch.cuda.current_stream(device).cuda_stream
    pad, mark = 64, -77

    def run(ints, call):
        ws = torch.full((ints + 2 * pad,), mark, dtype=torch.int32, device=device)
        assert call(ws.data_ptr() + 4 * pad, ints) == _lib.OMQ_OK
        assert bool((ws[:pad] == mark).all()) and bool((ws[pad + ints:] == mark).all())
        return int(count.item())

    assert run(_lib.bfs_workspace_ints(n), lambda ws, k: lib.omq_parallel_bfs_subtree(
        tp.data_ptr(), tc.data_ptr(), ne, 0, n, ins.data_ptr(), remap.data_ptr(),
        count.data_ptr(), ws, k, stream)) == k_e
    assert np.array_equal(_np(remap), remap_e)
    k = run(_lib.edges_workspace_ints(n), lambda ws, k: lib.omq_extract_subtree_edges(
        tp.data_ptr(), tc.data_ptr(), None, ne, ins.data_ptr(), remap.data_ptr(), n, n,
        out.data_ptr(), child.data_ptr(), acts.data_ptr(), count.data_ptr(), ws, k, stream))
    assert k == len(pe)
    assert np.array_equal(_np(out[:k]), pe) and np.array_equal(_np(child[:k]), ce)
