"""Per-move root operations on the GPU against the oracle: root policies, move selection
with a temperature, and root Dirichlet noise, bit for bit; a search with device noise."""
import numpy as np
import pytest
import torch

from omoknuni_quantum_amd import _lib
from omoknuni_quantum_amd.core.engine import SearchParams, WaveEngine
from omoknuni_quantum_amd.synthetic import games
from omoknuni_quantum_amd.synthetic.workloads import get
from oracle.oracle import Oracle, load
from oracle.parity import compare_wave, make_pair

pytestmark = pytest.mark.gpu


def test_policy_and_sampling_match_oracle(device):
    wl = get("C2").scaled(num_trees=8, num_simulations=512, wave_size=128, capacity=150_000)
    eng, orc, ev = make_pair(wl, device=device)
    eng.search(wl.num_simulations, wl.wave_size, ev)
    orc.search(wl.num_simulations, wl.wave_size)
    pol = eng.root_policies()
    lib = load()
    for t in range(wl.num_trees):
        assert np.array_equal(pol[t], orc.root_policy(t))
    for temperature in (0.0, 0.25, 1.0, 2.0):
        for counter in range(5):
            acts = eng.sample_actions(temperature, 1234, counter)
            for t in range(wl.num_trees):
                row = np.ascontiguousarray(pol[t])
                want = lib.orc_sample_action(row.ctypes.data, eng.A, temperature, 1234, counter, t)
                assert acts[t] == want, (temperature, counter, t)
                assert pol[t, acts[t]] > 0


def test_policy_corner_cases(device):
    """No children: uniform over the action space; children without visits: uniform over them."""
    model = games.gomoku(5)
    eng = WaveEngine(model, 2, 64, 4, 16, device, SearchParams())
    eng.reset()
    k = 6
    eng.first[64] = 0
    eng.nchild[64] = k
    eng.action[65:65 + k] = torch.tensor([3, 7, 8, 11, 20, 24], dtype=torch.int32)
    eng.N[65:65 + k] = 0
    eng.num_nodes[1] = 1 + k
    pol = eng.root_policies()
    assert np.all(pol[0] == 1.0 / 25)
    want = np.zeros(25)
    want[[3, 7, 8, 11, 20, 24]] = 1.0 / k
    assert np.array_equal(pol[1], want)


@pytest.mark.parametrize("name,alpha", [("C2", 0.3), ("C3", 0.03), ("C4", 1.5)])
def test_device_dirichlet_matches_oracle(device, name, alpha):
    wl = get(name).scaled(num_trees=6, capacity=1000)
    eng, orc, _ = make_pair(wl, device=device)
    eng.device_root_noise(alpha, 77, 2)
    got = eng.noise.view(eng.T, eng.A).cpu().numpy()
    for t in range(eng.T):
        want = orc.root_dirichlet(t, alpha, 77, 2)
        assert np.array_equal(got[t], want), (name, t)


def test_search_with_device_noise_matches_oracle(device):
    wl = get("C3").scaled(num_trees=3, num_simulations=2048, capacity=400_000)
    eng, orc, ev = make_pair(wl, device=device)
    eng.device_root_noise(wl.dirichlet_alpha, 5, 1)
    noise = eng.noise.view(eng.T, eng.A).cpu().numpy().copy()
    keys, legal, _ = wl.root_inputs()
    orc.set_roots(keys, legal, noise)
    eng.reset()
    for t in range(eng.T):
        orc.reset_tree(t)
    for i, w in enumerate([1] + [1024] * 2):
        eng.run_wave(w, ev)
        for t in range(eng.T):
            orc.wave(t, w)
        torch.cuda.synchronize()
        compare_wave(eng, orc, w, f"device noise wave {i}")


@pytest.mark.parametrize("kind,bs", [("gomoku", 22), ("go", 21)])
def test_root_ops_wide_boards(device, kind, bs):
    """Policies, move sampling and root noise on boards of 442-484 actions."""
    model = games.gomoku(bs) if kind == "gomoku" else games.go(bs)
    wl = get("C2" if kind == "gomoku" else "C3").scaled(
        model=model, num_trees=4, num_simulations=768, wave_size=256, max_stones=bs * bs // 4,
        capacity=1 + 4 * 256 * model.num_actions)
    eng, orc, ev = make_pair(wl, device=device)
    eng.search(wl.num_simulations, wl.wave_size, ev)
    orc.search(wl.num_simulations, wl.wave_size)
    pol = eng.root_policies()
    lib = load()
    for t in range(wl.num_trees):
        assert np.array_equal(pol[t], orc.root_policy(t))
    for temperature in (0.0, 1.0):
        for counter in range(3):
            acts = eng.sample_actions(temperature, 99, counter)
            for t in range(wl.num_trees):
                row = np.ascontiguousarray(pol[t])
                want = lib.orc_sample_action(row.ctypes.data, eng.A, temperature, 99, counter, t)
                assert acts[t] == want, (temperature, counter, t)
    eng.device_root_noise(0.03, 31, 4)
    got = eng.noise.view(eng.T, eng.A).cpu().numpy()
    for t in range(eng.T):
        assert np.array_equal(got[t], orc.root_dirichlet(t, 0.03, 31, 4)), t


def test_device_dirichlet_of_the_widest_root(device):
    """513 legal actions, one more than a row holds children: a Go root's pass."""
    wl = get("C3").scaled(model=games.GameModel("go", 513, 22), num_trees=2, capacity=1000)
    eng, orc, _ = make_pair(wl, device=device)
    legal = np.zeros((2, eng.model.legal_words), np.uint32)
    legal[:, :16], legal[:, 16] = 0xFFFFFFFF, 1
    keys = wl.root_inputs()[0]
    eng.set_roots(keys, legal)
    orc.set_roots(keys, legal, None)
    eng.device_root_noise(0.3, 9, 1)
    got = eng.noise.view(2, 513).cpu().numpy()
    for t in range(2):
        assert np.array_equal(got[t], orc.root_dirichlet(t, 0.3, 9, 1)), t


@pytest.mark.parametrize("model", [games.gomoku(5), games.gomoku(9), games.gomoku(15), games.go(19),
                                   games.chess_sparse()], ids=lambda m: f"{m.kind}{m.num_actions}")
def test_device_dirichlet_of_many_trees(device, model):
    """Forests of so many trees that a workgroup has as few threads as the row's entries need."""
    T = 514
    wl = get("C2" if model.is_board else "C4").scaled(
        model=model, num_trees=T, capacity=600, wave_size=1, max_stones=model.cells)
    eng, orc, _ = make_pair(wl, device=device)
    eng.device_root_noise(0.3, 9, 1)
    got = eng.noise.view(T, model.num_actions).cpu().numpy()
    for t in range(T):
        assert np.array_equal(got[t], orc.root_dirichlet(t, 0.3, 9, 1)), t


@pytest.mark.parametrize("name", ["C1", "C3", "C4"])
def test_root_children(device, name):
    """The root's child for an action and its visits: rows of 20-45, 225 and up to 362 children,
    the first, last and a middle child, absent actions, a lone root."""
    wl = get(name).scaled(num_trees=5, num_simulations=64, wave_size=32, capacity=40_000)
    eng, _, ev = make_pair(wl, device=device)
    assert eng.root_children([0] * 5).tolist() == [[-1, 0]] * 5  # (not searched yet)
    eng.search(wl.num_simulations, wl.wave_size, ev)
    trees = [eng.host_tree(t) for t in range(5)]
    for pick in (0, -1, 17):
        first = [int(tr["first"][0]) + 1 for tr in trees]
        node = [f + range(int(tr["nchild"][0]))[pick] for f, tr in zip(first, trees)]
        acts = [int(tr["action"][n]) for tr, n in zip(trees, node)]
        want = [[n, int(tr["N"][n])] for tr, n in zip(trees, node)]
        assert eng.root_children(acts).tolist() == want
    rows = [set(tr["action"][f:f + int(tr["nchild"][0])].tolist())
            for tr, f in zip(trees, first)]
    free = [next(a for a in range(eng.A + 1) if a not in row) for row in rows]
    assert (eng.root_children(free)[:, 0] == -1).all()
