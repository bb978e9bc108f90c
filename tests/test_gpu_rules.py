"""Gomoku terminal rule on the GPU (omq_gomoku_terminal through the C ABI) against the oracle:
terminal codes, legal counts and whole trees after every wave."""
import numpy as np
import pytest
import torch

from omoknuni_quantum_amd import _lib
from omoknuni_quantum_amd.core.engine import SearchParams, WaveEngine
from omoknuni_quantum_amd.synthetic import games
from omoknuni_quantum_amd.synthetic.evaluator import SyntheticEvaluator
from omoknuni_quantum_amd.synthetic.workloads import get
from oracle.oracle import Oracle
from oracle.parity import compare_wave, run_parity
from oracle.ref_np import gomoku_terminal, leaf_position

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rule", [_lib.OMQ_RULE_FREESTYLE, _lib.OMQ_RULE_RENJU])
def test_dense_boards_parity(device, rule):
    wl = get("C2").scaled(name=f"dense9-rule{rule}", model=games.gomoku(9), max_stones=45,
                          num_trees=8, num_simulations=512, wave_size=64, capacity=60_000)
    stats = {}
    assert run_parity(wl, rule=rule, device=device, stats=stats) >= 2
    assert stats["terminal"] > 50


def test_dense_boards_large_wave_parity(device):
    """Waves above OMQ_SELECT_RECORDS_MAX_WAVE: the leaf records come from omq_leaf_info, and the
    terminal check overwrites their legal counts after it."""
    wl = get("C2").scaled(name="dense15-large-wave", model=games.gomoku(15), max_stones=150,
                          num_trees=3, num_simulations=2048, wave_size=1024, capacity=200_000)
    assert wl.wave_size > _lib.OMQ_SELECT_RECORDS_MAX_WAVE
    stats = {}
    assert run_parity(wl, rule=_lib.OMQ_RULE_FREESTYLE, device=device, stats=stats) >= 2
    assert stats["terminal"] > 0


def _planted_boards(T, bs, seed):
    """Root positions with black and white fours with a gap (a move in the gap makes five)
    and black 2+3 split lines (a move in the gap makes an overline of six)."""
    rng = np.random.default_rng(seed)
    boards = np.zeros((T, bs, bs), np.int8)
    for t in range(T):
        b = boards[t]
        r = int(rng.integers(0, bs))
        b[r, 0:2] = 1
        b[r, 3:6] = 1                       # black 11_111: the gap gives six
        r2 = (r + 3) % bs
        b[r2, 1:3] = 2
        b[r2, 4:6] = 2                      # white 22_22: the gap gives five
        c = int(rng.integers(0, bs))
        rows = [x for x in range(bs) if x not in (r, r2)][:4]
        for x in rows:
            if b[x, c] == 0:
                b[x, c] = 1                 # a black column four
        if (b != 0).sum() % 2:
            empties = np.flatnonzero(b.reshape(-1) == 0)
            b.reshape(-1)[empties[int(rng.integers(0, len(empties)))]] = 2
    return boards


@pytest.mark.parametrize("rule", [_lib.OMQ_RULE_FREESTYLE, _lib.OMQ_RULE_RENJU])
def test_planted_overlines_parity(device, rule):
    T, bs, W, cap = 6, 9, 32, 40_000
    model = games.gomoku(bs)
    boards = _planted_boards(T, bs, 40 + rule)
    keys = games.root_keys(99, T)
    legal = games.legal_masks(model, boards, T)
    eng = WaveEngine(model, T, cap, W, 100, device, SearchParams(c_puct=1.4, virtual_loss=3.0))
    eng.set_roots(keys, legal)
    eng.set_gomoku_rules(boards, rule)
    orc = Oracle(model, T, cap, W, 100)
    orc.set_params(1.4, 3.0, 0, 0, 1.0, 0.0)
    orc.set_roots(keys, legal)
    orc.set_gomoku_rules(boards, rule)
    ev = SyntheticEvaluator()
    eng.reset()
    for t in range(T):
        orc.reset_tree(t)
    codes = np.zeros(4, np.int64)
    for i, w in enumerate([1] + [W] * 12):
        eng.run_wave(w, ev)
        for t in range(T):
            orc.wave(t, w)
            u = orc.last_wave(t, w)["uterm"]
            codes += np.bincount(u, minlength=4)
        torch.cuda.synchronize()
        compare_wave(eng, orc, w, f"planted rule {rule} wave {i}")
    assert codes[1] + codes[2] > 0


@pytest.mark.parametrize("rule", [_lib.OMQ_RULE_FREESTYLE, _lib.OMQ_RULE_RENJU])
@pytest.mark.parametrize("bs", [4, 5, 6, 8, 13, 19, 22])
def test_leaf_codes_of_dense_boards(device, bs, rule):
    """Every leaf's code against the numpy scan of its position, on boards nearly full of both
    colours (fives and overlines in all directions, draws), with given root players, and with
    stones of a third value (scanned cell by cell)."""
    T, W = 16, 16
    model = games.gomoku(bs)
    rng = np.random.default_rng(100 * bs + rule)
    boards = (1 + (rng.random((T, bs, bs)) < 0.35)).astype(np.int8)  # long lines of 1s
    for t in range(T):
        free = rng.permutation(bs * bs)[:2 + t % 3 * bs]
        boards[t].reshape(-1)[free] = 0
    boards[T - 2:][boards[T - 2:] == 2] = 3
    eng = WaveEngine(model, T, 20_000, W, 100, device, SearchParams(c_puct=1.4))
    eng.set_roots(games.root_keys(5, T), games.legal_masks(model, boards, T))
    for players in (None, rng.integers(1, 3, T).astype(np.int32)):
        eng.set_gomoku_rules(boards, rule, root_player=players)
        eng.reset()
        ev = SyntheticEvaluator(1.0)
        codes = set()
        for w in (1, W, W):
            eng.run_wave(w, ev)
            uterm = eng.uterm.view(T, W).cpu().numpy()
            ulegal = eng.ulegal.view(T, W).cpu().numpy()
            ufirst = eng.ufirst.view(T, W).cpu().numpy()
            plen = eng.path_len.view(T, W).cpu().numpy()
            paths = eng.paths.view(T, W, eng.MD).cpu().numpy()
            action = eng.action.view(T, eng.cap).cpu().numpy()
            for t in range(T):
                for u in range(int(eng.ucount[t])):
                    s = ufirst[t, u]
                    moves = [int(action[t, n]) for n in paths[t, s, 1:plen[t, s]]]
                    b, _, _ = leaf_position(boards[t], moves,
                                            None if players is None else players[t])
                    want = gomoku_terminal(b, rule == _lib.OMQ_RULE_RENJU) if moves else 0
                    assert uterm[t, u] == want, (t, u, moves)
                    assert want == 0 or ulegal[t, u] == 0
                    codes.add(want)
        assert len(codes) >= 2


@pytest.mark.parametrize("rule", [_lib.OMQ_RULE_FREESTYLE, _lib.OMQ_RULE_RENJU])
@pytest.mark.parametrize("bs,slots", [(9, 8192), (9, 8160), (11, 8192), (12, 8192)])
def test_leaf_codes_of_large_wave_buffers(device, bs, slots, rule):
    """Boards of up to two cells per lane in wave buffers around the size from where they are
    scanned, against the numpy scan."""
    T, W = 32, 8
    model = games.gomoku(bs)
    rng = np.random.default_rng(bs + rule)
    boards = (1 + (rng.random((T, bs, bs)) < 0.35)).astype(np.int8)
    for t in range(T):
        boards[t].reshape(-1)[rng.permutation(bs * bs)[:2 + t % 3 * bs]] = 0
    eng = WaveEngine(model, T, 5_000, slots // T, 100, device, SearchParams(c_puct=1.4))
    eng.set_roots(games.root_keys(5, T), games.legal_masks(model, boards, T))
    eng.set_gomoku_rules(boards, rule)
    eng.reset()
    ev = SyntheticEvaluator(1.0)
    codes = set()
    for w in (1, W, W):
        eng.run_wave(w, ev)
        MW = eng.MW
        uterm = eng.uterm.view(T, MW).cpu().numpy()
        ufirst = eng.ufirst.view(T, MW).cpu().numpy()
        plen = eng.path_len.view(T, MW).cpu().numpy()
        paths = eng.paths.view(T, MW, eng.MD).cpu().numpy()
        action = eng.action.view(T, eng.cap).cpu().numpy()
        for t in range(T):
            for u in range(int(eng.ucount[t])):
                s = ufirst[t, u]
                moves = [int(action[t, n]) for n in paths[t, s, 1:plen[t, s]]]
                b, _, _ = leaf_position(boards[t], moves, None)
                want = gomoku_terminal(b, rule == _lib.OMQ_RULE_RENJU) if moves else 0
                assert uterm[t, u] == want, (t, u, moves)
                codes.add(want)
    assert len(codes) >= 2
