"""The host-made root inputs against their definitions, one entry at a time: keys, legal masks and
counts, and the Go rules' root masks."""
from types import SimpleNamespace

import numpy as np
import pytest

from omoknuni_quantum_amd import _lib
from omoknuni_quantum_amd.core.mcts import MCTS
from omoknuni_quantum_amd.synthetic import games


@pytest.mark.parametrize("seed", [0, -3, 20260101, 2**63 + 5])
def test_root_keys(seed):
    want = [games.splitmix64((seed ^ t) & games.MASK64) for t in range(70)]
    assert games.root_keys(seed, 70).tolist() == want


@pytest.mark.parametrize("model", [games.gomoku(5), games.gomoku(15), games.go(9), games.go(19)])
def test_legal_masks_and_counts(model):
    boards = games.random_boards(6, model.board_size, model.cells, 4)
    masks = games.legal_masks(model, boards, 6)
    for t in range(6):
        legal = [a for a in range(model.num_actions)
                 if a == model.cells or boards[t].reshape(-1)[a] == 0]
        bits = [a for a in range(model.legal_words * 32) if masks[t, a // 32] >> (a % 32) & 1]
        assert bits == legal
        assert games.legal_counts(model, masks)[t] == len(legal)


@pytest.mark.parametrize("flags", [_lib.OMQ_GO_KO, _lib.OMQ_GO_KO | _lib.OMQ_GO_SUICIDE])
def test_go_root_legal(flags):
    bs, T = 5, 40
    boards = games.random_boards(T, bs, bs * bs, 9, min_stones=8)
    ko = np.random.default_rng(1).integers(-1, bs * bs + 2, T).astype(np.int32)
    me = SimpleNamespace(model=games.go(bs), _root_go_host=(np.zeros(T, np.int32), ko))
    masks = MCTS._go_root_legal(me, boards, flags)
    for t in range(T):
        legal = []
        for a in range(bs * bs):
            r, c = divmod(a, bs)
            near = [boards[t, y, x] for y, x in ((r - 1, c), (r + 1, c), (r, c - 1), (r, c + 1))
                    if 0 <= y < bs and 0 <= x < bs]
            closed = flags & _lib.OMQ_GO_SUICIDE and all(v != 0 for v in near)
            if boards[t, r, c] == 0 and a != ko[t] and not closed:
                legal.append(a)
        bits = [a for a in range(32) if masks[t, 0] >> a & 1]
        assert bits == legal + [bs * bs]


@pytest.mark.parametrize("layout", ["F", "transposed", "strided"])
@pytest.mark.parametrize("flags", [_lib.OMQ_GO_KO, _lib.OMQ_GO_KO | _lib.OMQ_GO_SUICIDE])
def test_go_root_legal_of_any_board_layout(flags, layout):
    """The masks of boards in other memory orders are those of the same boards in C order, the ko
    points excluded."""
    bs, T = 5, 12
    boards = games.random_boards(T, bs, bs * bs, 3, min_stones=8)
    ko = np.array([int(np.flatnonzero(b.reshape(-1) == 0)[0]) for b in boards], np.int32)
    me = SimpleNamespace(model=games.go(bs), _root_go_host=(np.zeros(T, np.int32), ko))
    want = MCTS._go_root_legal(me, boards, flags)
    assert not any(want[t, 0] >> int(ko[t]) & 1 for t in range(T))
    if layout == "F":
        other = np.asfortranarray(boards)
    elif layout == "transposed":
        other = np.ascontiguousarray(boards.transpose(0, 2, 1)).transpose(0, 2, 1)
    else:
        other = np.repeat(boards, 2, axis=2)[:, :, ::2]
    assert np.array_equal(other, boards) and not other.flags.c_contiguous
    assert np.array_equal(MCTS._go_root_legal(me, other, flags), want)
