"""A point's amplitudes and matrix element do not depend on the size of the call it comes in:
the launches of few events, whose colour orderings and helicity rows are spread over the chip,
give the bits of a launch in which one block walks every ordering and every row."""

import pytest
import torch

from oracle import oracle as O
from tests.helpers import phase_space_points
from madflow_amd.matrix import load_matrix


def _vals(m):
    rp, coup = O.default_params(ref_gs=True)
    return [rp[0], rp[1]] + [coup[c] for c in m.params[2:]]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("name", ["gg_ttxgg", "gg_ttxggg"])
def test_jamps_of_split_orderings(dev, name, precision):
    """Ranges of one word, ranges that begin inside a cycle of rotations, and whole cycles."""
    m, _ = load_matrix(name, precision=precision)
    hel = [-1, 1] + [1, -1] + [(-1) ** k for k in range(m.nexternal - 4)]
    base = torch.from_numpy(phase_space_points(name, 4097, seed=41)[0]).to(dev)
    ps = base.repeat(132000 // base.shape[0] + 1, 1, 1)     # more than 2,048 blocks: one range
    me, jamp = m._matrix(ps, hel, _vals(m), return_jamp=True)
    me, jamp = me[:45000].clone(), jamp[:45000].clone()
    for n in (1, 64, 257, 4097, 21824, 32768, 43712):
        print("jamps", name, precision, n, flush=True)
        me_n, jamp_n = m._matrix(ps[:n], hel, _vals(m), return_jamp=True)
        assert torch.equal(jamp_n, jamp[:n])
        assert torch.equal(me_n, me[:n])


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("name,large", [("gg_ttxgg", 600000), ("gg_ttxggg", 150000)])
def test_matrix_elements_of_split_rows(dev, name, large, precision):
    """large: enough events that no row range is split off (the colour sum of a tile's rows is one
    wave's); the sizes split them into ranges of one row, of some, and of half of them."""
    m, _ = load_matrix(name, precision=precision)
    base = torch.from_numpy(phase_space_points(name, 4097, seed=42)[0]).to(dev)
    m.workspace_limit = 48 << 30       # every row of every event in one pass
    ref = m.smatrix(base.repeat(large // base.shape[0] + 1, 1, 1), *_vals(m))
    assert torch.equal(ref[:4097], ref[4097:8194])
    for n in (1, 16, 17, 64, 65, 1000, 4097):
        print("rows", name, precision, n, flush=True)
        assert torch.equal(m.smatrix(base[:n], *_vals(m)), ref[:n])
    for n in (20000, 40000, 70000):
        print("rows", name, precision, n, flush=True)
        got = m.smatrix(base.repeat(n // base.shape[0] + 1, 1, 1), *_vals(m))
        assert torch.equal(got[:4097], ref[:4097])


@pytest.mark.gpu
@pytest.mark.parametrize("name,sizes", [("uux_ttxg", (110000, 120000, 131073, 240000, 262145)),
                                        ("ug_ttxu", (119000, 119200, 131073)),
                                        ("gg_ttx", (131072, 187000, 188000, 196609))])
def test_rows_side_by_side_or_in_turn(dev, name, sizes):
    """FP32 on both sides of the sizes (on 256 CUs) at which an event's rows go in turn on one lane."""
    m, _ = load_matrix(name, precision=32)
    base = torch.from_numpy(phase_space_points(name, 4097, seed=43)[0]).to(dev)
    ps = base.repeat(max(sizes) // base.shape[0] + 1, 1, 1)
    ref = m.smatrix(base, *_vals(m))
    for n in sizes:
        print("in turn", name, n, flush=True)
        got = m.smatrix(ps[:n], *_vals(m))
        assert torch.equal(got, ref.repeat(n // base.shape[0] + 1)[:n])
