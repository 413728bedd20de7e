"""A point's amplitudes do not depend on the size of the call it comes in: the launches of few
events, whose colour orderings are spread over the chip, give the bits of a launch in which one
block walks every ordering."""

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
