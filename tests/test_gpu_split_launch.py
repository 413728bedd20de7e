"""Calls of few events, whose helicity rows and colour orderings are spread over the chip,
against the same events inside a call large enough that they are not.

A row's arithmetic is the same either way; the rows' contributions, none negative, are added
in FP64 in another grouping.  Two such sums of R rows differ by at most 2 R 2^-53 relative.
"""

import pytest
import torch

from oracle import oracle as O
from tests.helpers import phase_space_points
from madflow_amd.matrix import load_matrix


def _call(m, ps):
    rp, coup = O.default_params(ref_gs=True)
    return m.smatrix(ps, rp[0], rp[1], *[coup[c] for c in m.params[2:]])


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("name,large", [("gg_ttxgg", 40000), ("gg_ttxggg", 35000)])
def test_split_orderings_and_rows(dev, name, large, precision):
    """Sizes at the edges of a 16-event colour tile and a 64-event block, one event, and sizes
    that split the orderings into few ranges or the helicity rows alone."""
    m, _ = load_matrix(name, precision=precision)
    sizes = (1, 15, 16, 17, 63, 64, 65, 257, 1000, 4097)
    ps = torch.from_numpy(phase_space_points(name, max(sizes), seed=31)[0]).to(dev)
    ref = _call(m, ps.repeat(large // ps.shape[0] + 1, 1, 1))
    for n in sizes:
        print("split", name, precision, n, flush=True)
        rel = (_call(m, ps[:n]) / ref[:n] - 1).abs().max().item()
        assert rel <= 2 * m.ncomb * 2.0 ** -53


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("name", ["gg_ttx", "gg_ttxg", "uux_ttx", "uux_ttxg", "uux_ttxgg", "ug_ttxu", "uxg_ttxux"])
def test_rows_side_by_side(dev, name, precision):
    """The fused kernels add an event's rows in one order however they are spread: every block
    size that small calls choose gives the bits of a large call, and those are the oracle's
    values within the precision's bar."""
    m, _ = load_matrix(name, precision=precision)
    sizes = (1, 3, 5, 63, 64, 65, 257, 1023, 1025, 2049, 4097, 16385)
    host = phase_space_points(name, max(sizes), seed=32)[0]
    ps = torch.from_numpy(host).to(dev)
    ref = _call(m, ps.repeat(300000 // ps.shape[0] + 1, 1, 1))
    for n in sizes:
        print("rows", name, precision, n, flush=True)
        assert torch.equal(_call(m, ps[:n]), ref[:n])
    rp, coup = O.default_params(ref_gs=True)
    want = torch.from_numpy(O.smatrix(name, host[:512], rp, coup, ref_compat=True)).to(dev)
    rel = (ref[:512] / want - 1).abs().max().item()
    print(name, precision, "against the oracle", rel, flush=True)
    # FP64 t t~ g g from u u~: its diagrams cancel up to 335-fold on uncut points
    assert rel < (5e-5 if precision == 32 else 3.4e-12 if name == "uux_ttxgg" else 1e-12)
