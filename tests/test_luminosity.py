"""The parton luminosity of hadronic points: one real value an event, whatever the caller's
density returns.  Other shapes and complex values are refused, as assigning the products to
the passing events is."""

import pytest
import torch

from madflow_amd import vegas
from madflow_amd.multichannel import MultiChannelIntegrand
from madflow_amd.vegas import MEIntegrand

SHAPES = [(), (1,), (5,), (1, 5), (1, 1, 5), (5, 1), (5, 5), (2, 5), (4,), (0,), (2, 1, 5)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.int64, torch.complex128])
@pytest.mark.parametrize("n", [5, 1])
def test_product_of_every_shape(n, dtype, shape):
    """Taken or refused, and valued, as the assignment to a mask's events; complex values are
    refused for a single event too, where the assignment drops the imaginary part."""
    shape = tuple(min(s, n) if s == 5 else s for s in shape)
    me = torch.arange(1, n + 1, dtype=torch.float64)
    lumi = (2 * torch.ones(shape)).to(dtype)
    ok = torch.tensor([True, False] * n)
    want = torch.zeros(2 * n, dtype=torch.float64)
    try:
        want[ok] = me * lumi
        if dtype.is_complex:
            raise RuntimeError("complex")
    except (RuntimeError, IndexError):
        with pytest.raises((ValueError, TypeError, RuntimeError)):
            vegas.with_luminosity(me, lumi)
    else:
        got = vegas.with_luminosity(me, lumi)
        assert got.shape == (n,) and got.dtype == torch.float64 and got.is_contiguous()
        assert torch.equal(got, want[ok])


PDFS = {
    "column": lambda x, q2: (x * (1 - x) ** 5).reshape(-1, 1),
    "complex": lambda x, q2: (x * (1 - x) ** 5).to(torch.complex128),
    "short": lambda x, q2: (x * (1 - x) ** 5)[1:],
}


@pytest.mark.gpu
@pytest.mark.parametrize("kind", sorted(PDFS))
@pytest.mark.parametrize("cls", [MEIntegrand, MultiChannelIntegrand])
def test_densities_of_another_shape_are_refused(dev, cls, kind):
    print("refused", cls.__name__, kind, flush=True)
    ig = cls("gg_ttx", 13000.0, pdf=PDFS[kind], seed=3, mapping="hadronic")
    with pytest.raises((ValueError, TypeError, RuntimeError)):
        ig.iteration(1000, 0, train=False)


@pytest.mark.gpu
@pytest.mark.parametrize("cls", [MEIntegrand, MultiChannelIntegrand])
def test_a_row_or_a_constant_is_taken(dev, cls):
    run = lambda pdf: cls("gg_ttx", 13000.0, pdf=pdf, seed=3, mapping="hadronic").iteration(1000, 0, train=False)["I"]
    assert run(lambda x, q2: x) == run(lambda x, q2: x.reshape(1, -1))
    # x f(x) = 1 as one number
    assert run(lambda x, q2: torch.ones_like(x)) == run(lambda x, q2: torch.ones((), device=x.device))
