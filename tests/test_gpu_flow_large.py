"""Large flow batches (a block of 64 samples, a transformed dimension per wave) against the same
samples in batches that the 16-sample kernel takes: every output element sums the same
products in the same order, so they are equal to the last bit."""

import pytest
import torch

from madflow_amd.flow import RQSFlow
from tests.test_gpu_flow import _perturbed


@pytest.mark.gpu
@pytest.mark.parametrize("D,layers", [(2, 2), (5, 3), (8, 8), (11, 4), (16, 6)])
def test_large_batch_equals_small_batches(dev, D, layers):
    """One sample past the switch at either width, a whole number of blocks, and ragged ends."""
    flow = RQSFlow(D, layers=layers, seed=3, device=dev)
    _perturbed(flow)
    sizes = (4097, 8193, 8256, 20031)
    x = torch.rand((max(sizes), D), generator=torch.Generator().manual_seed(2)).to(dev)
    x[5, 0], x[70, D - 1], x[4096, 0] = 0.0, 1.0, float("nan")
    for inverse in (False, True):
        parts = [flow._apply(x[a:a + 4096].contiguous(), inverse) for a in range(0, x.shape[0], 4096)]
        ref = [torch.cat([p[k] for p in parts]) for k in range(2)]
        for n in sizes:
            print("flow", D, layers, inverse, n, flush=True)
            out = flow._apply(x[:n].contiguous(), inverse)
            for got, want in zip(out, ref):
                assert torch.equal(got.view(torch.int32), want[:n].view(torch.int32))
