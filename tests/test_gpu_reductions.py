"""The reductions of an integration iteration at the edges of their launches: one event, a
block more or less, more events than one pass of every block; histograms of a block's
columns and of ragged ones; grids of the fewest and the most bins."""

import ctypes
import math

import numpy as np
import pytest
import torch

from madflow_amd import _lib
from madflow_amd.multichannel import MultiChannelIntegrand
from madflow_amd.phasespace_gpu import philox_uniforms
from madflow_amd.vegas import MEIntegrand, _ptr
from oracle import oracle as O


def _tensors(n, *cols):
    rng = np.random.default_rng(n)
    return [rng.exponential(size=(n, c) if c else n) ** 3 for c in cols]


@pytest.mark.gpu
@pytest.mark.parametrize("nbins", [2, 50, 64])
@pytest.mark.parametrize("n", [1, 255, 257, 300001])
def test_accumulate_sums_and_histogram(dev, n, nbins):
    print("accumulate", n, nbins, flush=True)
    ig = MEIntegrand("gg_ttx", 1000.0, mapping="diet", nbins=nbins, seed=5)
    b = ig._alloc(n)
    f = _tensors(n, 0)[0]
    fd = torch.from_numpy(f).to(dev)
    _lib.check(ig.lib.mfx_vegas_accumulate(ctypes.byref(ig.p), 0, n, 3, None, None, None, None, _ptr(fd), None,
                                           _ptr(b["ws"]), b["ws"].numel(), _ptr(b["result"]), _lib.stream_ptr(dev)))
    r = b["result"].cpu().numpy()
    y = philox_uniforms(n, ig.ndim, 5, 3, device=dev).cpu().numpy()
    # f and f^2 are compensated sums; a wave adds at most n / (4 blocks) + 64 squares to a bin plainly
    np.testing.assert_allclose(r[:2], [math.fsum(f), math.fsum(f * f)], rtol=4e-16 * np.log2(n + 2) + 1e-15)
    assert r[2] == f.max() and r[3] == n
    tol = (n / (4.0 * min(1024, -(-n // 256))) + 64) * 2.0 ** -53 + 1e-13
    for d in range(ig.ndim):
        hist = np.bincount((y[:, d] * nbins).astype(int), weights=f * f, minlength=nbins)
        np.testing.assert_allclose(r[6 + d * nbins:6 + (d + 1) * nbins], hist, rtol=tol)


@pytest.mark.gpu
@pytest.mark.parametrize("n,nch", [(1, 1), (256, 3), (300001, 8)])
def test_channel_moments(dev, n, nch):
    print("moments", n, nch, flush=True)
    lib = MultiChannelIntegrand("gg_ttx", 1000.0).lib
    me, w, ratios = _tensors(n, 0, 0, nch)
    t = [torch.from_numpy(x).to(dev) for x in (np.arange(n, dtype=np.int32), me, w, ratios)]
    ws, out = torch.empty(1024 * nch * 16, dtype=torch.uint8, device=dev), torch.empty(nch, dtype=torch.float64, device=dev)
    _lib.check(lib.mfx_mc_moments(n, nch, *[_ptr(x) for x in t], _ptr(ws), ws.numel(), _ptr(out), _lib.stream_ptr(dev)))
    ref = ((me * w) ** 2)[:, None] * ratios
    np.testing.assert_allclose(out.cpu().numpy(), [math.fsum(c) for c in ref.T], rtol=4e-16 * np.log2(n + 2) + 1e-15)


@pytest.mark.gpu
@pytest.mark.parametrize("nbins", [2, 3, 50, 64])
def test_refine_against_oracle(dev, nbins):
    print("refine", nbins, flush=True)
    rng = np.random.default_rng(nbins)
    edges = np.sort(np.concatenate([np.zeros((4, 1)), rng.random((4, nbins - 1)), np.ones((4, 1))], 1), 1)
    hist = rng.exponential(size=(4, nbins)) ** 4
    hist[1, nbins // 2:] = 0.0          # empty bins
    hist[2] = 0.0                       # nothing: the edges stay
    g, h = torch.from_numpy(edges).to(dev), torch.from_numpy(hist).to(dev)
    _lib.check(MEIntegrand("gg_ttx", 1000.0).lib.mfx_vegas_refine(_ptr(g), _ptr(h), 4, nbins, 1.5, _lib.stream_ptr(dev)))
    np.testing.assert_allclose(g.cpu().numpy(), O.vegas_refine(edges, hist, alpha=1.5), rtol=0, atol=1e-13)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 257, 65536, 300001, 3000001])
def test_compaction_offsets(dev, n):
    """Every block's offset, from one block to more blocks than threads of the scan."""
    from madflow_amd.vegas import unweight
    print("scan", n, flush=True)
    w = torch.from_numpy(_tensors(n, 0)[0]).to(dev)
    idx, keep = unweight(w, 4.0, seed=3)
    assert torch.equal(idx.long(), torch.nonzero(keep).reshape(-1))
