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
from madflow_amd.phasespace_gpu import PhaseSpaceGenerator, philox_uniforms, rambo
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
@pytest.mark.parametrize("n", [1, 63, 65, 300001])
@pytest.mark.parametrize("n_out,mapping,ndim,nbins", [(3, 1, 5, 64), (4, 0, 16, 3), (5, 2, 22, 50), (7, 2, 30, 16)])
def test_accumulate_of_an_external_proposal(dev, n_out, mapping, ndim, nbins, n):
    """Odd and large numbers of dimensions, one copy of the histogram a wave (22 of 50 bins) and
    two; coordinates at and beyond the ends of the range and not finite, weights not finite."""
    print("external", ndim, nbins, n, flush=True)
    gen = PhaseSpaceGenerator(n_out + 2, 13000.0)
    p = gen.p
    p.mapping, p.ndim, p.nbins = mapping, ndim, nbins
    rng = np.random.default_rng(n + ndim)
    y = rng.random((n, ndim), dtype=np.float32)
    f = rng.exponential(size=n)
    y[::7, 0], y[::5, 1], y[::11, 2], y[::13, 3], y[::17, 4] = 1.0, -0.5, 1.5, np.nan, np.inf
    f[3::9], f[5::31] = np.nan, np.inf
    yd, fd, fo = torch.from_numpy(y).to(dev), torch.from_numpy(f).to(dev), torch.empty(n, dtype=torch.float64, device=dev)
    ws = torch.empty(gen.lib.mfx_integrand_workspace_size(n, ndim, nbins), dtype=torch.uint8, device=dev)
    out = torch.empty(6 + ndim * nbins, dtype=torch.float64, device=dev)
    _lib.check(gen.lib.mfx_vegas_accumulate(ctypes.byref(p), 0, n, 0, _ptr(yd), None, None, None, _ptr(fd), _ptr(fo),
                                            _ptr(ws), ws.numel(), _ptr(out), _lib.stream_ptr(dev)))
    r = out.cpu().numpy()
    f = np.where(np.isfinite(f), f, 0.0)
    assert np.array_equal(fo.cpu().numpy(), f)
    np.testing.assert_allclose(r[:2], [math.fsum(f), math.fsum(f * f)], rtol=4e-16 * np.log2(n + 2) + 1e-15)
    assert r[2] == f.max() and r[3] == np.count_nonzero(f)
    yc = np.clip(np.where(np.isfinite(y), y, 0.0).astype(np.float64), 0.0, 1.0)
    tol = (n / (4.0 * min(1024, -(-n // 256))) + 64) * 2.0 ** -53 + 1e-13
    for d in range(ndim):
        bins = np.minimum((yc[:, d] * nbins).astype(int), nbins - 1)
        hist = np.bincount(bins, weights=f * f, minlength=nbins)
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


@pytest.mark.gpu
@pytest.mark.parametrize("process", ["gg_ttx", "gg_ttxgg"])
@pytest.mark.parametrize("n", [1, 257, 70001])
def test_hadronic_points(dev, process, n):
    """x1, x2 and Q^2 of the passing events, in their order, against selection by mask."""
    print("hadronic points", process, n, flush=True)
    ig = MEIntegrand(process, 13000.0, mapping="hadronic", pdf=lambda x, q2: x, seed=9)
    ig.register_cut("pt", particle=2, min_val=100.0)
    _, npass, _ = ig.chunk(0, n, 1)
    b = ig._bufs
    ok = b["flag"][:n] == 1
    x, q2 = torch.empty((2, npass), dtype=torch.float64, device=dev), torch.empty(npass, dtype=torch.float64, device=dev)
    _lib.check(ig.lib.mfx_hadronic_points(_ptr(b["dense"]), _ptr(b["slot"]), _ptr(b["x12"]), n, npass, ig.nexternal,
                                          _ptr(x), _ptr(q2), _lib.stream_ptr(dev)))
    assert torch.equal(x.T, b["x12"][:n][ok])
    out = b["all_ps"][:n][ok][:, 2:]
    mt = torch.sqrt(torch.clamp(out[..., 0] ** 2 - out[..., 3] ** 2, min=0.0)).sum(1)
    # E^2 - pz^2 loses (E / mT)^2 in the contraction of its products
    tol = 4e-16 * (1.0 + (out[..., 0] ** 2).sum(1) / mt ** 2)
    assert bool(((q2 / (0.5 * mt) ** 2 - 1).abs() <= 8 * tol).all())


@pytest.mark.gpu
def test_running_and_frozen_couplings_mixed(dev):
    """A coupling of one value beside couplings per event is broadcast into its plane."""
    from madflow_amd.matrix import load_matrix
    from madflow_amd.phasespace_gpu import sample_momenta
    m, _ = load_matrix("gg_ttxg", precision=64)
    ps = sample_momenta("gg_ttxg", 257, device=dev)
    one = lambda v: torch.full((257,), v, dtype=torch.complex128, device=dev)
    whole = m.smatrix(ps, 173.0, 1.5, one(-1.2), one(1.2j), one(1.44j))
    assert torch.equal(m.smatrix(ps, 173.0, 1.5, -1.2, one(1.2j), torch.tensor([1.44j], dtype=torch.complex128)), whole)
    assert torch.equal(m.smatrix(ps, 173.0, 1.5, one(-1.2), torch.tensor([1.2j], dtype=torch.complex128, device=dev), one(1.44j).cpu()), whole)


@pytest.mark.gpu
@pytest.mark.parametrize("n_out", [2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("massive", [False, True])
def test_generation_by_number_of_legs(dev, n_out, massive):
    """The generation kernels of two to five legs and the general one against RAMBO at each
    event's partonic energy, with a cut on the last leg."""
    print("legs", n_out, massive, flush=True)
    masses = [173.0 if massive and i < 2 else 0.0 for i in range(n_out)]
    gen = PhaseSpaceGenerator(n_out + 2, 13000.0, masses=masses)
    gen.p.shat_min = 2000.0 ** 2
    x = torch.rand((1025, gen.ndim), generator=torch.Generator().manual_seed(n_out), dtype=torch.float64).to(dev)
    ps, w, x1, x2, _ = gen.generate(x)
    p, wr = rambo(x[:, 2:].contiguous(), n_out, torch.sqrt(x1 * x2) * 13000.0, masses=masses)
    scale = (x1 * x2).sqrt() * 13000.0
    # sqrt(x1 x2) s is rounded once more here; a Newton step ends at 1e-14 of the energy
    assert ((ps[:, 2:] - p).abs().amax((1, 2)) / scale).max().item() < 1e-12
    tau = x1 * x2
    jac = (1.0 - (2000.0 / 13000.0) ** 2) * -torch.log(tau) * 389379365.6 / (2.0 * tau * 13000.0 ** 2)
    assert ((w / (wr * jac)) - 1).abs().max().item() < 1e-11
    gen.register_cut("pt", particle=n_out + 1, min_val=300.0)
    cut, _, _, _, idx = gen(x)
    want = torch.nonzero(torch.hypot(ps[:, -1, 1], ps[:, -1, 2]) > 300.0)
    assert torch.equal(idx.long(), want) and torch.equal(cut, ps[want[:, 0]])


@pytest.mark.gpu
def test_hadronic_points_of_undefined_momenta(dev):
    """The scale of an event whose transverse mass is not a number is not a number either, as
    elementwise operations give it; negative squares count as zero."""
    n = 8
    dense = torch.ones((n, 5, 4), dtype=torch.float64)
    dense[..., 0] = 3.0
    dense[1, 2, 0], dense[2, 4, 3] = math.nan, math.nan
    dense[3, 3, 0] = dense[3, 3, 3] = math.inf
    dense[4, 3, 0] = math.inf
    dense[5, 2, 0] = 0.5
    x12 = torch.rand((n, 2), dtype=torch.float64)
    d, x, s = dense.to(dev), x12.to(dev), torch.arange(n, dtype=torch.int32, device=dev)
    x_out, q2 = torch.empty((2, n), dtype=torch.float64, device=dev), torch.empty(n, dtype=torch.float64, device=dev)
    ig = MEIntegrand("gg_ttxg", 13000.0, mapping="hadronic", pdf=lambda x, q2: x)
    _lib.check(ig.lib.mfx_hadronic_points(_ptr(d), _ptr(s), _ptr(x), n, n, 5, _ptr(x_out), _ptr(q2), _lib.stream_ptr(dev)))
    out = dense[:, 2:]
    want = (0.5 * torch.sqrt(torch.clamp(out[..., 0] ** 2 - out[..., 3] ** 2, min=0.0)).sum(1)) ** 2
    assert bool(torch.isnan(want[1:4]).all())
    torch.testing.assert_close(q2.cpu(), want, rtol=1e-15, atol=0.0, equal_nan=True)
