"""Performance cases: the work that a user of the framework has it do, as cases that can be
timed and whose outputs can be checked.

Three kinds of work are covered, each through the entry points that a program calls:

* ``me``: ``Matrix_1_<proc>.smatrix`` on momenta that are in device memory, every process, both
  precisions, frozen couplings or couplings per event (running alpha_s);
* ``vegas`` / ``mc``: one iteration of the integration loop (points, cuts, matrix elements,
  accumulation and, when training, the refinement of the grid) on RAMBO, RAMBO on diet, the
  hadronic mapping and the multi-channel phase space;
* ``flow_grad`` / ``flow_sample``: the learned proposal, one gradient of a training batch and
  one batch of proposal points with their weights.

``listed()`` names twelve cases, ``draw(rng)`` makes more of the same ranges, ``prepare`` and
``run`` are one program each, ``work`` is what a pass cannot do without, and ``exact`` computes
what ``run`` returns in 64 bits from the physics alone (Feynman rules, colour tensors, the
published phase-space maps), with torch and numpy.
"""

import itertools
import math

import numpy as np
import torch

MT, WT = 173.0, 1.4915000200271606      # top mass and width (GeV)
GEV2PB = 389379365.6
NBINS = 50
KINDS = ("me", "vegas", "mc", "flow_grad", "flow_sample")

# outgoing legs after t t~, partonic c.m. energy (GeV), flops of one |M|^2 over every helicity
# row that does not vanish (the Feynman-diagram program's count)
PROCESSES = {
    "gg_ttx": ("gg", 0, 1000.0, 23041),
    "gg_ttxg": ("gg", 1, 2000.0, 259809),
    "gg_ttxgg": ("gg", 2, 3000.0, 3862785),
    "gg_ttxggg": ("gg", 3, 5000.0, 84556673),
    "uux_ttx": ("qq", 0, 1000.0, 2977),
    "uux_ttxg": ("qq", 1, 2000.0, 48353),
    "uux_ttxgg": ("qq", 2, 3000.0, 575841),
    "ug_ttxu": ("qg", 1, 2000.0, 48353),
    "uxg_ttxux": ("qg", 1, 2000.0, 48353),
}
# most events of one drawn call, FP32 (half of it in FP64): no more work than the largest listed
MOST_EVENTS = {"gg_ttx": 2000000, "gg_ttxg": 1000000, "gg_ttxgg": 800000, "gg_ttxggg": 50000,
               "uux_ttx": 2000000, "uux_ttxg": 2000000, "uux_ttxgg": 1000000, "ug_ttxu": 2000000, "uxg_ttxux": 2000000}


# ------------------------------------------------------------------------------ the cases
def _me(name, process, precision, nev, running=False):
    return dict(name=name, kind="me", process=process, precision=precision, nev=nev, running=running)


def listed():
    return [
        # the smallest calls: a few phase-space points of the simplest process, as a program
        # does that checks a matrix element or evaluates it event by event
        _me("me_ttx_f64_16", "gg_ttx", 64, 16),
        # a test-sized batch in the class's default precision
        _me("me_ttgg_f64_1000", "gg_ttxgg", 64, 1000),
        # a small ragged batch of the most expensive process
        _me("me_ttggg_f32_257", "gg_ttxggg", 32, 257),
        # an ordinary chunk with alpha_s running from event to event
        _me("me_ttg_f32_running", "gg_ttxg", 32, 500009, True),
        # quark-initiated, default precision, ragged
        _me("me_uuxgg_f64_30001", "uux_ttxgg", 64, 30001),
        # the production chunk of the benchmark's process
        _me("me_ttgg_f32_1M", "gg_ttxgg", 32, 1048576),
        # a production chunk of the most expensive process
        _me("me_ttggg_f32_50k", "gg_ttxggg", 32, 50000),
        # the first iterations of an integration: 1e6 points, the grid refined
        dict(name="vegas_ttx_f64_train", kind="vegas", process="gg_ttx", precision=64, mapping="rambo",
             npoints=1000000, train=True),
        # a hadron-collider run of the reference's size: 1e5 points an iteration, parton
        # densities, dynamic scale and running alpha_s, frozen grid
        dict(name="vegas_ttg_hadronic", kind="vegas", process="gg_ttxg", precision=32, mapping="hadronic",
             npoints=100000, train=False),
        # one production iteration on the multi-channel phase space
        dict(name="mc_ttgg_f32", kind="mc", process="gg_ttxgg", precision=32, npoints=500000),
        # one training batch of the learned proposal: forward, backward, weight gradients
        dict(name="flow_grad_8192", kind="flow_grad", dim=8, layers=8, nev=8192, beta=3.0),
        # one chunk of proposal points
        dict(name="flow_sample_1M", kind="flow_sample", dim=8, layers=8, nev=1000000, mix=0.3),
    ]


def _spread(rng, lo, hi):
    """An integer of [lo, hi], uniform in the logarithm, odd three times in four."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.75:
        n |= 1
    return max(lo, min(hi, n))


def draw(rng):
    kind = rng.choice(["me"] * 5 + ["vegas"] * 2 + ["mc", "flow_grad", "flow_sample"])
    if kind == "me":
        process, precision = rng.choice(sorted(PROCESSES)), rng.choice([32, 64])
        most = MOST_EVENTS[process] // (precision // 32)
        return dict(kind=kind, process=process, precision=precision, nev=_spread(rng, 1, most),
                    running=rng.random() < 0.3)
    if kind == "vegas":
        process = rng.choice(["gg_ttx", "gg_ttxg", "uux_ttx", "uux_ttxg", "ug_ttxu", "gg_ttxgg"])
        gg = PROCESSES[process][0] == "gg"
        return dict(kind=kind, process=process, precision=rng.choice([32, 64]),
                    mapping=rng.choice(["rambo", "diet", "hadronic"] if gg else ["rambo", "diet"]),
                    npoints=_spread(rng, 1000, 200000 if process == "gg_ttxgg" else 1000000), train=rng.random() < 0.5)
    if kind == "mc":
        process = rng.choice(["gg_ttxg", "gg_ttxgg", "uux_ttxg"])
        return dict(kind=kind, process=process, precision=rng.choice([32, 64]),
                    npoints=_spread(rng, 8000, 250000 if process == "gg_ttxgg" else 1000000))
    dim = rng.choice([4, 5, 7, 8, 10, 11])
    if kind == "flow_grad":
        return dict(kind=kind, dim=dim, layers=rng.choice([4, 6, 8]), nev=_spread(rng, 100, 16384),
                    beta=rng.choice([0.0, 3.0]))
    return dict(kind=kind, dim=dim, layers=rng.choice([4, 6, 8]), nev=_spread(rng, 1000, 1000000),
                mix=rng.choice([0.1, 0.3]))


# -------------------------------------------------------------------- what a program has in hand
def _gen(seed, device="cuda"):
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    return g


def _masses(process):
    return [MT, MT] + [0.0] * PROCESSES[process][1]


def _alpha_s(q2):
    """One-loop running from alpha_s(M_Z) = 0.118, five flavours."""
    b0 = (33.0 - 10.0) / (12.0 * math.pi)
    return 0.118 / (1.0 + 0.118 * b0 * torch.log(q2 / 91.188 ** 2))


def _gluon_density(x, q2):
    """A toy x f_g(x, Q^2) with the falling shape of a proton's gluon."""
    return 3.0 * x ** -0.2 * (1.0 - x) ** 5 * (1.0 + 0.1 * torch.log(q2 / 1.0e4))


def _cuts(process):
    """The benchmark's cuts: pT > 30 GeV of every massless outgoing leg and Delta R > 0.4."""
    k = PROCESSES[process][1]
    return dict(pt_min=30.0 if k else 0.0, dr_min=0.4 if k > 1 else 0.0)


def _momenta(process, nev, seed):
    """(nev, legs, 4) momenta of events that pass the cuts, in the partonic c.m. frame."""
    _, _, sqrts, _ = PROCESSES[process]
    m = _masses(process)
    g, parts, have = _gen(seed), [], 0
    while have < nev:
        n = max(1024, int(1.5 * (nev - have)))
        x = torch.rand((n, 4 * len(m)), generator=g, dtype=torch.float64, device="cuda").clamp_(1e-12, 1 - 1e-12)
        p, _ = _rambo(x, m, torch.full((n,), sqrts, dtype=torch.float64, device="cuda"))
        p = p[_pass_cuts(p, **_cuts(process))]
        parts.append(p)
        have += p.shape[0]
    p = torch.cat(parts)[:nev]
    return torch.cat([_incoming(torch.full((nev,), sqrts, dtype=torch.float64, device="cuda")), p], 1).contiguous()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "me":
        from madflow_amd.matrix import load_matrix
        matrix, module = load_matrix(case["process"], precision=case["precision"])
        model = module.get_model_param()
        if case["running"]:
            q = 100.0 + 900.0 * torch.rand(case["nev"], generator=_gen(seed + 7), dtype=torch.float64, device="cuda")
            params = model.evaluate(_alpha_s(q * q))
        else:
            model.freeze_alpha_s(0.118)
            params = model.evaluate()
        return dict(kind=kind, matrix=matrix, params=params, ps=_momenta(case["process"], case["nev"], seed))
    if kind == "vegas":
        from madflow_amd.vegas import MEIntegrand
        kw = dict(pdf=_gluon_density, alphas=_alpha_s) if case["mapping"] == "hadronic" else {}
        sqrts = 13000.0 if case["mapping"] == "hadronic" else PROCESSES[case["process"]][2]
        ig = MEIntegrand(case["process"], sqrts, precision=case["precision"], mapping=case["mapping"], seed=seed,
                         **_cuts(case["process"]), **kw)
        return dict(kind=kind, ig=ig, grid=ig.grid.clone(), n=case["npoints"], train=case["train"])
    if kind == "mc":
        from madflow_amd.multichannel import MultiChannelIntegrand
        ig = MultiChannelIntegrand(case["process"], PROCESSES[case["process"]][2], precision=case["precision"],
                                   seed=seed, **_cuts(case["process"]))
        return dict(kind=kind, ig=ig, n=case["npoints"])
    from madflow_amd.flow import RQSFlow
    masks = np.array([o["mask"] for o in _flow_layers(case["dim"], case["layers"])[0]])
    flow = RQSFlow(case["dim"], layers=case["layers"], seed=seed, masks=masks)
    flow.params.copy_(_flow_params(case, seed))
    flow.adam_step(torch.zeros_like(flow.params), lr=0.0)      # the bf16 copies follow the parameters
    g = _gen(seed + 1)
    y = torch.rand((case["nev"], case["dim"]), generator=g, device="cuda")
    if kind == "flow_grad":
        f = torch.exp(2.0 * torch.randn(case["nev"], generator=g, device="cuda", dtype=torch.float64))
        return dict(kind=kind, flow=flow, y=y, f=f, beta=case["beta"])
    return dict(kind=kind, flow=flow, y=y, mix=case["mix"])


def _flow_layers(dim, layers):
    """Per layer: its mask (1 = transformed) and the offsets of W1 (16, 128), b1, W2 (128, 128),
    b2, W3 (128, NP), b3 in the flat parameter vector; and the length of that vector."""
    out, at = [], 0
    for l in range(layers):
        mask = [1 if ((d >> (l // 2 % max(1, math.ceil(math.log2(dim))))) & 1) == (l + 1) % 2 else 0
                for d in range(dim)]
        NP = (sum(mask) * 49 + 15) // 16 * 16
        o = dict(mask=mask, NP=NP)
        for key, size in (("W1", 16 * 128), ("b1", 128), ("W2", 128 * 128), ("b2", 128), ("W3", 128 * NP), ("b3", NP)):
            o[key] = at
            at += size
        out.append(o)
    return out, at


def _flow_params(case, seed):
    """Parameters of a partly trained flow (splines of moderate strength, not the identity)."""
    layers, n = _flow_layers(case["dim"], case["layers"])
    p, g = torch.zeros(n, device="cuda"), _gen(seed + 2)
    for o in layers:
        na = case["dim"] - sum(o["mask"])
        for key, size, scale in (("W1", na * 128, na ** -0.5), ("W2", 128 * 128, 128 ** -0.5), ("W3", 128 * o["NP"], 0.05)):
            p[o[key]:o[key] + size] = scale * torch.randn(size, generator=g, device="cuda")
    return p


# ----------------------------------------------------------------------------------- one pass
def run(state):
    kind = state["kind"]
    if kind == "me":
        return state["matrix"].smatrix(state["ps"], *state["params"])
    if kind == "vegas":
        ig = state["ig"]
        if state["train"]:
            ig.grid = state["grid"].clone()      # every pass starts from the same grid
        r = ig.iteration(state["n"], 1, train=state["train"])
        out = {k: r[k] for k in ("I", "sigma", "wmax", "npass")}
        if state["train"]:
            out["grid"] = ig.grid
        return out
    if kind == "mc":
        r = state["ig"].iteration(state["n"], 1, train=False)
        return {k: r[k] for k in ("I", "sigma", "wmax", "npass")}
    if kind == "flow_grad":
        if state["beta"]:
            return state["flow"].grad(state["y"], None, state["f"], state["beta"])
        return state["flow"].grad(state["y"], state["f"])
    return state["flow"].sample_mixture(state["y"], state["y"], state["mix"])


def work(case):
    kind = case["kind"]
    if kind == "me":
        _, k, _, flops = PROCESSES[case["process"]]
        n = case["nev"]
        couplings = (2 if case["process"].endswith("_ttx") else 3) * 16 if case["running"] else 0
        return dict(bytes=n * ((4 + k) * 32 + 8 + couplings), flops=n * flops)
    if kind in ("vegas", "mc"):
        # the points need not leave the chip: in and out go the grid and the sums
        _, k, _, flops = PROCESSES[case["process"]]
        return dict(bytes=8 * 2 * NBINS * 4 * (k + 2), flops=case["npoints"] * flops)
    d, layers, n = case["dim"], case["layers"], case["nev"]
    nb = d / 2.0 * 49.0
    gemm = 2.0 * (d / 2.0 * 128 + 128 * 128 + 128 * nb) * layers
    weights = layers * (16 * 128 + 128 * 128 + 128 * nb)
    if kind == "flow_grad":
        return dict(bytes=int(n * (4 * d + 8) + 4 * weights * 2), flops=int(3 * n * gemm))
    return dict(bytes=int(n * (4 * d * 2 + 8) + 4 * weights), flops=int(n * gemm))


# --------------------------------------------------------------------------- phase space, 64 bits
def _incoming(sqrts):
    e = 0.5 * sqrts
    z = torch.zeros_like(e)
    return torch.stack([torch.stack([e, z, z, e], -1), torch.stack([e, z, z, -e], -1)], 1)


def _rescale(p, masses, sqrts):
    """RAMBO's massive rescaling of massless momenta p, and the log of its weight factor;
    masses: one row, or one for each event."""
    m = torch.as_tensor(masses, dtype=torch.float64, device=p.device).expand(p.shape[:2])
    xi = torch.sqrt(1.0 - (m.sum(1) / sqrts) ** 2)
    e2 = p[..., 0] ** 2
    for _ in range(40):
        ne = torch.sqrt(m * m + e2 * xi[:, None] ** 2)
        xi = xi - (ne.sum(1) - sqrts) / (xi * (e2 / ne).sum(1))
    ne = torch.sqrt(m * m + e2 * xi[:, None] ** 2)
    v = p[..., 0] * xi[:, None]
    logw = (2 * m.shape[1] - 3) * torch.log(xi) + torch.log((v / ne).prod(1) / (v * v / ne).sum(1) * sqrts)
    return torch.cat([ne[..., None], p[..., 1:] * xi[:, None, None]], -1), logw


def _flat_weight(n, sqrts):
    logw = math.log(math.pi / 2.0) * (n - 1) - 2.0 * math.lgamma(n - 1) - math.log(n - 1)
    return logw + (2 * n - 4) * torch.log(sqrts) - (3 * n - 4) * math.log(2.0 * math.pi)


def _rambo(x, masses, sqrts):
    """RAMBO (Kleiss, Stirling, Ellis 1986): uniforms (N, 4n) -> momenta (N, n, 4), weights."""
    n = len(masses)
    u = x.reshape(-1, n, 4)
    ct = 2.0 * u[..., 0] - 1.0
    st, ph, e = torch.sqrt(1.0 - ct * ct), 2.0 * math.pi * u[..., 1], -torch.log(u[..., 2] * u[..., 3])
    q = torch.stack([e, e * st * torch.sin(ph), e * st * torch.cos(ph), e * ct], -1)
    Q = q.sum(1)
    M = torch.sqrt(Q[:, 0] ** 2 - (Q[:, 1:] ** 2).sum(1))
    b, gam = (-Q[:, 1:] / M[:, None])[:, None], (Q[:, 0] / M)[:, None]
    bq = (b * q[..., 1:]).sum(-1)
    s = (sqrts / M)[:, None]
    p = torch.cat([((gam * q[..., 0] + bq) * s)[..., None],
                   (q[..., 1:] + b * (bq / (1.0 + gam) + q[..., 0])[..., None]) * s[..., None]], -1)
    p, logw = _rescale(p, masses, sqrts)
    return p, torch.exp(logw + _flat_weight(n, sqrts))


def _diet(x, masses, sqrts):
    """RAMBO on diet (Platzer 2013): uniforms (N, 3n - 4) -> momenta, weights."""
    n = (x.shape[1] + 4) // 3
    M, Q, p = sqrts, _incoming(sqrts).sum(1), []
    for i in range(n - 1):
        Mn = torch.zeros_like(M)
        if i < n - 2:
            k, lo, hi = n - 2 - i, torch.zeros_like(M), torch.ones_like(M)
            for _ in range(70):          # F(u) = (k + 1) u^k - k u^(k + 1) = x by bisection
                mid = 0.5 * (lo + hi)
                up = (k + 1) * mid ** k - k * mid ** (k + 1) > x[:, i]
                lo, hi = torch.where(up, lo, mid), torch.where(up, mid, hi)
            Mn = M * torch.sqrt(0.5 * (lo + hi))
        e = (M * M - Mn * Mn) / (2.0 * M)
        ct, ph = 2.0 * x[:, n - 2 + 2 * i] - 1.0, 2.0 * math.pi * x[:, n - 1 + 2 * i]
        st = torch.sqrt(torch.clamp(1.0 - ct * ct, min=0.0))
        k3 = torch.stack([e * st * torch.cos(ph), e * st * torch.sin(ph), e * ct], -1)
        b, gam = Q[:, 1:] / M[:, None], Q[:, 0] / M
        bk = (b * k3).sum(1)
        pi = torch.cat([(gam * e + bk)[:, None], k3 + b * (bk / (gam + 1.0) + e)[:, None]], 1)
        p.append(pi)
        Q, M = Q - pi, Mn
    p, logw = _rescale(torch.stack(p + [Q], 1), masses, sqrts)
    return p, torch.exp(logw + _flat_weight(n, sqrts))


def _pass_cuts(p, pt_min, dr_min):
    """The cuts on the massless legs 2.. of outgoing momenta p."""
    ok = torch.ones(p.shape[0], dtype=torch.bool, device=p.device)
    j = p[:, 2:]
    if pt_min > 0.0:
        ok &= (torch.hypot(j[..., 1], j[..., 2]) > pt_min).all(1)
    if dr_min > 0.0:
        pa = torch.sqrt((j[..., 1:] ** 2).sum(-1))
        eta, phi = 0.5 * torch.log((pa + j[..., 3]) / (pa - j[..., 3])), torch.atan2(j[..., 2], j[..., 1])
        for a, b in itertools.combinations(range(j.shape[1]), 2):
            dp = (phi[:, a] - phi[:, b]).abs()
            dp = torch.minimum(dp, 2.0 * math.pi - dp)
            ok &= (eta[:, a] - eta[:, b]) ** 2 + dp * dp > dr_min * dr_min
    return ok


def _philox(n, ndim, seed, iteration, first=0):
    """Uniforms of Philox4x32-10 (Salmon et al. 2011): counter (event, pair, iteration)."""
    u32 = np.uint64(0xFFFFFFFF)
    out = np.empty((n, ndim + 1))
    ev = np.arange(n, dtype=np.uint64) + np.uint64(first)
    for j in range((ndim + 1) // 2):
        c = [ev & u32, ev >> np.uint64(32), np.full(n, j, np.uint64), np.full(n, iteration, np.uint64)]
        k0, k1 = seed & 0xFFFFFFFF, 0x6D66
        for _ in range(10):
            p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
            c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & u32,
                 (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & u32]
            k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
        for h in range(2):
            m = ((c[2 * h] >> np.uint64(5)) << np.uint64(26)) | (c[2 * h + 1] >> np.uint64(6))
            out[:, 2 * j + h] = (m.astype(np.float64) + 0.5) / 9007199254740992.0
    return torch.from_numpy(np.ascontiguousarray(out[:, :ndim])).cuda()


def _refine(hist):
    """VEGAS refinement of a uniform grid (Lepage 1978, damping 1.5), one dimension."""
    n = len(hist)
    pad = np.concatenate([[0.0], hist, [0.0]])
    s = (pad[:-2] + pad[1:-1] + pad[2:]) / np.array([2.0] + [3.0] * (n - 2) + [2.0])
    r = s / s.sum()
    reg = np.array([((1.0 - v) / math.log(1.0 / v)) ** 1.5 if 0.0 < v < 1.0 else 0.0 for v in r])
    edges, ave = np.linspace(0.0, 1.0, n + 1), reg.mean()
    new, k, acc = edges.copy(), -1, 0.0
    for j in range(1, n):
        while acc < ave and k < n - 1:
            k += 1
            acc += reg[k]
        acc -= ave
        new[j] = edges[k + 1] - (edges[k + 1] - edges[k]) * acc / reg[k]
    return new


# ----------------------------------------------------------------------- matrix elements, 64 bits
def _gell_mann():
    t = np.zeros((8, 3, 3), dtype=complex)
    for a, (i, j) in enumerate([(0, 1), (0, 2), (1, 2)]):
        r, c = [(0, 1), (3, 4), (5, 6)][a]
        t[r, i, j] = t[r, j, i] = 0.5
        t[c, i, j], t[c, j, i] = -0.5j, 0.5j
    t[2] = np.diag([0.5, -0.5, 0.0])
    t[7] = np.diag([1.0, 1.0, -2.0]) / (2.0 * math.sqrt(3.0))
    f = -2j * np.einsum("abij,cji->abc", np.einsum("aij,bjk->abik", t, t) - np.einsum("bij,ajk->abik", t, t), t)
    return torch.from_numpy(t).cuda(), f.real


def _gamma():
    """Dirac matrices, Dirac representation, lower index."""
    s = np.array([[[0, 1], [1, 0]], [[0, -1j], [1j, 0]], [[1, 0], [0, -1]]])
    g = np.zeros((4, 4, 4), dtype=complex)
    g[0] = np.diag([1, 1, -1, -1])
    for k in range(3):
        g[k + 1, :2, 2:], g[k + 1, 2:, :2] = -s[k], s[k]
    return torch.from_numpy(g).cuda()


class _Feynman:
    """|M|^2 / g^(2 (2 + k)) of one process: every Feynman diagram as a pair (colour tensor,
    kinematics), summed over helicities and colours.  ``p`` (N, legs, 4); helicities are
    tensor axes, one for each leg.  A current is a list of terms (colour letters, colour
    tensor with the open index last, kinematics); momenta count as incoming."""

    def __init__(self, process, p):
        self.beams, k, _, _ = PROCESSES[process]
        self.T, f = _gell_mann()
        self.f = torch.from_numpy(f).cuda().to(torch.complex128)
        self.ff = torch.einsum("abe,cde->abcd", self.f, self.f)
        self.g = _gamma()
        self.p, self.L = p, p.shape[1]
        self.metric = torch.tensor([1.0, -1, -1, -1], dtype=torch.float64, device=p.device)
        antiquark_beam = process.startswith("uxg")
        out_leg = self.L - 1
        if self.beams == "gg":
            self.gluons, self.light, self.avg = [0, 1] + list(range(4, self.L)), None, 256.0 * math.factorial(k)
        elif self.beams == "qq":
            self.gluons, self.avg = list(range(4, self.L)), 36.0 * math.factorial(k)
            self.light = (self.spinor(1, "vbar", 0.0), -p[:, 1], self.spinor(0, "u", 0.0), p[:, 0], "q", "r")
        else:
            self.gluons, self.avg = [1] + list(range(4, out_leg)), 96.0
            if antiquark_beam:
                self.light = (self.spinor(0, "vbar", 0.0), -p[:, 0], self.spinor(out_leg, "v", 0.0), -p[:, out_leg],
                              "q", "r")
            else:
                self.light = (self.spinor(out_leg, "ubar", 0.0), p[:, out_leg], self.spinor(0, "u", 0.0), p[:, 0],
                              "q", "r")
        self.memo = {}

    def axis(self, leg, values):
        """(2, N, c) helicity components of a leg -> its own axis of (2, ..., N, c)."""
        shape = [1] * self.L + list(values.shape[1:])
        shape[leg] = 2
        return values.reshape(shape)

    def spinor(self, leg, kind, m):
        E, px, py, pz = self.p[:, leg].to(torch.complex128).unbind(-1)
        w = torch.sqrt(E + m)
        z, o = torch.zeros_like(E), torch.ones_like(E)
        comp = []
        for a, b in ((o, z), (z, o)):
            low = torch.stack([pz * a + (px - 1j * py) * b, (px + 1j * py) * a - pz * b], -1) / (E + m)[:, None]
            up = torch.stack([a, b], -1)
            comp.append(torch.cat([up, low] if kind[0] == "u" else [low, up], -1) * w[:, None])
        s = torch.stack(comp)
        if kind.endswith("bar"):
            s = s.conj() * torch.tensor([1, 1, -1, -1], device=s.device)
        return self.axis(leg, s)

    def polarisation(self, leg):
        _, px, py, pz = self.p[:, leg].unbind(-1)
        th, ph = torch.atan2(torch.hypot(px, py), pz), torch.atan2(py, px)
        z = torch.zeros_like(th)
        e1 = torch.stack([z, torch.cos(th) * torch.cos(ph), torch.cos(th) * torch.sin(ph), -torch.sin(th)], -1)
        e2 = torch.stack([z, -torch.sin(ph), torch.cos(ph), z], -1)
        return self.axis(leg, torch.stack([e1, e2]).to(torch.complex128))

    def momentum(self, X):
        """Incoming momentum of a set of gluon legs ('Q': the light quark pair)."""
        tot = torch.zeros_like(self.p[:, 0])
        for l in X:
            if l == "Q":
                tot = tot + self.light[3] - self.light[1]
            else:
                tot = tot + (self.p[:, l] if l < 2 else -self.p[:, l])
        return tot

    def dot(self, a, b):
        return (a * b * self.metric).sum(-1, keepdim=True)

    def slash(self, v):
        return torch.einsum("...m,mij->...ij", v.to(torch.complex128), self.g)

    def propagate(self, k, m):
        """i (k-slash + m) / (k^2 - m^2 + i m Gamma)."""
        den = (self.dot(k, k)[..., 0] - m * m + 1j * m * (WT if m else 0.0))
        eye = torch.eye(4, dtype=torch.complex128, device=k.device)
        return 1j * (self.slash(k) + m * eye) / den[..., None, None]

    def gluon(self, X):
        """Terms of the off-shell gluon current of the frozenset X (open adjoint index)."""
        if X in self.memo:
            return self.memo[X]
        terms = []
        if len(X) == 1 and "Q" not in X:
            (l,) = X
            terms = [(chr(97 + l), torch.eye(8, dtype=torch.complex128, device="cuda"), self.polarisation(l))]
            self.memo[X] = terms
            return terms
        legs = sorted(X, key=str)
        P = self.momentum(X)
        prop = -1j / self.dot(P, P)
        if "Q" in X:
            rest = X - {"Q"}
            for r in range(len(rest) + 1):
                for A in itertools.combinations(sorted(rest), r):
                    A = frozenset(A)
                    for (la, ca, ka), (lb, cb, kb) in itertools.product(self.row("light", A), self.column(rest - A)):
                        c = torch.einsum("%sx,zxy,%sy->%sz" % (la, lb, la + lb), ca, self.T, cb)
                        v = torch.einsum("...i,mij,...j->...m", ka, self.g, kb) * self.metric
                        terms.append((la + lb, c, 1j * v * prop))
        first, others = legs[0], legs[1:]
        for r in range(len(others)):
            for rest in itertools.combinations(others, r):
                A = frozenset((first,) + rest)
                B = X - A
                kA, kB = self.momentum(A), self.momentum(B)
                for (la, ca, a), (lb, cb, b) in itertools.product(self.gluon(A), self.gluon(B)):
                    c = torch.einsum("%sx,%sy,xyz->%sz" % (la, lb, la + lb), ca, cb, self.f)
                    v = (self.dot(a, b) * (kA - kB) + b * self.dot(2.0 * kB + kA, a) - a * self.dot(2.0 * kA + kB, b))
                    terms.append((la + lb, c, v * prop))
        for part in _three_parts(legs):
            A, B, C = (frozenset(x) for x in part)
            for (la, ca, a), (lb, cb, b), (lc, cc, d) in itertools.product(self.gluon(A), self.gluon(B), self.gluon(C)):
                ab, ad, bd = self.dot(a, b), self.dot(a, d), self.dot(b, d)
                # f^{abe} f^{cze}, f^{ace} f^{bze}, f^{aze} f^{bce} and their Lorentz structures
                for spec, v in (("xywz", b * ad - a * bd), ("xwyz", d * ab - a * bd), ("xzyw", d * ab - b * ad)):
                    c = torch.einsum("%sx,%sy,%sw,%s->%sz" % (la, lb, lc, spec, la + lb + lc), ca, cb, cc, self.ff)
                    terms.append((la + lb + lc, c, -1j * v * prop))
        self.memo[X] = terms
        return terms

    def row(self, line, X):
        """Terms of the outgoing end of a quark line ("top" or "light") that has absorbed X
        (open colour index, row spinor with its propagator)."""
        key = (line, X)
        if key in self.memo:
            return self.memo[key]
        left, kout, m = ((self.spinor(2, "ubar", MT), self.p[:, 2], MT) if line == "top" else
                         (self.light[0], self.light[1], 0.0))
        letter = "s" if line == "top" else self.light[4]
        if not X:
            terms = [(letter, torch.eye(3, dtype=torch.complex128, device="cuda"), left)]
        else:
            terms = [(l, c, torch.einsum("...i,...ij->...j", k, self.propagate(kout - self.momentum(X), m)))
                     for l, c, k in self.emissions(line, X)]
        self.memo[key] = terms
        return terms

    def emissions(self, line, X):
        """The row of ``line`` after its vertex with the last of the gluons X, no propagator."""
        for r in range(1, len(X) + 1):
            for A in itertools.combinations(sorted(X, key=str), r):
                A = frozenset(A)
                for (ll, cl, kl), (lg, cg, kg) in itertools.product(self.row(line, X - A), self.gluon(A)):
                    c = torch.einsum("%sx,%sw,wxy->%sy" % (ll, lg, ll + lg), cl, cg, self.T)
                    yield ll + lg, c, 1j * torch.einsum("...i,...ij->...j", kl, self.slash(kg))

    def column(self, X):
        """Terms of the incoming end of the light line that has absorbed X."""
        key = ("column", X)
        if key in self.memo:
            return self.memo[key]
        right, kin, letter = self.light[2], self.light[3], self.light[5]
        if not X:
            terms = [(letter, torch.eye(3, dtype=torch.complex128, device="cuda"), right)]
        else:
            terms = []
            prop = self.propagate(kin + self.momentum(X), 0.0)
            for r in range(1, len(X) + 1):
                for A in itertools.combinations(sorted(X), r):
                    A = frozenset(A)
                    for (lr, cr, kr), (lg, cg, kg) in itertools.product(self.column(X - A), self.gluon(A)):
                        c = torch.einsum("%sx,%sw,wyx->%sy" % (lr, lg, lr + lg), cr, cg, self.T)
                        k = torch.einsum("...ij,...jk,...k->...i", prop, self.slash(kg), kr)
                        terms.append((lr + lg, c, 1j * k))
        self.memo[key] = terms
        return terms

    def squared(self, gram):
        """(N,) |M|^2; gram: a cache of the colour Gram matrix (the same for every batch)."""
        X = frozenset(self.gluons + (["Q"] if self.light else []))
        v = self.spinor(3, "v", MT)
        amps, colours = [], []
        for l, c, k in self.emissions("top", X):
            amps.append((k * v).sum(-1))
            if "G" not in gram:
                order = "".join(sorted(l))
                colours.append(torch.einsum("%sy->%sy" % (l, order), c).reshape(-1))
        if "G" not in gram:
            C = torch.stack(colours)
            gram["G"] = C.conj() @ C.T
        n = self.p.shape[0]
        full = [2] * self.L + [n]
        A = torch.stack([a.expand(full) for a in amps]).reshape(len(amps), -1)
        return ((gram["G"] @ A) * A.conj()).sum(0).real.reshape(-1, n).sum(0) / self.avg


def _three_parts(legs):
    """Unordered partitions of legs into three non-empty parts."""
    seen = set()
    for lab in itertools.product(range(3), repeat=len(legs)):
        parts = [tuple(l for l, q in zip(legs, lab) if q == i) for i in range(3)]
        if all(parts):
            key = frozenset(parts)
            if key not in seen:
                seen.add(key)
                yield parts


# diagram terms and seconds of one batch, about, by the number of radiated legs
EXACT_TERMS = {0: 3, 1: 18, 2: 160, 3: 1900}
EXACT_SECONDS = {0: 0.01, 1: 0.02, 2: 0.12, 3: 0.9}


def _batch(process):
    k = PROCESSES[process][1]
    return max(64, int(2e9 / (16 * 2 ** (4 + k) * EXACT_TERMS[k])))


def _too_long(process, nev):
    return nev / _batch(process) * EXACT_SECONDS[PROCESSES[process][1]] > 15.0


def _squared(process, ps, gs):
    """|M|^2 of the momenta ps with the strong coupling gs (a number or one per event).  The
    polarisation vectors are scaled as the framework's default does (sqrt(1/2) in 32 bits)."""
    beams, k, _, _ = PROCESSES[process]
    batch = _batch(process)
    gram, out = {}, []
    for a in range(0, ps.shape[0], batch):
        out.append(_Feynman(process, ps[a:a + batch]).squared(gram))
    gluons = {"gg": 2, "qq": 0, "qg": 0}[beams] + k
    sqh = float(np.float32(math.sqrt(0.5)))
    return torch.cat(out) * (2.0 * sqh * sqh) ** gluons * gs ** (2 * (2 + k))


# ------------------------------------------------------------------------------- flow, 64 bits
def _spline(raw, v, inverse):
    """Rational-quadratic spline (Durkan et al. 2019), 16 bins on [0, 1]: value and log slope."""
    K, mn = 16, 1e-3
    edges = []
    for part in (raw[..., :K], raw[..., K:2 * K]):
        w = mn + (1.0 - K * mn) * torch.softmax(part, -1)
        c = torch.cumsum(w, -1)[..., :-1]
        edges.append(torch.cat([torch.zeros_like(w[..., :1]), c, torch.ones_like(w[..., :1])], -1))
    slope = mn + torch.nn.functional.softplus(raw[..., 2 * K:])
    k = (v[..., None] >= edges[1 if inverse else 0][..., 1:-1]).sum(-1, keepdim=True)
    (x0, x1), (y0, y1) = [(e.gather(-1, k)[..., 0], e.gather(-1, k + 1)[..., 0]) for e in edges]
    a, c = slope.gather(-1, k)[..., 0], slope.gather(-1, k + 1)[..., 0]
    s = (y1 - y0) / (x1 - x0)
    g = a + c - 2.0 * s
    if inverse:
        d = v - y0
        qa, qb, qc = (y1 - y0) * (s - a) + d * g, (y1 - y0) * a - d * g, -s * d
        xi = 2.0 * qc / (-qb - torch.sqrt(qb * qb - 4.0 * qa * qc))
    else:
        xi = (v - x0) / (x1 - x0)
    t = xi * (1.0 - xi)
    den = s + g * t
    ld = 2.0 * torch.log(s) + torch.log(c * xi * xi + 2.0 * s * t + a * (1.0 - xi) ** 2) - 2.0 * torch.log(den)
    if inverse:
        return x0 + xi * (x1 - x0), -ld
    return y0 + (y1 - y0) * (s * xi * xi + a * t) / den, ld


def _flow64(params, layers, x, inverse):
    """The coupling flow: (N, dim) points -> points, log of the determinant."""
    ld = torch.zeros(x.shape[0], dtype=torch.float64, device=x.device)
    for o in (reversed(layers) if inverse else layers):
        A = [d for d, m in enumerate(o["mask"]) if not m]
        B = [d for d, m in enumerate(o["mask"]) if m]
        NP = o["NP"]
        W = lambda key, shape: params[o[key]:o[key] + math.prod(shape)].reshape(shape)
        h = torch.relu(x[:, A] @ W("W1", (16, 128))[:len(A)] + W("b1", (128,)))
        h = torch.relu(h @ W("W2", (128, 128)) + W("b2", (128,)))
        raw = (h @ W("W3", (128, NP)) + W("b3", (NP,)))[:, :len(B) * 49].reshape(-1, len(B), 49)
        z, dl = _spline(raw, x[:, B], inverse)
        x = x.clone()
        x[:, B] = z
        ld = ld + dl.sum(1)
    return x, ld


# ------------------------------------------------------------------------------------ exact
def exact(case, seed):
    kind = case["kind"]
    gs0 = 2.0 * math.sqrt(math.pi * 0.118)
    if kind == "me":
        if _too_long(case["process"], case["nev"]):
            return None
        gs = gs0
        if case["running"]:
            q = 100.0 + 900.0 * torch.rand(case["nev"], generator=_gen(seed + 7), dtype=torch.float64, device="cuda")
            gs = 2.0 * torch.sqrt(math.pi * _alpha_s(q * q))
        return _squared(case["process"], _momenta(case["process"], case["nev"], seed), gs)
    if kind == "vegas":
        return _exact_vegas(case, seed, gs0)
    if kind == "mc":
        return _exact_mc(case, seed, gs0)
    params, layers = _flow_params(case, seed).double(), _flow_layers(case["dim"], case["layers"])[0]
    g = _gen(seed + 1)
    y = torch.rand((case["nev"], case["dim"]), generator=g, device="cuda").double()
    if kind == "flow_sample":
        nu = int(round(case["mix"] * case["nev"]))
        _, ldu = _flow64(params, layers, y[:nu], False)
        s, lds = _flow64(params, layers, y[nu:], True)
        ld = torch.cat([ldu, -lds])
        return torch.cat([y[:nu], s]), 1.0 / ((1.0 - case["mix"]) * torch.exp(ld) + case["mix"])
    f = torch.exp(2.0 * torch.randn(case["nev"], generator=g, device="cuda", dtype=torch.float64))
    params.requires_grad_(True)
    _, lq = _flow64(params, layers, y, False)
    v = (f / torch.exp(lq.detach())) ** case["beta"] if case["beta"] else f
    loss = -(v * lq).sum() / v.sum()
    loss.backward()
    return loss.detach(), params.grad


def _exact_vegas(case, seed, gs0):
    process, n = case["process"], case["npoints"]
    if _too_long(process, n):
        return None
    m = _masses(process)
    k = len(m)
    ndim = {"rambo": 4 * k, "diet": 3 * k - 4, "hadronic": 4 * k + 2}[case["mapping"]]
    y = _philox(n, ndim, seed, 1)
    sqrts = torch.full((n,), PROCESSES[process][2], dtype=torch.float64, device="cuda")
    if case["mapping"] == "hadronic":
        s = 13000.0 ** 2
        taumin = sum(m) ** 2 / s
        tau = y[:, 0] * (1.0 - taumin) + taumin
        x1 = tau ** y[:, 1]
        x2 = tau / x1
        sqrts = torch.sqrt(tau * s)
        p, w = _rambo(y[:, 2:], m, sqrts)
        w = w * (1.0 - taumin) * -torch.log(tau)
    else:
        p, w = (_rambo if case["mapping"] == "rambo" else _diet)(y, m, sqrts)
    ok = _pass_cuts(p, **_cuts(process)) & torch.isfinite(w)
    w = w * GEV2PB / (2.0 * sqrts * sqrts)
    ps = torch.cat([_incoming(sqrts), p], 1)[ok]
    gs = gs0
    if case["mapping"] == "hadronic":
        q2 = (0.5 * torch.sqrt(torch.clamp(p[ok][..., 0] ** 2 - p[ok][..., 3] ** 2, min=0.0)).sum(1)) ** 2
        # the dynamic scale is taken in the lab frame, where the transverse masses are the same
        gs = 2.0 * torch.sqrt(math.pi * _alpha_s(q2))
        w = w.clone()
        w[ok] = w[ok] * _gluon_density(x1[ok], q2) * _gluon_density(x2[ok], q2) / (x1[ok] * x2[ok])
    f = torch.zeros_like(w)
    f[ok] = w[ok] * _squared(process, ps, gs)
    I = float(f.mean())
    out = dict(I=I, sigma=math.sqrt(max((float((f * f).mean()) - I * I) / (n - 1.0), 0.0)), wmax=float(f.max()),
               npass=int(ok.sum()))
    if case["train"]:
        b = torch.clamp((y * NBINS).long(), max=NBINS - 1)
        hist = torch.stack([torch.bincount(b[:, d], weights=f * f, minlength=NBINS) for d in range(ndim)])
        out["grid"] = torch.from_numpy(np.stack([_refine(h) for h in hist.cpu().numpy()])).cuda()
    return out


def _boost(k, Q, M, sign=1.0):
    """Momenta k (N, n, 4) boosted by the velocity of Q (N, 4), mass M (-1: into its rest frame)."""
    b, gam = (sign * Q[:, 1:] / M[:, None])[:, None], (Q[:, 0] / M)[:, None]
    bk = (b * k[..., 1:]).sum(-1)
    return torch.cat([(gam * k[..., 0] + bk)[..., None], k[..., 1:] + b * (bk / (gam + 1.0) + k[..., 0])[..., None]], -1)


def _mass(p):
    return torch.sqrt(torch.clamp(p[..., 0] ** 2 - (p[..., 1:] ** 2).sum(-1), min=0.0))


def _diet_weight(p, M):
    """The weight that RAMBO on diet gives the momenta p, at rest with mass M."""
    pa = torch.sqrt((p[..., 1:] ** 2).sum(-1))
    n = p.shape[1]
    logw = (2 * n - 3) * torch.log(pa.sum(1) / M)
    logw = logw + torch.log((pa / p[..., 0]).prod(1) / (pa * pa / p[..., 0]).sum(1) * M)
    return torch.exp(logw + _flat_weight(n, M))


def _channels(process):
    """(type, legs, lo, hi): flat, a t-channel for each massless leg, an s-channel for each pair."""
    m, s, cuts = _masses(process), PROCESSES[process][2], _cuts(process)
    light = list(range(2, len(m)))
    m_lo = 0.9 * cuts["pt_min"] * cuts["dr_min"] if cuts["dr_min"] else 1e-3 * s
    return ([("flat", (), 0.0, 0.0)] + [("t", (a,), cuts["pt_min"], (s * s - sum(m) ** 2) / (2.0 * s)) for a in light] +
            [("s", ab, m_lo ** 2, (s - sum(m)) ** 2) for ab in itertools.combinations(light, 2)])


def _channel_points(channel, x, m, sqrts):
    """Momenta of a channel at the cube points x, and where they exist."""
    kind, legs, lo, hi = channel
    if kind == "flat":
        return _diet(x, m, sqrts)[0], torch.ones_like(sqrts, dtype=torch.bool)
    rest = [i for i in range(len(m)) if i not in legs]
    p = torch.zeros((x.shape[0], len(m), 4), dtype=torch.float64, device=x.device)
    ph = 2.0 * math.pi * x[:, 2]
    if kind == "t":
        pt = 1.0 / (1.0 / lo - x[:, 0] * (1.0 / lo - 1.0 / hi))
        y = (2.0 * x[:, 1] - 1.0) * torch.acosh(torch.clamp(hi / pt, min=1.0))
        k = torch.stack([pt * torch.cosh(y), pt * torch.cos(ph), pt * torch.sin(ph), pt * torch.sinh(y)], -1)
        X = _incoming(sqrts).sum(1) - k
        MX = _mass(X)
        ok = MX > sum(m)
        MX = torch.where(ok, MX, sqrts)
        p[:, rest] = _boost(_diet(x[:, 3:], [m[i] for i in rest], MX)[0], X, MX)
        p[:, legs[0]] = k
        return p, ok
    mG = torch.sqrt(lo * torch.exp(x[:, 0] * math.log(hi / lo)))
    ok = sqrts > sum(m) + mG
    mG = torch.where(ok, mG, torch.ones_like(mG))
    masses = torch.stack([torch.full_like(mG, m[i]) for i in rest] + [mG], 1)
    q, _ = _diet(x[:, 3:], masses, sqrts)
    p[:, rest] = q[:, :-1]
    ct = 2.0 * x[:, 1] - 1.0
    st = torch.sqrt(1.0 - ct * ct)
    n = torch.stack([torch.ones_like(ct), st * torch.cos(ph), st * torch.sin(ph), ct], -1) * (0.5 * mG)[:, None]
    back = torch.cat([n[:, :1], -n[:, 1:]], 1)
    p[:, list(legs)] = _boost(torch.stack([n, back], 1), q[:, -1], mG)
    return p, ok


def _channel_density(channel, p, m, sqrts):
    """1 / (dPhi/dx) of a channel at the momenta p; 0 outside its range."""
    kind, legs, lo, hi = channel
    if kind == "flat":
        return 1.0 / _diet_weight(p, sqrts)
    rest = [i for i in range(len(m)) if i not in legs]
    if kind == "t":
        k = p[:, legs[0]]
        pt = torch.hypot(k[:, 1], k[:, 2])
        ymax = torch.acosh(torch.clamp(hi / pt, min=1.0))
        X = _incoming(sqrts).sum(1) - k
        MX = _mass(X)
        w = pt ** 3 * (1.0 / lo - 1.0 / hi) * 2.0 * ymax / (8.0 * math.pi ** 2)
        w = w * _diet_weight(_boost(p[:, rest], X, MX, -1.0), MX)
        ok = (pt >= lo) & (pt <= hi) & (torch.asinh(k[:, 3] / pt).abs() <= ymax) & (MX > sum(m))
    else:
        G = p[:, list(legs)].sum(1)
        m2 = _mass(G) ** 2
        w = m2 * math.log(hi / lo) / (16.0 * math.pi ** 2) * _diet_weight(torch.cat([p[:, rest], G[:, None]], 1), sqrts)
        ok = (m2 >= lo) & (m2 <= hi)
    v = torch.where(ok, 1.0 / w, torch.zeros_like(w))
    return torch.where(torch.isfinite(v), v, torch.zeros_like(v))


def _exact_mc(case, seed, gs0):
    process, N = case["process"], case["npoints"]
    if _too_long(process, N):
        return None
    m, channels = _masses(process), _channels(process)
    K = len(channels)
    counts = [max(int(math.floor(N / K)), min(1000, N // K))] * K
    counts[0] += N - sum(counts)
    total, var, wmax, npass = 0.0, 0.0, 0.0, 0
    for c, (channel, n) in enumerate(zip(channels, counts)):
        sqrts = torch.full((n,), PROCESSES[process][2], dtype=torch.float64, device="cuda")
        p, ok = _channel_points(channel, _philox(n, 3 * len(m) - 4, seed, 1, c << 40), m, sqrts)
        g = sum(_channel_density(ch, p, m, sqrts) / K for ch in channels)
        ok &= _pass_cuts(p, **_cuts(process)) & (g > 0.0)
        ps = torch.cat([_incoming(sqrts), p], 1)[ok]
        f = torch.zeros(n, dtype=torch.float64, device="cuda")
        f[ok] = _squared(process, ps, gs0) * (N / K / n) / g[ok] * GEV2PB / (2.0 * sqrts[ok] ** 2)
        total += float(f.sum())
        var += max((float((f * f).mean()) - float(f.mean()) ** 2) / (n - 1.0), 0.0) * (n / N) ** 2
        wmax, npass = max(wmax, float(f.max())), npass + int(ok.sum())
    return dict(I=total / N, sigma=math.sqrt(var), wmax=wmax, npass=npass)
