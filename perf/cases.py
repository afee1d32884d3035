"""The measured cases of the SPECT projector and the algorithms that drive it.

Each case is one call that a user of the package makes: a projection or back
projection of one subset, an OSEM run, a whole reconstruction of new data
(sensitivities included), a gradient with respect to activity and attenuation,
a batch of uneven reconstructions, and a differentiated BSREM.  Sizes follow
the package's benchmark (64^3 to 192^3, 60 to 180 angles, 4.8 mm voxels, 25 cm
orbits, sigma(d) = 0.03 d + 0.1 cm); ragged grids and body-contour orbits come
from its parity tests.

Inputs are made with torch from the seed alone; ``exact`` computes the same
outputs in float64 with plain torch (grid_sample, matmul, cumsum).
"""
from __future__ import annotations

import math

import numpy as np
import torch
import torch.nn.functional as F

import pytomography_amd
from pytomography_amd.algorithms import OSEM
from pytomography_amd.autograd import poisson_log_likelihood
from pytomography_amd.batch import BatchedOSEM
from pytomography_amd.likelihoods import PoissonLogLikelihood
from pytomography_amd.metadata.SPECT import SPECTObjectMeta, SPECTProjMeta, SPECTPSFMeta
from pytomography_amd.priors import RelativeDifferencePrior
from pytomography_amd.projectors.SPECT import SPECTSystemMatrix
from pytomography_amd.transforms.SPECT import SPECTAttenuationTransform, SPECTPSFTransform
from pytomography_amd.unrolled import UnrolledBSREM

DX = 0.48                # voxel size, cm
SIGMA = (0.03, 0.1)      # sigma(d) = a d + b, cm
MIN_SIGMAS = 3
DELTA = 1e-11            # the package's delta in float32 and float64
BETA, GAMMA, FLOOR = 0.1, 2.0, 1e-4   # BSREM with the relative difference prior


def _case(name, kind, n, nz, angles, subsets, att=True, psf=True, orbit="circle", iters=1):
    c = dict(kind=kind, n=n, nz=nz, angles=angles, subsets=subsets, att=att, psf=psf,
             orbit=orbit, iters=iters)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # one subset's forward projection of a small object: launches and latency
        _case("forward_64x60_subset", "forward", 64, 64, 60, 8),
        # one OSEM iteration of a small object, as in a quick look or a phantom sweep
        _case("osem_64x60", "osem", 64, 64, 60, 8),
        # simulating the projections of every angle of a standard acquisition
        _case("forward_128x120", "forward", 128, 128, 120, 1),
        # one subset's back projection, the likelihood gradient of a user's own algorithm
        _case("backward_128x120_subset", "backward", 128, 128, 120, 8),
        # the standard reconstruction: one OSEM iteration, attenuation and PSF
        _case("osem_128x120", "osem", 128, 128, 120, 8),
        # the same without attenuation and PSF modelling
        _case("osem_128x120_plain", "osem", 128, 128, 120, 8, att=False, psf=False),
        # a cropped field of view on a body-contour orbit: odd sizes, subsets of
        # unequal length, a PSF table for every angle
        _case("osem_100x47_contour", "osem", 100, 47, 64, 6, orbit="contour"),
        # high resolution: one OSEM iteration
        _case("osem_192x180", "osem", 192, 192, 180, 12),
        # a whole reconstruction of new data on a known scanner geometry
        _case("recon_128x60", "recon", 128, 128, 60, 8, iters=2),
        # log-likelihood and its gradients for joint activity / attenuation estimation
        _case("grad_128x60", "grad", 128, 128, 60, 1),
        # a queue of uneven studies reconstructed together
        _case("batch_mix", "batch", 128, 0, 90, 8),
        # BSREM differentiated through its iterations (learned priors, hyperparameters)
        _case("unrolled_96x60", "unrolled", 96, 96, 60, 4, iters=2),
    ]


def draw(rng):
    kind = rng.choice(["forward", "backward", "osem", "osem", "recon", "grad", "unrolled"])
    top = {"recon": 112, "grad": 128, "unrolled": 88}.get(kind, 168)
    n = int(round(math.exp(rng.uniform(math.log(48), math.log(top)))))
    nz = rng.choice([n, n, rng.randint(33, n) if n > 33 else n])
    subsets = rng.choice([4, 5, 6, 8])
    angles = subsets * rng.randint(6, 15) + rng.choice([0, 0, 1, 3])
    att, psf = rng.choice([(True, True)] * 4 + [(False, True), (True, False), (False, False)])
    if kind in ("grad", "recon", "unrolled"):
        angles = min(angles, 64)
    if kind == "grad":
        att = True
        subsets = 1
    return _case(None, kind, n, nz, angles, subsets, att=att, psf=psf,
                 orbit=rng.choice(["circle", "circle", "contour"]),
                 iters=2 if kind in ("recon", "unrolled") else 1)


# ----------------------------------------------------------------- geometry
def _betas(case):
    return [k * 360.0 / case["angles"] for k in range(case["angles"])]


def _radii(case):
    """A circle, or a detector that follows an elliptical body contour."""
    if case["orbit"] == "circle":
        return [25.0] * case["angles"]
    return [round(22.0 + 3.0 * math.cos(2 * math.radians(b)), 3) for b in _betas(case)]


def _members(case):
    """The single problems of a case: itself, or a batch's uneven studies."""
    if case["kind"] != "batch":
        return [case]
    sizes = [(64, 60), (96, 90), (128, 60), (64, 120), (160, 60), (96, 60), (128, 120), (64, 90)]
    return [_case(None, "osem", n, n, a, case["subsets"]) for n, a in sizes]


def _subset(case):
    """The subset that a forward or backward case projects (None: every angle)."""
    return None if case["subsets"] == 1 else 1


def _rows(case, k):
    a = list(range(case["angles"]))
    return a if k is None else a[k::case["subsets"]]


# ------------------------------------------------------------------- inputs
def _gen(seed, dev):
    return torch.Generator(device=dev).manual_seed(int(seed))


def _ellipsoids(case, gen, dev, background):
    """Sum of six random ellipsoids inside the cylinder of the field of view."""
    n, nz = case["n"], case["nz"]
    u = torch.rand((6, 8), generator=gen, device=dev).tolist()
    x = torch.arange(n, device=dev, dtype=torch.float32).view(n, 1, 1)
    y = x.view(1, n, 1)
    z = torch.arange(nz, device=dev, dtype=torch.float32).view(1, 1, nz)
    out = torch.full((n, n, nz), background, device=dev)
    for r in u:
        semi = [min(5 + 35 * v, 0.45 * n) for v in r[:3]]
        room = max(n / 2 - 1 - max(semi[:2]), 0.0) * math.sqrt(r[3])
        cx = (n - 1) / 2 + room * math.cos(2 * math.pi * r[4])
        cy = (n - 1) / 2 + room * math.sin(2 * math.pi * r[4])
        cz = (nz - 1) * (0.2 + 0.6 * r[5])
        inside = ((x - cx) / semi[0]) ** 2 + ((y - cy) / semi[1]) ** 2 + ((z - cz) / semi[2]) ** 2 <= 1
        out += inside * (0.1 + 0.9 * r[6])
    return out


def _attenuation(case, gen, dev):
    """A water body with two bone inserts, 1/cm."""
    n, nz = case["n"], case["nz"]
    u = torch.rand((2, 6), generator=gen, device=dev).tolist()
    x = torch.arange(n, device=dev, dtype=torch.float32).view(n, 1, 1)
    y = x.view(1, n, 1)
    z = torch.arange(nz, device=dev, dtype=torch.float32).view(1, 1, nz)
    c, cz = (n - 1) / 2, (nz - 1) / 2
    mu = torch.zeros((n, n, nz), device=dev)
    mu[((x - c) / (0.42 * n)) ** 2 + ((y - c) / (0.36 * n)) ** 2 + ((z - cz) / (0.45 * nz)) ** 2 <= 1] = 0.15
    for r in u:
        s = [(0.05 + 0.07 * v) for v in r[:3]]
        ox, oy = (0.4 * r[3] - 0.2) * n, (0.4 * r[4] - 0.2) * n
        bz = (0.3 + 0.4 * r[5]) * (nz - 1)
        mu[((x - c - ox) / (s[0] * n)) ** 2 + ((y - c - oy) / (s[1] * n)) ** 2
           + ((z - bz) / (s[2] * nz)) ** 2 <= 1] = 0.25
    return mu


def _counts(case, activity, gen, dev):
    """Poisson counts over a scatter floor: the activity's line integrals at
    every angle, thinned by a constant for attenuation."""
    ref = _Reference(dict(case, att=False, psf=False), None, torch.float32, dev)
    expected = ref.forward(activity, None) * (40.0 / case["n"])
    scatter = torch.full_like(expected, 0.05 * float(expected.mean()) + 0.01)
    return torch.poisson((expected + scatter).clamp_(min=0), generator=gen), scatter


def _inputs(case, seed, dev):
    gen = _gen(seed, dev)
    d = {"activity": _ellipsoids(case, gen, dev, 0.0)}
    d["mu"] = _attenuation(case, gen, dev) if case["att"] else None
    kind = case["kind"]
    if kind == "backward":
        rows = len(_rows(case, _subset(case)))
        d["ratio"] = 0.5 + torch.rand((rows, case["n"], case["nz"]), generator=gen, device=dev)
    if kind in ("osem", "recon", "grad", "unrolled"):
        d["counts"], d["scatter"] = _counts(case, d["activity"], gen, dev)
    if kind in ("grad", "unrolled"):
        d["start"] = _ellipsoids(case, gen, dev, 0.2)
    return d


# ------------------------------------------------------- the package's calls
def _system_matrix(case, mu):
    om = SPECTObjectMeta((DX, DX, DX), (case["n"], case["n"], case["nz"]))
    pm = SPECTProjMeta((case["n"], case["nz"]), (DX, DX), _betas(case), radii=_radii(case))
    transforms = []
    if case["att"]:
        transforms.append(SPECTAttenuationTransform(mu))
    if case["psf"]:
        transforms.append(SPECTPSFTransform(SPECTPSFMeta(SIGMA, min_sigmas=MIN_SIGMAS)))
    sm = SPECTSystemMatrix(transforms, [], om, pm)
    if case["subsets"] > 1:
        sm.set_n_subsets(case["subsets"])
    return sm


def prepare(case, seed):
    dev = torch.device("cuda")
    pytomography_amd.set_device(dev)
    states = []
    for k, c in enumerate(_members(case)):
        d = _inputs(c, seed * 64 + k, dev)
        sm = _system_matrix(c, d["mu"])
        s = dict(d, sm=sm)
        if c["kind"] == "osem":
            # the plan, attenuation data and sensitivities that a program keeps
            # while it iterates
            s["likelihood"] = PoissonLogLikelihood(sm, d["counts"], additive_term=d["scatter"])
            s["likelihood"]._set_n_subsets(c["subsets"])
        elif c["kind"] == "unrolled":
            s["unrolled"] = UnrolledBSREM(sm, RelativeDifferencePrior(beta=BETA, gamma=GAMMA),
                                          additive_term=d["scatter"], n_iters=c["iters"],
                                          n_subsets=c["subsets"], addition_after_iteration=FLOOR)
        if c["kind"] in ("forward", "backward", "osem", "recon", "unrolled"):
            # attenuation data of the map, built with the first projection
            sm.forward(d["activity"], 0 if c["subsets"] > 1 else None)
        states.append(s)
    state = dict(case=case, members=states)
    if case["kind"] == "batch":
        state["batch"] = BatchedOSEM([s["likelihood"] for s in states], case["subsets"])
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    s = state["members"][0]
    if kind == "forward":
        return s["sm"].forward(s["activity"], _subset(case))
    if kind == "backward":
        return s["sm"].backward(s["ratio"], _subset(case))
    if kind == "osem":
        obj = OSEM(s["likelihood"])(case["iters"], case["subsets"])
        return {"object": obj, "projections_predicted": s["likelihood"].projections_predicted}
    if kind == "recon":
        lk = PoissonLogLikelihood(s["sm"], s["counts"], additive_term=s["scatter"])
        obj = OSEM(lk)(case["iters"], case["subsets"])
        return {"object": obj, "projections_predicted": lk.projections_predicted}
    if kind == "grad":
        f = s["start"].detach().requires_grad_(True)
        mu = s["mu"].detach().requires_grad_(True)
        value = poisson_log_likelihood(f, mu, s["sm"], s["counts"], s["scatter"])
        value.backward()
        return {"value": value.detach(), "grad_activity": f.grad, "grad_mu": mu.grad}
    if kind == "batch":
        for o in state["batch"].objects:
            o.fill_(1.0)
        return list(state["batch"].run(case["iters"]))
    if kind == "unrolled":
        g = s["counts"].detach().requires_grad_(True)
        x0 = s["start"].detach().requires_grad_(True)
        beta = torch.tensor(BETA, dtype=torch.float64, requires_grad=True)
        x = s["unrolled"](g, x0, beta)
        ((x - s["activity"]) ** 2).sum().backward()
        return {"object": x.detach(), "grad_counts": g.grad, "grad_start": x0.grad,
                "grad_beta": beta.grad}
    raise ValueError(kind)


# ---------------------------------------------------------------------- work
def work(case):
    """Inputs once, outputs once; per voxel and angle of each projection a
    bilinear sample, the attenuation product and the share in a PSF sum."""
    total = {"bytes": 0.0, "flops": 0.0}
    for c in _members(case):
        n2, nz, a = c["n"] ** 2, c["nz"], c["angles"]
        kind = c["kind"]
        vol, prj = 4.0 * n2 * nz, 4.0 * c["n"] * nz
        att = vol if c["att"] else 0.0
        voxel = n2 * nz * (8.0 + (1.0 if c["att"] else 0.0) + (4.0 if c["psf"] else 0.0))
        if kind in ("forward", "backward"):
            rows = len(_rows(c, _subset(c)))
            b, f = vol + att + rows * prj, rows * voxel
        elif kind in ("osem", "recon"):
            # per subset: object in and out, sensitivity, map; counts, scatter, prediction
            it = c["subsets"] * (3 * vol + att) + 3 * a * prj
            b, f = c["iters"] * it, c["iters"] * 2 * a * voxel
            if kind == "recon":  # the sensitivities, in float64
                b, f = b + c["subsets"] * (2 * vol + att), f + a * voxel
        elif kind == "grad":
            b, f = 4 * vol + 3 * a * prj, 4 * a * voxel
        else:  # unrolled: a sub-iteration, its recomputation and its reverse
            it = c["subsets"] * (12 * vol + 5 * att) + 10 * a * prj
            b, f = c["iters"] * it, c["iters"] * 6 * a * voxel
        total["bytes"] += b
        total["flops"] += f
    return total


# --------------------------------------------- the same in plain torch, float64
class _Reference:
    """Rotate, attenuate, blur and sum in plain torch: per angle the padded
    object is rotated by beta - 270 degrees (bilinear, zeros outside), weighted
    by exp(-(cumulative attenuation towards the detector at +x)), each plane
    blurred by its Gaussian along y and z, and summed along x; back projection
    runs the steps in reverse with the rotation by 270 - beta."""

    def __init__(self, case, mu, dtype, dev):
        self.case, self.dtype, self.dev = case, dtype, dev
        n = case["n"]
        self.pad = math.ceil((math.sqrt(2) * n - n) / 2)
        self.P = n + 2 * self.pad
        self.mu = None if mu is None else mu.to(dtype)
        self.beta = torch.tensor(_betas(case)).to(torch.float32).to(torch.float64).tolist()
        self.radii = _radii(case)
        self._blur = (None, None)

    def _rotate(self, x, degrees):
        """x [P, P, nz] rotated about the centre of the frame."""
        c, s = math.cos(math.radians(degrees)), math.sin(math.radians(degrees))
        theta = torch.tensor([[[c, -s, 0.0], [s, c, 0.0]]], dtype=self.dtype, device=self.dev)
        t = x.permute(2, 0, 1).unsqueeze(0)
        grid = F.affine_grid(theta, list(t.shape), align_corners=True)
        out = F.grid_sample(t, grid, mode="bilinear", padding_mode="zeros", align_corners=True)
        return out[0].permute(1, 2, 0)

    def _pad(self, x):
        return F.pad(x, [0, 0, self.pad, self.pad, self.pad, self.pad])

    def _factor(self, a, mu):
        m = self._rotate(self._pad(mu), self.beta[a] - 270.0) * DX
        return torch.exp(-(torch.cumsum(m.flip(0), 0).flip(0) - m / 2))

    def _matrices(self, radius):
        """Per plane the Toeplitz matrices of its taps along y and z."""
        if self._blur[0] != radius:
            P = self.P
            d = radius + ((P - 1) / 2 - np.arange(P)) * DX
            sigma = (SIGMA[0] * np.clip(d, 0, None) + SIGMA[1]) / DX
            h = int(math.ceil(sigma.max() * MIN_SIGMAS))
            s = torch.tensor(sigma, dtype=self.dtype, device=self.dev).view(P, 1, 1)
            t = torch.arange(-h, h + 1, device=self.dev, dtype=self.dtype).view(1, 1, -1)
            total = torch.exp(-t ** 2 / (2 * s ** 2 + DELTA)).sum(-1, keepdim=True)

            def toeplitz(m):
                k = torch.arange(m, device=self.dev, dtype=self.dtype)
                dist = (k.view(1, m, 1) - k.view(1, 1, m))
                w = torch.exp(-dist ** 2 / (2 * s ** 2 + DELTA)) / total
                return (w * (dist.abs() <= h)).contiguous()

            self._blur = (radius, (toeplitz(P), toeplitz(self.case["nz"])))
        return self._blur[1]

    def _psf(self, v, a):
        ty, tz = self._matrices(self.radii[a])
        return torch.matmul(torch.matmul(ty, v.contiguous()), tz)

    def project(self, f, a, mu):
        v = self._rotate(self._pad(f), self.beta[a] - 270.0)
        if mu is not None:
            v = v * self._factor(a, mu)
        if self.case["psf"]:
            v = self._psf(v, a)
        return v.sum(0)[self.pad:self.pad + self.case["n"]]

    def back(self, p, a):
        v = F.pad(p, [0, 0, self.pad, self.pad]).unsqueeze(0).expand(self.P, -1, -1)
        if self.case["psf"]:
            v = self._psf(v, a)
        if self.mu is not None:
            v = v * self._factor(a, self.mu)
        v = self._rotate(v, 270.0 - self.beta[a])
        return v[self.pad:self.pad + self.case["n"], self.pad:self.pad + self.case["n"]]

    def forward(self, f, k):
        f = f.to(self.dtype)
        return torch.stack([self.project(f, a, self.mu) for a in _rows(self.case, k)])

    def backward(self, p, k):
        p = p.to(self.dtype)
        out = 0
        for q, a in zip(p, _rows(self.case, k)):
            out = out + self.back(q, a)
        return out

    def sensitivity(self, k):
        rows = len(_rows(self.case, k))
        ones = torch.ones((rows, self.case["n"], self.case["nz"]), dtype=self.dtype, device=self.dev)
        return self.backward(ones, k)

    def subsets(self):
        return list(range(self.case["subsets"])) if self.case["subsets"] > 1 else [None]


def _exact_osem(case, d, dev):
    ref = _Reference(case, d["mu"], torch.float64, dev)
    g, s = d["counts"].double(), d["scatter"].double()
    norm = {k: ref.sensitivity(k) for k in ref.subsets()}
    f = torch.ones_like(d["activity"], dtype=torch.float64)
    for _ in range(case["iters"]):
        for k in ref.subsets():
            rows = _rows(case, k)
            pred = ref.forward(f, k) + s[rows]
            b = ref.backward(g[rows] / (pred + DELTA), k)
            f = (f + f * (1 / (norm[k] + DELTA)) * (b - norm[k])).clamp(min=0)
    return {"object": f, "projections_predicted": pred}


def _exact_grad(case, d, dev):
    ref = _Reference(case, None, torch.float64, dev)
    f = d["start"].double().requires_grad_(True)
    mu = d["mu"].double().requires_grad_(True)
    g, s = d["counts"].double(), d["scatter"].double()
    value = 0.0
    for a in range(case["angles"]):
        p = ref.project(f, a, mu) + s[a]
        part = (g[a] * torch.log(p) - p).sum()
        part.backward()
        value = value + part.detach()
    return {"value": value, "grad_activity": f.grad, "grad_mu": mu.grad}


def _prior_gradient(x, beta):
    """Gradient of the relative difference prior over the 26 replicated
    neighbours, weighted by inverse distance."""
    n0, n1, n2 = x.shape
    p = F.pad(x[None, None], (1,) * 6, mode="replicate")[0, 0]
    out = torch.zeros_like(x)
    for i in range(3):
        for j in range(3):
            for k in range(3):
                if (i, j, k) == (1, 1, 1):
                    continue
                w = 1 / math.sqrt((i - 1) ** 2 + (j - 1) ** 2 + (k - 1) ** 2)
                y = p[i:i + n0, j:j + n1, k:k + n2]
                t = (x - y).abs()
                out = out + w * (x - y) * (GAMMA * t + 3 * y + x + 2 * DELTA) / (x + y + GAMMA * t + DELTA) ** 2
    return beta * out


def _exact_unrolled(case, d, dev):
    ref = _Reference(case, d["mu"], torch.float64, dev)
    with torch.no_grad():
        norm = {k: ref.sensitivity(k) for k in ref.subsets()}
        total = sum(norm.values())
    g = d["counts"].double().requires_grad_(True)
    s = d["scatter"].double()
    x0 = d["start"].double().requires_grad_(True)
    beta = torch.tensor(BETA, dtype=torch.float64, device=dev, requires_grad=True)
    x = x0
    for _ in range(case["iters"]):
        for k in ref.subsets():
            rows = _rows(case, k)
            w = len(rows) / case["angles"]
            b = ref.backward(g[rows] / (ref.forward(x, k) + s[rows] + DELTA), k)
            y = x + x / (w * total + DELTA) * (b - norm[k] - _prior_gradient(x, beta * w))
            x = torch.where(y <= FLOOR, torch.full_like(y, FLOOR), y)
    ((x - d["activity"].double()) ** 2).sum().backward()
    return {"object": x.detach(), "grad_counts": g.grad, "grad_start": x0.grad,
            "grad_beta": beta.grad.cpu()}


def exact(case, seed):
    dev = torch.device("cuda")
    kind = case["kind"]
    if kind == "batch":
        return [_exact_osem(c, _inputs(c, seed * 64 + k, dev), dev)["object"]
                for k, c in enumerate(_members(case))]
    d = _inputs(case, seed * 64, dev)
    if kind in ("forward", "backward"):
        ref = _Reference(case, d["mu"], torch.float64, dev)
        if kind == "forward":
            return ref.forward(d["activity"], _subset(case))
        return ref.backward(d["ratio"], _subset(case))
    if kind in ("osem", "recon"):
        return _exact_osem(case, d, dev)
    return _exact_grad(case, d, dev) if kind == "grad" else _exact_unrolled(case, d, dev)
