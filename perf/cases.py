"""What users of nepx have it do, as measurable cases.

Kinds of case (each goes through the package's public entry points):
  md          NVT steps of one system: StepRunner.run_exact, the loop that Sim.run drives; the state goes on from
              pass to pass as a simulation's does, and a pass ends with the frame a dump writes (float32)
  md_beads    the same under the label potential (BeadPotential), to hold a network against what it learned
  replicas    many small systems in one arena, stepped together
  energy_grad nep_energy and its backward at a new configuration (minimisers, Monte Carlo, fits)
  components  DescriptorGenerator + ForceEvaluator, the method-by-method surface of a ported script
  layers      descriptor -> network -> adjoint on pairs at hand (nepx.ops), as a training loop calls them
  clouds      descriptors of site clouds that are on the GPU (nepx.ops.cloud_descriptor)
  featurise   NEP.get_g_fast on host arrays: a training set turned into descriptors
Sizes and densities are those of the benchmark workloads, the tests and the documented run
(200 tetrahedra in a box of side 33: 0.0056 bodies per unit volume).
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "anisotropic-ml_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import nepx  # noqa: E402
from nepx import label, ops  # noqa: E402
from nepx.autograd import nep_energy  # noqa: E402
from nepx.configs import make_system  # noqa: E402
from nepx.DescriptorGenerator import DescriptorGenerator  # noqa: E402
from nepx.engine import StepRunner  # noqa: E402
from nepx.ForceEvaluator import ForceEvaluator  # noqa: E402
from nepx.NEP import NEP  # noqa: E402

DEV = "cuda:0"
REF_DENSITY = 200 / 33.0 ** 3


def listed():
    return [
        # a small simulation, bound by the latency of a step: 512 cubes, 100 steps between checks (as Sim.run)
        dict(name="md_cubes_512", kind="md", shape="cube8", lmax=4, n=512, phi=0.30, steps=100),
        # the documented run: 200 tetrahedra, hypers 10 10 10, a 150-wide ReLU network
        dict(name="md_th_200", kind="md", shape="th_v1", lmax=10, n=200, phi=round(REF_DENSITY, 5), steps=32),
        # the same model on a system a hundred times as large
        dict(name="md_th_20001", kind="md", shape="th_v1", lmax=10, n=20001, phi=round(REF_DENSITY, 5), steps=4),
        # the headline: 32,768 tetrahedra at packing fraction 0.45
        dict(name="md_tets_32768", kind="md", shape="tet10", lmax=4, n=32768, phi=0.45, steps=4),
        # the largest: 262,144 cylinders
        dict(name="md_cylinders_262144", kind="md", shape="cyl12", lmax=6, n=262144, phi=0.35, steps=1),
        # 64 independent cube systems of 64 to 4,096 bodies, batched in one arena
        dict(name="replicas_64", kind="replicas", systems=64, largest=4096, steps=8),
        # a network's reference: cubes under the bead potential the labels came from
        dict(name="md_beads_4096", kind="md_beads", n=4096, phi=0.004, steps=16),
        # energy and gradient of one configuration, list included
        dict(name="energy_grad_tets_4097", kind="energy_grad", shape="tet10", lmax=4, n=4097, phi=0.45),
        # a ported script's step: descriptors and forces by the reference's method names, hypers 10 8 4
        dict(name="components_cubes_1024", kind="components", shape="cube_v2", lmax=4, n=1024, phi=0.006),
        # training and validation of the documented network: each layer on 100,001 pairs
        dict(name="layers_100001", kind="layers", shape="cube_v2", lmax=10, pairs=100001),
        # a training set of the 12-site cube clouds, resident on the GPU, hypers 10 8 4
        dict(name="clouds_1000003", kind="clouds", lmax=4, sites=12, clouds=1000003, weights=False),
        # the same from and to host arrays with type weights, hypers 10 10 10
        dict(name="featurise_50000", kind="featurise", lmax=10, sites=12, clouds=50000, weights=True),
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["md", "md", "md", "replicas", "md_beads", "energy_grad", "components", "layers", "clouds",
                       "featurise"])
    if kind in ("md", "energy_grad"):
        shape, lmax, lo, hi, d0, d1 = rng.choice([
            ("cube8", 4, 64, 32768, 0.2, 0.4), ("tet10", 4, 700, 32768, 0.3, 0.5), ("cyl12", 6, 128, 65536, 0.25, 0.4),
            ("th_v1", 4, 64, 40000, 0.004, 0.008), ("th_v1", 10, 64, 20000, 0.004, 0.008),
            ("cube_v2", 4, 64, 20000, 0.004, 0.008)])
        if kind == "energy_grad":
            hi = min(hi, 16384)
        n, phi = _log(rng, lo, hi), round(rng.uniform(d0, d1), 3)
        c = dict(kind=kind, shape=shape, lmax=lmax, n=n, phi=phi)
        if kind == "md":
            c["steps"] = 32 if n <= 2048 else 8 if n <= 16384 else 2
        return c
    if kind == "replicas":
        return dict(kind=kind, systems=rng.randint(8, 96), largest=_log(rng, 512, 4096), steps=8)
    if kind == "md_beads":
        return dict(kind=kind, n=_log(rng, 64, 4096), phi=round(rng.uniform(0.003, 0.006), 4), steps=16)
    if kind == "components":
        return dict(kind=kind, shape=rng.choice(["cube_v2", "th_v1"]), lmax=rng.choice([4, 10]),
                    n=_log(rng, 128, 8192), phi=round(rng.uniform(0.004, 0.008), 4))
    if kind == "layers":
        return dict(kind=kind, shape=rng.choice(["cube_v2", "th_v1"]), lmax=rng.choice([4, 10]),
                    pairs=_log(rng, 16, 200000))
    c = dict(kind=kind, lmax=rng.choice([4, 10]), sites=2 * rng.randint(3, 12), weights=rng.random() < 0.5)
    c["clouds"] = _log(rng, 64, 400000 if kind == "clouds" else 50000)
    return c


# ------------------------------------------------------------------ models
def _hypers(shape, lmax):
    if shape in ("cube8", "tet10"):
        return (11, 6, 4)
    if shape == "cyl12":
        return (17, 6, 6)
    return (10, 10, 10) if lmax == 10 else (10, 8, 4)


def _layers(shape, lmax):
    """Network of the model: (layers as [(W, b)], activation, energy range), seeded random weights."""
    hyp = _hypers(shape, lmax)
    d = nepx.n_descriptor(*hyp)
    if shape in ("cube8", "tet10"):
        widths, act, seed = [64, 64], "tanh", 7
    elif shape == "cyl12":
        widths, act, seed = [128, 128], "tanh", 7
    else:
        widths, act, seed = [150] * 4, "relu", 21
    s = nepx.get_shape(shape)
    rng = np.random.default_rng(seed)
    dims = [d] + widths + [1]
    layers = [(rng.standard_normal((b, a)) / math.sqrt(a), np.zeros(b)) for a, b in zip(dims[:-1], dims[1:])]
    return layers, act, s.en_min, s.en_max


def _net(shape, lmax):
    layers, act, e0, e1 = _layers(shape, lmax)
    return nepx.EnergyNet(layers, act=act, en_min=e0, en_max=e1, device=DEV)


def _phi(shape, n, phi):
    """Packing (or number density, for the reference's unit-volume shapes) capped so the box is two cutoffs wide."""
    s = nepx.get_shape(shape)
    return min(phi, n * s.volume / (2.05 * s.cutoff) ** 3)


def _spec(case, seed):
    if case["kind"] == "md_beads":
        reach = 2.0 * float(np.linalg.norm(label.cube_structure_beads(), axis=1).max()) + label.R0
        phi = min(case["phi"], case["n"] / (2.05 * reach) ** 3)
        return make_system("cube8", case["n"], phi, dt=0.002, seed=seed, rc=reach, non_overlap=False)
    return make_system(case["shape"], case["n"], _phi(case["shape"], case["n"], case["phi"]), kT=1.0, dt=0.001,
                       seed=seed, non_overlap=False)


def _replicas(case, seed):
    """Cube systems of 64 bodies to the case's largest (log-uniform), packing 0.2 to 0.5, kT 0.5 to 2: the sizes go with the
    case, the configurations with the seed."""
    size = np.random.default_rng(case["systems"])
    out = []
    for k in range(case["systems"]):
        n = int(round(math.exp(size.uniform(math.log(64), math.log(case["largest"])))))
        phi, kT = _phi("cube8", n, float(size.uniform(0.2, 0.5))), float(size.uniform(0.5, 2.0))
        out.append(make_system("cube8", n, phi, kT=kT, seed=1000 * seed + k, non_overlap=False))
    return out


def _cloud_points(case, seed):
    """Pairs of bodies as site clouds: each half about its own centre, the centres 2.5 to 5.8 apart."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    m, h = case["clouds"], case["sites"] // 2
    x = 0.9 * torch.randn((m, 2, h, 3), generator=g, device=DEV)
    d = torch.nn.functional.normalize(torch.randn((m, 1, 3), generator=g, device=DEV), dim=-1)
    x[:, 1] += d * (2.5 + 3.3 * torch.rand((m, 1, 1), generator=g, device=DEV))
    return x.reshape(m, 2 * h, 3).contiguous()


CLOUD_CUTOFF = 9.0


def _types(case):
    return [k % 5 for k in range(case["sites"])]


def _cloud_weights(case):
    t = np.asarray(_types(case), dtype=np.float64) + 1.0
    return np.sqrt(t) if t.max() > 4 else t


def _pairs_input(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    p = case["pairs"]
    nb = max(2, p // 3)
    qf = torch.nn.functional.normalize(torch.randn((nb, 4), generator=g, device=DEV), dim=1).contiguous()
    i = torch.randint(0, nb - 1, (p,), generator=g, device=DEV, dtype=torch.int32)
    j = i + 1 + (torch.rand(p, generator=g, device=DEV) * (nb - 1 - i)).to(torch.int32).clamp(max=nb)
    j = torch.minimum(j, torch.full_like(j, nb - 1))
    t = torch.zeros((p, 4), device=DEV)
    d = torch.nn.functional.normalize(torch.randn((p, 3), generator=g, device=DEV), dim=1)
    t[:, :3] = d * (2.5 + 3.3 * torch.rand((p, 1), generator=g, device=DEV))
    return qf, i.contiguous(), j.contiguous(), t


# ------------------------------------------------------------------ prepare and run
def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind in ("md", "md_beads", "replicas"):
        if kind == "replicas":
            specs, shape, hyp, net, pot = _replicas(case, seed), "cube8", (11, 6, 4), _net("cube8", 4), None
        elif kind == "md_beads":
            specs, shape, hyp, net, pot = [_spec(case, seed)], "cube8", (11, 6, 4), None, label.BeadPotential(device=DEV)
        else:
            specs, shape, pot = [_spec(case, seed)], case["shape"], None
            hyp, net = _hypers(shape, case["lmax"]), _net(shape, case["lmax"])
        ar = nepx.Arena(specs, nepx.get_shape(shape), hyp, net, device=DEV, potential=pot)
        st["runner"] = StepRunner(ar)
        st["runner"].init()
    elif kind == "energy_grad":
        spec = _spec(case, seed)
        st["arena"] = nepx.Arena([spec], nepx.get_shape(case["shape"]), _hypers(case["shape"], case["lmax"]),
                                 _net(case["shape"], case["lmax"]), device=DEV)
        st["pos"] = torch.from_numpy(spec.x).to(DEV, torch.float32).requires_grad_()
        st["rot"] = torch.zeros_like(st["pos"]).requires_grad_()
        st["quat"] = torch.from_numpy(spec.q).to(DEV, torch.float32)
    elif kind == "components":
        spec = _spec(case, seed)
        dg, fe = DescriptorGenerator(), ForceEvaluator()
        dg.setDevice(0)
        dg.setHyperParameters([*_hypers(case["shape"], case["lmax"]), 4.5])
        dg.setBoxSize(spec.L)
        dg.setShape(case["shape"])
        dg.move_data_to_device()
        fe.setDevice(0)
        fe.set_model(_net(case["shape"], case["lmax"]))
        fe.set_energy_range(*dg.get_en_min_max())
        fe.setNparticles(spec.n)
        fe.attach(dg)
        st.update(dg=dg, fe=fe, pos=torch.from_numpy(spec.x).to(DEV), quat=torch.from_numpy(spec.q).to(DEV))
        st["nlist"] = _pairs64(st["pos"], spec.L, spec.rc + 2.0)
    elif kind == "layers":
        st["model"] = nepx.make_pair_model(nepx.get_shape(case["shape"]), _hypers(case["shape"], case["lmax"]))
        st["net"] = _net(case["shape"], case["lmax"])
        st["pairs"] = _pairs_input(case, seed)
    elif kind == "clouds":
        st["x"] = _cloud_points(case, seed)
        st["w"] = torch.from_numpy(_cloud_weights(case)).to(DEV, torch.float32) if case["weights"] else None
    else:
        st["nep"] = NEP(_cloud_points(case, seed).cpu().numpy())
        st["nep"].set_hypers([*_hypers("cube_v2", case["lmax"]), CLOUD_CUTOFF])
        st["nep"].set_pts_types({"pts_types": _types(case)} if case["weights"] else {})
    return st


def _frame(ar, k):
    """State and forces of system k in float32, as a dump frame holds them."""
    F, T = ar.forces(k)
    cols = {"x": ["x", "y", "z"], "v": ["vx", "vy", "vz"], "q": ["q0", "q1", "q2", "q3"], "p": ["p0", "p1", "p2", "p3"]}
    out = {name: ar.tensor(keys, k).float() for name, keys in cols.items()}
    out["F"], out["T"] = F.float(), T.float()
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("md", "md_beads"):
        state["runner"].run_exact(case["steps"])
        return _frame(state["runner"].ar, 0)
    if kind == "replicas":
        state["runner"].run_exact(case["steps"])
        ar = state["runner"].ar
        cols = {"x": "x y z", "v": "vx vy vz", "q": "q0 q1 q2 q3", "p": "p0 p1 p2 p3", "F": "fx fy fz", "T": "tx ty tz"}
        return {name: torch.stack([ar.t[key] for key in keys.split()], 1).float() for name, keys in cols.items()}
    if kind == "energy_grad":
        state["pos"].grad = state["rot"].grad = None
        U = nep_energy(state["pos"], state["rot"], state["quat"], state["arena"])
        U.backward()
        return U.detach(), state["pos"].grad, state["rot"].grad
    if kind == "components":
        G, pp, n = state["dg"].generate_nep_descriptors(state["pos"], state["quat"], state["nlist"])
        F, T = state["fe"].evaluate_interactions(G, pp, n)
        return {"F": F.float(), "T": T.float()}
    if kind == "layers":
        qf, i, j, t = state["pairs"]
        G = ops.descriptor_forward(state["model"], qf, i, j, t)
        E, dG = ops.ffnn_forward_backward(state["net"], G)
        return {"G": G, "E": E, "dG": dG,
                "out": ops.descriptor_adjoint(state["model"], qf, i, j, t, dG, E=E, clip=100.0)}
    if kind == "clouds":
        return ops.cloud_descriptor(state["x"], *_hypers("cube_v2", case["lmax"]), CLOUD_CUTOFF, state["w"])
    return state["nep"].get_g_fast()


# ------------------------------------------------------------------ work
def _pair_flops(shape, lmax):
    """Contractions of one pair: angular sums forward and adjoint, network forward and backward."""
    nrad, nang, lm = _hypers(shape, lmax)
    widths = [w.shape for w, _ in _layers(shape, lmax)[0]]
    return (12 * 2 * nepx.get_shape(shape).n_sites * (nang + 1) * lm * (lm + 2)
            + 4 * sum(a * b for a, b in widths))


def _n_pairs(n, density, rc):
    return 0.5 * n * min(n - 1, density * 4.0 / 3.0 * math.pi * rc ** 3)


STATE_BYTES = 27 * 8 * 2  # a step reads and writes each particle's state, forces among it


def work(case):
    kind = case["kind"]
    if kind == "replicas":
        top = case["largest"]
        n = case["systems"] * (top - 64) / math.log(top / 64)  # mean of a log-uniform size
        p = _n_pairs(n, 0.35, 2.5)
        return {"bytes": case["steps"] * n * STATE_BYTES, "flops": case["steps"] * p * _pair_flops("cube8", 4)}
    if kind == "md_beads":
        p = _n_pairs(case["n"], case["phi"], 7.2)
        return {"bytes": case["steps"] * case["n"] * STATE_BYTES, "flops": case["steps"] * p * 152 * 152 * 8}
    if kind in ("md", "energy_grad", "components"):
        s = nepx.get_shape(case["shape"])
        p = _n_pairs(case["n"], _phi(case["shape"], case["n"], case["phi"]) / s.volume, s.cutoff)
        k = case.get("steps", 1)
        io = STATE_BYTES if kind == "md" else 7 * 8 + 7 * 8
        extra = p * 4 * (nepx.n_descriptor(*_hypers(case["shape"], case["lmax"])) + 4) if kind == "components" else 0
        return {"bytes": k * case["n"] * io + extra, "flops": k * p * _pair_flops(case["shape"], case["lmax"])}
    if kind == "layers":
        d = nepx.n_descriptor(*_hypers(case["shape"], case["lmax"]))
        return {"bytes": case["pairs"] * (24 + 4 * (2 * d + 13)) + case["pairs"] // 3 * 16,
                "flops": case["pairs"] * _pair_flops(case["shape"], case["lmax"])}
    nrad, nang, lm = _hypers("cube_v2", case["lmax"])
    d = nepx.n_descriptor(nrad, nang, lm)
    return {"bytes": case["clouds"] * 4 * (3 * case["sites"] + d),
            "flops": case["clouds"] * 2 * case["sites"] * (nang + 1) * lm * (lm + 2)}


# ------------------------------------------------------------------ values in 64 bits, by plain torch
def _mi(t, L):
    t = torch.where(t > 0.5 * L, t - L, t)
    return torch.where(t < -0.5 * L, t + L, t)


def _pairs64(x, L, r):
    """All i < j with |X_j - X_i| < r under the minimum image, sorted."""
    out = []
    step = max(1, 40_000_000 // len(x))
    for a in range(0, len(x), step):
        d = _mi(x[None, :, :] - x[a:a + step, None, :], L)
        ij = torch.nonzero((d * d).sum(-1) < r * r)
        ij[:, 0] += a
        out.append(ij[ij[:, 0] < ij[:, 1]])
    return torch.cat(out)


def _rotmat(q):
    w, x, y, z = q.unbind(-1)
    a = w * w - (x * x + y * y + z * z)
    return torch.stack([a + 2 * x * x, 2 * (x * y - w * z), 2 * (x * z + w * y),
                        2 * (x * y + w * z), a + 2 * y * y, 2 * (y * z - w * x),
                        2 * (x * z - w * y), 2 * (y * z + w * x), a + 2 * z * z], -1).reshape(q.shape[:-1] + (3, 3))


def _descriptor64(pts, r_nep, hyp, weights=None):
    """[g_rad | g_ang] of clouds (P, Nd, 3): Chebyshev radial functions, Legendre double sum."""
    nrad, nang, lmax = hyp
    c = pts - pts.mean(1, keepdim=True)
    r = c.norm(dim=-1)
    u = c / r[..., None]
    rho = r / r_nep
    x = 2.0 * (rho - 1.0) ** 2 - 1.0
    cheb = [torch.ones_like(x), x]
    for _ in range(nrad - 1):
        cheb.append(2.0 * x * cheb[-1] - cheb[-2])
    f = (torch.stack(cheb, 1) + 1.0) * (0.25 * (1.0 + torch.cos(math.pi * rho)))[:, None, :]
    if weights is not None:
        f = f * weights
    fa = f[:, :nang + 1]
    z = (u[:, :, None, :] * u[:, None, :, :]).sum(-1)
    g = []
    p0, p1 = torch.ones_like(z), z
    for l in range(1, lmax + 1):
        g.append((torch.matmul(fa, p1) * fa).sum(-1))
        p0, p1 = p1, ((2 * l + 1) * z * p1 - l * p0) / (l + 1)
    return torch.cat([f.sum(-1), torch.stack(g, 2).flatten(1)], 1)


class _Model64:
    def __init__(self, shape, lmax):
        s = nepx.get_shape(shape)
        self.hyp, self.r_nep = _hypers(shape, lmax), s.nep_cutoff
        self.sites = torch.from_numpy(np.asarray(s.sites, dtype=np.float32)).to(DEV, torch.float64)
        layers, self.act, self.e0, self.e1 = _layers(shape, lmax)
        self.layers = [(torch.from_numpy(w.astype(np.float32)).to(DEV, torch.float64),
                        torch.from_numpy(b).to(DEV, torch.float64)) for w, b in layers]
        per = (2 * s.n_sites) ** 2 * self.hyp[2] * 64 + 40000
        self.chunk = max(256, int(6e9 / per))

    def energy(self, G):
        h = G
        for w, b in self.layers[:-1]:
            h = torch.nn.functional.linear(h, w, b)
            h = torch.tanh(h) if self.act == "tanh" else torch.relu(h)
        w, b = self.layers[-1]
        return self.e0 + (self.e1 - self.e0) * torch.nn.functional.linear(h, w, b)[:, 0]

    def pairs(self, qi, qj, t):
        """G, E, dE/dG and (F_i, tau_i, tau_j) of pairs."""
        G, E, dG, o = [], [], [], []
        ns = len(self.sites)
        for a in range(0, len(t), self.chunk):
            s = slice(a, a + self.chunk)
            bi = torch.matmul(self.sites, _rotmat(qi[s]).transpose(1, 2))
            bj = torch.matmul(self.sites, _rotmat(qj[s]).transpose(1, 2))
            with torch.enable_grad():
                pts = torch.cat([bi, bj + t[s][:, None, :]], 1).detach().requires_grad_()
                g = _descriptor64(pts, self.r_nep, self.hyp)
                e = self.energy(g)
                dg, dp = torch.autograd.grad(e.sum(), [g, pts])
            G.append(g.detach())
            E.append(e.detach())
            dG.append(dg)
            o.append(torch.cat([-dp[:, :ns].sum(1), -torch.linalg.cross(bi, dp[:, :ns]).sum(1),
                                -torch.linalg.cross(bj, dp[:, ns:]).sum(1)], 1))
        if not o:
            z = lambda *k: torch.zeros(k, dtype=torch.float64, device=DEV)  # noqa: E731
            d = nepx.n_descriptor(*self.hyp)
            return z(0, d), z(0), z(0, d), z(0, 9)
        return torch.cat(G), torch.cat(E), torch.cat(dG), torch.cat(o)


def _beads64(qi, qj, t):
    """The bead potential's (E, F_i, tau_i, tau_j)."""
    beads = torch.from_numpy(label.cube_structure_beads().astype(np.float32)).to(DEV, torch.float64)
    eps, sig, r0 = float(np.float32(label.EPS)), float(np.float32(label.SIGMA)), float(np.float32(label.R0))
    E, o = [], []
    for a in range(0, len(t), 2048):
        s = slice(a, a + 2048)
        bi = torch.matmul(beads, _rotmat(qi[s]).transpose(1, 2))
        bj = torch.matmul(beads, _rotmat(qj[s]).transpose(1, 2))
        d = (bj + t[s][:, None, :])[:, None, :, :] - bi[:, :, None, :]
        r = d.norm(dim=-1)
        w = (r0 - r).clamp(min=0.0)
        E.append(eps * (w * w).sum((1, 2)) / sig ** 2)
        g = (-2.0 * eps / sig ** 2 * w / r)[..., None] * d
        o.append(torch.cat([g.sum((1, 2)), torch.linalg.cross(bi, g.sum(2)).sum(1),
                            -torch.linalg.cross(bj, g.sum(1)).sum(1)], 1))
    return torch.cat(E), torch.cat(o)


def _qmul(a, b):
    w = a[:, :1] * b[:, :1] - (a[:, 1:] * b[:, 1:]).sum(1, keepdim=True)
    return torch.cat([w, a[:, :1] * b[:, 1:] + b[:, :1] * a[:, 1:] + torch.linalg.cross(a[:, 1:], b[:, 1:])], 1)


def _rotor(k, h, moi, p, q):
    def perm(v):
        w, x, y, z = v.unbind(1)
        return torch.stack([[-x, w, z, -y], [-y, -z, w, x], [-z, y, -x, w]][k], 1)
    pp, qq = perm(p), perm(q)
    phi = (h * 0.25 / moi * (p * qq).sum(1, keepdim=True))
    return torch.cos(phi) * p + torch.sin(phi) * pp, torch.cos(phi) * q + torch.sin(phi) * qq


def _md64(specs, steps, forces_of_pairs):
    """NVT steps of systems side by side (Nose-Hoover translation and rotation, NO_SQUISH rotor)."""
    dev = lambda key: torch.from_numpy(np.concatenate([getattr(s, key) for s in specs])).to(DEV)  # noqa: E731
    x, v, q, p, m = dev("x"), dev("v"), dev("q"), dev("p"), dev("mass")[:, None]
    sysid = torch.from_numpy(np.repeat(np.arange(len(specs)), [s.n for s in specs])).to(DEV)
    per = lambda vals: torch.tensor(vals, dtype=torch.float64, device=DEV)  # noqa: E731
    L, dt, tau, kT = (per([getattr(s, k) for s in specs]) for k in ("L", "dt", "tau", "kT"))
    ndof, rndof, moi = per([s.ndof for s in specs]), per([s.rndof for s in specs]), per([s.moi for s in specs])
    th = {k: per([s.thermo[k] for s in specs]) for k in ("xi", "xi_r")}
    Lp, dtp, moip = L[sysid, None], dt[sysid, None], moi[sysid]
    starts = np.concatenate([[0], np.cumsum([s.n for s in specs])])

    def factors():
        kt = torch.zeros_like(L).index_add_(0, sysid, (0.5 * m * v * v).sum(1))
        qc = torch.cat([q[:, :1], -q[:, 1:]], 1)
        s = 0.5 * _qmul(qc, p)[:, 1:]
        kr = torch.zeros_like(L).index_add_(0, sysid, (0.5 * s * s / moip).sum(1))
        c = dt / tau / tau
        th["xi"] = th["xi"] + c * (2 * kt / ndof / kT - 1)
        th["xi_r"] = th["xi_r"] + c * (2 * kr / rndof / kT - 1)
        return torch.exp(-0.5 * th["xi"] * dt)[sysid, None], torch.exp(-0.5 * th["xi_r"] * dt)[sysid, None]

    theta, er = factors()
    for _ in range(steps):
        ij = torch.cat([_pairs64(x[a:b], s.L, s.rc) + int(a) for s, a, b in zip(specs, starts[:-1], starts[1:])])
        i, j = ij.unbind(1)
        o = forces_of_pairs(q[i], q[j], _mi(x[j] - x[i], Lp[i])).clamp(-100.0, 100.0)
        F = torch.zeros_like(x).index_add_(0, i, o[:, :3]).index_add_(0, j, -o[:, :3])
        T = torch.zeros_like(x).index_add_(0, i, o[:, 3:6]).index_add_(0, j, o[:, 6:])
        kick = 0.5 * dtp * F / m
        v = v * theta + kick
        tb = torch.matmul(_rotmat(q).transpose(1, 2), T[:, :, None])[:, :, 0]
        dp = dtp * _qmul(q, torch.cat([torch.zeros_like(tb[:, :1]), tb], 1))
        p = p * er + dp
        v = (v + kick) * theta
        x = _mi(x + v * dtp, Lp)
        p = (p + dp) * er
        for k, f in ((2, 0.5), (1, 0.5), (0, 1.0), (1, 0.5), (2, 0.5)):
            p, q = _rotor(k, f * dtp, moip[:, k:k + 1], p, q)
        q = q / q.norm(dim=1, keepdim=True)
        theta, er = factors()
    return dict(x=x, v=v, q=q, p=p, F=F, T=T)


def exact(case, seed):
    kind = case["kind"]
    f32 = lambda a: torch.from_numpy(np.asarray(a, dtype=np.float32)).to(DEV, torch.float64)  # noqa: E731
    if kind == "replicas":
        specs = _replicas(case, seed)
        mod = _Model64("cube8", 4)
        out = _md64(specs, case["steps"], lambda *a: mod.pairs(*a)[3])
        sizes = [s.n for s in specs]
        padded = {}
        for k, full in out.items():  # the arena pads each system to whole blocks of 256
            rows = []
            for part in full.split(sizes):
                pad = torch.zeros((-len(part) % 256, part.shape[1]), dtype=part.dtype, device=DEV)
                if k == "q":
                    pad[:, 0] = 1.0
                rows += [part, pad]
            padded[k] = torch.cat(rows)
        return padded
    if kind == "md_beads":
        return _md64([_spec(case, seed)], case["steps"], lambda *a: _beads64(*a)[1])
    if kind == "md":
        if work(case)["flops"] > 1.5e12 or case["n"] > 40000:
            return None
        mod = _Model64(case["shape"], case["lmax"])
        return _md64([_spec(case, seed)], case["steps"], lambda *a: mod.pairs(*a)[3])
    if kind in ("energy_grad", "components"):
        spec = _spec(case, seed)
        mod = _Model64(case["shape"], case["lmax"])
        grad = kind == "energy_grad"
        x, q = (f32(spec.x), f32(spec.q)) if grad else (torch.from_numpy(spec.x).to(DEV), torch.from_numpy(spec.q).to(DEV))
        ij = _pairs64(x, spec.L, spec.rc)
        i, j = ij.unbind(1)
        G, E, _, o = mod.pairs(q[i], q[j], _mi(x[j] - x[i], spec.L))
        o = o.clamp(-100.0, 100.0)
        F = torch.zeros_like(x).index_add_(0, i, o[:, :3]).index_add_(0, j, -o[:, :3])
        T = torch.zeros_like(x).index_add_(0, i, o[:, 3:6]).index_add_(0, j, o[:, 6:])
        return (E.sum(), -F, -T) if grad else {"F": F, "T": T}
    if kind == "layers":
        qf, i, j, t = _pairs_input(case, seed)
        mod = _Model64(case["shape"], case["lmax"])
        G, E, dG, o = mod.pairs(qf[i.long()].double(), qf[j.long()].double(), t[:, :3].double())
        o = o.clamp(-100.0, 100.0)
        z = torch.zeros_like(E)[:, None]
        return {"G": G, "E": E, "dG": dG, "out": torch.cat([o[:, :3], E[:, None], o[:, 3:6], z, o[:, 6:], z], 1)}
    x = _cloud_points(case, seed)
    w = torch.from_numpy(_cloud_weights(case).astype(np.float32)).to(DEV, torch.float64) if case["weights"] else None
    hyp = _hypers("cube_v2", case["lmax"])
    G = torch.cat([_descriptor64(c.double(), CLOUD_CUTOFF, hyp, w) for c in x.split(65536)])
    return G if kind == "clouds" else G.cpu().numpy()
