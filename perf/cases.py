"""Performance cases of jztree_amd's public entry points.

What they stand for, and the ranges draw() takes:

  knn          exact neighbours of one point set: from a thousand points, where a script calls it in
               a loop and launches and host work count, over 65,536 uniform points with k = 16, to
               2^24 clustered ones; k 4 to 64; open or periodic; rows in input or z order; float32
               and float64; 2 and 3 dims; the default settings, as a user without the autotuner has
               them, and leaves of 128 points, which it picks on large clustered sets
  knn_query    neighbours of a second point set among the first
  knn_learned  exact kNN with a trained radius proposer; 2^26 clustered points with k = 32 and leaf
               128 are the workload of bench.py and the largest case
  fof          friends-of-friends labels, from the few thousand points of a 2-D example to 2^26
  catalogue    friends-of-friends groups of particles with masses and velocities, their particles
               in group order and the catalogue, as a halo finder's snapshot loop calls it
  sets         a batch of independent uneven sets (kNN and FoF on one forest), captured once as a
               HIP graph and replayed on new positions, as a serving loop does
  zsort        z-order sort forward and its gradient backward

Sizes come from bench.py and the tests or lie between them; odd sizes are in every range.  Point
sets are uniform or clustered (Plummer halos with power-law member weights on a uniform
background), as in the benchmark, drawn on the GPU.
"""
from __future__ import annotations

import math
import random

import torch

import jztree_amd as jz
from jztree_amd.config import FofConfig, KNNConfig, TreeConfig, RegularizationConfig
from jztree_amd.data import ParticleData

DEV = "cuda"


def listed():
    return [
        # the smallest call: host work and launches
        dict(name="knn_1000_k8", op="knn", n=1000, k=8, dim=3, dtype="f32", cluster=0, box=0.0, order="input", leaf=48),
        # 65,536 uniform points, k = 16: the plain configuration of the tests and the quick start
        dict(name="knn_65536_k16", op="knn", n=65536, k=16, dim=3, dtype="f32", cluster=0, box=0.0, order="input",
             leaf=48),
        # an odd size, the widest one-pass k, rows in z order, periodic clustered points
        dict(name="knn_1000003_k64_z", op="knn", n=1000003, k=64, dim=3, dtype="f32", cluster=512, box=1.0, order="z",
             leaf=48),
        # a large snapshot with the default settings
        dict(name="knn_2e24_k32", op="knn", n=1 << 24, k=32, dim=3, dtype="f32", cluster=4096, box=1.0, order="input",
             leaf=48),
        # float64 positions searched in float64
        dict(name="knn_f64_200003_k16", op="knn", n=200003, k=16, dim=3, dtype="f64", cluster=0, box=0.0, order="input",
             leaf=48),
        # neighbours of 123,457 probes among 2^20 sources
        dict(name="knn_query_2e20_k8", op="knn_query", n=1 << 20, nq=123457, k=8, dim=3, dtype="f32", cluster=512,
             box=1.0, leaf=48),
        # the benchmark's kNN: 2^26 clustered points, trained proposer, leaf 128
        dict(name="knn_learned_2e26_k32", op="knn_learned", n=1 << 26, k=32, cluster=65536, box=1.0, leaf=128),
        # a small 2-D friends-of-friends example
        dict(name="fof_2d_12800", op="fof", n=12800, dim=2, cluster=16, b=0.2, box=1.0, order="z", leaf=48),
        # the benchmark's friends-of-friends: 2^26 clustered points
        dict(name="fof_2e26", op="fof", n=1 << 26, dim=3, cluster=65536, b=0.2, box=1.0, order="z", leaf=128),
        # groups, group order and catalogue of a snapshot with masses and velocities
        dict(name="catalogue_1000003", op="catalogue", n=1000003, cluster=512, b=0.2, box=1.0, leaf=48),
        # 64 uneven sets of 2^10 to 2^16 points as a replayed graph
        dict(name="sets_64", op="sets", nsets=64, lo=10, hi=16, k=8, b=0.2, leaf=48),
        # z-order sort and its gradient
        dict(name="zsort_grad_4194307", op="zsort", n=4194307, dim=3, dtype="f32", cluster=1024),
    ]


def _log_size(rng: random.Random, lo: int, hi: int) -> int:
    n = int(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    return n | 1 if rng.random() < 0.7 else n


def _halos(rng: random.Random, n: int) -> int:
    # small sets are uniform: a handful of halos in a few thousand points says little
    return 0 if n < 32768 or rng.random() < 0.3 else n // rng.choice([1024, 2048, 4096])


def draw(rng: random.Random) -> dict:
    op = rng.choice(["knn", "knn", "knn", "knn_query", "knn_learned", "fof", "fof", "catalogue", "sets", "zsort"])
    box = rng.choice([0.0, 1.0, 1.0])
    if op == "knn":
        dim, dtype = rng.choice([(3, "f32"), (3, "f32"), (3, "f32"), (2, "f32"), (3, "f64")])
        n = _log_size(rng, 1000, 1 << 24 if dtype == "f32" else 1 << 20)
        return dict(op=op, n=n, k=rng.choice([4, 8, 10, 16, 24, 32, 48, 64]), dim=dim, dtype=dtype,
                    cluster=_halos(rng, n), box=box, order=rng.choice(["input", "input", "z"]),
                    leaf=rng.choice([32, 48, 48, 64, 128]))
    if op == "knn_query":
        n = _log_size(rng, 4096, 1 << 22)
        return dict(op=op, n=n, nq=_log_size(rng, max(1000, n // 64), 2 * n), k=rng.choice([4, 8, 16, 32]), dim=3, dtype="f32",
                    cluster=_halos(rng, n), box=box, leaf=48)
    if op == "knn_learned":
        n = _log_size(rng, 1 << 18, 1 << 24)
        return dict(op=op, n=n, k=rng.choice([16, 32]), cluster=n // 1024, box=1.0,
                    leaf=rng.choice([64, 128]))
    if op == "fof":
        dim = rng.choice([3, 3, 3, 2])
        n = _log_size(rng, 4096, 1 << 25 if dim == 3 else 1 << 20)
        return dict(op=op, n=n, dim=dim, cluster=_halos(rng, n), b=round(rng.uniform(0.15, 0.25), 3), box=box,
                    order=rng.choice(["z", "input"]), leaf=rng.choice([48, 48, 64, 128]))
    if op == "catalogue":
        n = _log_size(rng, 4096, 1 << 22)
        return dict(op=op, n=n, cluster=n // 2048, b=0.2, box=1.0, leaf=48)
    if op == "sets":
        lo = rng.choice([8, 9, 10])
        return dict(op=op, nsets=rng.randrange(3, 128), lo=lo, hi=lo + rng.choice([3, 5, 6]), k=rng.choice([8, 16]),
                    b=0.2, leaf=rng.choice([32, 48]))
    return dict(op="zsort", n=_log_size(rng, 1000, 1 << 25), dim=rng.choice([3, 3, 2]),
                dtype=rng.choice(["f32", "f32", "f64"]), cluster=0 if rng.random() < 0.5 else 1024)


# ------------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------------

def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _points(n: int, dim: int, halos: int, dtype: str, g: torch.Generator) -> torch.Tensor:
    """n points in the unit box: 70% in `halos` Plummer halos (scale radius 0.002, member weights
    dN/dM ~ M^-1.9 on [32, 2^16]) and the rest uniform, in random order; halos = 0: all uniform."""
    dt = torch.float32 if dtype == "f32" else torch.float64
    f64 = dict(dtype=torch.float64, device=DEV)
    x = torch.empty((n, dim), dtype=dt, device=DEV)
    nh = int(round(0.7 * n)) if halos else 0
    step = 1 << 24  # drawn in slices: the float64 temporaries stay small
    if halos:
        u = torch.rand(halos, generator=g, **f64)
        w = (32.0 ** -0.9 + u * (65536.0 ** -0.9 - 32.0 ** -0.9)) ** (-1.0 / 0.9)
        cdf = torch.cumsum(w, 0)
        cdf = cdf / cdf[-1]
        cent = torch.rand((halos, dim), generator=g, **f64)
        for s in range(0, nh, step):
            m = min(step, nh - s)
            hid = torch.searchsorted(cdf, torch.rand(m, generator=g, **f64)).clamp_(max=halos - 1)
            uu = torch.rand(m, generator=g, **f64) * (0.999 - 1e-12) + 1e-12
            r = 0.002 / torch.sqrt(uu ** (-2.0 / 3.0) - 1.0)
            v = torch.randn((m, dim), generator=g, **f64)
            v /= torch.linalg.norm(v, dim=1, keepdim=True)
            x[s:s + m] = torch.remainder(cent[hid] + r[:, None] * v, 1.0).to(dt)
    for s in range(nh, n, step):
        m = min(step, n - s)
        x[s:s + m] = torch.rand((m, dim), generator=g, **f64).to(dt)
    one = torch.ones((), dtype=dt, device=DEV)
    x = torch.where(x >= one, torch.nextafter(one, torch.zeros_like(one)), x)
    return x[torch.randperm(n, generator=g, device=DEV)] if halos else x


def _knn_cfg(case: dict) -> KNNConfig:
    # the default settings with the case's leaf size; clustered sets need the larger node allocation
    # that the overflow message asks for, and so do the longer lists of a clustered set of few leaves
    return KNNConfig(alloc_fac_ilist=512. if case["cluster"] and case["n"] < 1 << 21 else 256.,
                     tree=TreeConfig(max_leaf_size=case["leaf"], coarse_fac=8.,
                                     alloc_fac_nodes=2. if case["cluster"] else 1.2, stop_coarsen=2048,
                                     mass_centered=False, regularization=RegularizationConfig()))


def _fof_cfg(case: dict) -> FofConfig:
    return FofConfig(alloc_fac_ilist=32. if case["n"] >= 1 << 20 else 128.,
                     tree=TreeConfig(max_leaf_size=case["leaf"], coarse_fac=8., alloc_fac_nodes=2., stop_coarsen=2048,
                                     mass_centered=False))


def _rlink(case: dict) -> float:
    return case["b"] * case["n"] ** (-1.0 / case.get("dim", 3))


def _set_sizes(case: dict) -> list:
    # the sizes belong to the plan, so they follow from the case; the points follow from the seed
    r = random.Random(1000 * case["nsets"] + case["lo"])
    return [int(2.0 ** r.uniform(case["lo"], case["hi"])) for _ in range(case["nsets"])]


def prepare(case: dict, seed: int) -> dict:
    g = _gen(seed)
    op = case["op"]
    st = dict(case=case)
    if op in ("knn", "knn_query"):
        st["x"] = _points(case["n"], case["dim"], case["cluster"], case["dtype"], g)
        st["cfg"] = _knn_cfg(case)
        if op == "knn_query":
            st["q"] = _points(case["nq"], case["dim"], 0, case["dtype"], g)
    elif op == "knn_learned":
        st["cfg"] = _knn_cfg(case)
        # the proposer of a user's program: trained once on another set of the same kind
        gp = _gen(case["k"])
        t = _points(case["n"], 3, case["cluster"], "f32", gp)
        feats, targets = jz.proposer.training_data([t], case["k"], st["cfg"], boxsize=case["box"])
        p = jz.proposer.RadiusProposer(case["k"], device=DEV, seed=0)
        p.train(feats, targets, steps=300)
        p.calibrate(feats, targets, quantile=0.999)
        st["proposer"] = p
        st["x"] = _points(case["n"], 3, case["cluster"], "f32", g)
    elif op == "fof":
        st["x"] = _points(case["n"], case["dim"], case["cluster"], "f32", g)
        st["cfg"], st["rlink"] = _fof_cfg(case), _rlink(case)
    elif op == "catalogue":
        n = case["n"]
        x = _points(n, 3, case["cluster"], "f32", g)
        mass = 0.5 + torch.rand(n, generator=g, device=DEV)
        vel = torch.randn((n, 3), generator=g, device=DEV)
        st["part"] = ParticleData(pos=x, mass=mass, vel=vel)
        st["cfg"], st["rlink"] = _fof_cfg(case), _rlink(case)
    elif op == "sets":
        sizes = _set_sizes(case)
        st["x"] = _points(sum(sizes), 3, 0, "f32", g)
        rl = [case["b"] * s ** (-1.0 / 3.0) for s in sizes]
        tree = TreeConfig(max_leaf_size=case["leaf"], coarse_fac=8., alloc_fac_nodes=1.1, stop_coarsen=2048)
        st["plan"] = jz.batch.CapturedSets(st["x"], sizes, k=case["k"], rlink=rl, boxsize=1.0, cfg_tree=tree)
    else:
        st["x"] = _points(case["n"], case["dim"], case["cluster"], case["dtype"], g).requires_grad_()
        st["grad"] = torch.randn(st["x"].shape, generator=g, device=DEV, dtype=st["x"].dtype)
    return st


# ------------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------------

def run(st: dict):
    case = st["case"]
    op = case["op"]
    if op == "knn":
        return jz.knn.knn(st["x"], case["k"], boxsize=case["box"] or None, output_order=case["order"], cfg=st["cfg"])
    if op == "knn_query":
        return jz.knn.knn(st["x"], case["k"], boxsize=case["box"] or None, part_query=st["q"], cfg=st["cfg"])
    if op == "knn_learned":
        return jz.proposer.knn_learned(st["x"], case["k"], st["proposer"], boxsize=case["box"], cfg=st["cfg"])
    if op == "fof":
        return jz.fof.fof_labels(st["x"], st["rlink"], boxsize=case["box"], cfg=st["cfg"], output_order=case["order"])
    if op == "catalogue":
        part, cata = jz.fof.fof_and_catalogue(st["part"], st["rlink"], boxsize=case["box"], cfg=st["cfg"])
        return dict(pos=part.pos, mass=part.mass, vel=part.vel, ngroups=cata.ngroups, count=cata.count,
                    offset=cata.offset, gmass=cata.mass, com_pos=cata.com_pos, com_vel=cata.com_vel,
                    radius=cata.com_inertia_radius)
    if op == "sets":
        return st["plan"].run(st["x"])
    posz, idz = jz.tree.zsort(st["x"])
    (gx,) = torch.autograd.grad(posz, st["x"], st["grad"])
    return posz.detach(), idz, gx


def work(case: dict) -> dict:
    op = case["op"]
    s = 8 if case.get("dtype") == "f64" else 4
    dim = case.get("dim", 3)
    if op in ("knn", "knn_learned", "knn_query"):
        # positions read once, k radii and ids written per query; at least k distances per query
        nq = case.get("nq", case["n"])
        rows = case["n"] + case.get("nq", 0)
        return dict(bytes=rows * dim * s + nq * case["k"] * (s + 4), flops=nq * case["k"] * 3 * dim)
    if op == "fof":
        # positions read, and (z order) the sorted positions and the labels written
        return dict(bytes=case["n"] * (dim * s * (2 if case["order"] == "z" else 1) + 4), flops=case["n"] * 3 * dim)
    if op == "catalogue":
        # position, mass and velocity read and written in group order
        return dict(bytes=case["n"] * 2 * 28, flops=case["n"] * 30)
    if op == "sets":
        n = sum(_set_sizes(case))
        return dict(bytes=n * (12 + 8 * case["k"] + 4), flops=n * case["k"] * 9)
    # positions and gradient read; sorted positions, indices and gradient written
    return dict(bytes=case["n"] * (4 * dim * s + s), flops=0)


# ------------------------------------------------------------------------------------------------
# 64-bit values
# ------------------------------------------------------------------------------------------------

def _exact_knn(q: torch.Tensor, x: torch.Tensor, k: int, box: float) -> torch.Tensor:
    """Radii of the k nearest by brute force in float64."""
    q, x = q.double(), x.double()
    out = torch.empty((len(q), k), dtype=torch.float64, device=q.device)
    step = max(1, (1 << 27) // len(x))
    for s in range(0, len(q), step):
        d2 = torch.zeros((min(step, len(q) - s), len(x)), dtype=torch.float64, device=q.device)
        for c in range(q.shape[1]):
            d = (q[s:s + step, None, c] - x[None, :, c]).abs_()
            if box:
                d = torch.minimum(d, box - d)
            d2 += d * d
        out[s:s + step] = torch.topk(d2, k, dim=1, largest=False, sorted=True)[0].sqrt_()
    return out


def exact(case: dict, seed: int):
    """Radii in float64 where a brute-force search takes seconds.  Ids, labels and sort permutations
    are whole numbers, the sort's positions and gradient are moved, not computed; catalogue values
    depend on a friends-of-friends run and are left to the bound of their type."""
    op = case["op"]
    if op in ("knn", "knn_query") and case["n"] * case.get("nq", case["n"]) <= 1 << 36:
        g = _gen(seed)
        x = _points(case["n"], case["dim"], case["cluster"], case["dtype"], g)
        if op == "knn_query":
            return _exact_knn(_points(case["nq"], case["dim"], 0, case["dtype"], g), x, case["k"], case["box"]), None
        if case["order"] == "z":
            return None  # rows in the order of the sort, which plain torch does not give
        return _exact_knn(x, x, case["k"], case["box"]), None
    return None
