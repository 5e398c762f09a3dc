"""Exact kNN on the GPU vs the oracle: neighbour ids bit-exact (ties by index), r2 bit-exact,
radii = correctly rounded sqrt of r2 and within 2 ulp of the float64 distance."""
import dataclasses
import math
import numpy as np
import pytest
import torch

from gen import clustered, uniform

pytestmark = pytest.mark.gpu


def _knn(x, k, dev, **kw):
    import jztree_amd as jz
    print(f"[knn] n={len(x)} k={k} {kw}", flush=True)
    t = torch.from_numpy(np.ascontiguousarray(x)).to(dev)
    rnn, inn = jz.knn.knn(t, k=k, **kw)
    torch.cuda.synchronize()
    return rnn.cpu().numpy(), inn.cpu().numpy()


def _check(x, k, rnn, inn, oracle, boxsize=0.0):
    r2o, io = oracle.knn(x, k, boxsize=boxsize)
    assert np.array_equal(inn.astype(np.int64), io), f"{np.sum(inn != io)} ids differ"
    assert np.array_equal(rnn, np.sqrt(r2o).astype(np.float32))


@pytest.mark.parametrize("k", [1, 4, 8, 12, 16, 32, 53, 64, 133])
def test_knn_k_sweep(dev, oracle, k):
    """checks/tests/test_knn.py:62-67 sizes: k from 1 to 133 (several passes above 64)."""
    x = uniform(1 << 14, seed=k)
    rnn, inn = _knn(x, k, dev)
    _check(x, k, rnn, inn, oracle)


def test_knn_config1(dev, oracle):
    """Plain kNN k=16 on 2^16 uniform points in the unit cube, non-periodic."""
    x = uniform(1 << 16, seed=0)
    rnn, inn = _knn(x, 16, dev)
    _check(x, 16, rnn, inn, oracle)


@pytest.mark.parametrize("boxsize", [0.03, 1.0, 170.0])
def test_knn_periodic(dev, oracle, boxsize):
    """checks/tests/test_knn.py:83-88"""
    x = uniform(1 << 14, seed=3, lo=0.0, hi=boxsize)
    x[x >= np.float32(boxsize)] = 0.0
    rnn, inn = _knn(x, 16, dev, boxsize=boxsize)
    _check(x, 16, rnn, inn, oracle, boxsize=boxsize)


@pytest.mark.parametrize("lohi", [(-0.3, 0.7), (0.1, 0.4), (-1.0, 0.0), (0.0, 1e6), (-1.0, 1.0)])
def test_knn_domains(dev, oracle, lohi):
    """checks/tests/test_knn.py:55-60"""
    x = uniform(1 << 14, seed=5, lo=lohi[0], hi=lohi[1])
    rnn, inn = _knn(x, 16, dev)
    _check(x, 16, rnn, inn, oracle)


def _clustered_cfg():
    """The default KNNConfig leaf allocation overflows on strongly clustered sets (as in the
    reference); a larger alloc_fac_nodes is the documented remedy."""
    import dataclasses
    from jztree_amd.config import KNNConfig
    c = KNNConfig()
    return dataclasses.replace(c, tree=dataclasses.replace(c.tree, alloc_fac_nodes=2.0))


def test_knn_clustered_and_duplicates(dev, oracle):
    x = clustered(1 << 16, nhalos=128, seed=4)
    x = np.concatenate([x, x[:4000]])  # exact duplicates: ties broken by index
    rnn, inn = _knn(x, 32, dev, cfg=_clustered_cfg())
    _check(x, 32, rnn, inn, oracle)


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("k", [12, 40])
def test_knn_many_copies_of_a_point(dev, oracle, fused, k):
    """More copies of a point than k, spread over several leaves (some of them mixed with other
    points, so their cells have a positive extent): the k-th distance of a copy is exactly 0, and
    its k neighbours are the copies with the smallest ids, wherever they sit."""
    rng = np.random.default_rng(k)
    x = np.concatenate([rng.random((20000, 3)), np.repeat(rng.random((3, 3)), 400, axis=0)]).astype(np.float32)
    x = x[rng.permutation(len(x))]
    rnn, inn = _knn(x, k, dev, fused=fused)
    _check(x, k, rnn, inn, oracle)


def test_knn_output_orders(dev):
    """checks/tests/test_knn.py:102-116: radii depend on the output order only; ids also on the input."""
    import jztree_amd as jz
    from jztree_amd.config import KNNConfig
    x = torch.from_numpy(uniform(1 << 15, seed=6)).to(dev)
    partz, idz, th = jz.tree.zsort_and_tree(x, KNNConfig().tree, data=torch.arange(len(x), device=dev))
    rnn00, inn00 = jz.knn.knn(x, k=16)
    rnn0z, inn0z = jz.knn.knn(x, k=16, output_order="z")
    rnnzz, innzz = jz.knn.knn(partz, k=16, th=th)
    idz = idz.long()
    assert torch.equal(rnn00[idz], rnn0z)
    assert torch.equal(rnn0z, rnnzz)
    assert torch.equal(inn00[idz], idz[innzz.long()].to(inn00.dtype))
    assert torch.equal(inn0z, innzz)


def test_knn_distance_ulp(dev):
    """Radii within 2 ulp of the float64 distance to the same neighbour."""
    x = clustered(1 << 15, nhalos=64, seed=8)
    rnn, inn = _knn(x, 16, dev, cfg=_clustered_cfg())
    d64 = np.linalg.norm(x.astype(np.float64)[:, None, :] - x.astype(np.float64)[inn], axis=-1)
    assert np.all(np.abs(rnn.astype(np.float64) - d64) <= 2 * np.spacing(rnn))


@pytest.mark.parametrize("case", ["uniform", "clustered_periodic", "small_one_plane", "k64", "two_planes"])
def test_fused_equals_reference_decomposition(dev, oracle, case):
    """The fused leaf-plane kernel returns exactly what KnnNode2Node + KnnLeaf2Leaf return, and both
    equal the oracle."""
    import jztree_amd as jz
    if case == "uniform":
        x, k, box = uniform(1 << 17, seed=11), 16, 0.0
    elif case == "clustered_periodic":
        x, k, box = clustered(1 << 17, nhalos=256, seed=12), 32, 1.0
    elif case == "small_one_plane":
        x, k, box = uniform(3000, seed=13), 8, 0.0
    elif case == "k64":
        x, k, box = clustered(1 << 16, nhalos=64, seed=14), 64, 1.0
    else:  # 2^19 points: two tree planes, so the parent lists and bounds come from KnnNode2Node
        x, k, box = clustered(1 << 19, nhalos=256, seed=16), 32, 1.0
    t = torch.from_numpy(x).to(dev)
    print(f"[fused] {case} n={len(x)} k={k}", flush=True)
    cfg = _clustered_cfg()
    r1, i1 = jz.knn.knn(t, k=k, boxsize=box, cfg=cfg, fused=True)
    r2_, i2 = jz.knn.knn(t, k=k, boxsize=box, cfg=cfg, fused=False)
    torch.cuda.synchronize()
    assert torch.equal(i1, i2) and torch.equal(r1, r2_)
    _check(x, k, r1.cpu().numpy(), i1.cpu().numpy(), oracle, boxsize=box)


def test_fused_bound_and_retry(dev, oracle):
    """A starting bound that is too small for some leaves triggers the in-call retry; results are
    unchanged."""
    import jztree_amd as jz
    x = clustered(1 << 16, nhalos=64, seed=15)
    t = torch.from_numpy(x).to(dev)
    cfg = _clustered_cfg()
    partz, originz, th = jz.tree.zsort_and_tree(t, cfg.tree, data=jz.data.RankIdx(
        rank=None, idx=torch.arange(len(x), dtype=torch.int32, device=dev)))
    size = th.size()
    tiny = torch.full((size,), 1e-12, dtype=torch.float32, device=dev)
    tiny[::2] = float("inf")
    r1, i1, retry = jz.knn._knn_fused(th, partz, 16, alloc_fac_ilist=cfg.alloc_fac_ilist, src_ids=originz.idx,
                                      init_r2=tiny)
    r2_, i2, _ = jz.knn._knn_fused(th, partz, 16, alloc_fac_ilist=cfg.alloc_fac_ilist, src_ids=originz.idx)
    jz.checks.flush()
    torch.cuda.synchronize()
    assert int(retry.sum()) > 0
    assert torch.equal(i1, i2) and torch.equal(r1, r2_)


def _leaf_max_r2k(jz, th, rz, k):
    """max over each leaf's queries of the k-th neighbour r2 (from z-ordered rows)."""
    from jztree_amd.tools import inverse_of_splits
    n = rz.shape[0]
    spl = th.splits_leaf_to_part()
    nl = int(th.num(0))
    leafof = inverse_of_splits(spl[: nl + 1].contiguous(), n).long()
    r2k = rz[:, k - 1].double() ** 2
    out = torch.zeros(th.size(), dtype=torch.float64, device=rz.device)
    return out.scatter_reduce(0, leafof, r2k, "amax", include_self=True).float()


@pytest.mark.gpu
@pytest.mark.parametrize("k,boxsize", [(16, 1.0), (32, 0.0), (32, 1.0), (12, 1.0), (40, 0.0)])
def test_bounded_matches_plain(dev, oracle, k, boxsize):
    """Bounded search from a proposed radius per leaf (lists + leaf kernel + retry) equals the plain
    search for bounds too small (retries), about right, too large, and for proposals with NaN and
    negative entries (a diverged network).  With k not a power of two (12, 40) the kernel's top-k
    is wider than k: a bound just above every leaf's exact radius must still flag no query."""
    import jztree_amd as jz
    x = clustered(1 << 16, nhalos=64, seed=21)
    t = torch.from_numpy(x).to(dev)
    cfg = _clustered_cfg()
    partz, originz, th = jz.tree.zsort_and_tree(t, cfg.tree, data=jz.data.RankIdx(
        rank=None, idx=torch.arange(len(x), dtype=torch.int32, device=dev)))
    il = jz.knn._knn_dual_walk(th, k, boxsize=boxsize, alloc_fac_ilist=cfg.alloc_fac_ilist)
    rz, iz = jz.knn._knn_leaf2leaf(il, th.splits_leaf_to_part(), partz, k=k, boxsize=boxsize, src_ids=originz.idx)
    exact = _leaf_max_r2k(jz, th, rz, k)
    mixed = exact.clone()
    mixed[::3] = 0.0
    wild = exact.clone()
    wild[::5] = float("nan")
    wild[1::5] = -1.0
    wild[2::5] = -float("inf")
    for fac, bound, grow, direct in [(0.25, exact * 0.25, None, True), (0.25, exact * 0.25, None, False),
                                     (0.25, exact * 0.25, 16.0, False), (1.0, exact * (1 + 1e-6), None, True),
                                     (3.0, exact * 3.0, None, True), ("mixed", mixed, None, True),
                                     ("mixed", mixed, None, False), ("nan_neg", wild, None, True),
                                     ("nan_neg", wild, None, False)]:
        st = {}
        r1, i1, retry = jz.knn._knn_bounded(th, partz, k, bound, boxsize=boxsize, grow=grow, direct_retry=direct,
                                            alloc_fac_ilist=cfg.alloc_fac_ilist, src_ids=originz.idx, stats=st)
        print(f"[bounded] k={k} box={boxsize} factor {fac}: {st}", flush=True)
        jz.checks.flush()
        torch.cuda.synchronize()
        assert torch.equal(i1, iz) and torch.equal(r1, rz), f"bound factor {fac}"
        nr = int(retry.sum())
        if fac in (0.25, "mixed"):
            assert nr > 0
        if fac in (1.0, 3.0):
            assert nr == 0
    # and the plain result is the oracle's
    inn = torch.empty_like(iz)
    inn[originz.idx.long()] = iz
    rnn = torch.empty_like(rz)
    rnn[originz.idx.long()] = rz
    _check(x, k, rnn.cpu().numpy(), inn.cpu().numpy(), oracle, boxsize=boxsize)


@pytest.mark.gpu
@pytest.mark.parametrize("k,boxsize", [(16, 1.0), (32, 0.0)])
def test_start_bound_fallback(dev, k, boxsize):
    """The plain search starts every query at its leaf's guaranteed radius; a start bound that
    rounds too small (forced here by shrinking it) sends the short leaves through the unbounded
    pass, and the result equals the unbounded kernel's."""
    import jztree_amd as jz
    x = clustered(1 << 16, nhalos=64, seed=23)
    t = torch.from_numpy(x).to(dev)
    cfg = _clustered_cfg()
    partz, originz, th = jz.tree.zsort_and_tree(t, cfg.tree, data=jz.data.RankIdx(
        rank=None, idx=torch.arange(len(x), dtype=torch.int32, device=dev)))
    il, leaf_r2, _ = jz.knn._knn_dual_walk(th, k, boxsize=boxsize, alloc_fac_ilist=cfg.alloc_fac_ilist,
                                           return_parents=True)
    spl = th.splits_leaf_to_part()
    rz, iz = jz.knn._knn_leaf2leaf(il, spl, partz, k=k, boxsize=boxsize, src_ids=originz.idx)
    for fac in (1.0, 0.3):
        print(f"[start bound] k={k} box={boxsize} factor {fac}", flush=True)
        r1, i1 = jz.knn._knn_leaf_start_bound(il, spl, partz, k, boxsize, leaf_r2 * fac, originz.idx)
        torch.cuda.synchronize()
        assert torch.equal(i1, iz) and torch.equal(r1, rz), f"factor {fac}"


def _cell_diag2_ref(lvl, dim):
    """Squared cell diagonal per level: sum of 4^l_i over the per-dim levels (python floor
    division as lvl_vec), exact powers of two from numpy.ldexp (a device pow is not exact)."""
    lv = lvl.cpu().numpy().astype(np.int64)
    o = (lv + 2000 * dim) // dim - 2000
    r = lv - o * dim
    d2 = np.zeros(lv.shape, dtype=np.float64)
    for i in range(dim):
        d2 = d2 + np.ldexp(1.0, 2 * (o + (r >= dim - i)))
    return torch.from_numpy(d2).to(lvl.device)


@pytest.mark.parametrize("k,boxsize", [(32, 1.0), (40, 0.0), (8, 1.0)])
def test_guaranteed_leaf_r2_bounds_true_kth(dev, oracle, k, boxsize):
    """The guaranteed leaf radius^2 (widened by 2^-10, as the bounded search and its retry pass use
    it) is at least the true k-th neighbour r2 of every query in the leaf: the oracle's canonical
    FP32 r2 of all 2^19 queries, clustered points (dense halos: small cells).  A leaf whose top-plane
    ancestor holds fewer than k particles has no bound from the tree (+inf); with 2^19 points the
    tree has two planes and nearly every leaf gets a finite bound, so the check is not vacuous."""
    import jztree_amd as jz
    from jztree_amd.knn import _guaranteed_leaf_r2
    from jztree_amd.tools import inverse_of_splits
    x = clustered(1 << 19, nhalos=256, seed=29)
    t = torch.from_numpy(x).to(dev)
    cfg = _clustered_cfg()
    partz, th = jz.tree.zsort_and_tree(t, cfg.tree)
    assert th.num_planes() >= 2
    cap = (_guaranteed_leaf_r2(th, k) * (1.0 + 2.0 ** -10)).to(torch.float32)
    nl = int(th.num(0))
    leafof = inverse_of_splits(th.splits_leaf_to_part()[: nl + 1].contiguous(), len(x)).long()
    r2o, _ = oracle.knn(partz.cpu().numpy(), k, boxsize=boxsize)
    r2k = torch.from_numpy(r2o[:, k - 1]).to(dev)
    bad = int((r2k > cap[leafof]).sum())
    assert bad == 0, f"{bad} queries have their k-th neighbour beyond the guaranteed radius"
    finite = float(torch.isfinite(cap[:nl]).float().mean())
    print(f"[cap] k={k} box={boxsize}: {finite:.4f} of {nl} leaves have a finite bound", flush=True)
    assert finite > 0.9


@pytest.mark.parametrize("n,leaf,k", [(1 << 14, 32, 32), (1 << 17, 64, 32), (1 << 17, 16, 40)])
def test_guaranteed_leaf_r2_matches_ancestor_walk(dev, n, leaf, k):
    """The per-plane kernel (jzt_plane_cap, top-down) equals walking each leaf up its ancestors
    to the first node with >= k particles and taking that cell's squared diagonal."""
    import jztree_amd as jz
    from jztree_amd.knn import _guaranteed_leaf_r2, _leaf_parent
    x = torch.from_numpy(clustered(n, nhalos=64, seed=11)).to(dev)
    cfg = jz.config.KNNConfig()
    tcfg = dataclasses.replace(cfg.tree, max_leaf_size=leaf, alloc_fac_nodes=2.0)
    _, th = jz.tree.zsort_and_tree(x, tcfg)
    size = th.size()
    ref = torch.full((size,), math.inf, dtype=torch.float64, device=dev)
    idx = torch.arange(size, device=dev)
    for p in range(th.num_planes()):
        npart = th.npart(p, size=size)
        d2 = _cell_diag2_ref(th.lvl.get(p, size), 3)
        take = (npart[idx] >= k) & torch.isinf(ref)
        ref = torch.where(take, d2[idx], ref)
        if p + 1 < th.num_planes():
            idx = _leaf_parent(th.ispl_n2n.get(p + 1, size + 1), size).long()[idx]
    got = _guaranteed_leaf_r2(th, k)
    nl = int(th.num(0))
    assert torch.equal(got[:nl], ref[:nl])


@pytest.mark.parametrize("k,boxsize,dim", [(8, 1.0, 3), (64, 1.0, 3), (40, 0.0, 3), (12, 1.0, 2), (70, 1.0, 3)])
def test_void_next_to_halo(dev, oracle, k, boxsize, dim):
    """Dense clumps on the box faces and in its corner, in a thin background: background leaves list whole
    clumps of which most or all particles are out of every query's reach, with and without the wrap."""
    import jztree_amd as jz
    rng = np.random.default_rng(11)
    cent = np.array([[0.0, 0.0, 0.0], [0.5, 0.999, 0.3], [0.25, 0.5, 0.5], [0.9995, 0.5, 0.7]])[:, :dim]
    x = np.concatenate([np.mod(c + 1e-3 * rng.standard_normal((2500, dim)), 1.0) for c in cent] + [rng.random((1500, dim))])
    x = np.minimum(x.astype(np.float32), np.float32(1) - np.float32(2.0 ** -24))
    x = np.ascontiguousarray(x[rng.permutation(len(x))])
    cfg = jz.config.KNNConfig(alloc_fac_ilist=1024.)
    cfg = dataclasses.replace(cfg, tree=dataclasses.replace(cfg.tree, alloc_fac_nodes=4.))
    rnn, inn = jz.knn.knn(torch.from_numpy(x).to(dev), k, boxsize=boxsize or None, cfg=cfg)
    r2o, io = oracle.knn(x, k, boxsize=boxsize)
    assert np.array_equal(inn.cpu().numpy().astype(np.int64), io)
    assert np.array_equal(rnn.cpu().numpy(), np.sqrt(r2o))


@pytest.mark.parametrize("leaf", [16, 31, 32, 33, 48, 63, 64, 65, 96, 97, 130])
@pytest.mark.parametrize("k,boxsize", [(1, 1.0), (8, 0.0), (33, 1.0), (70, 0.0)])
def test_leaf_query_chunks(dev, oracle, leaf, k, boxsize):
    """Leaf sizes around the 32 queries from which on two lanes share a query, and around whole chunks of
    64; chunks of sources that span several leaves."""
    import jztree_amd as jz
    x = uniform(3001, seed=leaf)
    cfg = jz.config.KNNConfig(alloc_fac_ilist=1024.)
    cfg = dataclasses.replace(cfg, tree=dataclasses.replace(cfg.tree, max_leaf_size=leaf, alloc_fac_nodes=3.))
    rnn, inn = _knn(x, k, dev, boxsize=boxsize or None, cfg=cfg)
    _check(x, k, rnn, inn, oracle, boxsize=boxsize)
