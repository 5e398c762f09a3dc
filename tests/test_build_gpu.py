"""The one-call hierarchy build (jzt_build_tree) and the walks' per-plane tables against the general steps: passing
the default level bound explicitly sends build_tree_hierarchy through those, so every array of the two
hierarchies, padding included, must be equal."""
import dataclasses

import numpy as np
import pytest
import torch

from gen import clustered

pytestmark = pytest.mark.gpu


def _equal(a, b, what):
    if a is None or b is None:
        assert a is None and b is None, what
    elif torch.is_tensor(a):
        assert a.dtype == b.dtype and a.shape == b.shape, what
        assert torch.equal(torch.nan_to_num(a, nan=-7.0) if a.is_floating_point() else a,
                           torch.nan_to_num(b, nan=-7.0) if b.is_floating_point() else b), what
        if a.is_floating_point():
            assert torch.equal(a.isnan(), b.isnan()), what
    elif dataclasses.is_dataclass(a):
        for f in dataclasses.fields(a):
            _equal(getattr(a, f.name), getattr(b, f.name), f"{what}.{f.name}")
    else:
        assert a == b, what


def _both(jz, part, cfg, **kw):
    pos = jz.data.get_pos(part)
    m = jz.data.LevelInfo(pos.shape[1], pos.dtype).max_lvl()
    new = jz.tree.build_tree_hierarchy(part, cfg, **kw)
    old = jz.tree.build_tree_hierarchy(part, cfg, lvl_bound=(m, m), **kw)
    jz.checks.flush()
    _equal(new, old, "th")
    size = new.size()
    t = jz.tree.plane_tables(new)
    for p in range(new.num_planes()):
        k = max(int(new.num(p)), 0)
        assert torch.equal(t.spl[p], new.ispl_n2n.get(p, size + 1)), p
        assert torch.equal(t.lvl[p][:k], new.lvl.get(p, size)[:k])
        assert torch.equal(t.npart[p][:k], new.npart(p, size=size)[:k].to(torch.int32))
        rows = jz.fof.PosLvl(pos=new.geom_cent.get(p, size), lvl=new.lvl.get(p, size)).pos_lvl()
        view = torch.int32 if rows.dtype == torch.float32 else torch.int64
        assert torch.equal(t.nodes[p][:k].view(view), rows[:k].view(view))
    return new


@pytest.mark.parametrize("n,dim,dtype,leaf,reg,stop", [
    (1, 3, np.float32, 48, True, 2048), (2, 3, np.float32, 4, False, 2048), (37, 2, np.float32, 48, False, 2048),
    (1000, 3, np.float32, 48, True, 2048), (1023, 3, np.float32, 8, True, 4), (4097, 5, np.float32, 16, True, 16),
    (5000, 3, np.float64, 16, True, 16), (3000, 10, np.float64, 32, True, 16), (40_001, 2, np.float64, 8, False, 64),
    (100_003, 3, np.float32, 16, True, 64), (100_003, 3, np.float32, 16, False, 64),
])
def test_build_equals_the_general_steps(dev, n, dim, dtype, leaf, reg, stop):
    import jztree_amd as jz
    rng = np.random.default_rng(n + dim)
    x = (clustered(n, nhalos=16, seed=n) if dim == 3 and n > 50_000 else rng.random((n, dim))).astype(dtype)
    x[: n // 9] = x[n - n // 9: n] if n // 9 else x[:0]  # duplicates
    cfg = jz.config.TreeConfig(max_leaf_size=leaf, coarse_fac=6., stop_coarsen=stop, alloc_fac_nodes=6.,
                               regularization=jz.config.RegularizationConfig() if reg else None)
    pz, _ = jz.tree.zsort(torch.from_numpy(x).to(dev))
    _both(jz, pz, cfg)
    _both(jz, jz.data.Pos(pos=pz, num=n), cfg)
    if n > 100:  # padded rows: NaN at the end, counted or given as a device count
        x[-n // 7:, 0] = np.nan
        pz, _ = jz.tree.zsort(torch.from_numpy(x).to(dev))
        th = _both(jz, pz, cfg)
        num = torch.tensor([n - n // 7 - 1], device=dev)
        _both(jz, jz.data.Pos(pos=pz, num=num), cfg)
        assert int(th.ispl_l2p_per_type[0, -1]) == int((~torch.isnan(pz[:, 0])).sum())


def test_build_of_batches_equals_the_general_steps(dev):
    import jztree_amd as jz
    sizes = [1, 700, 0, 33, 5000, 2, 48, 0]
    n = sum(sizes)
    x = torch.from_numpy(np.random.default_rng(3).random((n, 3), dtype=np.float32)).to(dev)
    off = jz.batch.set_offsets(sizes, dev)
    seg = jz.batch.set_ids(off, n)
    pz, _ = jz.batch.zsort_sets(x, off)
    for leaf, stop in ((48, 2048), (8, 16)):
        cfg = jz.config.TreeConfig(max_leaf_size=leaf, coarse_fac=6., stop_coarsen=stop, alloc_fac_nodes=3.)
        _both(jz, jz.data.Pos(pos=pz, num=n), cfg, set_id=seg, nsets=len(sizes))


def test_build_overflow_is_reported(dev):
    import jztree_amd as jz
    x = torch.from_numpy(clustered(1 << 15, nhalos=4, seed=1)).to(dev)
    pz, _ = jz.tree.zsort(x)
    cfg = jz.config.TreeConfig(max_leaf_size=8, alloc_fac_nodes=0.5)
    jz.tree.build_tree_hierarchy(pz, cfg)
    with pytest.raises(RuntimeError, match="allocation too small"):
        jz.checks.flush()
    with pytest.raises(RuntimeError, match="allocation too small"):
        jz.knn.knn(x, 8, cfg=jz.config.KNNConfig(tree=cfg))
    with pytest.raises(RuntimeError, match="allocation too small"):
        jz.fof.fof_labels(x, 0.01, cfg=jz.config.FofConfig(tree=cfg))
    ok = jz.config.KNNConfig(alloc_fac_ilist=1024., tree=dataclasses.replace(cfg, alloc_fac_nodes=8.))
    r, _ = jz.knn.knn(x, 8, cfg=ok)  # usable after
    assert torch.isfinite(r).all()


@pytest.mark.parametrize("dim,dtype", [(3, torch.float32), (2, torch.float64)])
@pytest.mark.parametrize("n", [16384, 16385, 200_003])
@pytest.mark.parametrize("tail", [0, 1, 300, 0.6])
def test_points_of_padded_positions(dev, n, dim, dtype, tail):
    """Points of a set whose last rows in z-order hold NaN: those with a NaN first coordinate are padding."""
    import jztree_amd as jz
    g = torch.Generator(device=dev).manual_seed(n)
    x = torch.rand((n, dim), generator=g, dtype=dtype, device=dev)
    m = tail if tail >= 1 else int(tail * n)
    x[:m] = float("nan")
    x[:m:5, 0] = 0.5  # a NaN in other coordinates only: a point
    posz, _ = jz.tree.zsort(x[torch.randperm(n, generator=g, device=dev)])
    print(f"[tail] n={n} dim={dim} {dtype} tail={m}", flush=True)
    th = jz.tree.build_tree_hierarchy(posz, jz.config.TreeConfig(max_leaf_size=48, alloc_fac_nodes=3.))
    jz.checks.flush()
    assert int(th.splits_leaf_to_part(0).max()) == int((~torch.isnan(x[:, 0])).sum())


@pytest.mark.parametrize("bad", ["int64", "short"])
def test_set_ids_are_checked(dev, bad):
    """The set of every row is int32, one a row; anything else is refused before a kernel reads it."""
    import jztree_amd as jz
    posz, _ = jz.tree.zsort(torch.rand((500, 3), device=dev))
    seg = torch.zeros(500, dtype=torch.int32, device=dev)
    seg = seg.long() if bad == "int64" else seg[:-1]
    with pytest.raises(AssertionError):
        jz.tree.build_tree_hierarchy(posz, jz.config.TreeConfig(alloc_fac_nodes=2.), set_id=seg, nsets=1)
    jz.checks.clear()
