"""Kernels of KnnNode2Node and its list sort, at the sizes where their split changes.

Segment sort: lengths around the powers of two of the one-wave sort (64 to 1024 entries), of the LDS sorts
(4096, 16384) and beyond, negative keys, equal keys, keys of any bits, against numpy's lexicographic order.
FofNode2Node: joined nodes and lists against all pairs, at every number of children per work item.
Node lists: every child's radius against the exact weighted selection and every list against all pairs,
with parents whose lists are short (one wave) and long (queued), fewer and more than 64 particles of
candidates per child, one and several children per work item."""
import dataclasses

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [
    [1, 2, 3, 0, 63, 64, 65, 127, 128, 129, 0, 255, 256, 257, 511, 512, 513, 1023, 1024],
    [1025, 5, 2048, 0, 4095, 4096, 4097, 70, 8191, 16384, 16385, 1],
])
def test_segment_sort_lengths(dev, lens):
    import jztree_amd._lib as L
    rng = np.random.default_rng(sum(lens))
    n = sum(lens)
    key = rng.normal(size=n).astype(np.float32)
    key[rng.random(n) < 0.3] = np.float32(0.25)  # equal keys: ordered by value
    key[rng.random(n) < 0.2] = np.float32(-0.5)
    key[rng.random(n) < 0.01] = np.float32(np.inf)
    val = rng.permutation(n).astype(np.int32)
    spl = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    t = [torch.from_numpy(a).to(dev) for a in (spl, key, val)]
    ko, vo = torch.empty_like(t[1]), torch.empty_like(t[2])
    L.call("jzt_segment_sort", L.stream(), L.ptr(t[0]), L.ptr(t[1]), L.ptr(t[2]), L.ptr(ko), L.ptr(vo), len(lens), n)
    ko, vo = ko.cpu().numpy(), vo.cpu().numpy()
    for a, b in zip(spl[:-1], spl[1:]):
        o = np.lexsort((val[a:b], key[a:b]))
        assert np.array_equal(ko[a:b], key[a:b][o]) and np.array_equal(vo[a:b], val[a:b][o]), (a, b)


@pytest.mark.parametrize("lens", [[3, 64, 65, 300, 1000, 1024], [1500, 5000, 17000]])
def test_segment_sort_any_key_bits(dev, lens):
    """Keys of every bit pattern, NaN ones and both zeros among them, in the float total order (by val among
    equal ones): every pair comes out once."""
    import jztree_amd._lib as L
    rng = np.random.default_rng(sum(lens))
    n = sum(lens)
    bits = rng.integers(0, 1 << 32, size=n, dtype=np.uint64).astype(np.uint32)
    bits[::5] = rng.integers(0x7f800000, 0x80000000, size=len(bits[::5]), dtype=np.uint64).astype(np.uint32)
    bits[1::5] = rng.integers(0xff800000, 1 << 32, size=len(bits[1::5]), dtype=np.uint64).astype(np.uint32)
    bits[::7], bits[1::7] = 0, 0x80000000
    bits[2::7], bits[3::7] = 0xffffffff, 0x7fffffff
    val = rng.integers(-2, 2, size=n).astype(np.int32)
    spl = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    t = [torch.from_numpy(a).to(dev) for a in (spl, bits.view(np.float32), val)]
    ko, vo = torch.empty_like(t[1]), torch.empty_like(t[2])
    L.call("jzt_segment_sort", L.stream(), L.ptr(t[0]), L.ptr(t[1]), L.ptr(t[2]), L.ptr(ko), L.ptr(vo), len(lens), n)
    ko, vo = ko.cpu().numpy().view(np.uint32), vo.cpu().numpy()
    order = np.where(bits >> 31, ~bits, bits | np.uint32(0x80000000))
    for a, b in zip(spl[:-1], spl[1:]):
        o = np.lexsort((val[a:b].view(np.uint32), order[a:b]))
        assert np.array_equal(ko[a:b], bits[a:b][o]) and np.array_equal(vo[a:b], val[a:b][o]), (a, b)


def _half_ext(lvl, dim):
    o = (lvl + 2000 * dim) // dim - 2000
    r = lvl - o * dim
    return np.stack([np.ldexp(0.5, o + (r >= dim - i)) for i in range(dim)], axis=1)


@pytest.mark.parametrize("nparents,kids,k,box", [
    (3, 5, 8, 0.0),       # a handful of nodes
    (130, 9, 40, 1.0),    # several child groups and rounds per parent, one wave per item
    (300, 32, 16, 1.0),   # dense lists of 300 entries: queued parents
    (300, 8, 200, 0.0),   # more candidates than a child keeps
])
def test_node_lists_against_all_pairs(dev, nparents, kids, k, box):
    import jztree_amd as jz
    from jztree_amd.data import InteractionList
    from jztree_amd.knn import PosLvlNum, _knn_node2node_ilist
    rng = np.random.default_rng(nparents + k)
    dim = 3
    nch = rng.integers(0, kids + 1, size=nparents)
    nch[0] = kids
    spl = np.concatenate([[0], np.cumsum(nch)]).astype(np.int32)
    n = int(spl[-1])
    lvl = rng.integers(-18, -9, size=n).astype(np.int32)
    cent = rng.random((n, dim)).astype(np.float32)
    npart = rng.integers(0, 4, size=n).astype(np.int32)
    npart[rng.random(n) < 0.1] = 300
    size_il = max(n * n, nparents * nparents, 64)
    t = lambda a: torch.from_numpy(a).to(dev)
    il = torch.zeros(size_il, dtype=torch.int32, device=dev)
    il[: nparents * nparents] = t(np.tile(np.arange(nparents, dtype=np.int32), nparents))
    dense = InteractionList(t((np.arange(nparents + 1) * nparents).astype(np.int32)), il,
                            rad2=torch.zeros(size_il, device=dev))
    out, radii = _knn_node2node_ilist(dense, t(spl), PosLvlNum(t(cent), t(lvl), t(npart)), k=k, boxsize=box,
                                      with_radii=True)
    jz.checks.flush()
    # the bounds are defined in float32: differences (subject to cancellation) are formed in it, the
    # fused sum of squares is rounded once per step
    e = _half_ext(lvl, dim).astype(np.float32)
    f32 = np.float32
    d = cent[None] - cent[:, None]  # target - child
    if box:
        d = np.where(d < -f32(0.5 * box), d + f32(box), d)
        d = np.where(d >= f32(0.5 * box), d - f32(box), d)
    w = e[:, None] + e[None]

    def norm2(v):
        r = np.zeros(v.shape[:-1], dtype=f32)
        for i in range(dim):
            x = v[..., i].astype(np.float64)
            r = (x * x + r).astype(f32)
        return r.astype(np.float64)

    dmin = norm2(np.maximum(np.abs(d) - w, f32(0.0)))
    dmax = norm2(np.abs(d) + w)
    r = radii.cpu().numpy().astype(np.float64)[:n]
    slack = 1.0 + 2.0 ** -16
    # float32 sums of three fused steps: a relative error below 2^-20
    tol = 2.0 ** -20
    for i in range(n):
        o = np.argsort(dmax[i], kind="stable")
        cum = np.cumsum(npart[o])
        exact = dmax[i][o][np.searchsorted(cum, k)] if cum[-1] >= k else np.inf
        if np.isinf(exact):
            assert np.isinf(r[i])
        else:
            assert r[i] >= exact * (1 - tol), (i, r[i], exact)
            if k <= 64:
                assert r[i] <= exact * slack * (1 + tol), (i, r[i], exact)
    ispl = out.ispl.cpu().numpy()
    src, r2 = out.isrc.cpu().numpy(), out.rad2.cpu().numpy()
    for i in range(n):
        a, b = ispl[i], ispl[i + 1]
        got = src[a:b]
        assert len(np.unique(got)) == len(got)
        inside = np.zeros(n, dtype=bool)
        inside[got] = True
        assert inside[dmin[i] < r[i] * (1 - tol)].all() and not inside[dmin[i] > r[i] * (1 + tol)].any(), i
        rr = r2[a:b]
        order = np.lexsort((got, rr))
        assert np.array_equal(order, np.arange(b - a)), i
        pos = rr >= 0
        assert np.allclose(rr[pos], dmin[i][got[pos]], rtol=2.0 ** -18, atol=0)
        assert (dmin[i][got[~pos]] <= 1e-12).all()


@pytest.mark.parametrize("nparents,kids", [(3, 9), (130, 20), (300, 12), (1100, 3)])  # every width of a work item
def test_fof_node_passes_against_all_pairs(dev, nparents, kids):
    """FofNode2Node on a dense parent list: nodes joined by guaranteed pairs share the smallest index of their
    set, and the lists hold every other pair that may link, each parent pair once."""
    import jztree_amd as jz
    from jztree_amd.data import InteractionList
    from jztree_amd.fof import PosLvl, _fof_node2node
    rng = np.random.default_rng(nparents)
    dim, f32 = 3, np.float32
    nch = rng.integers(0, kids + 1, size=nparents)
    nch[0] = kids
    spl = np.concatenate([[0], np.cumsum(nch)]).astype(np.int32)
    n = int(spl[-1])
    parent = np.repeat(np.arange(nparents), nch)
    lvl = rng.integers(-24, -12, size=n).astype(np.int32)
    cent = rng.random((n, dim)).astype(f32)
    cent[: n // 2] *= f32(0.1)
    rlink = 0.02
    t = lambda a: torch.from_numpy(a).to(dev)
    size_il = max(n * n, nparents * nparents, 64)
    il = torch.zeros(size_il, dtype=torch.int32, device=dev)
    il[: nparents * nparents] = t(np.tile(np.arange(nparents, dtype=np.int32), nparents))
    dense = InteractionList(t((np.arange(nparents + 1) * nparents).astype(np.int32)), il)
    ig, out = _fof_node2node(dense, t(spl), PosLvl(t(cent), t(lvl)), torch.arange(n, dtype=torch.int32, device=dev),
                             rlink=rlink, boxsize=1.0)
    jz.checks.flush()
    ig, ispl, src = ig.cpu().numpy()[:n], out.ispl.cpu().numpy(), out.isrc.cpu().numpy()
    e = _half_ext(lvl, dim).astype(f32)
    d = cent[None] - cent[:, None]
    d = np.where(d < -f32(0.5), d + f32(1), d)
    d = np.where(d >= f32(0.5), d - f32(1), d)
    w = e[:, None] + e[None]

    def norm2(v):
        r = np.zeros(v.shape[:-1], dtype=f32)
        for i in range(dim):
            x = v[..., i].astype(np.float64)
            r = (x * x + r).astype(f32)
        return r.astype(np.float64)

    dmin, dmax = norm2(np.maximum(np.abs(d) - w, f32(0))), norm2(np.abs(d) + w)
    diag = norm2(e) * 4
    r2 = float(f32(rlink * rlink))
    tol = 2.0 ** -20  # float32 sums of three fused steps
    once = parent[None] >= parent[:, None]
    bound = np.maximum(dmax, diag[None])
    surely = once & (bound <= r2 * (1 - 2.0 ** -16) * (1 - tol))
    maybe = once & (bound <= r2 * (1 - 2.0 ** -16) * (1 + tol))
    assert (surely == maybe).all()  # no pair at the edge of the test
    root = np.arange(n)
    for i, j in zip(*np.nonzero(surely)):
        a, b = root[i], root[j]
        if a != b:
            root[root == max(a, b)] = min(a, b)
    assert np.array_equal(ig, root)
    rest = once & ~surely & ((root[:, None] != root[None]) | np.eye(n, dtype=bool))
    need = rest & (dmin < r2 * (1 + 2.0 ** -16) * (1 - tol))
    may = rest & (dmin <= r2 * (1 + 2.0 ** -16) * (1 + tol))
    got = np.zeros((n, n), dtype=bool)
    for i in range(n):
        assert len(np.unique(src[ispl[i]:ispl[i + 1]])) == ispl[i + 1] - ispl[i]
        got[i, src[ispl[i]:ispl[i + 1]]] = True
    assert not (need & ~got).any() and not (got & ~may).any()
    assert need.any()


@pytest.mark.parametrize("n,dim,dtype,boxsize", [(200003, 3, "f32", 1.0), (150001, 2, "f32", 0.0),
                                                 (120001, 3, "f64", 1.0), (130001, 2, "f64", 1.0)])
def test_dense_top_distances(dev, monkeypatch, n, dim, dtype, boxsize):
    """Neighbours and groups with the super-nodes' distances in the dense list equal those without; the
    points are clustered towards the faces of the box."""
    import jztree_amd as jz
    rng = np.random.default_rng(n)
    x = np.concatenate([rng.random((n // 2, dim)), np.mod(0.02 * rng.standard_normal((n - n // 2, dim)), 1.0)])
    x = np.minimum(x, 1 - 2.0 ** -24).astype(np.float32 if dtype == "f32" else np.float64)
    t = torch.from_numpy(np.ascontiguousarray(x[rng.permutation(n)])).to(dev)
    kcfg, fcfg = jz.config.KNNConfig(alloc_fac_ilist=512.), jz.config.FofConfig(alloc_fac_ilist=256.)
    tree = lambda c: dataclasses.replace(c, tree=dataclasses.replace(c.tree, max_leaf_size=32, alloc_fac_nodes=2.5))
    kcfg, fcfg = tree(kcfg), tree(fcfg)
    rl = 0.2 * n ** (-1.0 / dim)
    out = []
    for least in (0, 1 << 40):
        monkeypatch.setattr(jz.tree, "_DENSE_R2_LEAVES", least)
        rnn, inn = jz.knn.knn(t, 10, boxsize=boxsize or None, cfg=kcfg)
        pz, ig = jz.fof.fof_labels(t, rl, boxsize=boxsize, cfg=fcfg)
        out.append((rnn, inn, pz, ig))
    for a, b in zip(*out):
        assert torch.equal(a, b)


def test_no_parents_give_empty_lists(dev):
    """Nodes without parents: lists of no entries, labels as given, nothing raised."""
    import jztree_amd as jz
    from jztree_amd.data import InteractionList
    from jztree_amd.fof import PosLvl, _fof_node2node
    from jztree_amd.knn import PosLvlNum, _knn_node2node_ilist
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device=dev)
    pos = torch.rand((5, 3), device=dev)
    il = InteractionList(i32(0), torch.zeros(64, dtype=torch.int32, device=dev), rad2=torch.zeros(64, device=dev))
    out = _knn_node2node_ilist(il, i32(0), PosLvlNum(pos=pos, lvl=i32(*[-12] * 5), npart=i32(*[1] * 5)), k=2)
    assert out.ispl.tolist() == [0] * 6
    ig, out = _fof_node2node(InteractionList(il.ispl, il.isrc), i32(0), PosLvl(pos=pos, lvl=i32(*[-12] * 5)),
                             i32(0, 1, 2, 3, 4), rlink=0.1)
    assert out.ispl.tolist() == [0] * 6 and ig.tolist() == [0, 1, 2, 3, 4]
    jz.checks.flush()
