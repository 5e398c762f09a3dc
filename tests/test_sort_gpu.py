"""Z-order sort on the GPU vs the oracle (bit-exact permutation)."""
import numpy as np
import pytest
import torch

from conftest import ZSORT_GOLDEN_IN, ZSORT_GOLDEN_OUT
from gen import clustered, uniform

pytestmark = pytest.mark.gpu


def _gpu_zsort(x, dev):
    import jztree_amd as jz
    print(f"[zsort] n={len(x)} dim={x.shape[1]} dtype={x.dtype}", flush=True)
    t = torch.from_numpy(np.ascontiguousarray(x)).to(dev)
    pz, idz = jz.tree.zsort(t)
    torch.cuda.synchronize()
    return pz.cpu().numpy(), idz.cpu().numpy()


def test_zsort_golden(dev):
    """checks/tests/test_tree.py:85-108"""
    xin = np.array(ZSORT_GOLDEN_IN, np.float32)
    pz, idz = _gpu_zsort(xin, dev)
    assert np.array_equal(pz[:-1], np.array(ZSORT_GOLDEN_OUT, np.float32)[:-1])
    assert np.all(np.isnan(pz[-1]))


@pytest.mark.parametrize("case", ["uniform16", "clustered", "dups", "negative", "specials", "2d", "wide",
                                  "f64", "tiny", "one"])
def test_zsort_matches_oracle(dev, oracle, case):
    rng = np.random.default_rng(3)
    if case == "uniform16":
        x = uniform(1 << 16, seed=0)
    elif case == "clustered":
        x = clustered(1 << 17, nhalos=256, seed=1)
    elif case == "dups":
        x = uniform(20000, seed=2)
        x = np.concatenate([x, x[:5000], x[:3000]])
        x[::7, 1] = x[0, 1]
        x[::11, 0] = 0.0
        x[::13, 2] = np.float32(1e-30)
    elif case == "negative":
        x = (rng.random((50000, 3)) * 4 - 2).astype(np.float32)
    elif case == "specials":
        x = (rng.random((5000, 3)) * 2 - 1).astype(np.float32)
        x[::9, 0] = np.inf
        x[::10, 1] = -np.inf
        x[::15, 2] = np.nan
        x[::23, 2] = np.float32(1e-42)
        x[::29, 1] = -0.0
    elif case == "2d":
        x = uniform(40000, dim=2, seed=4)
    elif case == "wide":
        x = uniform(40000, seed=5, lo=0.0, hi=1e6)
    elif case == "f64":
        x = rng.random((30000, 3))
    elif case == "tiny":
        x = uniform(5, seed=6)
    else:
        x = uniform(1, seed=7)
    pz, idz = _gpu_zsort(x, dev)
    opz, oidz = oracle.zsort(x)
    assert np.array_equal(idz.astype(np.int64), oidz)
    assert np.array_equal(pz, x[oidz], equal_nan=True)


def test_zsort_large_is_permutation_and_sorted(dev, oracle):
    """Full-size property checks: a bijection, and adjacent pairs never inverted."""
    x = clustered(1 << 22, nhalos=4096, seed=9)
    pz, idz = _gpu_zsort(x, dev)
    assert np.array_equal(np.sort(idz), np.arange(len(x)))
    assert np.array_equal(pz, x[idz])
    sample = np.random.default_rng(0).integers(0, len(x) - 1, 20000)
    assert all(oracle.z_exact_cmp(pz[i], pz[i + 1]) <= 0 for i in sample)


def test_zsort_gradient_backward(dev):
    """custom VJP (tree.py:111-138): the gradient scatters back through the permutation."""
    import jztree_amd as jz
    x = torch.from_numpy(uniform(1000, seed=8)).to(dev).requires_grad_(True)
    pz, idz = jz.tree.zsort(x)
    w = torch.arange(pz.numel(), dtype=torch.float32, device=dev).reshape(pz.shape)
    (pz * w).sum().backward()
    g = torch.empty_like(w)
    g[idz.long()] = w
    assert torch.equal(x.grad, g)


@pytest.mark.gpu
@pytest.mark.parametrize("kpt", [8, 16])
def test_zsort_tile_sizes(dev, oracle, kpt):
    """Every onesweep tile (keys per thread) sorts exactly as the default one and the oracle."""
    import jztree_amd as jz
    from gen import clustered
    x = clustered(200_003, nhalos=50, seed=9)
    x[:1000] = x[1000:2000]  # equal keys
    t = torch.from_numpy(x).to(dev)
    before = jz.autotune.get_knobs()
    try:
        jz.autotune.set_knobs(sort_kpt=kpt)
        print(f"[zsort tile] kpt={kpt}", flush=True)
        pz, iz = jz.tree.zsort(t)
        torch.cuda.synchronize()
    finally:
        jz.autotune.set_knobs(**before)
    p0, i0 = jz.tree.zsort(t)
    assert torch.equal(iz, i0) and torch.equal(pz, p0)
    assert np.array_equal(iz.cpu().numpy().astype(np.int64), oracle.zsort(x)[1])


# rounds of the one-workgroup sort (1024 keys each, up to 16384), tiles, the changes of tile shape
# (2^18, 2^21, 2^23) and more tiles than one look-back step reads
@pytest.mark.parametrize("n", [1, 2, 16, 17, 1023, 1024, 1025, 2047, 2049, 5000, 16383, 16384, 16385, 18433, (1 << 18) - 1, (1 << 18) + 1, (1 << 21) + 3,
                               (1 << 23) + 5])
def test_zsort_tiles(dev, oracle, n):
    x = clustered(n, nhalos=64, seed=n) if n > 4096 else uniform(n, seed=n)
    pz, idz = _gpu_zsort(x, dev)
    opz, oidz = oracle.zsort(x)
    assert np.array_equal(idz, oidz) and np.array_equal(pz, opz)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_zsort_equal_key_runs(dev, oracle, dtype):
    """Runs of equal keys around the length that one thread per row orders (16): copies of a point, and
    points that differ below the key's resolution."""
    rng = np.random.default_rng(5)
    parts = [rng.random((3000, 3)).astype(dtype), np.array([[1e6, 1., 1.]], dtype)]
    for length in (2, 3, 15, 16, 17, 18, 33, 34, 300):
        for _ in range(3):
            c = rng.random(3)
            parts.append(np.repeat(c[None], length, 0).astype(dtype))
            parts.append((c + 1e-3 * rng.random((length, 3))).astype(dtype))
    x = np.concatenate(parts)
    x = np.ascontiguousarray(x[rng.permutation(len(x))])
    pz, idz = _gpu_zsort(x, dev)
    opz, oidz = oracle.zsort(x)
    assert np.array_equal(idz, oidz) and np.array_equal(pz, opz)


@pytest.mark.parametrize("dtype,dim", [(torch.float32, 3), (torch.float64, 2)])
def test_zsort_gradient(dev, dtype, dim):
    """The gradient is the given one in input order; also of a strided one, of second order and batched."""
    import jztree_amd as jz
    g = torch.Generator(device=dev).manual_seed(1)
    x = torch.rand((1001, dim), dtype=dtype, device=dev, generator=g).requires_grad_()
    posz, idz = jz.tree.zsort(x)
    w = torch.randn((dim, 1001), dtype=dtype, device=dev, generator=g).T  # not contiguous
    ref = torch.empty_like(x)
    ref[idz.long()] = w
    (gx,) = torch.autograd.grad(posz, x, w, retain_graph=True)
    assert torch.equal(gx, ref)
    wr = w.clone().requires_grad_()
    (gx,) = torch.autograd.grad(posz, x, wr, create_graph=True)
    (gw,) = torch.autograd.grad(gx, wr, x.detach())
    assert torch.equal(gw, x.detach()[idz.long()])
    wb = torch.stack([w, 2 * w, -w])
    (gb,) = torch.autograd.grad(posz, x, wb, is_grads_batched=True)
    assert torch.equal(gb, torch.stack([ref, 2 * ref, -ref]))


@pytest.mark.parametrize("dim,dtype", [(2, np.float32), (3, np.float32), (2, np.float64), (3, np.float64)])
@pytest.mark.parametrize("kind", ["tight", "signed", "equal", "nan"])
def test_zsort_small(dev, oracle, dim, dtype, kind):
    """Sets for one workgroup whose points the top bits of the keys do not part, with signs, all equal,
    and with NaN rows next to the largest key."""
    rng = np.random.default_rng(9)
    x = rng.random((3000, dim))
    if kind == "tight":
        x = 0.3 + 1e-4 * x
        x[0] = 1.0
    elif kind == "signed":
        x = 2 * x - 1
        x[::17] = np.inf
        x[::19, 0] = -np.inf
    elif kind == "equal":
        x[:] = 0.25
    x = x.astype(dtype)
    if kind == "nan":
        x[::7] = np.nextafter(dtype(1), dtype(0))
        x[::11, 1] = np.nan
    x = np.ascontiguousarray(x)
    pz, idz = _gpu_zsort(x, dev)
    opz, oidz = oracle.zsort(x)
    assert np.array_equal(idz, oidz) and np.array_equal(pz, opz, equal_nan=True)


@pytest.mark.parametrize("dim,dtype", [(2, np.float32), (3, np.float32), (2, np.float64), (3, np.float64)])
@pytest.mark.parametrize("n,few", [(6, 1), (1000, 1), (1000, 8), (9001, 3)])
def test_zsort_small_nan_rows_next_to_the_top_corner(dev, oracle, dim, dtype, n, few):
    """A few NaN rows before and between points whose key bits are all ones (too few for a long run):
    the NaN rows come last, and a tree of the set counts the others."""
    import jztree_amd as jz
    rng = np.random.default_rng(n)
    x = rng.random((n, dim)).astype(dtype)
    rows = np.sort(rng.permutation(n)[:2 * few])
    x[rows[::2], 0] = np.nan  # every point of the corner has a NaN row before it
    x[rows[1::2]] = np.nextafter(dtype(1), dtype(0))
    pz, idz = _gpu_zsort(x, dev)
    opz, oidz = oracle.zsort(x)
    assert np.array_equal(idz, oidz) and np.array_equal(pz, opz, equal_nan=True)
    _, _, th = jz.tree.zsort_and_tree_origin(torch.from_numpy(x).to(dev), jz.config.TreeConfig(alloc_fac_nodes=2.))
    jz.checks.flush()
    assert int(th.splits_leaf_to_part(0).max()) == n - few


def _runs_set(rng, n, dim, dtype):
    """n rows in random order: runs of equal keys around the length that one thread per row orders (16) and far
    beyond, as copies of a point and as points that differ below the key's resolution, NaN rows, and
    single points."""
    parts = [np.full((1, dim), 1e6), np.full((n // 5, dim), np.nan)]
    for length in (2, 15, 16, 17, 18, 33, 300, 1500):
        for _ in range(2):
            c = rng.random(dim)
            parts.append(np.repeat(c[None], length, 0))
            parts.append(c + 1e-3 * rng.random((length, dim)))
            mixed = c + 1e-3 * rng.random((length, dim))  # copies and others in one run
            parts.append(mixed[rng.integers(0, min(3, length), length)])
    x = np.concatenate(parts)
    x = np.concatenate([x, rng.random((n - len(x), dim))])
    return np.ascontiguousarray(x[rng.permutation(n)].astype(dtype))


@pytest.mark.parametrize("dtype,dim", [(np.float32, 3), (np.float64, 3), (np.float32, 2), (np.float32, 5)])
@pytest.mark.parametrize("n", [16000, 20011, 150001])
def test_zsort_long_runs(dev, oracle, dtype, dim, n):
    """Long runs by one workgroup (n <= 16384) and by the passes over many."""
    x = _runs_set(np.random.default_rng(n), n, dim, dtype)
    pz, idz = _gpu_zsort(x, dev)
    opz, oidz = oracle.zsort(x)
    assert np.array_equal(idz, oidz) and np.array_equal(pz, opz, equal_nan=True)


@pytest.mark.parametrize("sizes", [[13000, 5, 14001, 1, 16000], [13000] * 3 + [1] * 300])
def test_zsort_sets_long_runs(dev, oracle, sizes):
    """The same runs in a batch, the same points in several sets: a run ends where its set does."""
    import jztree_amd as jz
    one = _runs_set(np.random.default_rng(3), 16000, 3, np.float32)
    x = np.concatenate([one[:s] for s in sizes])
    off = np.concatenate([[0], np.cumsum(sizes)])
    print(f"[zsort sets] {len(sizes)} sets, {len(x)} rows", flush=True)
    pz, idz = jz.batch.zsort_sets(torch.from_numpy(x).to(dev), jz.batch.set_offsets(sizes, dev))
    pz, idz = pz.cpu().numpy(), idz.cpu().numpy()
    for a, b in zip(off[:-1], off[1:]):
        _, oidz = oracle.zsort(x[a:b])
        assert np.array_equal(idz[a:b] - a, oidz), (a, b)
    assert np.array_equal(pz, x[idz], equal_nan=True)


def _lower_bits_sets(rng, n, dim):
    """Sets for the one-workgroup sort whose top key bits leave runs of more than 16 rows: in order, out of order
    by the lower bits, by less than the key, all but one row in one run, and a clump of few rows."""
    x = rng.random((n, dim))
    copies, near, below, far, clump = x.copy(), x.copy(), x.copy(), x.copy(), x.copy()
    copies[:n // 3] = x[0]
    copies[n // 3:n // 2] = x[1]
    c = rng.random((max(n // 60, 1), dim))
    near = (c[rng.integers(0, len(c), n)] + 1e-7 * rng.random((n, dim))) / 2
    below = np.concatenate([c[rng.integers(0, len(c), n - 1)] + 1e-9 * rng.random((n - 1, dim)), [[1e3] * dim]])
    far[n // 2] = 1e5
    clump[n // 2:n // 2 + 40] = 0.3 + 1e-7 * rng.random((40, dim))
    return dict(copies=copies, near=near, below=below, far=far, clump=clump)


@pytest.mark.parametrize("kind", ["copies", "near", "below", "far", "clump"])
@pytest.mark.parametrize("n", [100, 1025, 8192, 8193, 16384])
def test_zsort_small_lower_bits(dev, oracle, kind, n):
    """By itself (one workgroup up to 8192 rows) and for a call that asks for few launches (up to 16,384)."""
    import jztree_amd as jz
    for dim, dtype in ((3, np.float32), (3, np.float64), (2, np.float32)):
        x = np.ascontiguousarray(_lower_bits_sets(np.random.default_rng(n), n, dim)[kind].astype(dtype))
        _, oidz = oracle.zsort(x)
        t = torch.from_numpy(x).to(dev)
        for few in (False, True):
            pz, idz = jz.tree._zsort(t, few)
            assert np.array_equal(idz.cpu().numpy(), oidz), (dim, dtype, few)
            assert np.array_equal(pz.cpu().numpy(), x[oidz]), (dim, dtype, few)


@pytest.mark.parametrize("dtype,dim", [(torch.float32, 3), (torch.float64, 2)])
def test_zsort_gradient_forward_over_reverse(dev, dtype, dim):
    """A gradient that carries a tangent: both come back in input order, also through saved-tensor hooks, and
    batched."""
    import torch.autograd.forward_ad as fw
    import jztree_amd as jz
    g = torch.Generator(device=dev).manual_seed(2)
    x = torch.rand((1001, dim), dtype=dtype, device=dev, generator=g).requires_grad_()
    w, t = (torch.randn((1001, dim), dtype=dtype, device=dev, generator=g) for _ in range(2))
    with torch.autograd.graph.saved_tensors_hooks(lambda v: v.cpu(), lambda v: v.to(dev)):
        posz, idz = jz.tree.zsort(x)
    back = lambda v: torch.empty_like(v).index_copy_(0, idz.long(), v)
    with fw.dual_level():
        (gx,) = torch.autograd.grad(posz, x, fw.make_dual(w, t), retain_graph=True)
        p, dp = fw.unpack_dual(gx)
        assert torch.equal(p, back(w)) and torch.equal(dp, back(t))
    (gb,) = torch.autograd.grad(posz, x, torch.stack([w, t]), is_grads_batched=True)
    assert torch.equal(gb, torch.stack([back(w), back(t)]))


@pytest.mark.parametrize("kpt", [8, 16])
@pytest.mark.parametrize("n", [(1 << 18) + 1, (1 << 21) - 1, (1 << 21) + 3])
def test_zsort_tuned_tiles_of_larger_sets(dev, n, kpt):
    """The tuned number of keys per thread with 512 and 1024 threads a tile."""
    import jztree_amd as jz
    x = torch.rand((n, 3), device=dev, generator=torch.Generator(device=dev).manual_seed(n))
    p0, i0 = jz.tree.zsort(x)
    before = jz.autotune.get_knobs()
    try:
        jz.autotune.set_knobs(sort_kpt=kpt)
        print(f"[zsort tile] n={n} kpt={kpt}", flush=True)
        pz, iz = jz.tree.zsort(x)
        torch.cuda.synchronize()
    finally:
        jz.autotune.set_knobs(**before)
    assert torch.equal(iz, i0) and torch.equal(pz, p0)


def test_unsort_rows_of_many_elements(dev):
    """More elements than one launch holds threads."""
    import jztree_amd._lib as L
    n, width = 1031, 4_200_000
    assert n * width > 1 << 32
    rows = torch.empty((n, width), dtype=torch.int32, device=dev)
    rows.copy_(torch.arange(n, dtype=torch.int32, device=dev)[:, None])
    idz = torch.randperm(n, device=dev, generator=torch.Generator(device=dev).manual_seed(0)).to(torch.int32)
    out = torch.full_like(rows, -1)
    print("[unsort] 4.3e9 elements", flush=True)
    L.call("jzt_unsort_rows", L.stream(), L.ptr(rows), L.ptr(idz), n, width, 4, L.ptr(out))
    inv = torch.empty_like(idz)
    inv[idz.long()] = torch.arange(n, dtype=torch.int32, device=dev)
    for a in range(0, n, 100):
        assert bool((out[a:a + 100] == inv[a:a + 100, None]).all()), a
