"""Calls whose arguments need a copy (strided, or of another type): several copies made for one call must
not share memory."""
import dataclasses

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _strided(t):
    """The same values as a view that is not contiguous."""
    wide = torch.zeros(t.shape + (2,), dtype=t.dtype, device=t.device)
    wide[..., 0] = t
    return wide[..., 0]


@pytest.mark.parametrize("n", [100, 5000])
def test_search_of_strided_positions(dev, n):
    import jztree_amd as jz
    g = torch.Generator(device=dev).manual_seed(n)
    posz, _ = jz.tree.zsort(torch.rand((n, 3), device=dev, generator=g))
    q = torch.rand((n, 3), device=dev, generator=g)
    ref = jz.tree.search_sorted_z(posz, q)
    assert torch.equal(jz.tree.search_sorted_z(_strided(posz), _strided(q)), ref)


def test_tree_steps_of_strided_arrays(dev):
    import jztree_amd as jz
    n = 3000
    g = torch.Generator(device=dev).manual_seed(1)
    posz, _ = jz.tree.zsort(torch.rand((n, 3), device=dev, generator=g))
    lvl, lb, rb = jz.tree.determine_znode_boundaries(posz)
    lb, rb = lb[:-1].clamp(0, n - 1).contiguous(), rb[:-1].clamp(1, n).contiguous()
    ref = jz.tree.get_node_geometry(posz, lb, rb)
    for a, b in zip(ref, jz.tree.get_node_geometry(_strided(posz), _strided(lb), _strided(rb))):
        assert torch.equal(a.nan_to_num(), b.nan_to_num())
    spl = torch.arange(0, n + 1, 10, dtype=torch.int32, device=dev)
    ref = jz.tree.center_of_mass(spl, posz, 1.)
    for a, b in zip(ref, jz.tree.center_of_mass(_strided(spl), _strided(posz), 1.)):
        assert torch.equal(a, b)


def test_plane_tables_of_wider_integers(dev):
    """A hierarchy whose index arrays came back as int64 (a saved one, say) gives the same tables."""
    import jztree_amd as jz
    g = torch.Generator(device=dev).manual_seed(2)
    _, _, th = jz.tree.zsort_and_tree_origin(torch.rand((20000, 3), device=dev, generator=g),
                                             jz.config.TreeConfig(max_leaf_size=16, alloc_fac_nodes=2., stop_coarsen=64))
    jz.checks.flush()
    wide = lambda p: dataclasses.replace(p, data=p.data.long(), ispl=p.ispl.long(), fill_values=p.fill_values.long())
    th64 = dataclasses.replace(th, ispl_n2n=wide(th.ispl_n2n), ispl_n2l=wide(th.ispl_n2l), lvl=wide(th.lvl))
    a, b = jz.tree.plane_tables(th), jz.tree.plane_tables(th64)
    for p in range(th.num_planes()):
        m = int(th.num(p))
        assert torch.equal(a.spl[p], b.spl[p])
        for name in ("nodes", "lvl", "npart"):
            x, y = getattr(a, name)[p][:m].contiguous(), getattr(b, name)[p][:m].contiguous()
            assert np.array_equal(x.cpu().numpy().view(np.int32), y.cpu().numpy().view(np.int32)), (p, name)


def test_node_labels_of_wider_integers(dev):
    import jztree_amd as jz
    from jztree_amd.fof import _node_to_child_label
    ig = torch.tensor([0, 1, 1, 3], dtype=torch.int32, device=dev)
    lvl = torch.full((4,), -12, dtype=torch.int32, device=dev)
    spl = torch.tensor([0, 2, 5, 6, 9], dtype=torch.int32, device=dev)
    ref = _node_to_child_label(ig, lvl, spl, rlink=0.1, dim=3, size_child=9)
    assert torch.equal(_node_to_child_label(ig.long(), lvl.long(), spl.long(), rlink=0.1, dim=3, size_child=9), ref)
