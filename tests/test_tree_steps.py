"""Steps of the general hierarchy build that need no GPU."""
import pytest
import torch


@pytest.mark.parametrize("idx", [[3, 6], [0, 9], [9], [3, 9, 12, 40], [5, 5, 5]])
@pytest.mark.parametrize("width", [(), (3,)])
def test_delete_rows(idx, width):
    """Rows named once or several times, or past the end (a node allocation that overflowed, which is reported
    later): every write in range, the kept rows in order."""
    from jztree_amd.tree import _delete_rows
    x = torch.arange(10.).reshape((10,) + (1,) * len(width)).expand((10,) + width).clone()
    out = _delete_rows(x, torch.tensor(idx, dtype=torch.int32))
    gone = {min(i, 9) for i in idx}
    kept = [i for i in range(10) if i not in gone]
    assert out.shape == (10 - len(idx),) + width
    assert torch.equal(out, x[torch.tensor(kept)][:10 - len(idx)])
