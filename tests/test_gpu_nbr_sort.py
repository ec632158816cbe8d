"""The build's sorts by (type, cell) beyond one workgroup: the counting sort (few or many
atoms per cell, all atoms in one, its last workgroup's remainder) and the radix sort that
takes over when the cells outnumber the atoms four times.  Whole numbers: the order is
exactly numpy's stable one."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n,cells,spread", [
    (6145, 1, 1.0), (6145, 9, 1.0), (7001, 11, 0.09), (20001, 30, 1.0), (70001, 20, 1.0),
    (2000, 15, 1.0),      # fewer atoms than the one-workgroup sort takes, more cells
    (6145, 24, 1.0), (2000, 17, 1.0), (300, 30, 0.5)])   # radix: cells > 4 atoms
def test_order_is_stable_by_type_and_cell(n, cells, spread):
    from pantea_amd.engine import NeighborList

    rng = np.random.default_rng(n + cells)
    L = 1.0
    rc = L / (cells + 0.5)   # so many cells per dimension
    pos = rng.random((n, 3)) * spread * L
    types = rng.integers(1, 3, n).astype(np.int32)
    p = torch.as_tensor(pos, device="cuda")
    t = torch.as_tensor(types, device="cuda")
    counts = [int((types == 1).sum()), int((types == 2).sum())]
    nl = NeighborList(rc, 2).build(p, t, [L] * 3, counts)
    c = np.floor(pos * (1.0 / (L / cells))).astype(np.int64) % cells
    key = (types - 1) * cells ** 3 + (c[:, 2] * cells + c[:, 1]) * cells + c[:, 0]
    want = np.argsort(key, kind="stable")
    np.testing.assert_array_equal(nl.perm.cpu().numpy(), want)
    np.testing.assert_array_equal(nl.pos4.cpu().numpy(), np.concatenate([pos, types[:, None]], axis=1)[want])
