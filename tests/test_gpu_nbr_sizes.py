"""Neighbour lists at the edges of the small-build kernels (the one-workgroup sort and
offsets, cells split over workgroups), against all pairs in FP64 on the GPU: whole
numbers, so exactly equal.  The rows, the stable order by (type, input) within a cell's
type block, the positions and the reverse index are checked."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _mic(d, L):
    """Single-shift minimum image of atoms/distance.py:63-78."""
    d = torch.where(d > 0.5 * L, d - L, d)
    return torch.where(d < -0.5 * L, d + L, d)


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("n", [1, 2, 63, 65, 1024, 1025, 2048, 2049, 4096, 4097, 6144, 6145, 8192, 8193, 12289])
def test_list_at_kernel_edges(n, periodic):
    from pantea_amd.engine import NeighborList

    rng = np.random.default_rng(n)
    rc, L = 5.0, max(3.0, (n / 0.02) ** (1.0 / 3.0))
    pos = torch.as_tensor(rng.random((n, 3)) * L, device="cuda")
    types = np.sort(rng.integers(1, 3, n)).astype(np.int32)
    rng.shuffle(types)
    t = torch.as_tensor(types, device="cuda")
    counts = [int((types == 1).sum()), int((types == 2).sum())]
    nl = NeighborList(rc, 2).build(pos, t, [L] * 3 if periodic else None, counts)
    perm = nl.perm.long()
    assert torch.equal(torch.sort(perm).values, torch.arange(n, device="cuda"))
    assert torch.equal(nl.pos4[:, :3], pos[perm]) and torch.equal(nl.pos4[:, 3].int(), t[perm])
    p, row_off = pos[perm], nl.row_off.cpu().numpy()
    assert bool((nl.pos4[1:, 3] >= nl.pos4[:-1, 3]).all()) and row_off[0] == 0
    nbr, rev = nl.nbr[:nl.n_pairs].long(), nl.rev[:nl.n_pairs].long()
    total, longest = 0, 0
    for i0 in range(0, n, 512):
        d = p[i0:i0 + 512, None, :] - p[None, :, :]
        if periodic:
            d = _mic(d, torch.as_tensor(L, dtype=torch.float64, device="cuda"))
        s = d[..., 0] * d[..., 0]
        s = s + d[..., 1] * d[..., 1]
        s = s + d[..., 2] * d[..., 2]
        r = torch.sqrt(s)
        hit = (r <= rc) & (r > 0)
        rows, cols = torch.nonzero(hit, as_tuple=True)     # ascending within a row
        assert torch.equal(nbr[total:total + len(cols)], cols)
        per = hit.sum(1).cpu().numpy()
        np.testing.assert_array_equal(np.diff(row_off[i0:i0 + len(per) + 1]), per)
        centre = rows + i0
        e = torch.arange(total, total + len(cols), device="cuda")
        assert torch.equal(nbr[rev[e]], centre) and torch.equal(rev[rev[e]], e)
        total += len(cols)
        longest = max(longest, int(per.max()))
    assert total == nl.n_pairs == row_off[-1] and longest == nl.max_row
