"""A list that does not fit, built by a step that reads it before its totals are known.

pt_nbr_build_async_or_empty: more pairs than the arrays hold, or a row over 256 entries where
the second pass is not enqueued, leaves nbr and rev unwritten and every row empty, with the real
totals; a list that fits is the synchronous one.  Both offset kernels (one workgroup up to 8,192
atoms, three launches beyond).  MD: such steps are redone and the trajectory is the synchronous
one, bit for bit."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _clusters(k):
    """k clusters of 400 atoms, a few Bohr wide: rows longer than 256 entries."""
    from pantea_amd.atoms import Structure

    rng = np.random.default_rng(k)
    m = int(np.ceil(k ** (1.0 / 3.0)))
    L = 15.0 * m
    at = (np.stack(np.meshgrid(*[np.arange(m)] * 3), -1).reshape(-1, 3)[:k] + 0.5) * 15.0
    pos = (at[:, None, :] + 1.2 * rng.normal(size=(k, 400, 3))).reshape(-1, 3)
    return Structure.from_dict({"positions": np.mod(pos, L), "elements": ["H"] * (400 * k), "lattice": np.diag([L] * 3)})


def _water(n_mol):
    from pantea_amd import water
    from pantea_amd.atoms import Structure

    return Structure.from_dict(water.water_box(n_mol, water.box_for_density(n_mol), seed=2023))


@pytest.mark.parametrize("case", ["fits", "pairs", "row"])
@pytest.mark.parametrize("large", [False, True])
def test_list_that_does_not_fit_has_empty_rows(case, large):
    from pantea_amd import _lib
    from pantea_amd.atoms import host_box
    from pantea_amd.engine import NeighborList

    lib = _lib.load()
    s, rc = (_clusters(22 if large else 2), 4.0) if case == "row" else (_water(2800 if large else 128), 6.0)
    n = s.natoms
    assert (n > 8192) == large
    nl = NeighborList(rc, s.element_map.n_types).build(s.positions, s.atom_types, s.box_lengths, s.type_counts())
    assert (nl.max_row > 256) == (case == "row")
    cap = nl.n_pairs - (1 if case == "pairs" else 0)
    dev = s.positions.device
    perm = torch.full_like(nl.perm, -7)
    pos4 = torch.full_like(nl.pos4, -7.0)
    row_off = torch.full_like(nl.row_off, -7)
    nbr, rev = (torch.full((cap,), -7, dtype=torch.int32, device=dev) for _ in range(2))
    totals = torch.zeros(4, dtype=torch.int64, device=dev)
    ws = torch.empty(lib.pt_nbr_workspace_bytes(n, s.element_map.n_types), dtype=torch.uint8, device=dev)
    pos = s.positions.to(torch.float64).contiguous()
    types = s.atom_types.to(torch.int32).contiguous()
    box = host_box(s.box_lengths)
    _lib.check(lib.pt_nbr_build_async_or_empty(
        n, pos.data_ptr(), 3, types.data_ptr(), s.element_map.n_types, ctypes.cast(box, ctypes.c_void_p), rc,
        perm.data_ptr(), pos4.data_ptr(), row_off.data_ptr(), nbr.data_ptr(), rev.data_ptr(), cap, None,
        totals.data_ptr(), 200, ws.data_ptr(), ws.numel(), _lib.stream_ptr()), "pt_nbr_build_async_or_empty")
    assert totals.tolist() == [nl.n_pairs, nl.max_row, nl.n_pairs, 1]
    assert torch.equal(perm, nl.perm) and torch.equal(pos4, nl.pos4)
    if case == "fits":
        assert torch.equal(row_off, nl.row_off)
        assert torch.equal(nbr, nl.nbr[:cap]) and torch.equal(rev, nl.rev[:cap])
    else:
        assert not row_off.any()
        assert (nbr == -7).all() and (rev == -7).all()


@pytest.mark.parametrize("what,graph", [("pairs", False), ("pairs", True), ("row", False)])
def test_md_redoes_steps_whose_list_did_not_fit(what, graph):
    from pantea_amd.bench_models import make_nnp, teacher_acsf
    from pantea_amd.simulation import MDSimulator, System
    from pantea_amd.units import units

    s = _water(128)
    rc = 17.0 if what == "row" else 12.0
    pot = make_nnp(lambda e: teacher_acsf(e, rc), (25, 25), seed=2023)
    pot.fit_scaler([s])
    out = []
    for sync_free in (False, True):
        sysm = System.from_structure(s, pot, temperature=300.0, seed=2023, force_mode="full", precision="float64",
                                     sync_free=sync_free, graph=graph and sync_free)
        md = sysm._engine()
        if sync_free and what == "pairs":
            md.nl.cap = md.nl.n_pairs // 2       # (the arrays themselves stay larger)
        elif sync_free:
            assert md.nl.max_row > 256
            md.row_bound = 200                   # no second pass for the rows over 256
        MDSimulator(0.5 * units.FROM_FEMTO_SECOND, integrator="physical").run(sysm, 6)
        out.append((sysm.positions.cpu().numpy(), sysm.velocities.cpu().numpy(), md.redos))
    (x0, v0, _), (x1, v1, redos) = out
    assert redos >= 1
    np.testing.assert_array_equal(x1, x0)
    np.testing.assert_array_equal(v1, v0)
