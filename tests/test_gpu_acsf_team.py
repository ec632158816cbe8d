"""Descriptor launches of few centres (a team of wavefronts per centre) against launches of
many (one wavefront per centre): the same centres, listed often enough to cross the line,
must give the same descriptors, forces and tangents, for every table class, both
precisions and row lengths around the 64-entry chunks; several runs in one launch must
equal single launches.  Sums are taken in another order, so values agree to rounding:
a sum of a few thousand terms, 1e-13 in FP64 and 3e-6 in FP32 of the largest value."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TOL = {0: 1e-13, 1: 3e-6}


def _acsf(kind, rc):
    from pantea_amd.descriptors import ACSF, G2, G3, G9, CutoffFunction, NeighborElements

    cut, zetas, G = {"z14": ("tanh", (1.0, 4.0), G3), "p4": ("tanhu", (1.0, 2.0), G3), "z1": ("tanh", (1.0,), G3),
                     "generic": ("cos", (1.5, 3.0), G9)}[kind]
    cfn = CutoffFunction.from_type(cut, rc)
    radial = tuple((G2(cfn, r_shift=0.2, eta=e), NeighborElements(x)) for x in ("H", "O") for e in (0.01, 0.1, 0.7))
    # more functions than one radial group holds for one element
    radial += tuple((G2(cfn, r_shift=0.0, eta=0.02 * k), NeighborElements("H")) for k in range(1, 8))
    angular = tuple((G(cfn, eta=e, zeta=z, lambda0=l, r_shift=0.0), NeighborElements(j, k))
                    for j, k in (("H", "H"), ("H", "O"), ("O", "O")) for e in (0.005, 0.03) for z in zetas
                    for l in (1.0, -1.0))
    return ACSF("O", radial, angular)


def _system(rc, n_mol=100):
    from pantea_amd import water
    from pantea_amd.atoms import Structure
    from pantea_amd.engine import NeighborList

    s = Structure.from_dict(water.water_box(n_mol, water.box_for_density(n_mol), seed=3))
    nl = NeighborList(rc, 2).build(s.positions, s.atom_types, s.box_lengths, s.type_counts())
    return s, nl


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("kind,rc", [("z14", 12.0), ("z14", 9.9), ("p4", 10.0), ("z1", 12.0), ("generic", 12.0),
                                     ("z14", 4.0), ("z14", 1.0)])
def test_team_equals_single_wavefront(kind, rc, prec):
    from pantea_amd.engine import acsf_adjoint, acsf_forward, acsf_tangent

    s, nl = _system(rc)
    acsf = _acsf(kind, rc)
    dev = nl.pos4.device
    tab = acsf.device_table(s.element_map, dev)
    n_sf = acsf.num_symmetry_functions
    n = s.natoms
    dt = torch.float64 if prec == 0 else torch.float32
    few = torch.arange(n, dtype=torch.int32, device=dev)
    reps = 1536 // n + 2
    many = few.repeat(reps)
    g = torch.Generator(device="cpu").manual_seed(1)
    w = torch.randn((n, n_sf), generator=g, dtype=torch.float64).to(device=dev, dtype=dt)
    delta = torch.randn((n, 3), generator=g, dtype=torch.float64).to(dev)

    def close(a, b):
        scale = float(b.abs().max())
        assert float((a - b).abs().max()) <= TOL[prec] * scale if scale > 0 else float(a.abs().max()) == 0.0

    one = acsf_forward(nl, tab, prec, n, centers=few)
    ref = acsf_forward(nl, tab, prec, n * reps, centers=many)[:n]
    close(one, ref)
    close(acsf_tangent(nl, tab, prec, n, delta, False, centers=few),
          acsf_tangent(nl, tab, prec, n * reps, delta, False, centers=many)[:n])
    out = []
    for centers, k in ((few, 1), (many, reps)):
        f = torch.full((n * k, 3), np.nan, dtype=torch.float64, device=dev)
        e = torch.full((max(nl.n_pairs, 1), 3), np.nan, dtype=dt, device=dev)
        et = torch.full_like(e, np.nan)
        acsf_adjoint(nl, tab, prec, n * k, w.repeat(k, 1), n_sf, centers=centers, f_self=f, edge_grad=e)
        acsf_adjoint(nl, tab, prec, n * k, w.repeat(k, 1), n_sf, centers=centers, edge_grad=et, transposed=True)
        out.append((f[:n], e[:nl.n_pairs], et[:nl.n_pairs]))
    for a, b in zip(*out):
        if a.numel():
            close(a, b)
    # the team's sums do not depend on its wavefronts' timing
    again = torch.zeros_like(out[0][0])
    acsf_adjoint(nl, tab, prec, n, w, n_sf, centers=few, f_self=again)
    assert torch.equal(again, out[0][0])
    # a row beyond the staged length is reported, not staged
    if nl.max_row > 1:
        full, nl.max_row = nl.max_row, nl.max_row - 1
        try:
            cap = (nl.max_row + 3) // 4 * 4
            long = (nl.row_off[1:] - nl.row_off[:-1]) > cap
            bad = acsf_forward(nl, tab, prec, n, centers=few)
        finally:
            nl.max_row = full
        assert torch.isnan(bad[long]).all() and torch.equal(bad[~long], one[~long])


@pytest.mark.parametrize("prec", [0, 1])
def test_runs_equal_single_launches(prec):
    """Two tables of different classes and three unit-vector tangents, each in one call."""
    from pantea_amd.engine import (acsf_adjoint, acsf_adjoint_multi, acsf_forward, acsf_forward_multi, acsf_run,
                                   acsf_tangent, acsf_tangent_multi)

    s, nl = _system(10.0)
    dev = nl.pos4.device
    tabs = [_acsf(k, 10.0).device_table(s.element_map, dev) for k in ("z14", "generic", "z14")]
    blocks = [(0, 70), (70, 31), (101, 0)]
    ld = max(t.n_sf for t in tabs)
    dt = torch.float64 if prec == 0 else torch.float32
    w = torch.randn((200, ld), dtype=dt, device=dev)
    G, G1 = torch.zeros((200, ld), dtype=dt, device=dev), torch.zeros((200, ld), dtype=dt, device=dev)
    f, f1 = torch.zeros((200, 3), dtype=torch.float64, device=dev), torch.zeros((200, 3), dtype=torch.float64, device=dev)
    e, e1 = torch.zeros((nl.n_pairs, 3), dtype=dt, device=dev), torch.zeros((nl.n_pairs, 3), dtype=dt, device=dev)
    acsf_forward_multi(nl, prec, [acsf_run(t, c, b, out=G[b:]) for t, (b, c) in zip(tabs, blocks)], ld)
    acsf_adjoint_multi(nl, prec, [acsf_run(t, c, b, w=w[b:], f_self=f[b:]) for t, (b, c) in zip(tabs, blocks)], ld,
                       edge_grad=e, transposed=True)
    for t, (b, c) in zip(tabs, blocks):
        acsf_forward(nl, t, prec, c, center_begin=b, out=G1[b:], ld=ld)
        acsf_adjoint(nl, t, prec, c, w[b:], ld, center_begin=b, f_self=f1[b:], edge_grad=e1, transposed=True)
    assert torch.equal(G, G1) and torch.equal(f, f1) and torch.equal(e, e1)
    T = torch.zeros((3, 31, ld), dtype=dt, device=dev)
    acsf_tangent_multi(nl, prec, [acsf_run(tabs[0], 31, 5, out=T[d], direction=d) for d in range(3)], True, ld)
    for d in range(3):
        delta = torch.zeros((s.natoms, 3), dtype=torch.float64, device=dev)
        delta[:, d] = 1.0
        assert torch.equal(T[d], acsf_tangent(nl, tabs[0], prec, 31, delta, True, center_begin=5, ld=ld))
