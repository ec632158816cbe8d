"""Teams of eight and of four wavefronts against one wavefront per centre for the tables
that take other paths in a team: more angular groups than wait for their sums at once,
groups of two cutoffs (no shared cutoff values), radial groups of a cutoff of their own,
weights beyond the 64 columns a wavefront holds, no angular or no radial groups.  The same
values in another order: 1e-13 in FP64 and 3e-6 in FP32 of the largest value, as sums of a
few thousand terms."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TOL = {0: 1e-13, 1: 3e-6}
RC = 11.0


def _acsf(variant):
    from pantea_amd.descriptors import ACSF, G2, G3, CutoffFunction, NeighborElements

    def cut(rc):
        return CutoffFunction.from_type("tanh", rc)

    radial_rc = [9.0] if variant == "radial_cut" else [RC]
    n_radial = 40 if variant == "wide" else 5
    radial = tuple((G2(cut(rc), r_shift=0.1, eta=0.01 * k), NeighborElements(x)) for rc in radial_rc for x in ("H", "O")
                   for k in range(1, n_radial + 1))
    angular_rc = [RC, 8.0] if variant == "two_cutoffs" else [RC]
    # five eta values: a second group of each element pair
    etas = (0.001, 0.004, 0.01, 0.02, 0.05) if variant == "many_groups" else (0.005, 0.03)
    angular = tuple((G3(cut(rc), eta=e, zeta=z, lambda0=l, r_shift=0.0), NeighborElements(j, k))
                    for rc in angular_rc for j, k in (("H", "H"), ("H", "O"), ("O", "O")) for e in etas
                    for z in (1.0, 4.0) for l in (1.0, -1.0))
    return ACSF("O", () if variant == "no_radial" else radial, () if variant == "no_angular" else angular)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("variant", ["plain", "many_groups", "two_cutoffs", "radial_cut", "wide", "no_angular", "no_radial"])
def test_teams_equal_single_wavefront(variant, prec):
    from pantea_amd import water
    from pantea_amd.atoms import Structure
    from pantea_amd.engine import NeighborList, acsf_adjoint, acsf_forward, acsf_tangent

    n_mol = 60
    s = Structure.from_dict(water.water_box(n_mol, water.box_for_density(n_mol), seed=5))
    nl = NeighborList(RC, 2).build(s.positions, s.atom_types, s.box_lengths, s.type_counts())
    tab = _acsf(variant).device_table(s.element_map, "cuda")
    n = nl.n
    dt = torch.float64 if prec == 0 else torch.float32
    rng = np.random.default_rng(2)
    w0 = torch.as_tensor(rng.normal(size=(n, tab.n_sf)), device="cuda").to(dt)
    delta = torch.as_tensor(rng.normal(size=(n, 3)), device="cuda")
    got = {}
    for count in (n, 700, 2100):   # eight, four, one wavefronts per centre
        cen = torch.arange(count, device="cuda", dtype=torch.int32) % n
        G = acsf_forward(nl, tab, prec, count, centers=cen)
        T = acsf_tangent(nl, tab, prec, count, delta, False, centers=cen)
        f = torch.full((count, 3), float("nan"), dtype=torch.float64, device="cuda")
        acsf_adjoint(nl, tab, prec, count, w0[cen.long()].contiguous(), tab.n_sf, centers=cen, f_self=f)
        got[count] = [x.double().cpu().numpy() for x in (G, T, f)]
        for x in got[count]:
            assert np.isfinite(x).all()
    for k in range(3):
        one = got[2100][k]
        for count in (n, 700):
            x = got[count][k]
            scale = np.abs(one).max()
            for r in range(0, count, n):
                part = x[r:r + n]
                assert np.abs(part - one[:len(part)]).max() <= TOL[prec] * scale, (variant, count, k)
