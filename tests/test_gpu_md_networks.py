"""Networks that are replaced between captured MD steps, in the same dictionary: the next step
runs the new ones, as an eager step does.  Same kernels on the same inputs: bit for bit."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_replaced_networks_are_captured_again():
    from pantea_amd import water
    from pantea_amd.atoms import Structure
    from pantea_amd.bench_models import water_nnp
    from pantea_amd.simulation import MDSimulator, System
    from pantea_amd.units import units

    s = Structure.from_dict(water.water_box(64, water.box_for_density(64), seed=2023))
    pot, other = (water_nnp(s, hidden=(25, 25), seed=k) for k in (2023, 7))
    out = []
    for graph in (False, True):
        sysm = System.from_structure(s, pot, temperature=300.0, seed=2023, force_mode="full", precision="float64",
                                     graph=graph)
        sim = MDSimulator(0.5 * units.FROM_FEMTO_SECOND, integrator="physical")
        sim.run(sysm, 4)
        ff = sysm._engine().ff
        old = dict(ff.mlps)                       # (kept alive)
        ff.mlps = dict(old)
        sim.run(sysm, 4)
        ff.mlps.update(other._device_mlps(ff.dev))
        sim.run(sysm, 4)
        out.append((sysm.positions.cpu().numpy(), sysm.velocities.cpu().numpy()))
        ff.mlps.update(old)
    np.testing.assert_array_equal(out[1][0], out[0][0])
    np.testing.assert_array_equal(out[1][1], out[0][1])
