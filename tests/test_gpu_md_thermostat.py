"""A thermostat whose values change between runs (a heating ramp), on one object: captured and
eager steps give the same trajectory, and steps that are redone after a list overflow are redone
with the values they were first run with.  Same kernels on the same inputs: bit for bit."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _ramp(s, pot, graph, overflow):
    from pantea_amd.simulation import BrendsenThermostat, MDSimulator, System
    from pantea_amd.units import units

    dt = 0.5 * units.FROM_FEMTO_SECOND
    sysm = System.from_structure(s, pot, temperature=300.0, seed=2023, force_mode="full", precision="float64",
                                 graph=graph)
    md = sysm._engine()
    if overflow:   # the first rebuild has a longer row: redone at the next check, after the change below
        md.row_bound = md.nl.max_row - 8
    thermostat = BrendsenThermostat(300.0, 2.0 * dt)
    sim = MDSimulator(dt, thermostat=thermostat, integrator="physical")
    for temperature, tau in ((300.0, 2.0), (900.0, 2.0), (900.0, 5.0)):
        thermostat.target_temperature, thermostat.time_constant = temperature, tau * dt
        sim.run(sysm, 5)
    return sysm.positions.cpu().numpy(), sysm.velocities.cpu().numpy(), md.redos


@pytest.mark.parametrize("graph,overflow", [(True, False), (False, True), (True, True)])
def test_changed_thermostat_values(graph, overflow):
    from pantea_amd import water
    from pantea_amd.atoms import Structure
    from pantea_amd.bench_models import water_nnp

    s = Structure.from_dict(water.water_box(96, water.box_for_density(96), seed=2023))
    pot = water_nnp(s, hidden=(25, 25), seed=2023)
    x0, v0, _ = _ramp(s, pot, False, False)
    x1, v1, redos = _ramp(s, pot, graph, overflow)
    assert (redos >= 1) == overflow
    np.testing.assert_array_equal(x1, x0)
    np.testing.assert_array_equal(v1, v0)
