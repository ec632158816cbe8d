"""The batched loss gradient of a potential with more elements than a list has types (9
against 8), over structures that hold two, three and eight of them, against the sum of the
per-structure gradients.  The order of the sums differs: 1e-11 of the largest entry in FP64,
2e-5 in mixed precision."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

ELEMENTS = ("H", "O", "C", "N", "F", "Na", "Mg", "Al", "Si")


def _potential():
    from pantea_amd.descriptors import ACSF, G2, G3, CutoffFunction, DescriptorScaler, NeighborElements
    from pantea_amd.models import NeuralNetworkModel, NormalInitializer
    from pantea_amd.potential import AtomicPotential, NeuralNetworkPotential

    cfn = CutoffFunction.from_type("tanh", 6.0)
    radial = tuple((G2(cfn, r_shift=0.0, eta=0.05), NeighborElements(e)) for e in ELEMENTS)
    angular = tuple((G3(cfn, eta=0.02, zeta=1.0, lambda0=l, r_shift=0.0), NeighborElements("H", e))
                    for e in ("H", "O", "Si") for l in (1.0, -1.0))
    aps, params, scalers = {}, {}, {}
    for i, e in enumerate(ELEMENTS):
        model = NeuralNetworkModel(hidden_layers=((12, "tanh"),), kernel_initializer=NormalInitializer(1.0))
        acsf = ACSF(e, radial, angular)
        aps[e] = AtomicPotential(acsf, DescriptorScaler.from_type("scale"), model)
        params[e] = model.init(i, acsf.num_symmetry_functions)
        rows = np.random.default_rng(i).random((40, acsf.num_symmetry_functions)) * 3.0
        scalers[e] = DescriptorScaler.fit(torch.as_tensor(rows, device="cuda"))
    return NeuralNetworkPotential(directory=".", elements=ELEMENTS, atomic_potentials=aps, models_params=params,
                                  scalers_params=scalers)


@pytest.mark.parametrize("precision,tol", [("float64", 1e-11), ("mixed", 2e-5)])
def test_gradient_with_more_elements_than_types(precision, tol):
    from pantea_amd import water
    from pantea_amd.atoms import Structure
    from pantea_amd.student import StudentTrainer

    rng = np.random.default_rng(4)
    tr = StudentTrainer(_potential(), precision=precision)

    def water_with(n_mol, others):
        d = water.water_box(n_mol, water.box_for_density(n_mol), seed=n_mol)
        return Structure.from_dict({**d, "elements": list(others) + list(d["elements"])[len(others):]})

    for s in (water_with(20, ()), water_with(24, ("N",)), water_with(30, ELEMENTS[2:4] + ELEMENTS[5:]), water_with(33, ())):
        tr.add(s, 0.3 * s.natoms, torch.as_tensor(rng.normal(scale=0.1, size=(s.natoms, 3)), device="cuda"))
    tr.prepare(fit_scaler=False)
    assert [len(sn.blocks) for sn in tr.snapshots] == [2, 3, 8, 2]
    for indices in ([0], [2], [3, 1, 0, 2]):
        for g in tr.grad.values():
            g.zero_()
        tr.loss.zero_()
        for k in indices:
            tr._accumulate(tr.snapshots[k], 1.0 / len(indices))
        ref_loss, ref = tr.loss.clone(), {e: g.clone() for e, g in tr.grad.items()}
        loss, grad = tr.gradient(indices)
        assert torch.allclose(loss, ref_loss, rtol=tol, atol=0)
        for e, g in grad.items():
            assert float((g - ref[e]).abs().max()) <= tol * float(ref[e].abs().max())
