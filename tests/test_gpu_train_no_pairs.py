"""The batched loss gradient of structures without a neighbour pair (atoms further apart than
the cutoff), as a trainer's first batch and together with others, against the sum of the
per-structure gradients.  The order of the sums differs: 1e-11 of the largest entry in FP64,
2e-5 in mixed precision."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("precision,tol", [("float64", 1e-11), ("mixed", 2e-5)])
def test_gradient_of_structures_without_pairs(precision, tol):
    from pantea_amd import water
    from pantea_amd.atoms import Structure
    from pantea_amd.bench_models import water_student
    from pantea_amd.student import ASSET_DIR, StudentTrainer

    rng = np.random.default_rng(4)
    tr = StudentTrainer(water_student(ASSET_DIR), precision=precision)
    far = [[0.0, 0.0, 0.0], [30.0, 0.0, 0.0], [0.0, 30.0, 0.0]]
    for s in (Structure.from_dict({"positions": far, "elements": ["O", "H", "H"], "lattice": np.diag([90.0] * 3)}),
              Structure.from_dict({"positions": far[:1], "elements": ["H"]}),
              Structure.from_dict(water.water_box(20, water.box_for_density(20), seed=1))):
        tr.add(s, 0.3 * s.natoms, torch.as_tensor(rng.normal(scale=0.1, size=(s.natoms, 3)), device="cuda"))
    tr.prepare(fit_scaler=False)
    for indices in ([0], [1], [0, 1], [2, 0], [0]):
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
