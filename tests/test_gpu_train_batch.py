"""The batched loss gradient (one list over several structures) against the sum of the
per-structure gradients: structures of different sizes and boxes, one without a box, one of
a single element, one with an element the potential has no model for, repeated ones, and
batches split over several passes.  FP64 sums in another order: 1e-11 of the largest entry;
mixed precision: FP32 sums in another order, 2e-5."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TOL = {"float64": 1e-11, "mixed": 2e-5}


def _trainer(precision):
    from pantea_amd import water
    from pantea_amd.atoms import Structure
    from pantea_amd.bench_models import water_student
    from pantea_amd.student import ASSET_DIR, StudentTrainer

    rng = np.random.default_rng(4)
    tr = StudentTrainer(water_student(ASSET_DIR), precision=precision, w_energy=1.0, w_force=10.0)

    def add(s):
        tr.add(s, 0.3 * s.natoms, torch.as_tensor(rng.normal(scale=0.1, size=(s.natoms, 3)), device="cuda"))

    for n in (33, 71, 40, 128):
        add(Structure.from_dict(water.water_box(n, water.box_for_density(n), seed=n)))
    d = water.water_box(35, water.box_for_density(35), seed=1)
    add(Structure.from_dict({k: d[k] for k in ("positions", "elements")}))                    # no box
    d = water.water_box(40, water.box_for_density(40), seed=2)
    add(Structure.from_dict({**d, "elements": ["H"] * 120}))                                  # one element
    d = water.water_box(36, water.box_for_density(36), seed=3)
    add(Structure.from_dict({**d, "elements": ["He"] + d["elements"][1:]}))                   # no model for He
    tr.prepare(fit_scaler=False)
    return tr


@pytest.mark.parametrize("precision", ["float64", "mixed"])
@pytest.mark.parametrize("indices", [[0], [3, 1, 0, 2], [1, 1, 2], [4, 0, 5, 2], [6, 1]])
def test_batch_equals_sum_of_structures(precision, indices, monkeypatch):
    from pantea_amd import student

    tr = _trainer(precision)
    for g in tr.grad.values():
        g.zero_()
    tr.loss.zero_()
    for k in indices:
        tr._accumulate(tr.snapshots[k], 1.0 / len(indices))
    ref = tr.loss.clone(), {e: g.clone() for e, g in tr.grad.items()}
    for limit in (student._Batch.MAX_ATOMS, 220):
        monkeypatch.setattr(student._Batch, "MAX_ATOMS", limit)
        for _ in range(2):   # the second on used buffers
            loss, grad = tr.gradient(indices)
            assert torch.allclose(loss, ref[0], rtol=TOL[precision], atol=0)
            for e, g in grad.items():
                assert float((g - ref[1][e]).abs().max()) <= TOL[precision] * float(ref[1][e].abs().max())
