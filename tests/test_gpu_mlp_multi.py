"""pt_mlp_energy_grad_multi against the oracle's MLP: row counts at the edges of the
workgroup shapes (16 and 32 rows, 64 for narrow FP64 networks), networks of different
depth and width in one launch, and a launch without gradients."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# FP64: 64-bit products in another order than numpy; BF16x3: products of 16 mantissa bits
TOL = {"float64": 1e-12, "bf16x3": 2e-4}


def _net(n_in, hidden, seed):
    from pantea_amd.models import DeviceMLP, NeuralNetworkModel, NormalInitializer

    acts = ["tanh", "softplus", "tanh"][: len(hidden)]
    model = NeuralNetworkModel(tuple(zip(hidden, acts)), (1, "identity"), kernel_initializer=NormalInitializer())
    params = model.init(seed, n_in)
    rng = np.random.default_rng(seed)
    for k in params:
        params[k]["bias"] = rng.normal(size=params[k]["bias"].shape) * 0.1
    sub, mul = rng.random(n_in), 0.5 + rng.random(n_in)
    layers = [(params[f"layers_{2 * i}"]["kernel"], params[f"layers_{2 * i}"]["bias"], a)
              for i, a in enumerate(acts + ["identity"])]
    return DeviceMLP(model, params, n_in, np.stack([sub, mul]), 0.25, torch.device("cuda")), layers, sub, mul


@pytest.mark.parametrize("mode", ["float64", "bf16x3"])
@pytest.mark.parametrize("jobs", [
    [(52, (64, 64), 1), (52, (64, 64), 16), (52, (64, 64), 17), (52, (64, 64), 15), (52, (64, 64), 33)],
    [(34, (16, 16), 31), (34, (16, 16), 0), (34, (16, 16), 5)],
    [(34, (16, 16), 24576 + 13), (34, (16, 16), 65)],
    [(52, (64, 64), 20480 - 3), (52, (64, 33), 40)],
    [(20, (), 37), (96, (128, 7, 65), 50), (31, (32,), 64)],
])
def test_multi_matches_oracle(mode, jobs):
    from oracle import pyoracle
    from pantea_amd import _lib
    from pantea_amd.models import MLP_MODES, energy_grad_multi

    prec = _lib.PT_F64 if mode == "float64" else _lib.PT_F32
    dt = torch.float64 if mode == "float64" else torch.float32
    ld = max(j[0] for j in jobs) + 3
    rng = np.random.default_rng(len(jobs))
    call, ref = [], []
    for q, (n_in, hidden, n) in enumerate(jobs):
        mlp, layers, sub, mul = _net(n_in, hidden, 11 + q)
        G = rng.random((n, ld)) * 2.0
        call.append((mlp, n, torch.as_tensor(G, dtype=dt, device="cuda"),
                     torch.full((max(n, 1),), np.nan, dtype=torch.float64, device="cuda"),
                     torch.full((max(n, 1), ld), np.nan, dtype=dt, device="cuda")))
        y, g = pyoracle.mlp_forward_backward(layers, (G[:, :n_in] - sub) * mul + 0.25)
        ref.append((y, g * mul, n_in))
    energy_grad_multi(MLP_MODES[mode], call, ld, prec)
    for (mlp, n, _, e, d), (y, g, n_in) in zip(call, ref):
        if n == 0:
            continue
        e, d = e.cpu().numpy(), d.cpu().numpy()
        assert np.abs(e - y).max() < TOL[mode] * np.abs(y).max()
        assert np.abs(d[:, :n_in] - g).max() < TOL[mode] * np.abs(g).max()
        assert np.isnan(d[:, n_in:]).all()          # columns past the network's input stay untouched
    # energies alone: the same values, no gradient written
    again = [(m, n, G, torch.zeros_like(e), None) for m, n, G, e, _ in call]
    energy_grad_multi(MLP_MODES[mode], again, ld, prec)
    for a, b in zip(again, call):
        assert a[1] == 0 or torch.equal(a[3], b[3])
