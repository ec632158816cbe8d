"""pt_mlp_train_grad_multi and pt_mlp_jacobian_multi against double backward in FP64
torch on the host: row counts at the edges of the 16-row tiles, networks without and
with one to three hidden layers in one launch, several directions, and networks whose
buffers do not fit together.  Tolerance of FP64: products of at most 96 terms in another
order, 1e-12 of the largest entry; BF16x3 keeps 16 bits of each factor (2^-16 = 1.5e-5
per product and layer, forward and reverse): 5e-4."""

import numpy as np
import pytest

from test_gpu_mlp_multi import _net

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

JOBS = [
    [(52, (64, 64), 1), (34, (16, 16), 15), (34, (16, 16), 0), (52, (64, 64), 17)],
    [(20, (), 33), (31, (32,), 16), (20, (24, 8, 30), 31)],
    [(60, (90,), 5), (20, (24, 8, 40), 18)],            # 124 and 150 KB of LDS in FP64, 223 together
]


def _rows(layers, sub, mul, G, T, gy, seed):
    """d(gy y + seed T . dy/dG)/d(parameters) of one atom, flattened as W, b per layer."""
    ps = [torch.tensor(x, dtype=torch.float64, requires_grad=True) for W, b, _ in layers for x in (W, b)]
    x = torch.tensor((G - sub) * mul + 0.25, dtype=torch.float64, requires_grad=True)
    act = {"tanh": torch.tanh, "softplus": torch.nn.functional.softplus, "identity": lambda v: v}
    v = x
    for q, (_, _, a) in enumerate(layers):
        v = act[a](v @ ps[2 * q] + ps[2 * q + 1])
    y = v.sum()
    g, = torch.autograd.grad(y, x, create_graph=True)
    loss = gy * y + seed * (g * torch.tensor(T * mul)).sum()
    out = torch.autograd.grad(loss, ps, allow_unused=True)
    return np.concatenate([(torch.zeros_like(p) if o is None else o).numpy().ravel() for o, p in zip(out, ps)])


@pytest.mark.parametrize("jobs", JOBS)
def test_train_and_jacobian_match_double_backward(jobs):
    from pantea_amd import _lib
    from pantea_amd.models import MLP_MODES, jacobian_multi, train_grad_multi

    ld, ndir, sign = max(j[0] for j in jobs) + 3, 3, -0.7
    rng = np.random.default_rng(len(jobs))
    nets, host = [], []
    for q, (n_in, hidden, n) in enumerate(jobs):
        nets.append(_net(n_in, hidden, 31 + q))
        host.append((rng.random((n, ld)) * 2.0, rng.normal(size=(ndir, n, ld)), rng.normal(size=n)))
    dev = lambda x, dt=torch.float64: torch.as_tensor(x, dtype=dt, device="cuda").contiguous()
    rows = max(j[2] for j in jobs) * ndir

    def jacobians(which):
        """J of the jobs in `which` (one tangent stride serves a launch: all have max n rows)."""
        nmax = max(jobs[q][2] for q in which)
        T = [np.zeros((ndir, nmax, ld)) for _ in which]
        for t, q in zip(T, which):
            t[:, :jobs[q][2]] = host[q][1]
        ldj = max(nets[q][0].n_params for q in which) + 2
        J = [torch.full((rows, ldj), float("nan"), dtype=torch.float64, device="cuda") for _ in which]
        Gd, Td = [dev(host[q][0]) for q in which], [dev(t) for t in T]
        jacobian_multi(ndir, [(nets[q][0], jobs[q][2], Gd[k], Td[k], J[k].data_ptr()) for k, q in enumerate(which)],
                       nmax * ld, ld, sign, ldj)
        torch.cuda.synchronize()
        return J

    J = jacobians(range(len(jobs)))
    for q, (n_in, _, n) in enumerate(jobs):
        mlp, layers, sub, mul = nets[q]
        G, T, _ = host[q]
        Jq = J[q].cpu().numpy()
        for i in range(n):
            for d in range(ndir):
                ref = _rows(layers, sub, mul, G[i, :n_in], T[d, i, :n_in], 0.0, sign)
                assert np.abs(Jq[i * ndir + d, :mlp.n_params] - ref).max() < 1e-12 * max(np.abs(ref).max(), 1.0)
        assert np.isnan(Jq[:, mlp.n_params:]).all() and np.isnan(Jq[n * ndir:]).all()
    for mode, tol in (("float64", 1e-12), ("bf16x3", 5e-4)):
        f64 = mode == "float64"
        dt = torch.float64 if f64 else torch.float32
        grads = [torch.full((m[0].n_params,), 0.5, dtype=torch.float64, device="cuda") for m in nets]
        args = [(nets[q][0], jobs[q][2], dev(host[q][0], dt), dev(host[q][1][0], dt), dev(host[q][2]), grads[q])
                for q in range(len(jobs))]
        if f64 and max(m[0].n_params for m in nets) > 5000:   # the sums of a network alone are beyond the LDS
            with pytest.raises(_lib.HipLibraryError, match="exceed the device limit"):
                train_grad_multi(MLP_MODES[mode], args, ld, _lib.PT_F64, sign)
            continue
        train_grad_multi(MLP_MODES[mode], args, ld, _lib.PT_F64 if f64 else _lib.PT_F32, sign)
        torch.cuda.synchronize()
        for q, (n_in, _, n) in enumerate(jobs):
            mlp, layers, sub, mul = nets[q]
            G, T, gy = host[q]
            ref = np.full(mlp.n_params, 0.5) + sum((_rows(layers, sub, mul, G[i, :n_in], T[0, i, :n_in], gy[i], sign)
                                                    for i in range(n)), np.zeros(mlp.n_params))
            assert np.abs(grads[q].cpu().numpy() - ref).max() < tol * np.abs(ref).max()
