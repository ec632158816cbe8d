"""One workspace, made for more observations, serving updates of different observation counts
in turn, as KalmanFilter uses it: an energy update (m = 1) and force updates in both forms, the
workspace starting as NaN.  Against the oracle's explicit-inverse update; tolerance as for a
single update of this conditioning: P is 50 I + B B^T and r >= 0.01, so the inverse's rounding
stays below about 2e-8 of a correction below 1 % of P, and three updates add up: 6e-10 of the
largest entry."""

import numpy as np
import pytest

from oracle import kalman as okf

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n_w,ms", [(65, (1, 40, 130)), (400, (390, 1, 70)), (130, (300, 129, 1))])
def test_one_workspace_for_all_observation_counts(n_w, ms):
    from pantea_amd import _lib

    lib = _lib.load()
    rng = np.random.default_rng(n_w)
    st = okf.FilterState(rng.normal(size=n_w), kalman_type=1)
    B = rng.normal(size=(n_w, n_w)) * 0.02
    st.P = np.eye(n_w) * 50.0 + B @ B.T
    P_d = torch.as_tensor(st.P.T.copy(), device="cuda")
    W_d = torch.as_tensor(st.W[:, 0].copy(), device="cuda")
    size = lib.pt_kalman_workspace_bytes(n_w, 2 * max(ms) + 1000)
    ws = torch.full((size // 8,), float("nan"), dtype=torch.float64, device="cuda")
    info = torch.full((1,), -1, dtype=torch.int32, device="cuda")
    for m in ms:
        H = rng.normal(size=(n_w, m)) * 0.02
        xi = rng.normal(size=m)
        H_d = torch.as_tensor(H.T.copy(), device="cuda")
        x_d = torch.as_tensor(xi, device="cuda")
        r, c, q = st.lambda0, 1.0 / st.lambda0, st.q
        okf.ekf_update(st, xi, H)
        _lib.check(lib.pt_kalman_update(n_w, m, P_d.data_ptr(), H_d.data_ptr(), n_w, x_d.data_ptr(), W_d.data_ptr(),
                                        r, c, q, ws.data_ptr(), ws.numel() * 8, info.data_ptr(), _lib.stream_ptr()),
                   "pt_kalman_update")
        torch.cuda.synchronize()
        assert int(info.item()) == 0
        np.testing.assert_allclose(P_d.cpu().numpy().T, st.P, rtol=0, atol=6e-10 * np.abs(st.P).max())
        dW = st.W[:, 0] - W_d.cpu().numpy()
        assert np.abs(dW).max() <= 6e-10 * max(np.abs(st.W[:, 0]).max(), 1.0)
