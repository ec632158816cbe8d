"""pt_kalman_update where its products are split over K (K of at least 384 and too few tiles
to fill the chip): both forms, parts of unequal length, a K remainder, a workspace made for
more observations.  Against the oracle's explicit-inverse update.  Tolerance: P is
50 I + B B^T and r >= 0.01, so A's condition number stays below 1e5 and the inverse's rounding
below about 1e5 n eps = 2e-8 relative to the correction, which is below 1 % of P: 2e-10 of
the largest entry."""

import numpy as np
import pytest

from oracle import kalman as okf

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n_w,m", [(384, 65), (391, 130), (450, 1), (590, 70), (400, 800), (390, 391), (65, 700)])
def test_update_with_split_products(n_w, m):
    from pantea_amd import _lib

    lib = _lib.load()
    rng = np.random.default_rng(3 * n_w + m)
    st = okf.FilterState(rng.normal(size=n_w), kalman_type=1)
    B = rng.normal(size=(n_w, n_w)) * 0.02
    st.P = np.eye(n_w) * 50.0 + B @ B.T
    H = rng.normal(size=(n_w, m)) * 0.02
    xi = rng.normal(size=m)
    P_d = torch.as_tensor(st.P.T.copy(), device="cuda")
    W_d = torch.as_tensor(st.W[:, 0].copy(), device="cuda")
    H_d = torch.as_tensor(H.T.copy(), device="cuda")
    x_d = torch.as_tensor(xi, device="cuda")
    r, c, q = st.lambda0, 1.0 / st.lambda0, st.q
    okf.ekf_update(st, xi, H)
    # a workspace for more observations serves fewer; its content must not reach the result
    bytes_ = [lib.pt_kalman_workspace_bytes(n_w, k) for k in (m, m + 1, m + 64, 2 * m + 1000)]
    assert bytes_ == sorted(bytes_)
    ws = torch.full((bytes_[0] // 8,), float("nan"), dtype=torch.float64, device="cuda")
    info = torch.full((1,), -1, dtype=torch.int32, device="cuda")
    _lib.check(lib.pt_kalman_update(n_w, m, P_d.data_ptr(), H_d.data_ptr(), n_w, x_d.data_ptr(), W_d.data_ptr(),
                                    r, c, q, ws.data_ptr(), ws.numel() * 8, info.data_ptr(), _lib.stream_ptr()),
               "pt_kalman_update")
    torch.cuda.synchronize()
    assert int(info.item()) == 0
    P = P_d.cpu().numpy().T
    np.testing.assert_array_equal(P, P.T)
    np.testing.assert_allclose(P, st.P, rtol=0, atol=2e-10 * np.abs(st.P).max())
    dW = st.W[:, 0] - W_d.cpu().numpy()
    assert np.abs(dW).max() <= 2e-10 * max(np.abs(st.W[:, 0]).max(), 1.0)
