"""Calls of so many rows that a launch of one workgroup for each few of them would pass 2^32 lanes,
which the runtime cuts short without an error."""

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [67_108_863, 67_108_865, 67_200_000])
def test_row_norms(n):
    import torch

    from qml_amd.kernels import row_sqnorms_device

    X = torch.full((n, 1), 3.0, dtype=torch.float64, device="cuda")
    assert bool((row_sqnorms_device(X, n, 1) == 9.0).all())


@pytest.mark.parametrize("kind", ["gaussian", "laplacian"])
def test_predictions(kind):
    """268.5 million queries against one training row."""
    import torch

    from qml_amd import _lib

    m, n = 268_500_000, 1
    L = _lib.lib()
    Q = torch.zeros((m, 4), dtype=torch.float64, device="cuda")
    zeros = torch.zeros(m, dtype=torch.float64, device="cuda")
    a = torch.full((n,), 2.0, dtype=torch.float64, device="cuda")
    y = torch.zeros(m, dtype=torch.float64, device="cuda")
    ws = torch.empty(L.qmlh_predict_workspace(m, n) // 8, dtype=torch.float64, device="cuda")
    _lib.check(L.qmlh_krr_predict(
        _lib.PAIR_GAUSSIAN if kind == "gaussian" else _lib.PAIR_LAPLACIAN, Q.data_ptr(), m, 4,
        zeros.data_ptr(), Q.data_ptr(), n, 4, zeros.data_ptr(), a.data_ptr(), 4, 2.0,
        y.data_ptr(), ws.data_ptr(), ws.numel() * 8, None))
    assert bool((y == 2.0).all())
