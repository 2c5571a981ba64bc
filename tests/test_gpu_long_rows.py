"""Rows so far apart that byte offsets within a tile of rows pass 32 bits: the same values as for the
same features in short rows, bit for bit (one order of the products either way)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (rows, leading dimension): a 64-row tile passes 4 GiB from ld = 8.5e6 doubles on, a 128-row one
# from 4.2e6 on
SMALL, LARGE = (70, 8_600_000), (130, 4_300_000)


def _rows(n, ld, d, seed=0):
    """(n, ld) rows with random values in the first d features, and the same in short rows."""
    import torch

    X = torch.zeros((n, ld), dtype=torch.float64, device="cuda")
    X[:, :d] = torch.from_numpy(np.random.default_rng(seed).random((n, d))).cuda()
    return X, X[:, :48].contiguous()


@pytest.mark.parametrize("d", [5, 37, 48])
@pytest.mark.parametrize("op", ["linear", "gaussian", "predict"])
def test_tiles_of_64_rows(op, d):
    import torch

    from qml_amd import _lib
    from qml_amd.kernels import gaussian_mfma_device, row_sqnorms_device

    n, ld = SMALL
    X, S = _rows(n, ld, d)
    got = []
    for Y in (X, S):
        L = _lib.lib()
        nr = row_sqnorms_device(Y, n, d)
        if op == "gaussian":
            got.append(gaussian_mfma_device(Y, nr, n, Y, nr, n, d, 2.0, True))
            continue
        K = torch.zeros((n, n) if op == "linear" else (n,), dtype=torch.float64, device="cuda")
        if op == "linear":
            _lib.check(L.qmlh_linear_mfma(Y.data_ptr(), n, Y.shape[1], Y.data_ptr(), n, Y.shape[1],
                                          d, K.data_ptr(), n, 0, None))
        else:
            a = torch.arange(n, dtype=torch.float64, device="cuda")
            ws = torch.empty(L.qmlh_predict_workspace(n, n) // 8, dtype=torch.float64,
                             device="cuda")
            _lib.check(L.qmlh_krr_predict(
                _lib.PAIR_GAUSSIAN, Y.data_ptr(), n, Y.shape[1], nr.data_ptr(), Y.data_ptr(), n,
                Y.shape[1], nr.data_ptr(), a.data_ptr(), d, 2.0, K.data_ptr(), ws.data_ptr(),
                ws.numel() * 8, None))
        got.append(K)
    assert bool(torch.isfinite(got[1]).all()) and bool((got[0] == got[1]).all())


@pytest.mark.parametrize("d", [5, 37])
@pytest.mark.parametrize("op", ["deflated", "sweep"])
def test_tiles_of_128_rows(op, d):
    import torch

    from qml_amd import _lib
    from qml_amd.kernels import row_sqnorms_device
    from qml_amd.sweep import BatchedFit, SweepProblem

    n, ld = LARGE
    X, S = _rows(n, ld, d)
    y = torch.arange(n, dtype=torch.float64, device="cuda")
    got = []
    for Y in (X, S):
        if op == "sweep":
            fit = BatchedFit([SweepProblem(n, 2.0, 1e-3, "gaussian")], Y, d, y, nb=64, branches=1)
            got.append(fit.run().alpha.clone())
            continue
        nr = row_sqnorms_device(Y, n, d)
        K = torch.zeros((n, n), dtype=torch.float64, device="cuda")
        B = torch.zeros((n, n), dtype=torch.float32, device="cuda")
        u = torch.zeros(n, dtype=torch.float64, device="cuda")
        _lib.check(_lib.lib().qmlh_gaussian_deflated(
            Y.data_ptr(), n, Y.shape[1], nr.data_ptr(), d, 2.0, 1e-3, 0.0, K.data_ptr(), n,
            B.data_ptr(), n, None, n, u.data_ptr(), None))
        got.append(torch.cat([torch.tril(K.t()).flatten(), torch.tril(B.t()).double().flatten()]))
    assert bool(torch.isfinite(got[1]).all()) and bool((got[0] == got[1]).all())


@pytest.mark.parametrize("d", [5, 37])
def test_local_kernels_of_4_gib_and_more(d):
    """A set of 4 GiB stays in its own order; its first molecule alone fills more than a tile."""
    import torch

    from qml_amd import _lib
    from qml_amd.kernels import LocalSet, local_kernels_device

    counts = np.array([128, 1, 1])
    X, S = _rows(LARGE[0], LARGE[1], d)
    long, short = LocalSet(X, counts), LocalSet(S, counts)
    assert long.order_d is None
    long.d = short.d = d
    short.order_d = None
    got = [local_kernels_device(_lib.PAIR_GAUSSIAN, s, s, [2.0], True, expanded=True)
           for s in (long, short)]
    assert bool(torch.isfinite(got[1]).all()) and bool((got[0] == got[1]).all())
