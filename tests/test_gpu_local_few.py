"""Local kernels of few molecules run in the molecules' own order where that has fewer panel pairs:
no round of workgroups more than without an order, and the same bits as the call without one."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nmol", [190, 200, 40])
@pytest.mark.parametrize("kind,expanded", [("gaussian", True), ("gaussian", False),
                                           ("laplacian", False)])
def test_own_order(nmol, kind, expanded):
    import torch

    from qml_amd import _lib
    from qml_amd.kernels import LocalSet, _local_orders, local_kernels_device, local_panels

    counts = np.random.default_rng([nmol, 23]).integers(5, 24, size=nmol)
    d, ld = 30, 32
    X = torch.zeros((int(counts.sum()), ld), dtype=torch.float64, device="cuda")
    X[:, :d] = torch.from_numpy(np.random.default_rng(0).random((X.shape[0], d))).cuda()
    S = LocalSet(X, counts)
    own = torch.from_numpy(local_panels(S.offsets)).cuda()
    order, panels = _local_orders(S, S, True)[0]
    assert order is None and bool((panels == own).all())
    k = _lib.PAIR_GAUSSIAN if kind == "gaussian" else _lib.PAIR_LAPLACIAN
    sig = np.array([2.0, 4.0])
    got = local_kernels_device(k, S, S, sig, True, expanded=expanded)
    ref = torch.zeros_like(got)
    nr = S.norms().data_ptr() if expanded else None
    side = (X.data_ptr(), S.atoms, ld, nr, S.offsets_d.data_ptr(), own.data_ptr(),
            own.numel() - 1)
    _lib.check(_lib.lib().qmlh_local_kernels(k, *side, *side, S.d, sig.ctypes.data, 2,
                                             ref.data_ptr(), nmol, nmol * nmol, _lib.SYMMETRIC,
                                             None))
    assert bool((got == ref).all())


def test_order_by_size_where_it_pays():
    """Above the line, and where the molecules' own order has more panels."""
    import torch

    from qml_amd import _lib
    from qml_amd.kernels import LocalSet, _local_orders

    for counts in (np.random.default_rng([600, 23]).integers(5, 24, size=600),
                   np.array([120, 20] * 20)):
        S = LocalSet(torch.zeros((int(counts.sum()), 16), dtype=torch.float64, device="cuda"),
                     counts)
        ordered = S.npanels * (S.npanels + 1) // 2
        assert ordered > _lib.LOCAL_COUNT_PAIRS or S.own_panels.size > S.panels.size
        assert _local_orders(S, S, True)[0][0] is S.order_d
