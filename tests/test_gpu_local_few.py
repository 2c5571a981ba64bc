"""The order in which local kernels take the molecules: their own unless an order by size has fewer
panel pairs or skips enough trailing zeros; the same bits as the call without an order."""

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
    order, panels = _local_orders(S, S, True, True)[0]
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


def _padded(counts, d, dense):
    """Rows as an atomic Coulomb matrix pads them, or without zeros."""
    import torch

    X = torch.zeros((int(counts.sum()), d), dtype=torch.float64, device="cuda")
    for r, n in zip(np.cumsum(counts) - counts, counts):
        X[r:r + n, :d if dense else min(d, n * (n + 1) // 2)] = 1.0
    return X


@pytest.mark.parametrize("product", [True, False])
@pytest.mark.parametrize("d,dense,by_size", [(276, False, True), (276, True, False),
                                             (64, False, False), (64, True, False)])
def test_order_where_it_pays(product, d, dense, by_size):
    """More than LOCAL_COUNT_PAIRS panel pairs: by size where long rows are mostly padding."""
    from qml_amd import _lib
    from qml_amd.kernels import LocalSet, _local_orders

    counts = np.random.default_rng([600, 23]).integers(5, 24, size=600)
    S = LocalSet(_padded(counts, d, dense), counts)
    assert S.npanels * (S.npanels + 1) // 2 > _lib.LOCAL_COUNT_PAIRS
    assert (_local_orders(S, S, True, product)[0][0] is not None) == by_size
    few = LocalSet(S.X[:int(counts[:100].sum())], counts[:100])
    assert (_local_orders(S, few, False, product)[1][0] is not None) == by_size


def test_order_by_size_of_fewer_panels():
    from qml_amd.kernels import LocalSet, _local_orders

    counts = np.array([120, 20] * 20)
    S = LocalSet(_padded(counts, 16, True), counts)
    assert S.own_panels.size > S.panels.size
    assert _local_orders(S, S, True, True)[0][0] is S.order_d
