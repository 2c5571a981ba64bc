"""Local kernels of enough molecules that the panels' trailing zero features are counted and skipped
(more than 512 panel pairs), against the molecules' own order and all features."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LINE = 512  # panel pairs up to which the features are not counted


def _rows(counts, d, ld, seed):
    """Rows of each molecule: nonzero up to a length that grows with its size (all features from 23
    atoms), then zeros."""
    rng = np.random.default_rng(seed)
    X = np.zeros((int(np.sum(counts)), ld))
    r = 0
    for n in counts:
        length = d if n >= 23 else min(d, 1 + 3 * int(n))
        X[r:r + n, :length] = rng.random((n, length)) * 5
        r += n
    return X


def _plain(kind, SA, SB, sig, symmetric, expanded):
    """qmlh_local_kernels on panels of the molecules in their own order."""
    import torch

    from qml_amd import _lib
    from qml_amd.kernels import local_panels

    pa = torch.from_numpy(local_panels(SA.offsets)).cuda()
    pb = pa if symmetric else torch.from_numpy(local_panels(SB.offsets)).cuda()
    K = torch.full((sig.size, SB.nmol, SA.nmol), np.nan, dtype=torch.float64, device="cuda")
    _lib.check(_lib.lib().qmlh_local_kernels(
        kind, SA.X.data_ptr(), SA.atoms, SA.X.shape[1],
        SA.norms().data_ptr() if expanded else None, SA.offsets_d.data_ptr(), pa.data_ptr(),
        pa.numel() - 1, SB.X.data_ptr(), SB.atoms, SB.X.shape[1],
        SB.norms().data_ptr() if expanded else None, SB.offsets_d.data_ptr(), pb.data_ptr(),
        pb.numel() - 1, SA.d, sig.ctypes.data, sig.size, K.data_ptr(), SA.nmol,
        SA.nmol * SB.nmol, _lib.SYMMETRIC if symmetric else 0, None))
    return K


FORMS = [("gaussian", True), ("gaussian", False), ("laplacian", False)]


def _check(kind, expanded, A, B, symmetric):
    from qml_amd import _lib
    from qml_amd.kernels import _local_orders, local_kernels_device

    pairs = A.npanels * (A.npanels + 1) // 2 if symmetric else A.npanels * B.npanels
    assert pairs > LINE
    assert _local_orders(A, B, symmetric, expanded)[0][0] is not None  # and so the features counted
    k = _lib.PAIR_GAUSSIAN if kind == "gaussian" else _lib.PAIR_LAPLACIAN
    sig = np.array([6.0, 20.0])
    got = local_kernels_device(k, A, B, sig, symmetric, expanded=expanded)
    ref = _plain(k, A, B, sig, symmetric, expanded)
    # positive terms added in another order: at most 23 x 23 of them, by blocks; the rounding of a
    # distance is the same in both, skipped features being exact zeros
    ok = ~(ref.isnan() | got.isnan())
    assert bool(((got - ref).abs() <= 1e-13 * ref)[ok].all())
    return got, ref


@pytest.mark.parametrize("kind,expanded", FORMS)
@pytest.mark.parametrize("symmetric", [True, False])
@pytest.mark.parametrize("d,ld", [(139, 144), (128, 128), (129, 144)])
def test_skipped_features(kind, expanded, symmetric, d, ld):
    import torch

    from qml_amd.kernels import LocalSet

    rng = np.random.default_rng(d)
    na = np.concatenate([rng.integers(1, 24, size=598), [0, 130]])
    nb = np.concatenate([[0], rng.integers(1, 24, size=300)])
    A = LocalSet(torch.from_numpy(_rows(na, d, ld, 1)).cuda(), na)
    B = A if symmetric else LocalSet(torch.from_numpy(_rows(nb, d, ld, 2)).cuda(), nb)
    got, ref = _check(kind, expanded, A, B, symmetric)
    assert not bool(got.isnan().any()) and not bool(ref.isnan().any())


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("kind,expanded", FORMS)
@pytest.mark.parametrize("symmetric", [True, False])
def test_values_that_are_not_finite(kind, expanded, symmetric, value):
    """In a long molecule's last feature, which most panels it is paired with do not have. By
    products the distances are not finite either, and count as zero, whichever features are taken;
    by differences an infinite one adds nothing, and NaN reaches the molecules of its panel."""
    import torch

    from qml_amd.kernels import LocalSet

    d, ld, mol = 139, 144, 17
    na = np.random.default_rng(3).integers(1, 24, size=600)
    na[mol] = 23
    X = _rows(na, d, ld, 1)
    X[np.concatenate([[0], np.cumsum(na)])[mol] + 4, d - 1] = value
    A = LocalSet(torch.from_numpy(X).cuda(), na)
    nb = np.random.default_rng(4).integers(1, 24, size=300)
    B = A if symmetric else LocalSet(torch.from_numpy(_rows(nb, d, ld, 2)).cuda(), nb)
    for K in _check(kind, expanded, A, B, symmetric):
        if expanded or (value == value and not symmetric):
            assert not bool(K.isnan().any())
        elif value != value:
            assert bool(K[:, :, mol].isnan().all())
            assert int(K.isnan().any(0).sum()) < K[0].numel() // 4  # not the whole matrix
