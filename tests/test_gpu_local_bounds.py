"""Local kernels read no row beyond the set's atoms, also where the offsets on the device do."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,expanded", [("gaussian", True), ("gaussian", False),
                                           ("laplacian", False)])
def test_offsets_beyond_the_rows(kind, expanded):
    import torch

    from qml_amd import _lib
    from qml_amd.kernels import local_panels, row_sqnorms_device

    d, ld, atoms = 20, 32, 10
    X = torch.zeros((16, ld), dtype=torch.float64, device="cuda")
    X[:, :d] = torch.from_numpy(np.random.default_rng(0).random((16, d))).cuda()
    norms = row_sqnorms_device(X, 16, d)
    k = _lib.PAIR_GAUSSIAN if kind == "gaussian" else _lib.PAIR_LAPLACIAN
    sig = np.array([2.0])
    got = []
    for offsets in ([0, 4, 9, 13, 16], [0, 4, 9, 10, 10]):  # the same ten rows
        off = np.array(offsets, dtype=np.int64)
        offs = torch.from_numpy(off).cuda()
        panels = torch.from_numpy(local_panels(off)).cuda()
        K = torch.zeros((4, 4), dtype=torch.float64, device="cuda")
        nr = norms.data_ptr() if expanded else None
        side = (X.data_ptr(), atoms, ld, nr, offs.data_ptr(), panels.data_ptr(),
                panels.numel() - 1)
        _lib.check(_lib.lib().qmlh_local_kernels(k, *side, *side, d, sig.ctypes.data, 1,
                                                 K.data_ptr(), 4, 16, 0, None))
        got.append(K)
    assert bool((got[0] == got[1]).all())
    assert bool((got[0][3] == 0).all()) and bool((got[0][:3, :3] > 0).all())
