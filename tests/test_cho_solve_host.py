"""cho_solve leaves the caller's matrix alone until the device's work is known to have ended."""

import numpy as np
import pytest


class Lost(RuntimeError):
    pass


@pytest.mark.parametrize("where", ["solution", "info"])
def test_matrix_untouched_when_the_wait_fails(monkeypatch, where):
    import torch

    import qml_amd.math as qmath

    class Info:
        def item(self):
            raise Lost

    def potrs(Ad, n, xd, *a, **k):
        if where == "solution":
            raise Lost

    monkeypatch.setattr(qmath, "device", lambda: torch.device("cpu"))
    monkeypatch.setattr(qmath, "potrf_device", lambda *a, **k: Info())
    monkeypatch.setattr(qmath, "potrs_device", potrs)
    A = np.arange(25.0).reshape(5, 5)
    before = A.copy()
    with pytest.raises(Lost):
        qmath.cho_solve(A, np.ones(5))
    assert np.array_equal(A, before)
