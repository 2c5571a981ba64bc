"""Atomic Coulomb matrices where the largest molecule that the caller names is too small: every
molecule of up to 256 atoms is computed all the same."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _batch(natoms, seed=0):
    import torch

    rng = np.random.default_rng(seed)
    natoms = np.asarray(natoms)
    total = int(natoms.sum())
    offsets = np.concatenate([[0], np.cumsum(natoms)]).astype(np.int64)
    to = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    cmol = np.repeat(np.arange(natoms.size, dtype=np.int64), natoms)
    central = np.arange(total, dtype=np.int64) - offsets[cmol]
    return (to(rng.integers(1, 10, total).astype(np.float64)), to(rng.normal(0, 2.5, (total, 3))),
            to(offsets), to(central), to(cmol))


@pytest.mark.parametrize("sorting", ["distance", "row-norm"])
@pytest.mark.parametrize("cutoff,decay", [(1e6, -1), (4.0, 1.0)])
@pytest.mark.parametrize("hint", [-1, 0, 5, 31, 32])
def test_hint_below_the_largest_molecule(sorting, cutoff, decay, hint):
    from qml_amd.representations import generate_atomic_coulomb_matrices_device

    batch = _batch([5, 33, 1, 32, 31, 200, 0, 6])
    kw = dict(sorting=sorting, central_cutoff=cutoff, central_decay=decay)
    ref, ref_status = generate_atomic_coulomb_matrices_device(*batch, 200, **kw, max_atoms=256)
    out, status = generate_atomic_coulomb_matrices_device(*batch, 200, **kw, max_atoms=hint)
    assert int(ref_status) == 0 and int(status) == 0
    assert bool((out == ref).all()) and bool((out.abs().sum(1) > 0).all())


def test_status_of_both_kernels():
    """Too many atoms for the rows (1) below the hint and above it, an index out of range (4), a
    molecule of more than 256 atoms (2)."""
    from qml_amd.representations import generate_atomic_coulomb_matrices_device

    for natoms, size, bad, want in (([12, 40], 40, False, 0), ([12, 40], 12, False, 1),
                                    ([12, 5], 10, False, 1), ([12, 40], 40, True, 4),
                                    ([12, 300], 40, False, 2), ([12, 40, 300], 12, True, 7)):
        Z, R, O, central, cmol = _batch(natoms)
        if bad:
            central[3] = 12
            cmol[7] = len(natoms)
        got = [generate_atomic_coulomb_matrices_device(Z, R, O, central, cmol, size,
                                                       max_atoms=m) for m in (10, 256)]
        assert [int(s) for _, s in got] == [want, want]
        assert bool((got[0][0] == got[1][0]).all())


def test_status_keeps_the_first_kernels_word():
    """On a stream of the caller's own the second launch reads it after the call has returned."""
    import torch

    from qml_amd.representations import generate_atomic_coulomb_matrices_device

    batch = _batch([12, 40])
    status = generate_atomic_coulomb_matrices_device(*batch, 40, max_atoms=10)[1]
    assert status.shape == (1,) and status.dtype == torch.int32
    assert status.untyped_storage().nbytes() == 8


def test_rows_are_timed_once():
    """The launch that looks for rows left over counts none of its own: a call with a hint is one
    launch of its rows to the timers, as a call without."""
    from qml_amd import _lib
    from qml_amd.representations import generate_atomic_coulomb_matrices_device

    batch = _batch([5, 12, 23])
    for hint in (None, 23):
        _lib.timer_enable(True)
        generate_atomic_coulomb_matrices_device(*batch, 23, max_atoms=hint)
        _, launches, rows = _lib.timer_read("cm")
        _lib.timer_enable(False)
        assert (launches, rows) == (1, 40)
