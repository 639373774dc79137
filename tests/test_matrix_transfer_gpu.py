"""Matrices to the device and back in column blocks through two staging slots:
sizes of one, two, three and many blocks (4 MiB each), and the exported
array's life."""
import ctypes
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 700, 725, 1023, 1024, 1300, 2100])
def test_block_copies_round_trip(n):
    print(f"[matrix transfer] n={n}", flush=True)
    import progress_amd as P
    a = np.random.default_rng(n).standard_normal((n, n))
    m = P.Matrix.from_numpy(a)
    # (1/2 + c mu) I - c H with c = -1, mu = 1/2: H itself, now on the device only
    P.lib().prg_normalize_implicit_fermi(m.h, -1.0, 0.5)
    got = m.numpy()
    assert got.flags.f_contiguous and got.flags.writeable
    assert np.array_equal(got, a)
    got[0, 0] += 1.0  # the array is the caller's own
    assert np.array_equal(m.numpy(), a)
    m.close()
    column = got[:, -1]
    del got
    gc.collect()
    kept = [np.full((n, n), 7.0) for _ in range(2)]  # would take a freed buffer's place
    assert np.array_equal(column[1:], a[1:, -1]) and kept[0][0, 0] == 7.0


class Handle(ctypes.Structure):
    """Leading fields of the library's matrix handle."""
    _fields_ = [("N", ctypes.c_int), ("M", ctypes.c_int), ("type", ctypes.c_int),
                ("host", ctypes.c_void_p), ("dev", ctypes.c_void_p), ("ld", ctypes.c_int),
                ("host_valid", ctypes.c_bool), ("dev_valid", ctypes.c_bool)]


@pytest.mark.parametrize("n", [7, 300, 362, 363, 800])
def test_export_leaves_what_a_host_access_needs(n):
    """An export brings the handle's own copy up to date from the same
    download, except that of an output of 1 MiB or more that no host routine
    has touched; host routines and later exports see the same values."""
    print(f"[matrix export] n={n}", flush=True)
    import progress_amd as P
    a = np.random.default_rng(n).standard_normal((n, n))
    imported = P.Matrix.from_numpy(a)
    P.lib().prg_normalize_implicit_fermi(imported.h, -1.0, 0.5)  # H itself, on the device only
    output = P.Matrix.zeros(n)
    z = np.eye(n)
    mz = P.Matrix.from_numpy(z)
    P.lib().prg_orthogonalize(imported.h, mz.h, output.h, 0.0, b"dense", 0)  # I A I
    for m, kept in ((imported, True), (output, 8 * n * n < 1 << 20)):
        head = Handle.from_address(m.h.value)
        assert head.N == n and head.dev_valid and not head.host_valid
        assert np.array_equal(m.numpy(), a)
        assert head.host_valid == kept
        assert P.lib().bml_trace(m.h) == sum(float(a[i, i]) for i in range(n))
        assert head.host_valid
        assert np.array_equal(m.numpy(), a)
        m.close()
    mz.close()
