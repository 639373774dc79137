"""Matrices to the device and back in column blocks through two staging slots:
sizes of one, two, three and many blocks (4 MiB each), and the exported
array's life."""
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
