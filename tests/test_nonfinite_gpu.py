"""A Hamiltonian with one entry that is not finite is refused by the implicit
Fermi solvers, whichever triangle holds it and whatever their products read."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def P():
    import progress_amd
    progress_amd.set_precision(progress_amd.PREC_FP64)
    return progress_amd


@pytest.mark.parametrize("prec", ["PREC_FP64", "PREC_BF16SPLIT"])
@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("at", [(3, 90), (90, 3), (140, 131), (5, 5)])
def test_non_finite_hamiltonian_is_refused(P, at, value, prec, n=150):
    import torch
    print(f"[non-finite] {value} at {at}, {prec}", flush=True)
    x = np.random.default_rng(n).standard_normal((n, n)) / np.sqrt(n)
    h = 0.5 * (x + x.T)
    h[at] = value
    ld = P.padded_ld(n)
    d = torch.zeros((ld, ld), dtype=torch.float64, device="cuda")
    d[:n, :n] = torch.from_numpy(h)
    P.set_product_precision(getattr(P, prec))
    try:
        with pytest.raises(P.ProgressError, match="non-finite"):
            P.implicit_fermi_device(d, torch.zeros_like(d), n, 4, 0.0, 5.0, 3e-2)
        with pytest.raises(P.ProgressError, match="non-finite"):
            P.implicit_fermi(h, 4, 2, n / 2, 0.0, 5.0, 1, 10, 1e-4, 3e-2)
    finally:
        P.set_product_precision(P.PREC_FP64)
