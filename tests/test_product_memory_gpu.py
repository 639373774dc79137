"""Device memory of the iterative solvers' mixed-precision products: the planes
of three operands at most, however many of them are held."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def P():
    import progress_amd
    progress_amd.set_precision(progress_amd.PREC_FP64)
    return progress_amd


@pytest.mark.parametrize("prec,tol,plane_bytes,product_bytes",
                         [("PREC_INT8CRT", 1e-9, 12, 36 * 12 * 256 * 256),
                          ("PREC_BF16SPLIT", 3e-2, 4, 0)])
def test_plane_sets_of_an_implicit_fermi_solve(P, prec, tol, plane_bytes, product_bytes, n=2048,
                                               levels=2):
    import torch
    print(f"[product memory] {prec}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn((n, n), dtype=torch.float64, device="cuda", generator=g) / n ** 0.5
    h, p = 0.5 * (x + x.T), torch.zeros_like(x)
    P.lib().prg_progress_shutdown()  # gives the kept workspaces back
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    P.set_product_precision(getattr(P, prec))
    P.set_int8_moduli(12)
    try:
        P.implicit_fermi_device(h, p, n, levels, 0.0, 5.0, tol)
    finally:
        P.set_product_precision(P.PREC_FP64)
        P.set_int8_moduli(11)
    used = before - torch.cuda.mem_get_info()[0]
    # levels + 1 iterates, as many inverses less one, P^2, Y, its inverse, I,
    # Newton-Schulz's three and CG's three; 2 MiB of rounding each and 16 for
    # sums and tables
    matrices = 2 * levels + 1 + 10
    sets = 3 * plane_bytes * n * n
    assert used <= matrices * (8 * n * n + (2 << 20)) + sets + product_bytes + (24 << 20)
    assert bool(torch.isfinite(p).all())
