"""The FP16 / BF16 hi+lo tiles (LDS-DMA slabs, blocked planes) at one, two and
more tiles, and at sizes that are no multiple of anything: products against
float64, and SP2 steps whose result must be exactly symmetric.

A product drops lo lo (2^-2b relative, b the bits of the 16-bit format: 8 or
11), rounds lo to b bits (2^-2b again, for each operand) and adds in FP32:
|error| <= (3 * 2^-2b + n 2^-24) (|A| |B|) entrywise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def P():
    import progress_amd
    progress_amd.set_precision(progress_amd.PREC_FP64)
    return progress_amd


@pytest.mark.parametrize("n", [1, 31, 65, 128, 130, 257, 500, 1100])
def test_bf16_product(P, n):
    import torch
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, n)) / np.sqrt(n)
    a = 0.5 * (x + x.T)
    b = a @ a + 0.5 * a
    b = 0.5 * (b + b.T)
    ld = P.padded_ld(n)
    pad = torch.zeros((3, ld, ld), dtype=torch.float64, device="cuda")
    pad[0, :n, :n] = torch.from_numpy(a)
    pad[1, :n, :n] = torch.from_numpy(b)
    pad[2] = 7.0
    torch.cuda.synchronize()
    P.set_product_precision(P.PREC_BF16SPLIT)
    try:
        P.symmetric_product_device(pad[0], pad[1], pad[2], n)
    finally:
        P.set_product_precision(P.PREC_FP64)
    c = pad[2].cpu().numpy()
    bound = (3 * 2.0 ** -16 + n * 2.0 ** -24) * (np.abs(a) @ np.abs(b)) + 1e-300
    assert np.all(np.abs(c[:n, :n] - a @ b) <= np.maximum(bound, bound.T))
    assert np.array_equal(c, c.T)
    assert not c[n:].any() and not c[:, n:].any()


@pytest.mark.parametrize("prec,bits", [("PREC_F16SPLIT", 11), ("PREC_BF16SPLIT", 8)])
@pytest.mark.parametrize("n", [40, 128, 300, 650])
def test_split_sp2_of_a_gapped_hamiltonian(P, n, prec, bits):
    """A gap of half the spectrum does not amplify the products' rounding: the
    density is within the error of a step, and it is symmetric to the bit."""
    import torch
    rng = np.random.default_rng(n)
    q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    e = np.concatenate([rng.uniform(-3, -1, n // 2), rng.uniform(1, 3, n - n // 2)])
    h = (q * e) @ q.T
    ld = P.padded_ld(n)
    dh = torch.zeros((ld, ld), dtype=torch.float64, device="cuda")
    dh[:n, :n] = torch.from_numpy(0.5 * (h + h.T))
    rho = torch.zeros_like(dh)
    P.sp2_alg2_device(dh, rho, n, (n // 2) / n, 1, 100, "Abs", 1e-10, precision=getattr(P, prec))
    d = rho[:n, :n].cpu().numpy()
    c = q[:, :n // 2]
    # a few steps' rounding, n entries per row
    assert np.linalg.norm(d - 2 * c @ c.T) <= 16 * n * (2.0 ** (-2 * bits) + 2.0 ** -24)
    assert np.array_equal(d, d.T)
