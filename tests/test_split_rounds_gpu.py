"""FP16 / BF16 hi+lo products whose last round of 128 x 128 tiles is cut into
quarters (528 tiles: 512 whole and 16 cut) and whose only round is not (171):
the same bounds as the smaller sizes, which are cut throughout."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def P():
    import progress_amd
    progress_amd.set_precision(progress_amd.PREC_FP64)
    return progress_amd


@pytest.mark.parametrize("n", [2300, 4000])
def test_bf16_product(P, n):
    """lo lo dropped, lo rounded, FP32 sums: |error| <= (3 * 2^-16 + n 2^-24)
    (|A| |B|) entrywise."""
    import torch
    ld = P.padded_ld(n)
    gen = torch.Generator(device="cuda").manual_seed(n)
    a = torch.zeros((ld, ld), dtype=torch.float64, device="cuda")
    x = torch.randn((n, n), dtype=torch.float64, device="cuda", generator=gen) / n ** 0.5
    a[:n, :n] = 0.5 * (x + x.T)
    b = a @ a + 0.5 * a
    b = 0.5 * (b + b.T)
    c = torch.full_like(a, 7.0)
    torch.cuda.synchronize()
    P.set_product_precision(P.PREC_BF16SPLIT)
    try:
        P.symmetric_product_device(a, b, c, n)
    finally:
        P.set_product_precision(P.PREC_FP64)
    bound = (3 * 2.0 ** -16 + n * 2.0 ** -24) * (a.abs() @ b.abs())
    assert bool(((c - a @ b).abs() <= torch.maximum(bound, bound.T)).all())
    assert torch.equal(c, c.T)


@pytest.mark.parametrize("prec,bits", [("PREC_F16SPLIT", 11), ("PREC_BF16SPLIT", 8)])
@pytest.mark.parametrize("n", [2300, 4000])
def test_split_sp2_of_a_gapped_hamiltonian(P, n, prec, bits):
    """H = Q diag(e) Q with the reflection Q = I - 2 v v^T: the density
    2 Q diag(e < 0) Q is known without an eigensolver."""
    import torch
    rng = np.random.default_rng(n)
    v = rng.standard_normal(n)
    v /= np.linalg.norm(v)
    e = np.concatenate([rng.uniform(-3, -1, n // 2), rng.uniform(1, 3, n - n // 2)])
    vt, et = torch.from_numpy(v).cuda(), torch.from_numpy(e).cuda()

    def conjugate(d):
        """Q diag(d) Q."""
        dv = d * vt
        m = torch.diag(d) - 2 * torch.outer(vt, dv) - 2 * torch.outer(dv, vt)
        return m + 4 * (vt @ dv) * torch.outer(vt, vt)

    ld = P.padded_ld(n)
    h = torch.zeros((ld, ld), dtype=torch.float64, device="cuda")
    h[:n, :n] = conjugate(et)
    h = 0.5 * (h + h.T)
    rho = torch.zeros_like(h)
    torch.cuda.synchronize()
    P.sp2_alg2_device(h, rho, n, (n // 2) / n, 1, 100, "Abs", 1e-10, precision=getattr(P, prec))
    d = rho[:n, :n]
    ref = 2 * conjugate((et < 0).double())
    # a few steps' rounding, n entries per row
    assert float((d - ref).norm()) <= 16 * n * (2.0 ** (-2 * bits) + 2.0 ** -24)
    assert torch.equal(d, d.T)
