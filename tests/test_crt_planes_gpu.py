"""int8 CRT products whose residue planes come from the upper triangle's blocks:
sizes of one block, of blocks that overhang the 256-wide padding and of many
blocks, for moduli counts on both sides of the shortcut residues (12) and at
the ends of the range, against the oracle's exact arithmetic."""
import numpy as np
import pytest

import progress_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def P():
    import progress_amd
    return progress_amd


@pytest.mark.parametrize("moduli", [6, 11, 12, 13, 14])
@pytest.mark.parametrize("n", [1, 63, 64, 129, 300, 520])
def test_product_equals_the_oracle(P, n, moduli):
    import torch
    rng = np.random.default_rng(1000 * moduli + n)
    x = rng.standard_normal((n, n)) / np.sqrt(n)
    a = 0.5 * (x + x.T)
    b = a @ a - 0.7 * a
    b = 0.5 * (b + b.T)
    ld = P.padded_ld(n)
    pad = torch.zeros((3, ld, ld), dtype=torch.float64, device="cuda")
    pad[0, :n, :n] = torch.from_numpy(a)
    pad[1, :n, :n] = torch.from_numpy(b)
    pad[2] = 7.0
    torch.cuda.synchronize()
    P.set_product_precision(P.PREC_INT8CRT)
    P.set_int8_moduli(moduli)
    try:
        P.symmetric_product_device(pad[0], pad[1], pad[2], n)
    finally:
        P.set_int8_moduli(11)
        P.set_product_precision(P.PREC_FP64)
    c = pad[2].cpu().numpy()
    ref = O.crt_product(a, b, moduli)
    # the fraction sum's rounding: moduli terms of up to 1/2, scaled by the
    # range M s_A s_B / 2^2a (at most 4 times what the norms need, 72 at 14)
    na, nb = np.sqrt((a * a).sum(0)).max(), np.sqrt((b * b).sum(0)).max()
    tol = 4 * moduli * np.finfo(float).eps * 72 * 16 * na * nb
    assert np.max(np.abs(c[:n, :n] - ref)) <= tol
    assert np.array_equal(c, c.T)
    assert not c[n:].any() and not c[:, n:].any()


@pytest.mark.parametrize("moduli", [13, 14])
@pytest.mark.parametrize("n", [1025, 1500, 1900, 2200])
def test_shared_blocks_of_larger_matrices(P, n, moduli):
    """The moduli of a block over 5, 4, 2 and 1 workgroups, against float64
    (n eps of the norms): the fraction sum's rounding as above, and the
    operands' of 2^-(a + 1) of a scale of at most twice their norm."""
    import torch
    print(f"[crt planes] n={n} moduli={moduli}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn((n, n), dtype=torch.float64, device="cuda", generator=g) / n ** 0.5
    a = 0.5 * (x + x.T)
    b = a @ a - 0.7 * a
    b = 0.5 * (b + b.T)
    ld = P.padded_ld(n)
    pad = torch.zeros((3, ld, ld), dtype=torch.float64, device="cuda")
    pad[0, :n, :n], pad[1, :n, :n], pad[2] = a, b, 7.0
    torch.cuda.synchronize()
    P.set_product_precision(P.PREC_INT8CRT)
    P.set_int8_moduli(moduli)
    try:
        P.symmetric_product_device(pad[0], pad[1], pad[2], n)
    finally:
        P.set_int8_moduli(11)
        P.set_product_precision(P.PREC_FP64)
    c = pad[2]
    scale_bits = O.crt_constants(moduli, square=False)[2]
    eps = np.finfo(float).eps
    rounding = n * eps + 4 * moduli * eps * 72 * 16 + 4 * n ** 0.5 * 2.0 ** -scale_bits
    bound = rounding * float(a.norm(dim=0).max() * b.norm(dim=0).max())
    assert float((c[:n, :n] - a @ b).abs().max()) <= bound
    assert torch.equal(c, c.T)
    assert not bool(c[n:].any()) and not bool(c[:, n:].any())
