"""Full FP64 products (operands that are not symmetric) at sizes that take the
staged 128-wide tiles (leading dimensions 2048, 2816 and 3968) and at their
neighbours that do not: products, two-product sums with an input term, the
partial sums and <C, E>.

Each entry of a product is a sum of n terms in another order: it may differ by
n eps (|A| |B|) from another correct one (twice that is allowed)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


@pytest.fixture(scope="module")
def P():
    import progress_amd
    progress_amd.set_precision(progress_amd.PREC_FP64)
    return progress_amd


def _random(n, seed, scale=1.0):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    return scale * torch.randn((n, n), dtype=torch.float64, device="cuda", generator=g)


def _padded(P, x):
    import torch
    n = x.shape[0]
    out = torch.zeros((P.padded_ld(n),) * 2, dtype=torch.float64, device="cuda")
    out[:n, :n] = x
    return out


@pytest.mark.parametrize("n", [1930, 2048, 2700, 2816, 2817, 3841])
def test_congruences(P, n):
    """Z^T A Z and Z A Z^T of matrices without any symmetry."""
    print(f"[full products] n={n}", flush=True)
    import torch
    a, z = _random(n, n), _random(n, n + 1)
    ma, mz = P.Matrix.from_numpy(a.cpu().numpy()), P.Matrix.from_numpy(z.cpu().numpy())
    out = P.Matrix.zeros(n)
    for call, x, y in ((P.lib().prg_orthogonalize, z.T, z), (P.lib().prg_deorthogonalize, z, z.T)):
        call(ma.h, mz.h, out.h, 0.0, b"dense", 0)
        got = torch.from_numpy(out.numpy().copy(order="C")).cuda()
        bound = 4 * n * EPS * (x.abs() @ (a.abs() @ y.abs()))
        assert bool(((got - x @ (a @ y)).abs() <= bound).all())
    for m in (ma, mz, out):
        m.close()


@pytest.mark.parametrize("n", [2050, 2700])
def test_two_products_and_an_input_term(P, n):
    """The SP2 adjoint of a cotangent that is not symmetric: S = X G + G X, and
    2 G - S, the input term, where the branch is 2 X - X^2."""
    print(f"[full products] adjoint n={n}", flush=True)
    import torch
    h = _random(n, n, 1.0 / n ** 0.5)
    h = 0.5 * (h + h.T)
    gout = _random(n, n + 1)
    lo, hi, pp = -3.0, 3.0, [1, 0, 1]
    grad = _padded(P, torch.zeros_like(h))
    # the library's matrices are column major: it sees the transposes
    P.sp2_adjoint_device(_padded(P, h), _padded(P, gout.T), grad, n, pp, lo, hi, 2)
    xs = [(hi * torch.eye(n, dtype=torch.float64, device="cuda") - h) / (hi - lo)]
    for s in pp:
        x = xs[-1]
        xs.append(x @ x if s else 2 * x - x @ x)
    g = 2 * gout
    for k in (2, 1, 0):
        s = xs[k] @ g + g @ xs[k]
        g = s if pp[k] else 2 * g - s
    ref = -g / (hi - lo)
    got = grad[:n, :n].T
    # ||X|| <= 1: a step at most doubles (square) or quadruples the norm, and
    # adds 2 n eps of it
    assert float((got - ref).norm()) <= 2 * 3 * 2 * n * EPS * float(ref.norm() + 8 * gout.norm())


def test_sums_and_elementwise_product(P, n=2700):
    """PCG (a residual's norm decides the stop, B - A X has an input term) and
    the canonical gradient (<P P, A>), which is that of A - kappa I."""
    print(f"[full products] sums n={n}", flush=True)
    import torch
    eye = torch.eye(n, dtype=torch.float64, device="cuda")
    h = _random(n, n, 1.0 / n ** 0.5)
    h = 0.5 * (h + h.T)
    m = (eye + 0.2 * h).cpu().numpy()
    x = torch.from_numpy(np.ascontiguousarray(P.pcg(m, np.eye(n), np.eye(n), 1e-10)[0])).cuda()
    assert float((eye - torch.from_numpy(m).cuda() @ x).norm()) <= 2e-5  # its square <= 1e-10
    a = _random(n, 7)
    a = 0.5 * (a + a.T)
    levels, beta = 6, 5.0
    g1, g2, p = (_padded(P, torch.zeros_like(h)) for _ in range(3))
    P.implicit_fermi_adjoint_device(_padded(P, h), _padded(P, a), g1, n, levels, 0.1, beta, 1e-10,
                                    canonical=True, dP=p)
    d = p[:n, :n]
    w = beta * (d - d @ d)
    kappa = float((w * a).sum() / w.diagonal().sum())
    P.implicit_fermi_adjoint_device(_padded(P, h), _padded(P, a - kappa * eye), g2, n, levels, 0.1,
                                    beta, 1e-10)
    assert float((g1 - g2).norm()) <= 1e-10 * float(g2.norm())
