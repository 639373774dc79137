"""FP64 products at sizes that take the staged 128-wide tiles and at neighbours
that do not.  Operands that are not symmetric (leading dimensions 2048, 2816 and
3968): products, two-product sums with an input term, the partial sums and
<C, E>; symmetric ones (8064): products, SP2 steps and the response.

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


def test_symmetric_products_and_steps(P, n=8010):
    """A B + beta C + gamma I for commuting A, B through an adjoint (the two-product
    sum), the product itself, and replayed SP2 steps, whose results are
    symmetric to the bit."""
    print(f"[staged symmetric] n={n}", flush=True)
    import torch
    x = _random(n, n, 1.0 / n ** 0.5)
    h = 0.5 * (x + x.T)
    del x
    a, c = _padded(P, h), _padded(P, torch.zeros_like(h))
    c += 7.0
    torch.cuda.synchronize()
    P.gemm_counters(reset=True)
    P.symmetric_product_device(a, a, c, n)
    ld = P.padded_ld(n)
    assert ld == 8064 and P.gemm_counters(reset=True)[2] == 63 * 64 / 2 * 2.0 * 128 * 128 * 8032
    h2 = h @ h
    habs = h.abs()
    assert bool(((c[:n, :n] - h2).abs() <= 2 * n * EPS * (habs @ habs)).all())
    assert torch.equal(c, c.T) and not bool(c[n:].any())
    lo, hi, pp = -3.0, 3.0, [1, 0, 1]
    P.sp2_seq_device(a, c, n, pp, lo, hi)
    xs = [-h / (hi - lo)]
    xs[0].diagonal().add_(hi / (hi - lo))
    for s in pp:
        xs.append(xs[-1] @ xs[-1] if s else 2 * xs[-1] - xs[-1] @ xs[-1])
    # x <- x^2 or 2 x - x^2 keeps [0, 1]: a step adds at most n eps to an entry
    # and at most doubles what the steps before left
    assert float((c[:n, :n] - 2 * xs[-1]).abs().max()) <= 2 * 2 ** len(pp) * n * EPS
    assert torch.equal(c, c.T)
    gout = _random(n, n + 1)
    gout = 0.5 * (gout + gout.T)
    P.sp2_adjoint_device(a, _padded(P, gout), c, n, pp, lo, hi, 2)
    g = 2 * gout
    for k in (2, 1, 0):
        s = xs[k] @ g
        s = s + s.T
        g = s if pp[k] else 2 * g - s
    ref = -g / (hi - lo)
    assert float((c[:n, :n] - ref).norm()) <= 2 * 3 * 2 * n * EPS * float(ref.norm() + 8 * gout.norm())
    assert torch.equal(c, c.T)


def test_density_and_response(P, n=8010):
    """Both matrices of the response's steps, for H = Q diag(e) Q with the
    reflection Q = I - 2 v v^T, whose density and response are known."""
    print(f"[staged response] n={n}", flush=True)
    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    v = torch.randn(n, dtype=torch.float64, device="cuda", generator=g)
    v /= v.norm()
    u = torch.rand(n, dtype=torch.float64, device="cuda", generator=g)
    occ = torch.arange(n, device="cuda") < n // 2
    e = torch.where(occ, -3 + 2 * u, 1 + 2 * u)

    def conjugate(m):
        m = m - 2 * torch.outer(v, v @ m)
        return m - 2 * torch.outer(m @ v, v)

    h = conjugate(torch.diag(e))
    h = 0.5 * (h + h.T)
    h1 = _random(n, 5, 1.0 / n ** 0.5)
    h1 = 0.5 * (h1 + h1.T)
    rho, rsp = P.compute_response_sp2(h.cpu().numpy(), h1.cpu().numpy(), (n // 2) / n, 1, 100, "Abs",
                                      1e-10)
    f = occ.double()
    df, de = f[:, None] - f[None, :], e[:, None] - e[None, :]
    quotient = torch.where(df != 0, df / torch.where(de != 0, de, torch.ones_like(de)),
                           torch.zeros_like(de))
    ref = 2 * conjugate(conjugate(h1) * quotient)
    rho, rsp = torch.from_numpy(rho).cuda(), torch.from_numpy(rsp).cuda()
    assert float((rho - 2 * conjugate(torch.diag(f))).norm()) < 4e-9
    assert float((rsp - ref).norm()) < 1e-7 * float(ref.norm())
    assert torch.equal(rsp, rsp.T) and torch.equal(rho, rho.T)
