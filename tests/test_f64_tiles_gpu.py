"""The FP64 MFMA tiles (products and SP2 steps) at the sizes where their edges
and dispatch can go wrong: single chunks of K, sizes that are not multiples of
the tile, the last row pairs, and both sides of each change of the tile edge
(16, 32, 48) and of the bookkeeping (inside the step or in its own launch).

Products against numpy in float64: each entry is a sum of n terms in another
order, so it may differ by n eps sum_k |a_ik b_kj| (twice that is allowed)."""
import numpy as np
import pytest

import progress_oracle as O

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps

SIZES = [1, 2, 15, 17, 33, 47, 100, 129, 352, 385, 500, 640, 701, 1000, 1153, 1500, 2305]


@pytest.fixture(scope="module")
def P():
    import progress_amd
    progress_amd.set_precision(progress_amd.PREC_FP64)
    return progress_amd


@pytest.mark.parametrize("n", SIZES)
def test_symmetric_product(P, n):
    """A B for commuting symmetric A, B (polynomials of one matrix)."""
    import torch
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, n)) / np.sqrt(n)
    a = 0.5 * (x + x.T)
    b = a @ a + 0.3 * a
    b = 0.5 * (b + b.T)
    ld = P.padded_ld(n)
    pad = torch.zeros((3, ld, ld), dtype=torch.float64, device="cuda")
    pad[0, :n, :n] = torch.from_numpy(a)
    pad[1, :n, :n] = torch.from_numpy(b)
    pad[2] = 7.0  # the product overwrites all of it
    torch.cuda.synchronize()
    P.symmetric_product_device(pad[0], pad[1], pad[2], n)
    c = pad[2].cpu().numpy()
    bound = 2 * n * np.finfo(float).eps * (np.abs(a) @ np.abs(b)) + 1e-300
    # the lower triangle is the upper one mirrored: it may differ by the
    # asymmetry that b's own rounding leaves in the exact product
    exact = a @ b
    skew = np.abs(exact - exact.T)
    assert np.all(np.abs(c[:n, :n] - exact) <= bound + bound.T + skew)
    assert np.array_equal(c, c.T)
    assert not c[n:].any() and not c[:, n:].any()


@pytest.mark.parametrize("n", [17, 130, 500, 900, 1400])
def test_general_products(P, n):
    """Z^T A Z: products of operands that are not symmetric."""
    rng = np.random.default_rng(n)
    a, z = rng.standard_normal((n, n)), rng.standard_normal((n, n))
    out = P.orthogonalize(a, z)
    ref = z.T @ a @ z
    absref = np.abs(z.T) @ (np.abs(a) @ np.abs(z))
    assert np.all(np.abs(out - ref) <= 4 * n * np.finfo(float).eps * absref)


@pytest.mark.parametrize("n", [1, 2, 17, 48, 129, 352, 385, 639, 700, 1153, 1409, 2320])
def test_replayed_steps(P, n):
    """A replayed branch sequence equals the same steps in numpy: x <- x^2 or
    2x - x^2 keeps [0, 1], so each step adds at most n eps to an entry and at
    most doubles what the steps before left."""
    import torch
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, n)) / np.sqrt(n)
    h = 0.5 * (x + x.T)
    lo, hi = -3.0, 3.0
    pp = [1, 0, 0, 1, 1]
    ld = P.padded_ld(n)
    dh = torch.zeros((ld, ld), dtype=torch.float64, device="cuda")
    dh[:n, :n] = torch.from_numpy(h)
    rho = torch.zeros_like(dh)
    P.sp2_seq_device(dh, rho, n, pp, lo, hi)
    x = (hi * np.eye(n) - h) / (hi - lo)
    for s in pp:
        x = x @ x if s else 2 * x - x @ x
    r = rho[:n, :n].cpu().numpy()
    assert np.max(np.abs(r - 2 * x)) <= 2 * 2 ** len(pp) * n * np.finfo(float).eps
    assert np.array_equal(r, r.T)


@pytest.mark.parametrize("n", [30, 400, 1201])
def test_response_steps(P, n):
    """Density and response of a gapped Hamiltonian against the oracle's
    recursion (the same branches; the response is of order 1 / gap)."""
    rng = np.random.default_rng(n)
    q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    e = np.concatenate([rng.uniform(-3, -1, n // 2), rng.uniform(1, 3, n - n // 2)])
    h = (q * e) @ q.T
    h = 0.5 * (h + h.T)
    h1 = rng.standard_normal((n, n)) / np.sqrt(n)
    h1 = 0.5 * (h1 + h1.T)
    rho, rsp = P.compute_response_sp2(h, h1, (n // 2) / n, 1, 100, "Abs", 1e-10)
    c, v = q[:, :n // 2], q[:, n // 2:]
    # Rayleigh-Schroedinger: sum over occupied-virtual pairs
    u = (c.T @ h1 @ v) / (e[:n // 2, None] - e[None, n // 2:])
    ref = 2 * (c @ u @ v.T)
    ref = ref + ref.T
    assert np.linalg.norm(rho - 2 * c @ c.T) < 1e-9
    assert np.linalg.norm(rsp - ref) < 1e-7 * np.linalg.norm(ref)
    assert np.array_equal(rsp, rsp.T)


@pytest.mark.parametrize("thr,kind", [(0.0, None), (1e-3, "ELLPACK")])
@pytest.mark.parametrize("n", [2, 15, 16, 17, 33, 100, 127, 128])
def test_replayed_steps_of_a_matrix_without_symmetry(P, n, thr, kind):
    """Up to 128 rows a matrix need not be symmetric: its steps are those of the
    dense product (each at most doubles the error and adds 2 n eps of
    || |X|^2 ||), thresholded in the sparse formats."""
    rng = np.random.default_rng(n)
    h = rng.standard_normal((n, n)) / np.sqrt(n)
    pp = [1, 0, 0, 1]
    ppa, vv, ic = P._ivec(len(pp), pp), P._dvec(len(pp)), P._ivec(1, [len(pp)])
    got = P._h_rho(P.lib().prg_sp2_alg2_seq, h, thr, P._ip(ppa), P._ip(ic), P._dp(vv), 0,
                   matrix_type=getattr(P, kind) if kind else None)
    lo, hi = O.gershgorin(h)
    x = (hi * np.eye(n) - h) / (hi - lo)
    drop = lambda a: np.where(np.abs(a) > thr, a, 0.0)
    bound, idem = 0.0, []
    for s in pp:
        bound = 3 * bound * max(1.0, np.linalg.norm(x)) + 2 * n * EPS * np.linalg.norm(
            np.abs(x) @ np.abs(x))
        y = drop(x @ x)
        idem.append(np.linalg.norm(x - y))
        x = drop(y if s else 2 * x - y)
    assert np.linalg.norm(got - 2 * x) <= 2 * bound
    assert np.allclose(np.asarray(vv[:len(pp)]), idem, rtol=0, atol=2 * bound + 1e-14)


def test_response_steps_with_their_own_bookkeeping_launch(P, n=2320):
    """Above 1280 tiles (leading dimension 2432 on) the response's step launch
    neither absorbs nor plans.  H = Q diag(e) Q with the reflection
    Q = I - 2 v v^T: density and response are known without an eigensolver."""
    print(f"[response] n={n}", flush=True)
    rng = np.random.default_rng(n)
    v = rng.standard_normal(n)
    v /= np.linalg.norm(v)
    e = np.concatenate([rng.uniform(-3, -1, n // 2), rng.uniform(1, 3, n - n // 2)])

    def conjugate(m):
        """Q m Q."""
        m = m - 2 * np.outer(v, v @ m)
        return m - 2 * np.outer(m @ v, v)

    h = conjugate(np.diag(e))
    h = 0.5 * (h + h.T)
    h1 = rng.standard_normal((n, n)) / np.sqrt(n)
    h1 = 0.5 * (h1 + h1.T)
    rho, rsp = P.compute_response_sp2(h, h1, (n // 2) / n, 1, 100, "Abs", 1e-10)
    f = (np.arange(n) < n // 2).astype(float)
    de = e[:, None] - e[None, :]
    quotient = np.where(f[:, None] != f[None, :], (f[:, None] - f[None, :]) / np.where(de, de, 1.0), 0.0)
    ref = 2 * conjugate(conjugate(h1) * quotient)
    assert np.linalg.norm(rho - 2 * conjugate(np.diag(f))) < 1e-9
    assert np.linalg.norm(rsp - ref) < 1e-7 * np.linalg.norm(ref)
    assert np.array_equal(rsp, rsp.T)


@pytest.mark.parametrize("n", [700, 2320])
def test_thresholded_steps(P, n, thr=1e-6):
    """The sparse formats' thresholding, with the bookkeeping in the step's
    launch (700) and in its own (2320), against the elementwise rule."""
    import torch
    print(f"[thresholded steps] n={n}", flush=True)
    i = np.arange(n)
    d = np.abs(i[:, None] - i[None, :])
    rng = np.random.default_rng(n)
    h = -np.exp(-d / 8.0) * (1.0 + 0.1 * rng.standard_normal((n, n)))
    h[d > 64] = 0.0
    h = 0.5 * (h + h.T)
    pp = [1, 0, 1, 1, 0]
    ppa, vv, ic = P._ivec(len(pp), pp), P._dvec(len(pp)), P._ivec(1, [len(pp)])
    rho = P._h_rho(P.lib().prg_sp2_alg2_seq, h, thr, P._ip(ppa), P._ip(ic), P._dp(vv), 0,
                   matrix_type=P.ELLPACK)
    r = np.abs(h).sum(0) - np.abs(np.diag(h))
    lo, hi = (np.diag(h) - r).min(), (np.diag(h) + r).max()

    def drop(a):
        return torch.where(a.abs() > thr, a, torch.zeros_like(a))

    x = torch.from_numpy((hi * np.eye(n) - h) / (hi - lo)).cuda()
    idem = []
    for s in pp:
        y = drop(x @ x)
        idem.append(float((x - y).norm()))
        x = drop(y if s else 2 * x - y)
    got = torch.from_numpy(rho.copy(order="C")).cuda()
    diff = (got - 2 * x).abs()
    zeros = int((x == 0).sum())
    assert n < zeros < n * n  # the threshold decides, and not everywhere
    # an entry whose sums end on both sides of the threshold may be dropped in
    # one of them only, which moves what it enters by as much
    assert int((diff > 1e-12).sum()) <= n and float(diff.max()) <= 8 * thr
    assert np.allclose(np.asarray(vv[:len(pp)]), idem, rtol=0, atol=1e-9)
    assert bool((got == got.T).all())


# (n, tiles of the upper triangle, edge): the edges of prg_f64_tile.h over the
# leading dimensions 256, 768, 1024 and 3072
@pytest.mark.parametrize("n,tiles,edge", [(129, 136, 16), (700, 300, 32), (1000, 253, 48),
                                          (2999, 2080, 48)])
def test_counted_flops_of_symmetric_products(P, n, tiles, edge):
    """The executed flops are those of the launched tiles, K up to n's multiple
    of 32."""
    import torch
    ld = P.padded_ld(n)
    a = torch.zeros((ld, ld), dtype=torch.float64, device="cuda")
    a[:n, :n] = torch.eye(n, dtype=torch.float64, device="cuda")
    expected = tiles * 2.0 * edge * edge * (-(-n // 32) * 32)
    P.gemm_counters(reset=True)
    P.symmetric_product_device(a, a, torch.empty_like(a), n)
    assert P.gemm_counters(reset=True) == (1.0, 2.0 * n ** 3, expected)
    assert P.sp2_step_flops(n) == expected


# full products: 32-wide tiles over ld 1024, staged 128-wide ones over 4096
@pytest.mark.parametrize("n,tiles,edge", [(1000, 1024, 32), (4060, 1024, 128)])
def test_counted_flops_of_full_products(P, n, tiles, edge):
    m, out = P.Matrix.from_numpy(np.eye(n)), P.Matrix.zeros(n)
    P.gemm_counters(reset=True)
    P.lib().prg_orthogonalize(m.h, m.h, out.h, 0.0, b"dense", 0)
    products, alg, executed = P.gemm_counters(reset=True)
    assert products == 2.0 and alg == 4.0 * n ** 3
    assert executed == 2 * tiles * 2.0 * edge * edge * (-(-n // 32) * 32)
    m.close()
    out.close()
