"""FP16 / BF16 hi+lo products whose last round of 128 x 128 tiles is cut into
quarters (528 tiles: 512 whole and 16 cut) and whose only round is not (171):
the same bounds as the smaller sizes, which are cut throughout, and for SP2 one
for every 64 x 64 block, which a lost tile cannot meet."""
import numpy as np
import pytest


def reflected(d, v, outer):
    """Q diag(d) Q with the reflection Q = I - 2 v v^T (arrays or tensors)."""
    dv = d * v
    m = -2 * outer(v, dv) - 2 * outer(dv, v) + 4 * (v @ dv) * outer(v, v)
    i = list(range(len(d)))
    m[i, i] += d
    return m


def worst_block(got, ref, edge=64):
    """Largest error norm of a block of `edge` rows and columns over the
    block's own norm (the last block of an overhanging size may be smaller)."""
    worst = 0.0
    for a in range(0, len(ref), edge):
        rows, exact = got[a:a + edge], ref[a:a + edge]
        for b in range(0, len(ref), edge):
            e = exact[:, b:b + edge]
            worst = max(worst, float(((rows[:, b:b + edge] - e) ** 2).sum() / (e ** 2).sum()) ** 0.5)
    return worst


def block_bound(n, bits, steps=30):
    """A step's product is off by (3 * 2^-2b + sqrt(n) 2^-24) of |X| |X| (lo lo
    dropped, lo rounded; FP32 sums of random signs), and |X| |X| is at most 6
    times |X| in norm off the diagonal: x_i + x_j <= 2 times from the diagonal,
    4 from the n entries of order 4 / n."""
    return steps * 6 * (3 * 2.0 ** (-2 * bits) + n ** 0.5 * 2.0 ** -24)


@pytest.mark.parametrize("lost", [False, True])
def test_block_bound_sees_a_lost_quarter_tile(lost, n=512):
    """On the CPU in float64: a 64 x 64 block (and its mirror) that no step
    writes exceeds the bound of either precision, and nothing else does."""
    rng = np.random.default_rng(n)
    v = rng.standard_normal(n)
    v /= np.linalg.norm(v)
    e = np.concatenate([rng.uniform(-3, -1, n // 2), rng.uniform(1, 3, n - n // 2)])
    x = 0.5 * np.eye(n) - reflected(e, v, np.outer) / 6.0
    for _ in range(30):
        y = x @ x
        x = y if abs(np.trace(y) - n // 2) < abs(2 * np.trace(x) - np.trace(y) - n // 2) else 2 * x - y
        if lost:
            x[448:, 384:448] = 0.0
            x[384:448, 448:] = 0.0
    worst = worst_block(x, reflected((e < 0).astype(float), v, np.outer))
    print(f"[lost={lost}] worst block {worst:.2e}, bounds {block_bound(n, 8):.2e} {block_bound(n, 11):.2e}")
    assert (worst > block_bound(n, 8)) if lost else (worst < block_bound(n, 11))


@pytest.fixture(scope="module")
def P():
    import progress_amd
    progress_amd.set_precision(progress_amd.PREC_FP64)
    return progress_amd


@pytest.mark.gpu
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


@pytest.mark.gpu
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
    ld = P.padded_ld(n)
    h = torch.zeros((ld, ld), dtype=torch.float64, device="cuda")
    h[:n, :n] = reflected(et, vt, torch.outer)
    h = 0.5 * (h + h.T)
    rho = torch.zeros_like(h)
    torch.cuda.synchronize()
    P.sp2_alg2_device(h, rho, n, (n // 2) / n, 1, 100, "Abs", 1e-10, precision=getattr(P, prec))
    d = rho[:n, :n]
    ref = 2 * reflected((et < 0).double(), vt, torch.outer)
    # a few steps' rounding, n entries per row
    assert float((d - ref).norm()) <= 16 * n * (2.0 ** (-2 * bits) + 2.0 ** -24)
    worst = worst_block(d.cpu().numpy(), ref.cpu().numpy())
    print(f"[{prec} n={n}] worst block {worst:.2e}, bound {block_bound(n, bits):.2e}", flush=True)
    assert worst <= block_bound(n, bits)
    assert torch.equal(d, d.T)
