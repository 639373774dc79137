"""The 48-wide tiles of the batched subgraph SP2 loop
(src/prg_subgraphloop_mod.F90:36-126): part sizes around the tile edges, and
the last iteration, which computes only the tiles that hold core rows."""
import numpy as np
import pytest

import progress_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def P():
    import progress_amd
    progress_amd.set_precision(progress_amd.PREC_FP64)
    return progress_amd


EPS = np.finfo(float).eps


@pytest.mark.parametrize("panel", ["", "48"])
@pytest.mark.parametrize("sizes,ncore", [
    ((1, 15, 16, 17, 33), 1), ((47, 48, 49, 63), 5), ((64, 65, 95, 96, 97), 50),
    ((143, 144, 145), 48), ((200, 257), 300)])
def test_direct_tiles_match_oracle(P, sizes, ncore, panel, monkeypatch):
    print(f"[subgraph 48-wide tiles] sizes={sizes} core={ncore} panel={panel!r}", flush=True)
    n, rng = sum(sizes), np.random.default_rng(sum(sizes))
    h = np.zeros((n, n))
    parts, at = [], 0
    for k in sizes:
        a = rng.standard_normal((k, k))
        h[at:at + k, at:at + k] = (a + a.T) / 2
        parts += [list(range(c, min(c + ncore, at + k))) for c in range(at, at + k, ncore)]
        at += k
    g = np.where(h != 0.0, 1.0, 0.0)
    lo, hi = O.gershgorin(h)
    if panel:
        monkeypatch.setenv("PRG_BATCH_TILE", panel)
    for imax in (1, 2, 7):
        seq = [1, 0, 0, 1, 0, 1, 1][:imax]
        gp = P.set_partition(parts, n)
        rho, vv = P.subgraph_sp2_loop(h, g, gp, seq, imax, lo, hi)
        assert P.subgraph_config()[0] == 48
        ref, vv_ref = O.subgraph_sp2_loop(h, g, parts, seq, imax, lo, hi)
        # |d(x^2)|, |d(2x - x^2)| <= 2 on [0, 1]: every step at most doubles an
        # error and adds the product's k eps
        tol = 2.0 ** (imax + 2) * max(sizes) * EPS * np.sqrt(n)
        assert np.linalg.norm(rho - ref) < tol
        assert np.allclose(vv, vv_ref, rtol=0, atol=tol * np.sqrt(n))


def test_padded_panels_take_staged_tiles(P, monkeypatch):
    """Many parts of 128 rows (2 panels of 64, 3 of 48): the staged tiles, with
    the 48-wide ones' result up to the order of the sums."""
    k, blocks, imax = 128, 8, 4
    print(f"[subgraph staged tiles] parts={k * blocks} of {k} rows", flush=True)
    rng = np.random.default_rng(5)
    h = np.zeros((k * blocks, k * blocks))
    for b in range(blocks):
        a = rng.standard_normal((k, k))
        h[b * k:(b + 1) * k, b * k:(b + 1) * k] = (a + a.T) / 2
    g = np.where(h != 0.0, 1.0, 0.0)
    lo, hi = O.gershgorin(h)
    parts = [[i] for i in range(k * blocks)]
    rho, vv = P.subgraph_sp2_loop(h, g, P.set_partition(parts, k * blocks), [1, 0, 1, 0], imax,
                                  lo, hi)
    assert P.subgraph_config()[:3] == (64, 1, 16)
    monkeypatch.setenv("PRG_BATCH_TILE", "48")
    ref, vv_ref = P.subgraph_sp2_loop(h, g, P.set_partition(parts, k * blocks), [1, 0, 1, 0],
                                      imax, lo, hi)
    assert P.subgraph_config()[0] == 48
    tol = 2.0 ** (imax + 2) * k * EPS * np.sqrt(k * blocks)
    assert np.linalg.norm(rho - ref) < tol
    assert np.allclose(vv, vv_ref, rtol=0, atol=tol * np.sqrt(k * blocks))


@pytest.mark.parametrize("k,parts,panel", [(64, 640, 64), (80, 560, 48), (128, 512, 64),
                                           (144, 432, 48), (256, 512, 64)])
def test_tiles_of_uniform_parts(P, k, parts, panel):
    """The rule's choice where the padding decides (64, 128 and 256 rows waste
    nothing on 64-wide panels, 80 and 144 a quarter or more), and the result."""
    blocks, imax = -(-parts // k), 3
    n = k * blocks
    print(f"[subgraph rule] parts={parts} of {k} rows", flush=True)
    rng = np.random.default_rng(k)
    h = np.zeros((n, n))
    for b in range(blocks):
        a = rng.standard_normal((k, k))
        h[b * k:(b + 1) * k, b * k:(b + 1) * k] = (a + a.T) / 2
    g = np.where(h != 0.0, 1.0, 0.0)
    lo, hi = O.gershgorin(h)
    cores = [[i] for i in range(parts)]
    rho, vv = P.subgraph_sp2_loop(h, g, P.set_partition(cores, n), [1, 0, 1], imax, lo, hi)
    assert P.subgraph_config()[:3] == (panel, 1, 16)
    x = (hi * np.eye(n) - h) / (hi - lo)
    for s in (1, 0, 1):
        x = x @ x if s else 2 * x - x @ x
    tol = 2.0 ** (imax + 2) * k * EPS * np.sqrt(n)
    assert np.linalg.norm((rho - 2 * x)[:parts]) < tol


def test_direct_tiles_round_no_worse_than_staged_ones(P, monkeypatch, n=300, imax=6):
    """Against the same steps in extended precision (64-bit mantissas): the sums
    over four waves' quarters of K leave an error within that of the staged
    tiles' sequential ones, plus a quarter for the input's luck."""
    if np.finfo(np.longdouble).nmant < 63:
        pytest.skip("no extended precision here")
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n))
    h = (a + a.T) / 2
    lo, hi = O.gershgorin(h)
    seq = [1, 0, 0, 1, 0, 1]
    x = (np.longdouble(hi) * np.eye(n, dtype=np.longdouble) - h) / (np.longdouble(hi) - lo)
    for s in seq:
        x = x.dot(x) if s else 2 * x - x.dot(x)
    err = {}
    for panel in ("48", "64"):
        monkeypatch.setenv("PRG_BATCH_TILE", panel)
        monkeypatch.setenv("PRG_BATCH_DEPTH", "1")
        monkeypatch.setenv("PRG_BATCH_KSLAB", "16")
        gp = P.set_partition([list(range(n))], n)
        rho, _ = P.subgraph_sp2_loop(h, np.ones((n, n)), gp, seq, imax, lo, hi)
        assert P.subgraph_config()[0] == int(panel)
        err[panel] = float(np.sqrt(((rho - 2 * x) ** 2).sum()) / np.sqrt((4 * x ** 2).sum()))
    print(f"[subgraph rounding] error of 48-wide tiles {err['48']:.2e}, staged {err['64']:.2e}",
          flush=True)
    assert err["48"] <= 1.25 * err["64"]
