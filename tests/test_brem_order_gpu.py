"""Bremsstrahlung of rows put in class order against the same rows cell by cell (GPU).

The order is taken from 1e8 cells and 20,480 rows on; calls of a part of the rows stay below and
evaluate every cell.  Energies on and beside the class edges, below, at and above
the bins, beyond both ends of the classes; bins in no order; rows without weight,
of negative weight and without length.  Either route is within 1e-6 of the sum of
the cells' sizes (the bound of the oracle test), so they differ by at most twice
that."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COMPS = {1: [("C", 0.1136)], 2: [("Si", 0.04), ("N", 0.053)],
         4: [("C", 0.02), ("N", 0.015), ("Al", 0.01), ("W", 0.01)]}


@pytest.mark.parametrize("n_el,n_E,weights", [(1, 1025, "none"), (2, 1024, "signed"), (4, 700, "zeros"),
                                              (2, 300, "none"), (4, 61, "signed")])
def test_order_equals_cell_by_cell(device, n_el, n_E, weights):
    import torch

    from pyrite_amd.spectrum.lines import BremScorer

    rng = np.random.default_rng([n_el, n_E])
    n = 100_000_000 // n_E + 77
    grid = rng.permutation(np.geomspace(1000.0, 200_000.0, n_E))
    sc = BremScorer(COMPS[n_el], grid, 1.0e6, np.array([np.cos(0.2), 0.0, np.sin(0.2)]), device)
    T = np.exp(rng.uniform(np.log(0.1), np.log(4.0e4), n)).astype(np.float32)
    edges = (2.0 ** np.arange(-2, 15)[:, None] * (1 + np.arange(8) / 8)).ravel().astype(np.float32)
    T[: edges.size] = edges
    T[edges.size: 2 * edges.size] = np.nextafter(edges, np.float32(0))
    T[2 * edges.size: 2 * edges.size + n_E] = (grid * 1e-3).astype(np.float32)
    L = rng.exponential(2.0e4, n).astype(np.float32)
    L[rng.random(n) < 0.05] = 0.0
    v = rng.normal(0.0, 1.0, (n, 3))
    seg = {"r_mid": rng.uniform(0.0, 1.0e6, (n, 3)).astype(np.float32),
           "v_hat": (v / np.linalg.norm(v, axis=1, keepdims=True)).astype(np.float32), "L": L, "E": T}
    w = None
    if weights != "none":
        w = np.where(rng.random(n) < 0.3, 0.0, rng.uniform(0.1, 1.0, n)).astype(np.float32)
        if weights == "signed":
            w *= rng.choice([-1.0, 1.0], n).astype(np.float32)
    seg = {k: torch.as_tensor(np.ascontiguousarray(a), device=device) for k, a in seg.items()}
    w = None if w is None else torch.as_tensor(w, device=device)
    whole, again, parts, size = (torch.zeros(n_E, dtype=torch.float64, device=device) for _ in range(4))
    sc.reduce(seg, whole, w)
    sc.reduce(seg, again, w)
    assert torch.equal(whole, again)
    for lo in range(0, n, (n + 2) // 3):
        hi = min(lo + (n + 2) // 3, n)
        part = {k: a[lo:hi] for k, a in seg.items()}
        sc.reduce(part, parts, None if w is None else w[lo:hi])
        sc.reduce(part, size, None if w is None else w[lo:hi].abs())
    err, bound = (whole - parts).abs(), 2.0e-6 * size + 1.0e-12 * size.max()
    assert bool(torch.all(err <= bound)), float((err / bound).max())


def _workspace(n, n_E):
    from pyrite_amd import _lib

    args = _lib.BremArgs()
    args.n_seg, args.n_E, args.n_el = n, n_E, 1
    return _lib.workspace_bytes("hr_brem_workspace_bytes", ctypes.byref(args))


@pytest.mark.parametrize("n,n_E", [(100, 1_000_000), (1000, 100_000), (20_479, 60_000), (20_480, 65_537),
                                   (24, 4_200_000), (1_000_000, 70_000)])
def test_few_rows_or_many_bins_take_the_direct_workspace(device, n, n_E):
    """At most 16 blocks per CU and window of bins, one row each: 16 x 256 CUs x 1,024 bins x 8 B."""
    assert _workspace(n, n_E) <= max(16 * 256 * 1024 * 8, 8 * n_E)


def test_few_rows_and_many_bins_match_the_oracle(oracle, device):
    """Past the cells that the order asks for, with few rows: as many bins as 1,000 rows need."""
    import torch

    from pyrite_amd.spectrum import attenuation
    from pyrite_amd.spectrum.lines import BremScorer

    rng = np.random.default_rng(3)
    n, n_E = 1000, 100_100
    grid, comp, n_hat = np.linspace(1000.0, 50_000.0, n_E), COMPS[1], np.array([np.cos(0.2), 0.0, np.sin(0.2)])
    v = rng.normal(0.0, 1.0, (n, 3))
    seg = {"r_mid": rng.uniform(0.0, 1.0e6, (n, 3)).astype(np.float32),
           "v_hat": (v / np.linalg.norm(v, axis=1, keepdims=True)).astype(np.float32),
           "L": rng.exponential(2.0e4, n).astype(np.float32),
           "E": np.exp(rng.uniform(np.log(200.0), np.log(1.0e4), n)).astype(np.float32)}
    sc = BremScorer(comp, grid, 1.0e6, n_hat, device)
    out = torch.zeros(n_E, dtype=torch.float64, device=device)
    sc.reduce({k: torch.as_tensor(a, device=device) for k, a in seg.items()}, out)
    pick = np.unique(np.concatenate([[0, n_E - 1], rng.integers(0, n_E, 2000)]))
    mu = attenuation.mu_total_inv_ang(comp, grid[pick]).astype(np.float32)
    want = oracle.brem_reduce(seg, 1.0e6, n_hat, [6.0], [0.1136e24], grid[pick], mu)
    got = out.cpu().numpy()[pick]
    assert np.all(np.abs(got - want) <= 1e-6 * np.abs(want) + 1e-12 * want.max())
