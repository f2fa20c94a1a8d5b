"""Flat field and grouped term in one pass against the two separate ones (GPU).

Groups of no, one and many lines, ends on and beside the 128 lines a block stages
and the 8 it sums in FP32, one chunk and many.  Both routes sum the same FP32
cells, in FP32 groups of at most 8 that start elsewhere: they may differ by the
bound the field test uses on either (2e-6 of the lines' L1 size), and the grouped
term by that carried through the square."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = {
    "one_line": [1],
    "empty_groups": [0, 0, 3, 0, 5, 0],
    "tile_edges": [127, 1, 128, 129, 255, 256, 257, 1, 7, 8, 9],
    "one_long": [1500],
    "histories": None,
}


@pytest.mark.parametrize("n_E", [5, 300, 1100])
@pytest.mark.parametrize("sizes", list(SIZES))
def test_one_pass_equals_two(device, sizes, n_E):
    import torch

    from pyrite_amd.spectrum.coherent import N_FIELDS, CoherentScorer
    from pyrite_amd.spectrum.geometry import cone_detector
    from pyrite_amd.spectrum.lines import line_tables

    rng = np.random.default_rng([len(sizes), n_E])
    E_grid = np.linspace(3000.0, 4500.0, n_E)
    n_hats, weights = cone_detector(np.pi / 2, np.deg2rad(0.5), 0.01, 2)
    count = SIZES[sizes] or rng.integers(0, 45, 3000).tolist()
    n = int(np.sum(count))
    sc = CoherentScorer(line_tables("hopg", [(0, 0, 2)], E_grid), "hopg", E_grid, 1.0e6, n_hats, weights, device,
                        grouped=True)
    # records of lines across and beside the grid: centre, width, phases, amplitudes, path, formation
    rec = np.empty((N_FIELDS, sc.n_rows, n))
    rec[0], rec[1] = rng.uniform(2500.0, 5000.0, rec[0].shape), rng.uniform(0.1, 12.0, rec[0].shape)
    rec[2], rec[3] = rng.uniform(0.0, 1.0e3, rec[0].shape), rng.uniform(0.0, 1.0e6, rec[0].shape)
    rec[4:8] = rng.normal(0.0, 1.0, rec[4:8].shape) * (rng.random(rec[0].shape) < 0.8)
    rec[8], rec[9] = rng.uniform(0.0, 1.0e7, rec[0].shape), rng.uniform(-1.0e5, 1.0e5, rec[0].shape)
    q = rng.normal(0.0, 0.3, rec[0].shape)
    rec[10], rec[11], rec[12] = 2.0 * np.cosh(q), -2.0 * np.sinh(q), q
    rec_d = torch.as_tensor(rec, device=device).contiguous()
    gs = torch.as_tensor(np.concatenate([[0], np.cumsum(count)]), device=device)
    sc._launch_field(rec_d, n)
    sc._launch_grouped(rec_d, n, gs)
    field, grouped = sc.field.cpu().numpy(), sc.grouped.cpu().numpy()
    sc.reset()
    sc._launch_both(rec_d, n, gs)
    # |profile| <= cosh(q) sin(v)/v + ..: at most apb/2 + |bma|/2 + |q| (apb + |bma|)/2
    size = np.abs(rec[4:8]).max(0) * 2 * (0.5 * (rec[10] + np.abs(rec[11])) * (1 + np.abs(q)))
    bound = 2 * 2e-6 * size.sum(-1)
    assert np.all(np.abs(sc.field.cpu().numpy() - field) <= bound[:, None, None] + 1e-300)
    per = np.add.reduceat(np.concatenate([size, np.zeros((sc.n_rows, 1))], 1), np.minimum(gs[:-1].cpu().numpy(), n), 1)
    per = np.where(np.asarray(count) > 0, per, 0.0)
    g_bound = (4 * 2 * 2e-6 * 2 * per**2).sum(-1)
    assert np.all(np.abs(sc.grouped.cpu().numpy() - grouped) <= g_bound[:, None] + 1e-300)
    assert n == 0 or np.abs(field).max() > 0
