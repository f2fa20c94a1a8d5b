"""Windows of every length around the lines where their lanes change (GPU).

A line's window stays with its lane up to 8 bins, goes to 16 lanes up to 128 and
to the whole wave above; lengths on both sides of each, mixed within a wave, on
grids where they are windows and where a quarter of the grid makes them broad.
The bar is that of the windowed route (1e-6 per bin plus 1e-12 of the peak)."""

import numpy as np
import pytest

from tests.test_window_gpu import _close, _stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_E", [30, 500, 4096])
@pytest.mark.parametrize("n_lines", [1, 63, 65, 1500])
def test_every_window_length_matches_the_oracle(oracle, device, n_E, n_lines):
    import torch

    from pyrite_amd import _lib

    rng = np.random.default_rng([n_E, n_lines])
    E0, dE, x_c = 1000.0, 24.0, 100.0
    reach = rng.choice([1, 2, 3, 4, 5, 7, 8, 31, 63, 64, 65, 300, 3000], n_lines)  # 2 reach + 1 bins
    E_r = E0 + dE * (rng.integers(-40, n_E + 40, n_lines) + rng.uniform(-0.4, 0.4, n_lines))
    a = x_c / (dE * (reach - 0.45))  # |eps| <= 0.4 dE keeps the reach
    w = np.where(rng.random(n_lines) < 0.2, 0.0, rng.uniform(0.1, 1.0, n_lines)).astype(np.float32)
    w[0] = 0.7
    want = oracle.window_reduce(E_r, a, w, E0, dE, n_E, x_c)
    t = [torch.as_tensor(v, device=device) for v in (E_r, a, w)]
    out = torch.zeros(n_E, dtype=torch.float64, device=device)
    ws = _lib.DeviceScratch(device).get(_lib.workspace_bytes("hr_window_reduce_workspace_bytes", n_lines, n_E))
    _lib.call("hr_window_reduce", t[0].data_ptr(), t[1].data_ptr(), t[2].data_ptr(), n_lines, n_E, E0, dE, x_c,
              out.data_ptr(), ws, _stream())
    _close(out.cpu().numpy(), want)
