"""Tails of the windowed route on grids beside the blocks of 256 bins (GPU).

Short windows, so that nearly all of a bin's value is tails, of lines on the grid
and up to one grid length beside it; the bar of the windowed route (1e-6 per bin
plus 1e-12 of the peak)."""

import numpy as np
import pytest

from tests.test_window_gpu import _close, _stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_E", [1, 5, 63, 255, 256, 257, 511, 513, 1030])
def test_tails_match_the_oracle(oracle, device, n_E):
    import torch

    from pyrite_amd import _lib

    rng = np.random.default_rng(n_E)
    E0, dE, x_c, n_lines = 1000.0, 24.0, 10.0, 400
    E_r = E0 + dE * (rng.integers(-n_E, 2 * n_E, n_lines) + rng.uniform(-0.4, 0.4, n_lines))
    a = x_c / (dE * (rng.choice([1, 2], n_lines) - 0.45))
    w = rng.uniform(0.1, 1.0, n_lines).astype(np.float32)
    want = oracle.window_reduce(E_r, a, w, E0, dE, n_E, x_c)
    t = [torch.as_tensor(v, device=device) for v in (E_r, a, w)]
    out = torch.zeros(n_E, dtype=torch.float64, device=device)
    ws = _lib.DeviceScratch(device).get(_lib.workspace_bytes("hr_window_reduce_workspace_bytes", n_lines, n_E))
    _lib.call("hr_window_reduce", t[0].data_ptr(), t[1].data_ptr(), t[2].data_ptr(), n_lines, n_E, E0, dE, x_c,
              out.data_ptr(), ws, _stream())
    _close(out.cpu().numpy(), want)
