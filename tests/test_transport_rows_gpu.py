"""Rows where the transport step's element table and Poisson search change route (GPU).

The step keeps the element constants of up to 32 (layer, element) slots in LDS
and builds them per row beyond; it searches the three Poisson numbers of a row
together while each mean is at most 64 and one after another above.  Each side
of both lines against the oracle, row for row, with the bar of the full
histories (1e-9 of the value or of 1: host and device mathematics differ in the
last bits and the rows add those up)."""

import numpy as np
import pytest

from tests.test_transport_gpu import _gpu_run, _oracle_run
from tests.transport_cases import Case

pytestmark = pytest.mark.gpu


def _stack(n):
    """n thin films, silicon and a silicon-carbon compound in turn: two slots each."""
    comps = ([("Si", 0.05)], [("Si", 0.025), ("C", 0.05)])
    return [(400.0 * i, 400.0 * (i + 1), comps[i % 2]) for i in range(n)]


@pytest.mark.parametrize("case", [
    Case("slots_32", 40.0, 64, _stack(16), seed=21, straggle=True),
    Case("slots_34", 40.0, 64, _stack(17), seed=21, straggle=True),
    # hydrogen loses the most per free path: means of 50 to several hundred per row
    Case("hydrogen", 2000.0, 48, [(0.0, 1.0e8, [("H", 0.04)])], seed=22, straggle=True),
    Case("hydrogen_mixed_in", 1000.0, 32, [(0.0, 2.0e7, [("H", 0.06), ("C", 0.02)])], seed=23, straggle=True),
    Case("helium_like_cut", 50.0, 64, [(0.0, 1.0e6, [("H", 0.04)])], seed=24, E_cut=1.0, straggle=True),
], ids=lambda c: c.name)
def test_rows_match_the_oracle(oracle, device, case):
    cap = 4096
    g, o = _gpu_run(case, device, cap=cap), _oracle_run(oracle, case, cap=cap)
    np.testing.assert_array_equal(g[1], o[1])
    np.testing.assert_array_equal(g[2], o[2])
    assert o[1].max() <= cap and o[1].sum() > 2 * case.Ne
    for k in ("seg_mid", "seg_E", "seg_len", "seg_E_end", "seg_t_end"):
        for e in range(case.Ne):
            a, b = (x[0][k][e * cap:e * cap + int(o[1][e])] for x in (g, o))
            assert np.max(np.abs(a - b) / np.maximum(np.abs(b), 1.0)) < 1e-9, (k, e)
