"""What is timed when this package's speed is measured: twelve calls of its public entry points.

Each case is one call a program makes on inputs it already holds on the device:

* scoring of given segments -- dense lines on uniform and non-uniform grids, windowed
  lines per pixel, bremsstrahlung, coherent fields with and without the grouped term;
* transport alone -- the flat entry on a film, the core on thick graphite, a campaign of
  targets through the work queue;
* whole cases -- transport and scoring together: a small batch, the default batch on two
  streams, detector-cone splitting, and continuation rounds of a thick silicon target.

``exact`` restates the scoring formulas in 64 bits with torch and numpy; Monte Carlo
transport has no closed value per history (its draws decide discrete events), so the
transport and whole-case entries have none.
"""

import math

import numpy as np
import torch

from pyrite_amd import _lib
from pyrite_amd.backend import require_device
from pyrite_amd.pipeline import CaseConfig, CasePipeline
from pyrite_amd.queue import QueueCase, TransportQueue
from pyrite_amd.spectrum import attenuation
from pyrite_amd.spectrum.coherent import CoherentScorer, escape_phase_rate, gaussian_longitudinal_factor
from pyrite_amd.spectrum.crystal import allowed_reflections
from pyrite_amd.spectrum.geometry import cone_detector, tilted_geometry
from pyrite_amd.spectrum.lines import BremScorer, LineScorer, line_tables, mc_brem_spectrum, synthetic_line_tables
from pyrite_amd.transport.api import simulate_trajectories
from pyrite_amd.transport.core import DeviceTables, TransportControl, alloc_rows, make_hip_transport_core
from pyrite_amd.transport.tables import build_layer_tables, build_transport_lut

TARGETS = {  # crystal key, composition (element, atoms per cubic angstrom), beam energy [keV], mean segment [A]
    "hopg": ("hopg", [("C", 0.1136)], 5000.0, 2.5e4),
    "silicon": ("silicon", [("Si", 0.04994)], 10000.0, 3.0e4),
}
COMPOSITIONS = {
    "graphite": [("C", 0.1136)],
    "silicon": [("Si", 0.04994)],
    "silicon nitride": [("Si", 0.0419), ("N", 0.0559)],
    "four elements": [("C", 0.02), ("N", 0.015), ("Al", 0.01), ("W", 0.01)],
}
# transport rows of one history, to price the work of a case (measured means)
ROWS = {"hopg": 41, "silicon": 303, "film": 120, "graphite": 60, "Si": 300, "Ge": 1500, "W": 4000}
FILM = [("Si", 0.025), ("C", 0.05)]


def listed():
    """The measured cases, smallest calls first."""
    return [
        # a quick look at a target: one detector ray, a few hundred histories; launches and host calls count
        dict(name="step_small", kind="step", target="hopg", Ne=256, n_side=1, n_bins=201, batches=1, split=False),
        # the default case (100 um graphite, 5 MeV, 3x3 rays, brem, 1024 bins) over two overlapped batches
        dict(name="step_hopg", kind="step", target="hopg", Ne=32_768, n_side=3, n_bins=1024, batches=2, split=False),
        # the same case with detector-cone splitting: a batch and the generation of its copies
        dict(name="step_split", kind="step", target="hopg", Ne=20_000, n_side=3, n_bins=1024, batches=1, split=True),
        # a thick target streamed through continuation rounds: mixed precision, windowed lines, 4096 bins
        dict(name="stream_silicon", kind="stream", n=16_384, lanes=16_384, rows=32, n_bins=4096, reflections=16),
        # the flat entries: 40 keV electrons stopping in a compound film, then its bremsstrahlung on the host
        dict(name="flat_film", kind="flat", Ne=3001, E0=40.0, substeps=True, n_bins=320),
        # the transport core alone: the rows of one launch of the default case in the driver's own grid
        dict(name="core_hopg", kind="core", target="hopg", Ne=20_000, cap=256),
        # a campaign of uneven targets in one work-queue launch
        dict(name="queue_campaign", kind="queue", scale=1.0),
        # dense line spectrum of given segments: uniform grid, 3x3 rays, an odd segment count
        dict(name="lines_uniform", kind="lines", target="hopg", n=300_017, n_side=3, n_bins=1024, grid="uniform",
             weighted=False),
        # the same on a logarithmic grid (general reducer), few rays, weighted rows (copies)
        dict(name="lines_log_grid", kind="lines", target="silicon", n=20_011, n_side=2, n_bins=777, grid="log",
             weighted=True),
        # windowed spectra per pixel: 64 reflections, 4096 bins
        dict(name="lines_pixels", kind="pixels", n=12_007, n_g=64, n_side=8, n_bins=4096),
        # bremsstrahlung of a compound over every energy of a shower, 10 MeV down to the cutoff
        dict(name="brem_shower", kind="brem", composition="silicon nitride", n=150_001, n_bins=2000, E_lo=5.0,
             E_hi=10_000.0, weighted=True),
        # coherent fields of whole histories and the decoherence blend
        dict(name="coherent_blend", kind="coherent", n=4001, slots=41, n_side=2, n_bins=1024, grouped=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges the listed ones stand for."""
    kind = rng.choice(["step", "stream", "flat", "core", "queue", "lines", "lines", "pixels", "brem", "brem",
                       "coherent"])
    if kind == "step":
        split = rng.random() < 0.3
        return dict(kind=kind, target="hopg", Ne=_log_int(rng, 100, 20_000 if split else 32_768),
                    n_side=rng.randint(1, 3), n_bins=rng.randint(150, 1400), batches=1 if split else rng.randint(1, 2),
                    split=split)
    if kind == "stream":
        n = _log_int(rng, 500, 16_384)
        return dict(kind=kind, n=n, lanes=max(64, n // rng.randint(1, 3)), rows=rng.choice([8, 17, 32]),
                    n_bins=rng.randint(500, 4096), reflections=rng.randint(1, 16))
    if kind == "flat":
        return dict(kind=kind, Ne=_log_int(rng, 50, 3000), E0=rng.uniform(15.0, 40.0), substeps=rng.random() < 0.5,
                    n_bins=rng.randint(50, 400))
    if kind == "core":
        return dict(kind=kind, target=rng.choice(["hopg", "silicon"]), Ne=_log_int(rng, 100, 20_000),
                    cap=rng.choice([32, 256]))
    if kind == "queue":
        return dict(kind=kind, scale=rng.uniform(0.1, 1.0))
    if kind == "lines":
        return dict(kind=kind, target=rng.choice(["hopg", "silicon"]), n=_log_int(rng, 200, 150_000),
                    n_side=rng.randint(1, 3), n_bins=_log_int(rng, 40, 3000), grid=rng.choice(["uniform", "log"]),
                    weighted=rng.random() < 0.5)
    if kind == "pixels":
        return dict(kind=kind, n=_log_int(rng, 200, 12_000), n_g=rng.randint(1, 64), n_side=rng.randint(1, 8),
                    n_bins=rng.randint(100, 4096))
    if kind == "brem":
        E_hi = math.exp(rng.uniform(math.log(100.0), math.log(10_000.0)))
        E_lo = E_hi * rng.choice([0.001, 0.1, 0.9, 0.98])
        return dict(kind=kind, composition=rng.choice(sorted(COMPOSITIONS)), n=_log_int(rng, 200, 150_000),
                    n_bins=_log_int(rng, 40, 4096), E_lo=max(5.0, E_lo), E_hi=E_hi, weighted=rng.random() < 0.5)
    return dict(kind=kind, n=_log_int(rng, 20, 4000), slots=rng.randint(5, 41), n_side=rng.randint(1, 3),
                n_bins=rng.randint(100, 1100), grouped=rng.random() < 0.5)


# ------------------------------------------------------------------ inputs
def _grid(case, lo=1000.0, hi=50_000.0):
    n = int(case["n_bins"])
    if case.get("grid") == "log":
        return np.geomspace(lo, hi, n)
    edges = np.linspace(lo, hi, n + 1)
    return 0.5 * (edges[:-1] + edges[1:])


def _segments(rng, n, thickness, E_lo, E_hi, mean_len, spread):
    """FP32 segment records: positions in the slab, a beam tilted by 0.5 degrees with some
    spread, exponential lengths, energies log-uniform."""
    r = np.stack([rng.normal(0, 1e4, n), rng.normal(0, 1e4, n), rng.uniform(0.0, thickness, n)], 1)
    d = np.stack([rng.normal(0, spread, n) - math.sin(math.radians(0.5)), rng.normal(0, spread, n), np.ones(n)], 1)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    seg = {"r_mid": r, "v_hat": d, "L": rng.exponential(mean_len, n),
           "E": np.exp(rng.uniform(math.log(E_lo), math.log(E_hi), n))}
    return {k: np.ascontiguousarray(v, dtype=np.float32) for k, v in seg.items()}


def _row_weights(rng, case, n):
    """Weights of split copies: powers of two, a share of them zero (rouletted)."""
    if not case["weighted"]:
        return None
    return np.where(rng.random(n) < 0.25, 0.0, 2.0 ** rng.integers(-6, 1, n)).astype(np.float32)


def _rays(n_side):
    return cone_detector(math.pi / 2, math.radians(0.5), 0.01, n_side)


def _line_inputs(case, seed):
    rng = np.random.default_rng([11, seed])
    key, comp, E0, mean_len = TARGETS[case["target"]]
    grid = _grid(case)
    hkl = [(0, 0, 2)] if key == "hopg" else [(1, 1, 1), (2, 2, 0), (3, 3, 3), (4, 4, 4)]
    tables = line_tables(key, hkl, grid, comp)
    n_hats, weights = _rays(case["n_side"])
    seg = _segments(rng, case["n"], 1.0e6, 0.98 * E0, E0, mean_len, 1.0e-2)
    return grid, tables, n_hats, weights, seg, _row_weights(rng, case, case["n"]), 1.0e6


def _pixel_inputs(case, seed):
    rng = np.random.default_rng([12, seed])
    grid = _grid(case, 1000.0, 100_000.0)
    tables = synthetic_line_tables(case["n_g"], grid, rng)
    n_hats, weights = _rays(case["n_side"])
    seg = _segments(rng, case["n"], 5.0e6, 1000.0, 20_000.0, 1.0e4, 1.0e-3)
    return grid, tables, n_hats, weights, seg, None, 5.0e6


def _brem_inputs(case, seed):
    rng = np.random.default_rng([13, seed])
    grid = _grid(case)
    comp = COMPOSITIONS[case["composition"]]
    seg = _segments(rng, case["n"], 1.0e6, case["E_lo"], case["E_hi"], 2.0e4, 0.3)
    tilt = math.radians(0.5)
    n_hat = np.array([math.cos(tilt), 0.0, math.sin(tilt)])
    return grid, comp, n_hat, seg, _row_weights(rng, case, case["n"]), 1.0e6


def _coherent_inputs(case, seed):
    """FP64 slot rows of histories that run through the slab one segment after another."""
    rng = np.random.default_rng([14, seed])
    n, slots = case["n"], case["slots"]
    key, comp, E0, mean_len = TARGETS["hopg"]
    grid = _grid(case)
    tables = line_tables(key, [(0, 0, 2)], grid, comp)
    n_hats, weights = _rays(case["n_side"])
    count = rng.integers(0, slots + 1, n)
    L = rng.exponential(mean_len * 0.9, (n, slots))
    d = np.stack([np.cumsum(rng.normal(0, 3e-3, (n, slots)), 1) - math.sin(math.radians(0.5)),
                  np.cumsum(rng.normal(0, 3e-3, (n, slots)), 1), np.ones((n, slots))], 2)
    d /= np.linalg.norm(d, axis=2, keepdims=True)
    end = np.cumsum(L[:, :, None] * d, 1)
    E_end = E0 - np.cumsum(L, 1) * 4.0e-5
    rows = {"seg_mid": end - 0.5 * L[:, :, None] * d, "seg_dir": d, "seg_len": L,
            "seg_E": np.concatenate([np.full((n, 1), E0), E_end[:, :-1]], 1), "seg_E_end": E_end,
            "seg_t0": np.cumsum(L, 1) - L}
    rows = {k: np.ascontiguousarray(v.reshape((n * slots, 3) if v.ndim == 3 else n * slots)) for k, v in rows.items()}
    factor = gaussian_longitudinal_factor(grid, 1.0e-4)
    return grid, tables, n_hats, weights, rows, count.astype(np.int64), factor, 1.0e6


def _dev():
    return require_device().torch_device


def _put(arrays):
    return {k: torch.as_tensor(v, device=_dev()) for k, v in arrays.items()}


def _queue_cases(case, seed):
    """Graphite, silicon, germanium and tungsten from 10 um to 400 um, 1 to 20 MeV."""
    spec = [("graphite", 1.0e6, 5000.0, 60_000), ("graphite", 4.0e6, 20000.0, 20_000), ("Si", 2.0e6, 10000.0, 20_000),
            ("Si", 5.0e5, 1000.0, 8000), ("Ge", 5.0e5, 10000.0, 10_000), ("Ge", 1.0e5, 3000.0, 20_000),
            ("W", 1.0e5, 10000.0, 8000), ("W", 3.0e5, 20000.0, 3000)]
    return [QueueCase(Ne=max(1, int(Ne * case["scale"])), thickness_ang=t, E0_keV=E, material=m,
                      tilt_deg=0.4 * i, seed=1000 * seed + i + 1) for i, (m, t, E, Ne) in enumerate(spec)]


# Slot-row bytes a pipeline may hold: the grid of the largest listed batch fits one arena.
ARENA_BYTES = 8 << 30


def _pipeline(case, seed):
    kw = dict(seed=1 + seed)
    if case["kind"] == "stream":
        return CasePipeline(CaseConfig.silicon_1mm_10MeV(
            Ne=case["n"], n_bins=case["n_bins"], hkl_list=allowed_reflections("silicon", case["reflections"]), **kw),
            arena_bytes=256 << 20)
    return CasePipeline(CaseConfig(Ne=case["Ne"], n_side=case["n_side"], n_bins=case["n_bins"],
                                   cone_split={} if case["split"] else None, **kw), arena_bytes=ARENA_BYTES)


def _core(case, seed):
    """Tables, the core, the entry state, and a zeroed grid of ``cap`` slots per electron."""
    silicon = case["target"] == "silicon"
    _key, comp, E0, _L = TARGETS[case["target"]]
    layers = build_layer_tables([(0.0, 1.0e7 if silicon else 1.0e6, comp)])
    tables = DeviceTables(layers, build_transport_lut(5.0, E0, layers), _dev())
    control = TransportControl(straggle_on=True)
    n = case["Ne"]
    full = lambda value, *shape: torch.full(shape, value, dtype=torch.float64, device=_dev())  # noqa: E731
    beam, _n_hat = tilted_geometry(math.pi / 2, math.radians(1.0 if silicon else 0.5))
    entry = {"clock": full(0.0, n), "pos": full(0.0, n, 3), "dirs": torch.as_tensor(beam, device=_dev()).repeat(n, 1),
             "E": full(E0, n)}
    keys = torch.empty(n, dtype=torch.uint64, device=_dev())
    _lib.call("hr_stream_keys", 1 + seed, 0, n, keys.data_ptr(), torch.cuda.current_stream().cuda_stream)
    rows = {k: v.zero_() for k, v in alloc_rows(n, case["cap"], True, _dev()).items()}
    return {"case": case, "core": make_hip_transport_core(tables, control), "keys": keys, "entry": entry,
            "state": {k: v.clone() for k, v in entry.items()}, "rows": rows,
            "alive": torch.ones(n, dtype=torch.uint8, device=_dev()), "E_cut": full(5.0, n), "straggle": full(0.0, n),
            "count": torch.zeros(n, dtype=torch.int64, device=_dev()),
            "code": torch.zeros(n, dtype=torch.int8, device=_dev())}


# ------------------------------------------------------------------ prepare and run
def prepare(case, seed):
    """Inputs, tables and handles a program holds before the call."""
    kind = case["kind"]
    if kind in ("step", "stream"):
        return {"case": case, "pipe": _pipeline(case, seed)}
    if kind == "core":
        return _core(case, seed)
    if kind == "flat":
        return {"case": case, "seed": 1 + seed}
    if kind == "queue":
        return {"case": case, "queue": TransportQueue(_queue_cases(case, seed), _dev())}
    if kind == "brem":
        grid, comp, n_hat, seg, w, thickness = _brem_inputs(case, seed)
        return {"case": case, "scorer": BremScorer(comp, grid, thickness, n_hat, _dev()), "seg": _put(seg),
                "w": None if w is None else torch.as_tensor(w, device=_dev())}
    if kind == "coherent":
        grid, tables, n_hats, weights, rows, count, factor, thickness = _coherent_inputs(case, seed)
        return {"case": case, "scorer": CoherentScorer(tables, "hopg", grid, thickness, n_hats, weights, _dev(),
                                                       grouped=case["grouped"]),
                "rows": _put(rows), "count": torch.as_tensor(count, device=_dev()),
                "factor": factor if case["grouped"] else None}
    inputs = _line_inputs if kind == "lines" else _pixel_inputs
    grid, tables, n_hats, weights, seg, w, thickness = inputs(case, seed)
    return {"case": case, "scorer": LineScorer(tables, grid, thickness, n_hats, weights, _dev()), "seg": _put(seg),
            "w": None if w is None else torch.as_tensor(w, device=_dev())}


def run(state):
    """One pass."""
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        pipe = state["pipe"]
        pipe.spec_lines.zero_()
        pipe.spec_brem.zero_()
        if case["split"]:
            pipe.step(0, case["batches"])
            pipe.flush_copies()
        else:
            pipe.run_steps(0, case["batches"])
        return {"lines": pipe.spec_lines, "brem": pipe.spec_brem}
    if kind == "stream":
        pipe = state["pipe"]
        pipe.spec_lines.zero_()
        pipe.spec_brem.zero_()
        res = pipe.stream(0, case["n"], lanes=case["lanes"], rows_per_round=case["rows"])
        return {"lines": pipe.spec_lines, "brem": pipe.spec_brem, "rows": res.n_segments}
    if kind == "flat":
        seg = simulate_trajectories(case["E0"], case["Ne"], thickness_ang=3.0e4, composition=FILM, seed=state["seed"],
                                    straggling=True, max_dE_frac=0.05 if case["substeps"] else 0.0)
        grid = _grid(case, 1000.0, 1000.0 * case["E0"])
        brem = mc_brem_spectrum(seg, grid, FILM, np.array([0.6, 0.0, -0.8]))
        keys = ("final_E_keV", "final_pos", "final_dirs", "exit_code", "seg_count", "straggle_dE_keV")
        return {"brem": brem, **{k: seg[k] for k in keys}}
    if kind == "core":
        now = state["state"]
        for k, v in state["entry"].items():
            now[k].copy_(v)
        state["core"]((0, case["Ne"], case["cap"], state["keys"]),
                      (state["alive"], now["clock"], now["pos"], now["dirs"], now["E"], state["E_cut"]),
                      state["rows"], (state["count"], state["code"]), (True, state["straggle"]),
                      stream=torch.cuda.current_stream().cuda_stream)
        return {**state["rows"], **now, "straggle": state["straggle"], "count": state["count"], "code": state["code"]}
    if kind == "queue":
        return state["queue"].run()
    sc = state["scorer"]
    if kind == "lines":
        return sc.spectrum(state["seg"], case["n"], row_weight=state["w"])
    if kind == "pixels":
        return sc.window_spectra(state["seg"], case["n"])
    if kind == "brem":
        return sc.spectrum(state["seg"], case["n"], row_weight=state["w"])
    sc.reset()
    sc.add_slots([(0, case["n"], case["slots"], state["rows"], state["count"])], case["n"])
    out = {"spectrum": sc.spectrum(factor=state["factor"]), "field": sc.field}
    if case["grouped"]:
        out["grouped"] = sc.grouped
    return out


# ------------------------------------------------------------------ work and tolerance
# Operations of one unit, an FMA as two and a transcendental as 20 (40 in FP64): transport step,
# line prologue, sinc^2 cell, brem cell, coherent cell.
STEP_OPS, LINE_OPS, SINC_OPS, BREM_OPS, FIELD_OPS = 330, 540, 48, 125, 141
ROW_BYTES = 113


def work(case):
    kind = case["kind"]
    n_E = case.get("n_bins", 0)
    if kind == "step":
        rows = ROWS["hopg"] * case["Ne"] * case["batches"]
        lines = rows * case["n_side"] ** 2
        return {"bytes": rows * 2 * ROW_BYTES,
                "flops": rows * STEP_OPS + lines * (LINE_OPS + 0.5 * SINC_OPS * n_E) + rows * n_E * BREM_OPS}
    if kind == "stream":
        rows = ROWS["silicon"] * case["n"]
        lines = rows * 9 * case["reflections"]
        return {"bytes": rows * 2 * ROW_BYTES,
                "flops": rows * (STEP_OPS + n_E * BREM_OPS) + lines * (LINE_OPS + 6 * SINC_OPS)}
    if kind == "flat":
        rows = case["Ne"] * ROWS["film"]
        return {"bytes": rows * ROW_BYTES, "flops": rows * (STEP_OPS + 0.3 * n_E * 2 * BREM_OPS)}
    if kind == "core":
        rows = case["Ne"] * ROWS[case["target"]]
        return {"bytes": min(rows, case["Ne"] * case["cap"]) * ROW_BYTES, "flops": rows * STEP_OPS}
    if kind == "queue":
        rows = sum(q.Ne * ROWS[q.material] * q.thickness_ang / 1.0e6 for q in _queue_cases(case, 0))
        return {"bytes": 8 * 12 * 8, "flops": rows * STEP_OPS}
    n = case["n"]
    if kind == "coherent":
        lines = 0.5 * n * case["slots"] * case["n_side"] ** 2
        cells = lines * n_E * (2 if case["grouped"] else 1)
        return {"bytes": 0.5 * n * case["slots"] * 88 + case["n_side"] ** 2 * 4 * n_E * 8,
                "flops": lines * LINE_OPS + 0.5 * cells * FIELD_OPS}
    if kind == "brem":
        share = 0.75 if case["weighted"] else 1.0
        return {"bytes": n * 36 + n_E * 24, "flops": share * n * n_E * len(COMPOSITIONS[case["composition"]]) * BREM_OPS}
    if kind == "pixels":
        lines = n * case["n_g"] * case["n_side"] ** 2
        return {"bytes": n * 32 + case["n_side"] ** 2 * n_E * 8, "flops": lines * (LINE_OPS + 6 * SINC_OPS)}
    lines = n * case["n_side"] ** 2 * (1 if case["target"] == "hopg" else 4)
    live = 0.5 * (0.75 if case["weighted"] else 1.0)
    return {"bytes": n * 36 + n_E * 16, "flops": lines * (LINE_OPS + live * SINC_OPS * n_E)}


def tolerance(case):
    """Relative errors another correct implementation at this precision shows."""
    if case["kind"] in ("core", "queue"):
        # FP64 throughout: rows differ by the rounding of the math library only
        return {"rel": 1.0e-9}
    if case["kind"] == "coherent":
        # FP32 profiles and phase rotations of fields that cancel, squared: up to 5e-7 against 64 bits
        return {"rel": 2.0e-6}
    # FP32 cells with FP64 phases and sums: up to 2.5e-7 against 64 bits, 5e-7 in a single cell
    return {"rel": 1.0e-6}


# ------------------------------------------------------------------ the same results in 64 bits
HBARC, ALPHA, MC2_EV = 1973.269804, 1.0 / 137.035999, 510998.95


def _t(x):
    return torch.as_tensor(np.asarray(x, dtype=np.float64), device="cuda" if torch.cuda.is_available() else "cpu")


def _interp(grid, f, x, i):
    """Linear interpolation in the bracket (i-1, i), the end values outside the grid."""
    y = f[i - 1] + (x - grid[i - 1]) / (grid[i] - grid[i - 1]) * (f[i] - f[i - 1])
    y = torch.where(x <= grid[0], f[0], y)
    return torch.where(x >= grid[-1], f[-1], y)


def _escape_path(z, thickness, nz):
    depth = z.clamp(0.0, thickness)
    inv = 1.0 / max(abs(nz), 1.0e-12)
    return depth * inv if nz < 0.0 else (thickness - depth) * inv


def _exact_kinematics(tables, n_hat, thickness, z, v, L, E, g):
    """Resonance, width slope and both complex amplitudes of every segment for reflection ``g``."""
    grid = _t(tables.E_tab)
    nx, ny, nz = (float(c) for c in n_hat)
    G = [float(c) for c in tables.g[g]]
    gamma = 1.0 + E / (MC2_EV / 1.0e3)
    beta = torch.sqrt(1.0 - 1.0 / gamma**2)
    vel = [beta * v[:, k] for k in range(3)]
    miss = (v[:, 0] - nx) ** 2 + (v[:, 1] - ny) ** 2 + (v[:, 2] - nz) ** 2
    denom_row = 1.0 / (gamma**2 * (1.0 + beta)) + 0.5 * beta * miss
    slope_z = torch.where((z < 0.0) | (z > thickness), torch.zeros_like(z), torch.full_like(z, -1.0 / nz))
    inv_E = HBARC / (gamma * MC2_EV)
    g2 = sum(c * c for c in G)
    n_dot_g = G[0] * nx + G[1] * ny + G[2] * nz
    vdg = vel[0] * G[0] + vel[1] * G[1] + vel[2] * G[2]
    r_num, r_den = 0.5 * g2 * inv_E, n_dot_g * inv_E
    vacuum = denom_row + r_den
    denom, previous, delta = vacuum, vacuum, torch.zeros_like(vacuum)
    table = _t(tables.delta_tab)
    for _ in range(3):
        x = HBARC * ((vdg - r_num) / denom)
        i = torch.searchsorted(grid, x).clamp(1, grid.numel() - 1)
        delta = _interp(grid, table, x, i)
        previous, denom = denom, vacuum - delta * (vel[2] * slope_z)
    settled = ((denom - previous).abs() <= 1.0e-3 * denom.abs()) & (2.0 * delta.abs() * slope_z**2 < 1.0)
    omega = (vdg - r_num) / denom
    E_res = HBARC * omega
    oe = omega * inv_E
    keep = (settled & (E_res > tables.lo_keep) & (E_res > 10.0) & (E_res < tables.hi_keep) & (denom > 0.0)
            & (oe <= 1.0 - 1.0 / gamma))
    safe = torch.where(keep, E_res, torch.full_like(E_res, float(tables.lo_keep) + 1.0))
    i = torch.searchsorted(grid, safe).clamp(1, grid.numel() - 1)
    row = int(tables.row[g])
    chi = torch.complex(*(_interp(grid, _t(t[row]), safe, i) for t in (tables.chi_re, tables.chi_im)))
    u = torch.complex(*(_interp(grid, _t(t[row]), safe, i) for t in (tables.u_re, tables.u_im)))
    frac = torch.log(torch.minimum(torch.maximum(safe, grid[i - 1]), grid[i]) / grid[i - 1])
    frac = frac / torch.log(grid[i] / grid[i - 1])
    mu = torch.zeros_like(safe)
    for el in tables.log_mu:
        lm = _t(el)
        y = lm[i - 1] + frac * (lm[i] - lm[i - 1])
        y = torch.where(safe <= grid[0], lm[0], torch.where(safe >= grid[-1], lm[-1], y))
        mu = mu + torch.exp(y)
    h = HBARC / MC2_EV
    k_dot_v = omega * ((1.0 - denom) + r_den)
    k_dot_g = omega * (n_dot_g + delta * (slope_z * G[2]))
    k2 = omega**2 * torch.where(slope_z == 0.0, torch.ones_like(delta), 1.0 - 2.0 * delta + (delta * slope_z) ** 2)
    n_1 = h * g2 - 2.0 * gamma * vdg
    n_2 = n_1 + 2.0 * h * k_dot_g
    n_f = h * (g2 + 2.0 * k_dot_g + k2) - 2.0 * gamma * (vdg + k_dot_v)
    e_1 = torch.sqrt(gamma**2 + h * n_1)
    e_2 = torch.sqrt(gamma**2 + h * (h * k2 - 2.0 * gamma * k_dot_v))
    e_f = torch.sqrt(gamma**2 + h * n_f)
    amplitude = []
    e_s = np.cross(n_hat, tables.g[g])
    if np.linalg.norm(e_s) < 1e-12:
        e_s = np.cross(n_hat, [0.0, 1.0, 0.0])
    e_s = e_s / np.linalg.norm(e_s)
    e_p = np.cross(e_s, n_hat)
    for e in (e_s, e_p / np.linalg.norm(e_p)):
        v_dot_e = vel[0] * e[0] + vel[1] * e[1] + vel[2] * e[2]
        k_dot_e = omega * delta * (slope_z * e[2])
        g_dot_e = float(G[0] * e[0] + G[1] * e[1] + G[2] * e[2])
        pxr = (-n_f * (g_dot_e + k_dot_e) - k2 * (2.0 * gamma * v_dot_e - h * (g_dot_e + k_dot_e))) / (gamma + e_f)
        pxr = pxr / (g2 + 2.0 * k_dot_g)
        x = 2.0 * gamma * v_dot_e - h * k_dot_e
        cbs = 2.0 * g_dot_e * (e_1 + gamma) / ((e_1 + e_f) * n_1)
        cbs = cbs + x * (n_1 * n_f / (gamma + e_f) * (gamma + e_f + e_1 + e_2)
                         - 2.0 * (e_1 + gamma) * (gamma + e_2) * k_dot_g) / ((e_1 + e_f) * (gamma + e_2) * n_1 * n_2)
        amplitude.append(chi * pxr + u * cbs)
    half = 0.5 * L * v[:, 2]
    return dict(keep=keep, E_res=E_res, omega=omega, slope=denom / (1.0 - oe), mu=mu, amplitude=amplitude,
                t_L=L / beta, path0=_escape_path(z - half, thickness, nz), path1=_escape_path(z + half, thickness, nz),
                denom_row=denom_row, r_num=r_num, r_den=r_den, vdg=vdg, inv_E=inv_E)


def _mean_escape(t0, t1):
    """Mean of exp(-t) for t running evenly from t0 to t1."""
    d = (t1 - t0).abs()
    ratio = torch.where(d > 1.0e-4, -torch.expm1(-d) / d.clamp(min=1.0e-300), 1.0 - 0.5 * d + d * d / 6.0)
    return torch.exp(-torch.minimum(t0, t1)) * ratio


def _exact_lines(inputs, case, d, g):
    """(E_r, a, w) of the live lines of ray ``d`` and reflection ``g``."""
    _grid_E, tables, n_hats, weights, seg, row_weight, thickness = inputs
    v = _t(seg["v_hat"])
    k = _exact_kinematics(tables, n_hats[d], thickness, _t(seg["r_mid"])[:, 2], v, _t(seg["L"]), _t(seg["E"]), g)
    power = sum(a.real**2 + a.imag**2 for a in k["amplitude"])
    w = ALPHA * k["omega"] / (4.0 * math.pi**2 * HBARC) * k["t_L"] ** 2 * power * float(tables.wm[g])
    w = w * _mean_escape(k["path0"] * k["mu"], k["path1"] * k["mu"]) * float(weights[d]) / case["n"]
    if row_weight is not None:
        w = w * _t(row_weight)
    live = k["keep"] & torch.isfinite(w) & (w > 0.0)
    return k["E_res"][live], (k["slope"] * k["t_L"])[live] / (2.0 * HBARC), w[live]


def _exact_dense(case, seed):
    inputs = _line_inputs(case, seed)
    E = _t(inputs[0])
    out = torch.zeros_like(E)
    for d in range(len(inputs[3])):
        for g in range(len(inputs[1].wm)):
            E_r, a, w = _exact_lines(inputs, case, d, g)
            for lo in range(0, E_r.numel(), 1 << 15):
                s = slice(lo, lo + (1 << 15))
                out += w[s] @ torch.sinc(a[s, None] * (E[None, :] - E_r[s, None]) / math.pi) ** 2
    return out


def _exact_pixels(case, seed, x_c=100.0):
    """Exact profile on the nodes within x_c of a line, its cycle-averaged expansion beyond."""
    inputs = _pixel_inputs(case, seed)
    E = _t(inputs[0])
    n, E0, dE = E.numel(), float(inputs[0][0]), float((inputs[0][-1] - inputs[0][0]) / max(1, inputs[0].size - 1))
    out = torch.zeros((len(inputs[3]), n), dtype=E.dtype, device=E.device)
    step = torch.arange(-(2 * n), n + n, device=E.device, dtype=E.dtype) * dE  # offsets of a node to a bin
    inv = torch.where(step == 0.0, 0.0, 1.0 / step)
    # offsets[e, q] = e - (q - n) for node slots q in [0, 3n)
    index = torch.arange(n, device=E.device)[:, None] - torch.arange(3 * n, device=E.device)[None, :] + n + 2 * n
    for d in range(len(inputs[3])):
        moments = torch.zeros((3, 3 * n), dtype=E.dtype, device=E.device)
        parts = [_exact_lines(inputs, case, d, g) for g in range(len(inputs[1].wm))]
        E_r, a, w = (torch.cat(p) for p in zip(*parts))
        ok = a > 0.0
        E_r, a, w = E_r[ok], a[ok], w[ok]
        node = torch.round((E_r - E0) / dE)
        eps = E_r - (E0 + node * dE)
        reach = torch.ceil((eps.abs() + x_c / a) / dE)
        lo = (node - reach).clamp(min=0.0)
        hi = (node + reach).clamp(max=n - 1.0)
        windowed = (node >= -n) & (node < 2 * n) & ((hi - lo + 1.0) < 0.25 * n)
        for s in (slice(k, k + 4096) for k in range(0, int((~windowed).sum()), 4096)):
            Eb, ab, wb = E_r[~windowed][s], a[~windowed][s], w[~windowed][s]
            out[d] += wb @ torch.sinc(ab[:, None] * (E[None, :] - Eb[:, None]) / math.pi) ** 2
        order = torch.argsort(reach[windowed])
        E_r, a, w, node, eps, reach, lo, hi = (t[windowed][order] for t in (E_r, a, w, node, eps, reach, lo, hi))
        m2 = 0.5 / a**2
        m3, m4 = 2.0 * eps * m2, 3.0 * eps**2 * m2
        for k, m in enumerate((m2, m3, m4)):
            moments[k].index_add_(0, node.long() + n, w * m)
        start = 0
        while start < E_r.numel():  # lines of similar reach together
            stop = min(E_r.numel(), start + (1 << 17))
            width = int(reach[start:stop].max())
            if width > 64:
                stop = min(stop, start + 4096)
                width = int(reach[start:stop].max())
            s = slice(start, stop)
            off = torch.arange(-width, width + 1, device=E.device, dtype=E.dtype)
            e = node[s, None] + off
            x = off * dE
            ix = torch.where(off == 0.0, 0.0, 1.0 / x)
            cell = torch.sinc(a[s, None] * ((E0 + e * dE) - E_r[s, None]) / math.pi) ** 2
            cell = cell - (m2[s, None] + (m3[s, None] + m4[s, None] * ix) * ix) * ix**2
            cell = torch.where((e >= lo[s, None]) & (e <= hi[s, None]), w[s, None] * cell, 0.0)
            out[d].index_add_(0, e.clamp(0, n - 1).long().reshape(-1), cell.reshape(-1))
            start = stop
        used = moments.abs().sum(0) > 0.0
        K = inv[index[:, used]]
        out[d] += (K**2) @ moments[0, used] + (K**3) @ moments[1, used] + (K**4) @ moments[2, used]
    return out


def _exact_brem(case, seed):
    """Born cross section with the Elwert factor, averaged over the escape along each segment."""
    grid, comp, n_hat, seg, row_weight, thickness = _brem_inputs(case, seed)
    from pyrite_amd.transport.elements import TRANSPORT_ELEMENTS

    m = MC2_EV / 1.0e3
    k = _t(grid) * 1.0e-3
    mu = _t(attenuation.mu_total_inv_ang(comp, grid).astype(np.float32))
    T, L, z, vz = _t(seg["E"]), _t(seg["L"]), _t(seg["r_mid"])[:, 2], _t(seg["v_hat"])[:, 2]
    p_i = torch.sqrt(T * (T + 2.0 * m)) / m
    b_i = p_i / (1.0 + T / m)
    w = torch.ones_like(T) if row_weight is None else _t(row_weight)
    path = [_escape_path(z + sgn * 0.5 * L * vz, thickness, float(n_hat[2])) for sgn in (-1.0, 1.0)]
    total = torch.zeros_like(k)
    for lo in range(0, T.numel(), 1 << 14):
        s = slice(lo, lo + (1 << 14))
        T_f = T[s, None] - k[None, :]
        good = T_f > 1.0e-6
        T_f = torch.where(good, T_f, torch.ones_like(T_f))
        p_f = torch.sqrt(T_f * (T_f + 2.0 * m)) / m
        inv_b = (1.0 + T_f / m) / p_f
        born = torch.log((p_i[s, None] + p_f) ** 2 * m * m / (k[None, :] * (T[s, None] + T_f + 2.0 * m)))
        escape = _mean_escape(path[0][s, None] * mu[None, :], path[1][s, None] * mu[None, :])
        elwert = torch.zeros_like(T_f)
        for el, density in comp:
            c = 2.0 * math.pi * float(TRANSPORT_ELEMENTS[el]["Z"]) * ALPHA
            front = (density * 1.0e24 * L * 1.0e-8 * (16.0 / 3.0) * ALPHA * 7.9407877e-26
                     * float(TRANSPORT_ELEMENTS[el]["Z"]) ** 2 * b_i * -torch.expm1(-c / b_i) / p_i**2)
            elwert = elwert + (w * front)[s, None] / -torch.expm1(-c * inv_b)
        total += torch.where(good, elwert * born / _t(grid)[None, :] * inv_b * escape, 0.0).sum(0)
    return total / (4.0 * math.pi * case["n"])


def _exact_coherent(case, seed):
    """Fields of every segment with their phases and formation factors; squares per history."""
    grid, tables, n_hats, weights, rows, count, factor, thickness = _coherent_inputs(case, seed)
    n, slots = case["n"], case["slots"]
    live = (np.arange(slots)[None, :] < count[:, None]).reshape(-1)
    owner = torch.as_tensor(np.repeat(np.arange(n), slots)[live], device=_t(0.0).device)
    r, v, L, t0 = (_t(rows[k][live]) for k in ("seg_mid", "seg_dir", "seg_len", "seg_t0"))
    T = _t(0.5 * (rows["seg_E"] + rows["seg_E_end"])[live])
    E, dom = _t(grid), _t(escape_phase_rate("hopg", grid))
    n_E = E.numel()
    field = torch.zeros((len(weights), 4, n_E), dtype=E.dtype, device=E.device)
    grouped = torch.zeros((len(weights), n_E), dtype=E.dtype, device=E.device)
    chunk = max(1, (1 << 24) // n_E)
    bounds = np.concatenate([[0], np.cumsum(count)])
    for d, n_hat in enumerate(n_hats):
        k = _exact_kinematics(tables, n_hat, thickness, r[:, 2], v, L, T, 0)
        centre = (k["vdg"] - k["r_num"]) / (k["denom_row"] + k["r_den"])
        x = centre * k["inv_E"]
        kappa = 1.0 / (1.0 - x)
        age = t0 + 0.5 * k["t_L"]
        nh = _t(n_hat)
        retard = (age - r @ nh + kappa * (x * k["denom_row"] + k["r_den"]) * age) / HBARC
        lattice = r @ _t(tables.g[0]) + kappa * (x * k["vdg"] - k["r_num"]) * age
        width = kappa * (k["denom_row"] + k["r_den"]) * k["t_L"] / (2.0 * HBARC)
        scale = torch.sqrt(ALPHA * k["omega"].clamp(min=0.0) / (4.0 * math.pi**2 * HBARC)) * k["t_L"]
        tau0, tau1 = k["path0"] * k["mu"], k["path1"] * k["mu"]
        q = 0.25 * (tau1 - tau0)
        keep = k["keep"]
        first = 0
        while first < n:
            last = int(np.searchsorted(bounds, bounds[first] + chunk, side="right")) - 1
            last = min(max(last, first + 1), n)
            s = slice(int(bounds[first]), int(bounds[last]))
            lateral = 0.5 * (k["path1"] - k["path0"])[s, None] * dom
            arg = width[s, None] * (E - HBARC * centre[s, None]) - lateral
            phase = retard[s, None] * E - lattice[s, None] - 0.5 * (k["path0"] + k["path1"])[s, None] * dom
            w = torch.complex(-q[s, None].expand_as(arg), arg)
            ratio = torch.where(w.abs() < 1.0e-5, 1.0 + w * w / 6.0, torch.sinh(w) / torch.where(w == 0, 1.0, w))
            F = torch.exp(-0.25 * (tau0 + tau1))[s, None] * ratio * torch.exp(1j * phase)
            sums = []
            for a in k["amplitude"]:
                c = torch.where(keep[s], scale[s] * a[s], torch.zeros_like(a[s]))
                sums.append(torch.where(keep[s, None], c[:, None] * F, torch.zeros_like(F)))
            for pol in range(2):
                total = sums[pol].sum(0)
                field[d, 2 * pol] += total.real
                field[d, 2 * pol + 1] += total.imag
                if case["grouped"]:
                    per = torch.zeros((last - first, n_E), dtype=F.dtype, device=F.device)
                    per.index_add_(0, owner[s] - first, sums[pol])
                    grouped[d] += (per.real**2 + per.imag**2).sum(0)
            first = last
    power = (field**2).sum(1)
    if case["grouped"]:
        F = _t(factor)
        power = (1.0 - F) * grouped + F * power
    out = {"spectrum": (_t(weights)[:, None] * power * float(tables.wm[0])).sum(0) / n, "field": field}
    if case["grouped"]:
        out["grouped"] = grouped
    return out


def exact(case, seed):
    """The case's results in 64 bits, or None for Monte Carlo transport."""
    kind = case["kind"]
    if kind in ("step", "stream", "flat", "core", "queue"):
        return None
    return {"lines": _exact_dense, "pixels": _exact_pixels, "brem": _exact_brem, "coherent": _exact_coherent}[kind](
        case, seed)
