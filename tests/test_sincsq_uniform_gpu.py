"""The sinc^2 reductions at the edges of their windows, runs, chunks and tiles (GPU).

Against the FP64 profile in numpy.  The bound: a cell's factor x carries the
rounding of the sine, the two of the distance, the reciprocal's ulp and the
product (6 x 2^-24), squared and summed in FP32 groups of four, 1e-6 of the sum
in all; the stepped sines are off by at most 1e-10 of their envelope, which a
square turns into 2e-10 of the envelope (w at the centre, w/(pi u)^2 beyond)."""

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _lines(rng, n, E0, dE, n_E):
    """Lines across the grid and beyond it, of every width: far narrower than a bin
    to far wider than the grid; some centred on a bin or half way, some without
    weight, one flat (a = 0) and one of negative weight."""
    E_r = E0 + dE * rng.uniform(-1.5 * n_E - 3, 2.5 * n_E + 3, n)
    on = rng.random(n)
    k = rng.integers(0, n_E, n)
    E_r = np.where(on < 0.2, E0 + dE * k, np.where(on < 0.3, E0 + dE * (k + 0.5), E_r))
    a = np.exp(rng.uniform(np.log(1e-9), np.log(2e3), n)) / abs(dE)
    w = np.where(rng.random(n) < 0.2, 0.0, rng.uniform(1e-3, 1.0, n)).astype(np.float32)
    if n > 6:
        a[3] = 0.0
        w[3], w[5] = 0.5, -0.25
    return E_r, a, w


def _reduce(E_r, a, w, E0, dE, n_E, device):
    import torch

    from pyrite_amd import _lib

    t = [torch.as_tensor(v, device=device) for v in (E_r, a, w)]
    out = torch.full((n_E,), 0.125, dtype=torch.float64, device=device)
    args = _lib.SincsqArgs()
    args.n_lines, args.E_r, args.a, args.w = E_r.size, *(v.data_ptr() for v in t)
    args.n_E, args.E_grid, args.uniform, args.E0, args.dE = n_E, None, 1, E0, dE
    args.out = out.data_ptr()
    args.ws = _lib.DeviceScratch(device).get(_lib.workspace_bytes("hr_sincsq_workspace_bytes", C.byref(args)))
    _lib.check(_lib.load().hr_sincsq_reduce(C.byref(args), C.c_void_p(torch.cuda.current_stream().cuda_stream)),
               "hr_sincsq_reduce")
    return out.cpu().numpy() - 0.125


@pytest.mark.parametrize("n_E", [1, 2, 63, 64, 255, 256, 257, 777, 1024, 1025, 1400, 3001])
@pytest.mark.parametrize("n_lines", [1, 8, 9, 700, 40_000])
def test_uniform_reduction_matches_fp64(device, n_E, n_lines):
    rng = np.random.default_rng([n_E, n_lines])
    E0, dE = 1000.0, (47.9, -3.5)[n_E % 2]
    if n_lines > 1000 and n_E > 1100:
        n_lines = 5000
    E_r, a, w = _lines(rng, n_lines, E0, dE, n_E)
    got = _reduce(E_r, a, w, E0, dE, n_E, device)
    k = np.arange(n_E)
    want, envelope = np.zeros(n_E), np.zeros(n_E)
    for s in range(0, n_lines, 4096):
        al = (a[s:s + 4096] / np.pi)[:, None]
        u = k[None, :] * (al * dE) + al * (E0 - E_r[s:s + 4096])[:, None]
        wl = w[s:s + 4096].astype(float)[:, None]
        r = u - np.rint(u)
        cell = np.where(u == 0.0, 1.0, np.sin(np.pi * r) / (np.pi * np.where(u == 0.0, 1.0, u))) ** 2
        want += (wl * cell).sum(0)
        envelope += (np.abs(wl) / np.maximum(1.0, (np.pi * u) ** 2)).sum(0)
        want_abs = (np.abs(wl) * cell).sum(0) if s == 0 else want_abs + (np.abs(wl) * cell).sum(0)
    assert np.isfinite(got).all()
    assert np.all(np.abs(got - want) <= 1e-6 * want_abs + 1e-9 * envelope + 1e-15), \
        float(np.max(np.abs(got - want) / (1e-6 * want_abs + 1e-9 * envelope + 1e-15)))


def test_step_of_zero_takes_the_general_reducer(device):
    """A uniform grid whose bins coincide: every bin the same profile."""
    E_r, a, w = np.array([10.0, 12.0]), np.array([0.7, 0.2]), np.array([1.0, 0.5], dtype=np.float32)
    got = _reduce(E_r, a, w, 11.0, 0.0, 5, device)
    want = float((w * np.sinc(a * (11.0 - E_r) / np.pi) ** 2).sum())
    np.testing.assert_allclose(got, want, rtol=1e-6)


def _errors(rng, device, n, n_E, du, centre, draws):
    """Relative error of the spectrum (2-norm) and of its sum, of `draws` sets of `n`
    lines whose width is a decade of bins about ``du`` turns and whose centres are
    ``centre(k)`` for bins k."""
    E0, dE = 1000.0, 47.9
    norm, mean = [], []
    for _ in range(draws):
        d = du * 10.0 ** rng.uniform(-0.5, 0.5, n)
        E_r = E0 + dE * centre(rng.integers(0, n_E, n), d)
        a, w = np.pi * d / dE, rng.uniform(1e-3, 1.0, n).astype(np.float32)
        got, want = _reduce(E_r, a, w, E0, dE, n_E, device), np.zeros(n_E)
        for s in range(0, n, 65536):
            al = (a[s:s + 65536] / np.pi)[:, None]
            u = np.arange(n_E)[None, :] * (al * dE) + al * (E0 - E_r[s:s + 65536])[:, None]
            r = u - np.rint(u)
            cell = np.where(u == 0.0, 1.0, np.sin(np.pi * r) / (np.pi * np.where(u == 0.0, 1.0, u))) ** 2
            want += (w[s:s + 65536].astype(float)[:, None] * cell).sum(0)
        norm.append(np.linalg.norm(got - want) / np.linalg.norm(want))
        mean.append((got - want).sum() / want.sum())
    return float(np.sqrt(np.mean(np.square(norm)))), float(np.mean(mean))


# An FP32 rounding leaves 2^-24 / sqrt(3) x sqrt(E 1/m^2) = 2.5e-8 of a value m of logarithmic
# density (root mean square).  A cell of the central half period carries the polynomial's last
# step twice (squared), the square's, and the weighted sum's: sqrt(4 + 1 + 1) of these.  Cells
# beyond it, with 12 % of the profile's squared 2-norm (integral of sinc^4), carry up to 1.2e-7:
# the phase's rounding twice, the reciprocal's 2.8e-8 and the products' besides.
CENTRAL = 6.2e-8
PROFILE = (0.88 * CENTRAL**2 + 0.12 * 1.2e-7**2) ** 0.5


@pytest.mark.parametrize("n", [1, 20])
@pytest.mark.parametrize("du", [1e-3, 0.03, 0.3])
def test_lines_wider_than_a_bin_carry_one_rounding_at_the_centre(device, n, du):
    rng = np.random.default_rng([n, int(1e4 * du)])
    norm, _ = _errors(rng, device, n, 512, du, lambda k, d: k + rng.uniform(-0.5, 0.5, k.size), 60)
    assert norm < PROFILE


@pytest.mark.parametrize("n", [1, 20, 2000])
def test_narrow_lines_on_a_bin_carry_one_rounding_at_the_centre(device, n):
    rng = np.random.default_rng(n)
    norm, _ = _errors(rng, device, n, 512, 30.0, lambda k, d: k + rng.uniform(-0.4, 0.4, k.size) / d, 60)
    assert norm < CENTRAL


def test_sums_of_many_distant_cells_have_no_common_error(device):
    """The cells' common relative error: the weights' and sums' roundings have none, the
    reciprocal's mean (6.4e-9, twice in a square) is taken off.  What is left is the
    statistical rest of 2e5 lines that fall between bins, 1.1e-7 / sqrt(2e5) with the
    spread of their sizes, and the profiles' (0.5 units in the ninth digit)."""
    rng = np.random.default_rng(5)
    _, mean = _errors(rng, device, 200_000, 40, 300.0, lambda k, d: k + rng.uniform(0.2, 0.8, k.size), 2)
    assert abs(mean) < 4e-9


def test_lines_without_a_finite_phase_have_a_profile_of_one(device):
    E_r = np.array([np.nan, 1200.0, np.inf, 1300.0])
    a = np.array([0.1, np.inf, 0.1, np.nan])
    w = np.array([1.0, 2.0, 4.0, 8.0], dtype=np.float32)
    np.testing.assert_array_equal(_reduce(E_r, a, w, 1000.0, 47.9, 300, device), 15.0)


@pytest.mark.parametrize("n_E", [1_048_577, 1_500_000, 2_097_152])
def test_static_scratch_takes_grids_of_two_million_bins(device, n_E):
    """The static array holds the partial rows of every grid up to 2^21 bins, at line
    counts that take chunks of 64 (1,024 lines and more where windows outnumber blocks)."""
    import torch

    from pyrite_amd import _lib

    rng = np.random.default_rng(n_E)
    E0, dE, n = 1000.0, 0.05, 1100
    E_r, a, w = E0 + dE * n_E * rng.random(n), 3.0 * rng.random(n) / dE, rng.random(n).astype(np.float32)
    t = [torch.as_tensor(v, device=device) for v in (E_r, a, w)]
    out = torch.zeros(n_E, dtype=torch.float64, device=device)
    args = _lib.SincsqArgs()
    args.n_lines, args.E_r, args.a, args.w = n, *(v.data_ptr() for v in t)
    args.n_E, args.E_grid, args.uniform, args.E0, args.dE, args.out = n_E, None, 1, E0, dE, out.data_ptr()
    _lib.check(_lib.load().hr_sincsq_reduce_static(C.byref(args), C.c_void_p(torch.cuda.current_stream().cuda_stream)),
               "hr_sincsq_reduce_static")
    got = out.cpu().numpy()
    np.testing.assert_allclose(got, _reduce(E_r, a, w, E0, dE, n_E, device), rtol=0, atol=1e-14)
    k = np.unique(np.concatenate([[0, n_E - 1], rng.integers(0, n_E, 300), np.rint((E_r[:100] - E0) / dE).astype(int)]))
    k = k[k < n_E]
    want = (w.astype(float)[:, None] * np.sinc((a / np.pi)[:, None] * (E0 + dE * k - E_r[:, None])) ** 2).sum(0)
    assert np.all(np.abs(got[k] - want) <= 1e-6 * want + 1e-9)


# Lines that make a wave's chunk 16, 32 and 64 on 256 CUs and one window of bins (8 below the
# first): 16 waves a CU with four chunks each, 256 x 16 x 4 x the chunk.  Chunks of 64 also take
# four times the resident blocks.
CHUNK_LINES = {16: 262_144, 32: 524_288, 64: 1_048_576}


@pytest.mark.parametrize("n_E", [61, 777])
@pytest.mark.parametrize("chunk", list(CHUNK_LINES))
def test_long_chunks_match_fp64(device, chunk, n_E):
    """Ragged last chunks, runs of lines without weight as long as several chunks, and eighths
    that are alive, dead and partly dead, against torch in FP64."""
    import torch

    from pyrite_amd import _lib

    rng = np.random.default_rng([chunk, n_E])
    n, E0, dE = CHUNK_LINES[chunk] + 77, 1000.0, 47.9
    E_r, a, w = _lines(rng, n, E0, dE, n_E)
    w[:chunk * 8] = rng.uniform(0.5, 1.0, chunk * 8)          # every eighth alive
    w[chunk * 8:chunk * 24] = 0.0                              # whole chunks dead
    w[chunk * 24:chunk * 40].reshape(-1, 8)[::3] = 0.0         # every third eighth dead
    w[chunk * 40:chunk * 56].reshape(-1, 8)[:, 1:7] = 0.0      # eighths with their ends alive
    dead = np.repeat(rng.random(n // 1000 + 1) < 0.3, 1000)[:n]
    w[chunk * 56:][dead[chunk * 56:]] = 0.0
    args = _lib.SincsqArgs()
    args.n_lines, args.n_E, args.uniform, args.E0, args.dE = n, n_E, 1, E0, dE
    rows = _lib.workspace_bytes("hr_sincsq_workspace_bytes", C.byref(args)) // (8 * n_E)
    if torch.cuda.get_device_properties(device).multi_processor_count == 256:
        assert rows == (4096 if chunk == 64 else 1024)
    got = _reduce(E_r, a, w, E0, dE, n_E, device)
    t = [torch.as_tensor(v, dtype=torch.float64, device=device) for v in (E_r, a, w)]
    want, size, envelope = (torch.zeros(n_E, dtype=torch.float64, device=device) for _ in range(3))
    k = torch.arange(n_E, dtype=torch.float64, device=device)
    for s in range(0, n, 1 << 16):
        Er, al, wl = (v[s:s + (1 << 16), None] for v in t)
        al = al / np.pi
        u = k * (al * dE) + al * (E0 - Er)
        r = u - torch.round(u)
        cell = torch.where(u == 0.0, 1.0, torch.sin(np.pi * r) / (np.pi * torch.where(u == 0.0, 1.0, u))) ** 2
        want += (wl * cell).sum(0)
        size += (wl.abs() * cell).sum(0)
        envelope += (wl.abs() / torch.clamp((np.pi * u) ** 2, min=1.0)).sum(0)
    bound = (1e-6 * size + 1e-9 * envelope + 1e-15).cpu().numpy()
    assert np.all(np.abs(got - want.cpu().numpy()) <= bound), float(np.max(np.abs(got - want.cpu().numpy()) / bound))


@pytest.mark.parametrize("n_E", [2, 63, 65, 256, 257, 700, 1024, 1025])
@pytest.mark.parametrize("n", [1, 63, 65, 1200, 140_000])
def test_general_grid_matches_fp64(device, n, n_E):
    """A grid without a step at the edges of tiles of 64 lines, runs of 64 bins and windows of
    1,024, one block to a tile until 8 a CU share them."""
    import torch

    from pyrite_amd import _lib

    rng = np.random.default_rng([n, n_E])
    grid = np.geomspace(1000.0, 50_000.0, n_E)
    E_r, a, w = _lines(rng, n, 1000.0, 49_000.0 / n_E, n_E)
    t = [torch.as_tensor(v, device=device) for v in (E_r, a, w, grid)]
    out = torch.zeros(n_E, dtype=torch.float64, device=device)
    args = _lib.SincsqArgs()
    args.n_lines, args.E_r, args.a, args.w = n, *(v.data_ptr() for v in t[:3])
    args.n_E, args.E_grid, args.uniform, args.out = n_E, t[3].data_ptr(), 0, out.data_ptr()
    need = _lib.workspace_bytes("hr_sincsq_workspace_bytes", C.byref(args))
    blocks = 8 * torch.cuda.get_device_properties(device).multi_processor_count // ((n_E + 1023) // 1024)
    assert need == 8 * n_E * min(blocks, (n + 63) // 64)
    args.ws = _lib.DeviceScratch(device).get(need)
    _lib.check(_lib.load().hr_sincsq_reduce(C.byref(args), C.c_void_p(torch.cuda.current_stream().cuda_stream)),
               "hr_sincsq_reduce")
    want, size = (torch.zeros(n_E, dtype=torch.float64, device=device) for _ in range(2))
    for s in range(0, n, 1 << 15):
        Er, al, wl = (v[s:s + (1 << 15), None].double() for v in t[:3])
        u = al / np.pi * (t[3] - Er)
        cell = torch.where(u == 0.0, 1.0,
                           torch.sin(np.pi * (u - torch.round(u))) / (np.pi * torch.where(u == 0.0, 1.0, u))) ** 2
        want += (wl * cell).sum(0)
        size += (wl.abs() * cell).sum(0)
    assert bool(torch.all((out - want).abs() <= 1.0e-6 * size + 1.0e-15))
