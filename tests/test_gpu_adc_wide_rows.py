"""Density control of sets with view-dependent colour (SH rows of 9, 15 and 21 floats) and their moments, the
prune by screen radius, and the values that an MCMC relocation leaves."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

WIDTHS = {"mean3d": 3, "rotation": 4, "logscale": 3, "opacity": 1, "sh0": 3, "sh1": 9, "sh2": 15, "sh3": 21}
BASE = ("mean3d", "rotation", "logscale", "opacity", "sh0")


def _rows(n, seed, sh, kept=0.8):
    """Rows of which the share `kept` passes the opacity cut, a third of them candidates; sh0's first float
    names the row, and no moment is 0."""
    rng = np.random.default_rng(seed)
    names = list(WIDTHS)[: 5 + sh]
    f = {k: rng.normal(size=(n, WIDTHS[k])) for k in names}
    f["logscale"] = rng.uniform(-6.0, -3.0, (n, 3))
    f["opacity"] = np.where(rng.random(n) < kept, rng.uniform(-1.0, 3.0, n), -8.0)
    f["sh0"][:, 0] = np.arange(n)
    f = {k: np.ascontiguousarray(v, np.float32) for k, v in f.items()}
    mom = {k: tuple((rng.random(v.shape) + 0.5).astype(np.float32) for _ in range(2)) for k, v in f.items()}
    return f, mom


def _buffer(a, cap, width):
    t = torch.zeros((cap, width) if width > 1 else (cap,), dtype=torch.float32, device="cuda")
    t[: a.shape[0]] = torch.from_numpy(a.reshape(a.shape[0], width) if width > 1 else a)
    return t


def _device(f, mom, cap):
    return ({k: _buffer(v, cap, WIDTHS[k]) for k, v in f.items()},
            {k: tuple(_buffer(m, cap, WIDTHS[k]) for m in v) for k, v in mom.items()})


@pytest.mark.parametrize("n,room,sh,algorithm,kept", [
    (1, 3, 1, 0, 1.0), (255, 300, 1, 1, 0.8), (256, 300, 2, 0, 0.8), (257, 60, 3, 1, 0.8), (1025, 1200, 3, 0, 1.0),
    (5000, 900, 2, 1, 0.9), (5000, 900, 3, 1, 0.5),
])
@pytest.mark.parametrize("screen", [None, "prunes", "too early"])
def test_refine_of_wide_rows(oracle, n, room, sh, algorithm, kept, screen):
    """Degree 0's fields equal the oracle's; every SH row is its source's, its moments the source's or, appended,
    0. With a screen radius the rows from before the growth are also subject to it, from the first reset on
    (gsx/src/gsx-cpu/adc/default.c:252-254)."""
    from gsx_amd.backend import DensityControl
    from oracle.oracle import AdcParams
    f, mom = _rows(n, 11 * n + sh, sh, kept)
    rng = np.random.default_rng(n + sh)
    aux = {"grad_acc": rng.random(n) * 1e-3, "absgrad_acc": rng.random(n) * 1e-3, "visible_counter": np.full(n, 2.0)}
    aux = {k: v.astype(np.float32) for k, v in aux.items()}
    cap = n + room
    params = dict(algorithm=algorithm, pruning_opacity_threshold=0.1, opacity_clamp_value=0.3, max_world_scale=0.0,
                  duplicate_grad_threshold=1e-4, duplicate_scale_threshold=0.02, duplicate_absgrad_threshold=2e-4,
                  scene_scale=1.0, refine_every=100, start_refine=0, end_refine=1000, max_num_gaussians=cap,
                  reset_every=200 if screen == "too early" else 70)
    print(f"[case] wide refine n={n} room={room} sh={sh} algorithm={algorithm} screen={screen}", flush=True)
    ref_f, ref_m, ref_counts = oracle.adc_step({k: f[k].copy() for k in BASE}, {k: mom[k] for k in BASE},
                                               {k: v.copy() for k, v in aux.items()},
                                               AdcParams(**params, global_step=100, seed=5), cap)
    radius = rng.random(n).astype(np.float32)
    radius[n // 2] = np.nan
    source = ref_f["sh0"][:, 0].astype(np.int64)
    appended = ref_m["sh0"][0][:, 0] == 0.0
    stay = np.ones(source.size, bool)
    if screen == "prunes":
        stay = appended | (radius[source] < 0.7)
        if not stay.any():  # one row always survives, the first
            pytest.skip("no row is left")
    d, m = _device(f, mom, cap)
    d.update({k: _buffer(v, cap, 1) for k, v in aux.items()})
    if screen is not None:
        d["max_screen_radius"] = _buffer(radius, cap, 1)
        params["max_screen_scale"] = 0.7
    o = {k: torch.zeros_like(v) for k, v in d.items()}
    om = {k: tuple(torch.zeros_like(t) for t in v) for k, v in m.items()}
    count, in_out, counts = DensityControl(params, seed=5).step(100, n, sh, d, m, cap, o, om)
    torch.cuda.synchronize()
    gone = int((~stay).sum())
    assert list(counts) == [ref_counts[0] + gone, *ref_counts[1:]]
    assert count == source.size - gone and in_out == (ref_counts[0] + gone > 0)
    res_f, res_m = (o, om) if in_out else (d, m)
    for k in f:
        want = ref_f[k] if k in BASE else f[k][source]
        assert np.array_equal(res_f[k][:count].cpu().numpy(), want[stay]), k
        for j in (0, 1):
            want = np.where(appended.reshape([-1] + [1] * (f[k].ndim - 1)), 0.0, mom[k][j][source])
            assert np.array_equal(res_m[k][j][:count].cpu().numpy(), want[stay].astype(np.float32)), (k, j)
    for k in set(d) - set(f):
        assert float(res_f[k][:count].abs().max()) == 0.0, k


def _libm():
    lib = ctypes.CDLL("libm.so.6")
    for name, args in (("expf", 1), ("logf", 1), ("powf", 2)):
        fn = getattr(lib, name)
        fn.restype, fn.argtypes = ctypes.c_float, [ctypes.c_float] * args
    return lib


def _relocated(lib, opacity, logscale, draws, min_opacity):
    """gsx/src/gsx-cpu/adc/mcmc.c:283-343 in its own float operations: the opacity that a source drawn `draws`
    times and its copies share, and their scales."""
    one = np.float32(1.0)
    so = one / (one + np.float32(lib.expf(-opacity)))
    ratio = min(draws + 1, 51)
    clamped = min(max(so, np.float32(0.0)), one - np.float32(1e-6))
    new = one - np.float32(lib.powf(one - clamped, one / np.float32(ratio)))
    denom = np.float32(0.0)
    for a in range(1, ratio + 1):
        for k in range(a):
            choose, lower = 1.0, min(k, a - 1 - k)
            for j in range(1, lower + 1):
                choose = choose * (a - 1 - (lower - j)) / j
            sign = one if k % 2 == 0 else -one
            denom = denom + np.float32(choose) * sign * np.float32(lib.powf(new, np.float32(k + 1))) / np.sqrt(
                np.float32(k + 1))
    scale = one if abs(denom) <= np.float32(1e-8) else so / denom
    new = min(max(new, np.float32(min_opacity)), one - np.float32(1e-6))
    c = min(max(new, np.float32(1e-6)), one - np.float32(1e-6))
    return (np.float32(lib.logf(c / (one - c))),
            [np.float32(lib.logf(np.float32(lib.expf(s)) * scale)) for s in logscale])


@pytest.mark.parametrize("sh", [0, 1, 2, 3])
@pytest.mark.parametrize("n,live,grow", [(300, 0.9, 0.0), (1025, 0.5, 0.0), (257, 0.03, 0.0), (300, 1.0, 0.3),
                                         (1025, 1.0, 3.0)])
def test_mcmc_rows_and_values(n, live, grow, sh):
    """Either a relocation (some rows dead) or a growth: every row made is its source's in every field, the
    sources' opacities and scales are corrected for the number of their copies, the moments of relocated
    sources and of appended rows are cleared, and nothing else changes."""
    from gsx_amd.backend import DensityControl
    f, mom = _rows(n, 3 * n + sh, sh, live)
    threshold = 0.02
    cap = int(n * (1.0 + grow)) + 2
    d, m = _device(f, mom, cap)
    control = DensityControl(dict(algorithm=2, pruning_opacity_threshold=threshold, opacity_clamp_value=0.3,
                                  refine_every=100, start_refine=0, end_refine=1000,
                                  max_num_gaussians=cap if grow > 0.0 else 0, grow_ratio=grow, noise_strength=0.0), seed=9)
    print(f"[case] mcmc rows n={n} live={live} grow={grow} sh={sh}", flush=True)
    count, in_out, counts = control.step(100, n, sh, d, m, cap, {}, None)
    torch.cuda.synchronize()
    dead = f["opacity"] == -8.0
    assert not in_out and counts[0] == int(dead.sum()) and counts[2] == int(dead.sum()) + count - n
    assert count == n + int(n * grow)
    got = {k: v[:count].cpu().numpy() for k, v in d.items()}
    source = got["sh0"][:, 0].astype(np.int64)
    made = np.ones(count, bool)
    made[:n] = dead
    assert np.array_equal(source[~made], np.flatnonzero(~made)) and not dead[source].any()
    draws = np.bincount(source[made], minlength=n)
    lib, want = _libm(), {k: f[k][source].copy() for k in f}
    for s in np.flatnonzero(draws):
        values = _relocated(lib, f["opacity"][s], f["logscale"][s], int(draws[s]), threshold)
        at = source == s
        want["opacity"][at], want["logscale"][at] = values
    for k in f:
        assert np.array_equal(got[k], want[k]), k
    for k in f:
        for j in (0, 1):
            ref = np.zeros((count,) + mom[k][j].shape[1:], np.float32)
            ref[:n] = mom[k][j]
            if dead.any():
                ref[:n][draws > 0] = 0.0
            assert np.array_equal(m[k][j][:count].cpu().numpy(), ref), (k, j)
