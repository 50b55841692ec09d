"""MCMC draws where the running float sum of the weights stays tiny for long (nearly transparent rows and a
pruning threshold near 0): the same sources as the sequential sum gives, and no chunk-by-chunk walk."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

WIDTHS = {"mean3d": 3, "rotation": 4, "logscale": 3, "opacity": 1, "sh0": 3}


def _rows(opacity, cap):
    n = opacity.shape[0]
    d = {k: torch.zeros((cap, w) if w > 1 else (cap,), dtype=torch.float32, device="cuda") for k, w in WIDTHS.items()}
    d["rotation"][:, 3] = 1.0
    d["logscale"][:] = -4.0
    d["opacity"][:n] = torch.from_numpy(opacity)
    d["sh0"][:n, 0] = torch.arange(n, dtype=torch.float32)
    return d


def _control(cap, threshold=0.0):
    from gsx_amd.backend import DensityControl
    return DensityControl(dict(algorithm=2, pruning_opacity_threshold=threshold, opacity_clamp_value=0.3, refine_every=100,
                               start_refine=0, end_refine=1000, max_num_gaussians=cap, grow_ratio=10.0,
                               noise_strength=0.0), seed=21)


def _logits(kind, n, rng):
    if kind == "tiny":        # 1e-15 to 1e-12: the sum stays below 2^-12
        return rng.uniform(-34.0, -28.0, n)
    if kind == "denormal":    # weights and sums around the least normal float, 1.2e-38
        return rng.uniform(-88.7, -86.0, n)
    if kind == "gap":         # nothing at all (exp overflows), then tiny, then an opaque row
        a = np.where(np.arange(n) < n // 2, -200.0, -30.0)
        a[-1] = 0.0
        return a
    a = rng.uniform(-30.0, -20.0, n)  # "steps": an ever larger row now and then
    a[::997] = -28.0 + 28.0 * np.arange(n)[::997] / n
    return a


# chunks of 1024 weights, 16 to a step of the sums below the lowest binade
@pytest.mark.parametrize("n", [5, 1024, 1025, 16 * 1024, 17 * 1024 + 1, 33 * 1024 - 1, 300_001])
@pytest.mark.parametrize("kind", ["tiny", "denormal", "gap", "steps"])
def test_draws_of_tiny_weights(kind, n):
    from gsx_amd import _lib, scenes
    from gsx_amd.backend import ptr, stream_handle
    room = max(3, n // 5)
    opacity = _logits(kind, n, np.random.default_rng(n)).astype(np.float32)
    # threshold -1: no row is dead, whatever its weight
    d, control = _rows(opacity, n + room), _control(n + room, -1.0)
    logits = d["opacity"][:n].clone()
    w = torch.empty_like(logits)
    _lib.check(_lib.load().gsx_hip_unary_f32(ptr(logits), ptr(w), n, 1, stream_handle()))
    print(f"[case] tiny weights {kind} n={n}", flush=True)
    count, in_out, _ = control.step(100, n, 0, d, None, n + room, {}, None)
    torch.cuda.synchronize()
    assert count == n + room and not in_out
    cdf = np.cumsum(w.cpu().numpy(), dtype=np.float32)  # in order, each addition rounded to float
    u = scenes.pcg32_stream(21, room, False)
    want = np.minimum(np.searchsorted(cdf, u * cdf[-1], side="right"), n - 1)
    assert np.array_equal(d["sh0"].cpu().numpy()[n:, 0].astype(np.int64), want)


def test_tiny_weights_take_no_walk_of_their_chunks():
    """1M rows of opacity 1e-13: 2.4 times the refine of ordinary ones (560 against 235 us); a chunk of 1024
    weights after the other it took 11 times as long (2690 us), the sum on the host 3.4 times (800 us)."""
    n = 1_000_000
    cap = n + n // 10

    def best(opacity):
        d, times = _rows(opacity, cap), []
        logits = d["opacity"][:n].clone()
        for _ in range(6):
            d["opacity"][:n] = logits
            control = _control(cap)
            torch.cuda.synchronize()
            start = time.perf_counter()
            control.step(100, n, 0, d, None, cap, {}, None)
            torch.cuda.synchronize()
            times.append(time.perf_counter() - start)
        return min(times)

    ordinary = best(np.random.default_rng(0).normal(0.0, 2.0, n).astype(np.float32))
    tiny = best(np.full(n, -30.0, np.float32))
    print(f"[case] ordinary {ordinary * 1e6:.0f} us, tiny {tiny * 1e6:.0f} us", flush=True)
    assert tiny <= 5.0 * ordinary
