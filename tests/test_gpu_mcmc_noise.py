"""The MCMC position noise: row i's normals come from draws 6i .. 6i + 5 of the step's stream."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

PARAMS = dict(algorithm=2, pruning_opacity_threshold=0.005, opacity_clamp_value=0.3, refine_every=100, start_refine=0,
              end_refine=1000, max_num_gaussians=0, grow_ratio=0.0, noise_strength=50.0, mean3d_learning_rate=0.01)


def _rows(n):
    g = torch.Generator(device="cuda").manual_seed(n)
    uniform = lambda shape, lo, hi: torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo  # noqa: E731
    return {"mean3d": torch.zeros((n, 3), device="cuda"), "rotation": uniform((n, 4), -1.0, 1.0),
            "logscale": uniform((n, 3), -4.0, -1.0), "opacity": uniform((n,), -8.0, -4.0),
            "sh0": torch.zeros((n, 3), device="cuda")}


def _step(control, rows):
    n = rows["opacity"].shape[0]
    count, in_out, _ = control.step(101, n, 0, rows, None, n, {}, None)  # no refine at step 101
    assert count == n and not in_out


# 3072 workgroups of 256 threads: from 786433 rows on a thread takes several
@pytest.mark.parametrize("n", [1, 255, 257, 786_432, 786_433, 1_600_001])
def test_noise(n):
    from gsx_amd import scenes
    from gsx_amd.backend import DensityControl
    rows = _rows(n)
    print(f"[case] mcmc noise n={n}", flush=True)
    _step(DensityControl(PARAMS, seed=17), rows)
    got = rows["mean3d"].double().cpu().numpy()
    r = {k: v.double().cpu().numpy() for k, v in rows.items()}
    u = scenes.pcg32_stream(17, 6 * n, False).astype(np.float64).reshape(n, 3, 2)
    radius = np.sqrt(-2.0 * np.log(np.maximum(u[..., 0], 1e-7)))
    normal = radius * np.cos(2.0 * np.pi * u[..., 1])
    q = r["rotation"] / np.linalg.norm(r["rotation"], axis=1, keepdims=True)
    x, y, z, w = q.T
    m = np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                  2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                  2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], 1).reshape(n, 3, 3)
    var = np.exp(2.0 * r["logscale"])
    opacity = 1.0 / (1.0 + np.exp(-r["opacity"]))
    gate = 1.0 / (1.0 + np.exp(-100.0 * ((1.0 - opacity) - 0.995)))
    size = 0.5 * gate * var.max(1) * np.linalg.norm(radius, axis=1)
    # the rows' covariances times their normals, through the axes
    want = np.einsum("nij,nj->ni", m, var * np.einsum("nji,nj->ni", m, normal)) * (0.5 * gate)[:, None]
    # the gate's argument is off by 100 times the roundings of 1 - opacity, of 0.995 and of the opacity (6e-6 of the
    # result and more), the angle of a normal by its own (4e-7 of the radius, however small its cosine), a covariance's
    # entries and the other factors by some ten roundings (6e-7 each)
    assert float((np.abs(got - want).max(1) / size).max()) < 2e-5


def test_two_steps_draw_what_one_does():
    from gsx_amd.backend import DensityControl
    n, first = 1_600_001, 786_500
    whole = _rows(n)
    parts = [{k: v[:first].clone() for k, v in whole.items()}, {k: v[first:].clone() for k, v in whole.items()}]
    print(f"[case] mcmc noise {n} rows, and {first} and the others", flush=True)
    _step(DensityControl(PARAMS, seed=4), whole)
    control = DensityControl(PARAMS, seed=4)
    for p in parts:
        _step(control, p)
    torch.cuda.synchronize()
    assert torch.equal(whole["mean3d"], torch.cat([p["mean3d"] for p in parts]))


def test_noise_takes_no_jump_for_every_row():
    """4M rows beside a fill of as many normals (12M): 1.2 times its time; with a jump for every row 1.5 times, with two
    1.75 times."""
    from gsx_amd import _lib
    from gsx_amd.backend import DensityControl, ptr, stream_handle
    n = 4_000_000
    rows, control = _rows(n), DensityControl(PARAMS, seed=3)
    normals = torch.empty(3 * n, device="cuda")

    def best(f):
        times = []
        for _ in range(8):
            torch.cuda.synchronize()
            start = time.perf_counter()
            for _ in range(10):
                f()
            torch.cuda.synchronize()
            times.append((time.perf_counter() - start) / 10)
        return min(times)

    fill = best(lambda: _lib.check(_lib.load().gsx_hip_fill_randn_f32(ptr(normals), 3 * n, 1, 3, 1.0, stream_handle())))
    noise = best(lambda: _step(control, rows))
    print(f"[case] 12M normals {fill * 1e6:.0f} us, the noise of 4M rows {noise * 1e6:.0f} us", flush=True)
    assert noise <= 1.37 * fill
