"""Scale and rotation gradients of footprints of a pixel or two, against 64 bits. The blend backward sums a regular
tile's second moments per 8 x 8 quadrant and moves them to each Gaussian's mean; about the quadrant's centre alone
these sums are much larger than what is left of them, and the gradients lost up to a bit."""
import importlib.util
import os

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def cases():
    spec = importlib.util.spec_from_file_location("perf_cases", os.path.join(ROOT, "perf", "cases.py"))
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


def _errors(cases, case, seed, grow):
    """Relative 2-norm errors of the rotation and logscale gradients of an L1 loss."""
    s = cases.prepare(dict(case, kind="fwdbwd", sh=0, loss="l1", borrow=False), seed)
    s["tensors"].logscale += grow
    raw = {f: getattr(s["tensors"], f).double().requires_grad_(True) for f in cases.FIELDS[:5]}
    pending = cases._render64(s["block"], raw, train=True)
    _, grad = cases._point64(pending["image"], s["target"].double(), "l1", 1.0)
    want = cases._backward64(pending, raw, grad)
    got = cases.run(s)["grads"]
    torch.cuda.synchronize()
    errors = {}
    for field in ("rotation", "logscale"):
        size = float(want[field].norm())
        errors[field] = float((got[field].double() - want[field]).norm()) / size if size > 0.0 else 0.0
    print("  " + ", ".join(f"{f}: {e * 1e6:.2f}e-6" for f, e in errors.items()), flush=True)
    return errors


# (scene, n, width, height, added to the log scales): relative 2-norm errors of (rotation, logscale) with every
# term formed per contribution, in 1e-6. About the quadrant's centre: 2.50 and 1.23, 3.42 and 1.76.
@pytest.mark.parametrize("scene,n,width,height,grow,rotation,logscale", [
    ("cube", 5000, 96, 64, 0.0, 1.54, 0.84),
    ("plane", 5000, 257, 257, -0.5, 1.95, 0.97),
])
def test_small_footprints(cases, scene, n, width, height, grow, rotation, logscale):
    """At most 1.25 times the error of the per-contribution form (measured: 1.07 at most)."""
    print(f"[case] gradient precision {scene} n={n} {width}x{height} {grow}", flush=True)
    errors = _errors(cases, dict(scene=scene, n=n, width=width, height=height), 3, grow)
    for field, bound in (("rotation", rotation), ("logscale", logscale)):
        assert errors[field] <= 1.25e-6 * bound, field


# An image, or a tile at its edge, of a few pixels: the moments of the only pixel that takes an entry, moved to a mean that
# lies nearer to the pixel than the origin does, leave little of themselves. Largest errors of a seed with every term
# formed per contribution: 2.6e-6; with moments 21e-6 (1x1) and 4.5e-6 (1x33).
@pytest.mark.parametrize("width,height", [(1, 1), (1, 3), (3, 2), (17, 1), (1, 33)])
@pytest.mark.parametrize("n", [64, 700])
def test_tiles_of_few_pixels(cases, n, width, height):
    print(f"[case] few pixels n={n} {width}x{height}", flush=True)
    for seed in range(12):
        errors = _errors(cases, dict(scene="cube", n=n, width=width, height=height), seed, 0.0)
        assert max(errors.values()) <= 1.25e-6 * 2.6, (seed, errors)
