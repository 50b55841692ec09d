"""The blend kernels at the sizes where their walks change: lists that end just before, at and just
after a bucket (8 entries), a wave of entries (64), the first staged batch (64) and a later one (256),
on images whose last tiles are partial, against the CPU oracle: image bit-exact, gradients within
1e-3 relative L2 per field (the bar of test_gpu_render, whose inputs these resemble)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

GRAD_TOL = 1e-3


def _stack(n, seed, width, height, sharp=0):
    """n translucent Gaussians in front of each other, wider than a tile for even indices and a few
    pixels for odd ones, so that every list is long and the pixels do not saturate; the first
    `sharp` are needles (axis ratio 50, their covariance's 2500) across the image."""
    from gsx_amd import scenes
    rng = np.random.default_rng(seed)
    mean = np.stack([rng.uniform(-0.3, 0.3, n), rng.uniform(-0.3, 0.3, n), rng.uniform(-0.5, 0.5, n)], 1)
    ls = np.where((np.arange(n) % 2 == 0)[:, None], rng.uniform(-1.5, -0.5, (n, 3)), rng.uniform(-4.5, -3.5, (n, 3)))
    ls[:sharp, 0], ls[:sharp, 1:] = -0.6, -0.6 - np.log(50.0)
    op = rng.uniform(-4.5, -3.0, n)  # opacity 0.011 to 0.047
    op[:sharp] = 0.0
    sh0 = rng.normal(0.0, 0.5, (n, 3))
    sc = scenes.Scene(*[np.ascontiguousarray(a, np.float32) for a in (mean, rng.normal(size=(n, 4)), ls, op, sh0)])
    return sc, scenes.camera(width, height, 60.0, background=(0.2, 0.5, 0.1))


@pytest.mark.parametrize("n,width,height,sharp", [
    (1, 1, 1, 0), (2, 16, 16, 0), (7, 17, 16, 0), (8, 16, 17, 1), (9, 33, 15, 0), (63, 16, 16, 0), (64, 16, 16, 2),
    (65, 24, 24, 0), (72, 16, 16, 72), (128, 40, 8, 5), (129, 16, 16, 0), (319, 16, 16, 0), (320, 31, 31, 40),
    (321, 16, 16, 0), (577, 20, 12, 1), (1500, 48, 32, 10),
])
def test_blend_at_list_lengths(oracle, n, width, height, sharp):
    from gsx_amd.backend import Camera, GaussianTensors, Renderer
    sc, block = _stack(n, 1000 + n, width, height, sharp)
    cam, g = Camera.from_block(block), GaussianTensors.from_scene(sc)
    print(f"[case] blend n={n} {width}x{height} needles={sharp}", flush=True)
    ref, _ = oracle.render(sc, block)
    r = Renderer(width, height)
    img = r.render(cam, g, train=False)
    torch.cuda.synchronize()
    assert np.array_equal(img.cpu().numpy(), ref)
    img = r.render(cam, g, train=True, borrow_train_state=False)
    rng = np.random.default_rng(n)
    grad = rng.normal(size=(3, height, width)).astype(np.float32)
    grads = g.zeros_like_grads()
    r.backward(torch.from_numpy(grad).cuda(), grads)
    torch.cuda.synchronize()
    assert np.array_equal(img.cpu().numpy(), ref)
    want = oracle.render_backward(sc, block, grad)
    for f in ("mean3d", "rotation", "logscale", "opacity", "sh0"):
        a = getattr(grads, f).cpu().numpy().astype(np.float64).ravel()
        b = want[f].astype(np.float64).ravel()
        rel = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)
        assert rel <= GRAD_TOL, (f, rel)
