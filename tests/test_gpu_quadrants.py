"""The blend kernels look at an entry only in the 8 x 8 quadrants that its ellipse may reach: thin, turned
Gaussians that cut corners, faint ones whose cut lies near their centre, round and huge ones give the
oracle's image bit for bit, and its gradients."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# log scales of the axes, raw opacity
KINDS = {"thin": ((-1.5, -6.5, -6.5), 1.0), "needles": ((0.5, -8.0, -8.0), 2.0), "faint": ((-3.0, -5.0, -4.0), -5.4),
         "small": ((-6.5, -6.0, -7.0), 0.0), "discs": ((-1.0, -1.5, -7.0), -1.0)}


@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("n", [70, 900])
def test_quadrants(oracle, kind, n):
    from gsx_amd import scenes
    from gsx_amd.backend import Camera, GaussianTensors, Renderer
    logscale, opacity = KINDS[kind]
    w = scenes.config0(n=n, width=203, height=117)
    rng = np.random.default_rng(n)
    w.scene.logscale[:] = np.asarray(logscale) + 0.2 * rng.normal(size=(n, 3))
    w.scene.opacity[:] = opacity + 0.1 * rng.normal(size=n)
    cam, g = Camera.from_block(w.camera), GaussianTensors.from_scene(w.scene)
    print(f"[case] quadrants {kind} n={n}", flush=True)
    ref, _ = oracle.render(w.scene, w.camera)
    r = Renderer(203, 117)
    for train in (False, True):
        img = r.render(cam, g, train=train, borrow_train_state=False)
        torch.cuda.synchronize()
        assert np.array_equal(img.cpu().numpy(), ref), train
    grad = rng.normal(size=(3, 117, 203)).astype(np.float32)
    grads = g.zeros_like_grads()
    r.backward(torch.from_numpy(grad).cuda(), grads)
    want = oracle.render_backward(w.scene, w.camera, grad)
    for f in ("mean3d", "rotation", "logscale", "opacity", "sh0"):
        a, b = getattr(grads, f).cpu().numpy().astype(np.float64).ravel(), want[f].astype(np.float64).ravel()
        # sums of float terms in another order: 1e-3 of the norm, as the other gradient tests
        assert np.linalg.norm(a - b) <= 1e-3 * np.linalg.norm(b), f
