"""Boxes of more than 1024 tiles (emitted by waves of their own) and runs of several reduction chunks, none,
a few and many of them among small ones: tile lists and gradients against the oracle."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


# (n, big ones): a workgroup lists 256 ranks, and a search step compares 64 workgroups; the depth sort
# scans its counts in a launch of its own from 65 chunks of 2048 on
@pytest.mark.parametrize("n,big", [(1, 1), (255, 3), (257, 257), (5000, 70), (64 * 256 + 300, 4), (64 * 256, 0),
                                   (66 * 256 + 1, 130), (20000, 19900),
                                   (64 * 2048, 2), (64 * 2048 + 1, 2)])
def test_big_boxes(oracle, n, big):
    from gsx_amd import scenes
    from gsx_amd.backend import Camera, GaussianTensors, Renderer
    w = scenes.config0(n=n, width=1601, height=1200)
    w.scene.logscale[:] = -6.0 + 0.1 * np.random.default_rng(n).normal(size=w.scene.logscale.shape)
    which = np.random.default_rng(n + 1).choice(n, big, replace=False)
    w.scene.logscale[which] = 0.5 if n != 20000 else -0.9  # (from 16384 on, waves take several)
    w.scene.opacity[which] = -3.0
    cam, g = Camera.from_block(w.camera), GaussianTensors.from_scene(w.scene)
    print(f"[case] big boxes n={n} big={big}", flush=True)
    r = Renderer(1601, 1200)
    r.render(cam, g, train=True, borrow_train_state=False)
    keys, gaussians = oracle.tile_keys(w.scene, w.camera, 16)
    count = r.stats().instance_count
    assert count == len(keys)

    def pull(ptr):
        a = np.empty(count, np.uint32)
        r.lib.gsx_hip_memcpy_dtoh(a.ctypes.data_as(ctypes.c_void_p), ptr, a.nbytes)
        return a

    buffers = r.buffers()
    assert np.array_equal(pull(buffers.sorted_tiles), (keys >> np.uint64(32)).astype(np.uint32))
    assert np.array_equal(pull(buffers.instance_gaussian)[pull(buffers.sorted_values)], gaussians)
    if big <= 4:  # the oracle's backward visits every pixel of a box
        grad = np.random.default_rng(n).normal(size=(3, 1200, 1601)).astype(np.float32)
        grads = g.zeros_like_grads()
        r.backward(torch.from_numpy(grad).cuda(), grads)
        want = oracle.render_backward(w.scene, w.camera, grad)
        for f in ("mean3d", "logscale", "opacity", "sh0"):
            a, b = getattr(grads, f).cpu().numpy().astype(np.float64).ravel(), want[f].astype(np.float64).ravel()
            assert np.linalg.norm(a - b) <= 1e-3 * np.linalg.norm(b), f
