"""Tile lists on both sides of the 16-bit tile index (65536 tiles): the sorted tiles and their Gaussians equal
the oracle's, two looks at the buffers agree, and the backward finds the same tiles."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("width,height,n", [(16, 16, 40), (4081, 4096, 500), (4096, 4096, 500), (4097, 4096, 500),
                                            (9000, 2000, 300),
                                            (2800, 2800, 3000)])  # 15 bits: a pass of 8 and one of 7
def test_sorted_tiles_around_the_narrow_limit(oracle, width, height, n):
    from gsx_amd import scenes
    from gsx_amd.backend import Camera, GaussianTensors, Renderer
    w = scenes.config0(n=n, width=width, height=height)
    cam, g = Camera.from_block(w.camera), GaussianTensors.from_scene(w.scene)
    print(f"[case] tiles {width}x{height} n={n}", flush=True)
    r = Renderer(width, height)
    r.render(cam, g, train=True, borrow_train_state=False)
    keys, gaussians = oracle.tile_keys(w.scene, w.camera, 16)
    count = r.stats().instance_count
    assert count == len(keys) > 0

    def pull(ptr):
        a = np.empty(count, np.uint32)
        r.lib.gsx_hip_memcpy_dtoh(a.ctypes.data_as(ctypes.c_void_p), ptr, a.nbytes)
        return a

    buffers = r.buffers()
    tiles = pull(buffers.sorted_tiles)
    assert np.array_equal(tiles, (keys >> np.uint64(32)).astype(np.uint32))
    assert np.array_equal(pull(buffers.instance_gaussian)[pull(buffers.sorted_values)], gaussians)
    assert np.array_equal(pull(r.buffers().sorted_tiles), tiles)
    if width * height <= 1 << 24:  # the backward's reduction looks up the same indices
        grad = np.random.default_rng(n).normal(size=(3, height, width)).astype(np.float32)
        grads = g.zeros_like_grads()
        r.backward(torch.from_numpy(grad).cuda(), grads)
        want = oracle.render_backward(w.scene, w.camera, grad)
        for f in ("mean3d", "logscale", "opacity", "sh0"):
            a, b = getattr(grads, f).cpu().numpy().astype(np.float64).ravel(), want[f].astype(np.float64).ravel()
            assert np.linalg.norm(a - b) <= 1e-3 * np.linalg.norm(b), f
