"""Density control at the edges of its kernels' blocks (256 rows), lists and counts: refines against
the C oracle bit for bit, and the MCMC draws against a sequential float sum of the weights."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

WIDTHS = {"mean3d": 3, "rotation": 4, "logscale": 3, "opacity": 1, "sh0": 3}


def _rows(n, seed, kept):
    """n rows of which about the share `kept` pass the opacity cut, a third of them candidates."""
    rng = np.random.default_rng(seed)
    f = {"mean3d": rng.normal(size=(n, 3)), "rotation": rng.normal(size=(n, 4)),
         "logscale": rng.uniform(-6.0, -3.0, (n, 3)),
         "opacity": np.where(rng.random(n) < kept, rng.uniform(-1.0, 3.0, n), -8.0), "sh0": rng.normal(size=(n, 3))}
    aux = {"grad_acc": rng.random(n) * 1e-3, "absgrad_acc": rng.random(n) * 1e-3,
           "visible_counter": rng.integers(0, 4, n).astype(np.float64)}
    mom = {k: (rng.normal(size=v.shape), rng.random(v.shape)) for k, v in f.items()}
    c = lambda a: np.ascontiguousarray(a, np.float32)  # noqa: E731
    return ({k: c(v) for k, v in f.items()}, {k: c(v) for k, v in aux.items()},
            {k: (c(a), c(b)) for k, (a, b) in mom.items()})


def _buffer(a, cap, width):
    t = torch.zeros((cap, width) if width > 1 else (cap,), dtype=torch.float32, device="cuda")
    t[: a.shape[0]] = torch.from_numpy(a.reshape(a.shape[0], width) if width > 1 else a)
    return t


@pytest.mark.parametrize("n,room,kept,algorithm", [
    (1, 4, 1.0, 0), (1, 0, 0.0, 1), (2, 4, 0.0, 1), (255, 300, 0.7, 0), (256, 300, 0.7, 1), (257, 17, 1.0, 1),
    (300, 300, 0.0, 0), (512, 1, 0.9, 1), (511, 40, 1.0, 0), (1025, 0, 0.5, 1), (5000, 900, 0.8, 1),
    (70_001, 9_000, 0.9, 1),
])
@pytest.mark.parametrize("with_out", [True, False])
def test_refine_edges(oracle, n, room, kept, algorithm, with_out):
    """Counts, row order, rows, moments and statistics equal the oracle's; without out rows a refine that
    prunes is refused and one that does not stays in place."""
    from gsx_amd.backend import DensityControl, GsxHipError
    from oracle.oracle import AdcParams
    fields, aux, moments = _rows(n, 7 * n + room, kept)
    cap = n + room
    params = dict(algorithm=algorithm, pruning_opacity_threshold=0.1, opacity_clamp_value=0.3, max_world_scale=0.0,
                  duplicate_grad_threshold=2e-4, duplicate_scale_threshold=0.02, duplicate_absgrad_threshold=4e-4,
                  scene_scale=1.0, refine_every=100, start_refine=0, end_refine=1000, max_num_gaussians=cap,
                  reset_every=0)
    print(f"[case] refine n={n} room={room} kept={kept} algorithm={algorithm} out={with_out}", flush=True)
    ref_f, ref_m, ref_counts = oracle.adc_step({k: v.copy() for k, v in fields.items()}, moments,
                                               {k: v.copy() for k, v in aux.items()},
                                               AdcParams(**params, global_step=100, seed=3), cap)
    d = {k: _buffer(v, cap, WIDTHS[k]) for k, v in fields.items()}
    d.update({k: _buffer(v, cap, 1) for k, v in aux.items()})
    m = {k: (_buffer(a, cap, WIDTHS[k]), _buffer(b, cap, WIDTHS[k])) for k, (a, b) in moments.items()}
    o = {k: torch.zeros_like(v) for k, v in d.items()} if with_out else {}
    om = {k: (torch.zeros_like(a), torch.zeros_like(b)) for k, (a, b) in m.items()} if with_out else None
    control = DensityControl(params, seed=3)
    if not with_out and ref_counts[0] > 0:
        with pytest.raises(GsxHipError, match="out rows are required"):
            control.step(100, n, 0, d, m, cap, o, om)
        torch.cuda.synchronize()
        return
    count, in_out, counts = control.step(100, n, 0, d, m, cap, o, om)
    torch.cuda.synchronize()
    assert list(counts) == list(ref_counts)
    assert count == ref_f["mean3d"].shape[0] and in_out == (ref_counts[0] > 0)
    res_f, res_m = (o, om) if in_out else (d, m)
    for k in WIDTHS:
        assert np.array_equal(res_f[k][:count].cpu().numpy().reshape(ref_f[k].shape), ref_f[k]), k
        for j in (0, 1):
            got = res_m[k][j][:count].cpu().numpy().reshape(ref_m[k][j].shape)
            assert np.array_equal(got, ref_m[k][j]), (k, j)
    for k in aux:
        assert float(res_f[k][:count].abs().max()) == 0.0


def _logits(kind, n, rng):
    if kind == "spread":
        return rng.normal(0.0, 2.0, n)
    if kind == "equal":      # 0.5 each: every addition from 2^23 on would be a tie
        return np.zeros(n)
    if kind == "powers":     # weights with few bits, so that ties are common: 1 / (1 + (2^k - 1)) = 2^-k
        return -np.log(2.0 ** rng.integers(1, 20, n) - 1.0 + 1e-12)
    return rng.uniform(-14.0, -10.0, n)  # "small": 1e-6 to 5e-5, the sum stays below 1 for long


@pytest.mark.parametrize("n,kind,dead", [
    (1, "spread", 0.0), (2, "equal", 0.0), (16, "powers", 0.0), (17, "small", 0.0), (1023, "spread", 0.3),
    (1024, "powers", 0.0), (1025, "equal", 0.1), (4096, "small", 0.0), (50_001, "powers", 0.2),
    (300_000, "small", 0.0), (1_100_000, "equal", 0.0), (1_500_001, "spread", 0.05),
])
def test_mcmc_draws_follow_the_sequential_float_sum(n, kind, dead):
    """The sources of relocated and appended rows are those that the CPU's sampler draws
    (gsx/src/gsx-cpu/adc/mcmc.c:118-170): the first row whose running float sum of weights exceeds
    u * total, u the next of the pcg32 stream. Sources are read off an untouched field (sh0)."""
    from gsx_amd import _lib, scenes
    from gsx_amd.backend import DensityControl, ptr, stream_handle
    rng = np.random.default_rng(n)
    opacity = _logits(kind, n, rng).astype(np.float32)
    threshold = 1e-9
    if dead > 0.0:
        opacity[rng.random(n) < dead] = -40.0
    room = max(3, n // 5)
    cap = n + room
    fields = {"mean3d": rng.normal(size=(n, 3)), "rotation": rng.normal(size=(n, 4)),
              "logscale": rng.uniform(-4, -3, (n, 3)), "opacity": opacity,
              "sh0": np.stack([np.arange(n), np.arange(n) * 0.5, np.ones(n)], 1)}
    d = {k: _buffer(np.ascontiguousarray(v, np.float32), cap, WIDTHS[k]) for k, v in fields.items()}

    def weights(t):
        w = torch.empty_like(t)
        lib = _lib.load()
        _lib.check(lib.gsx_hip_unary_f32(ptr(t), ptr(w), t.numel(), 1, stream_handle()))
        torch.cuda.synchronize()
        return w.cpu().numpy()

    def sources(w, u):
        cdf = np.cumsum(np.maximum(w, np.float32(0)), dtype=np.float32)  # numpy accumulates in order
        return np.minimum(np.searchsorted(cdf, u * cdf[-1], side="right"), len(w) - 1)

    w = weights(d["opacity"][:n].contiguous())
    is_dead = w <= np.float32(threshold)
    draws = scenes.pcg32_stream(21, int(is_dead.sum()) + room, False)
    control = DensityControl(dict(algorithm=2, pruning_opacity_threshold=threshold, opacity_clamp_value=0.3,
                                  refine_every=100, start_refine=0, end_refine=1000, max_num_gaussians=cap,
                                  grow_ratio=10.0, noise_strength=0.0), seed=21)
    print(f"[case] mcmc draws n={n} {kind} dead={int(is_dead.sum())}", flush=True)
    count, in_out, counts = control.step(100, n, 0, d, None, cap, {}, None)
    torch.cuda.synchronize()
    assert count == cap and not in_out and counts[0] == int(is_dead.sum())
    got = d["sh0"].cpu().numpy()[:, 0].astype(np.int64)
    live = np.flatnonzero(~is_dead)
    relocated = live[sources(w[live], draws[: int(is_dead.sum())])] if is_dead.any() else np.zeros(0, np.int64)
    now = np.arange(n)
    now[is_dead] = relocated
    assert np.array_equal(got[:n], now)
    # the appended rows draw from the opacities that the relocation left; their own change is undone by
    # reading the weights from a run of the relocation alone
    if is_dead.any():
        again = {k: _buffer(np.ascontiguousarray(v, np.float32), cap, WIDTHS[k]) for k, v in fields.items()}
        alone = DensityControl(dict(algorithm=2, pruning_opacity_threshold=threshold, opacity_clamp_value=0.3,
                                    refine_every=100, start_refine=0, end_refine=1000, max_num_gaussians=0,
                                    grow_ratio=0.0, noise_strength=0.0), seed=21)
        alone.step(100, n, 0, again, None, cap, {}, None)
        w = weights(again["opacity"][:n].contiguous())
    assert np.array_equal(got[n:], now[sources(w, draws[int(is_dead.sum()):])])
