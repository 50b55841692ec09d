"""An MCMC growth whose rows hold more floats than a launch has threads (2^32)."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_growth_of_more_floats_than_threads():
    from gsx_amd.backend import DensityControl
    n, grown = 1000, 204_530_000  # sh3: 21 floats a row, 2^32 + 162 704
    cap = n + grown
    print(f"[case] mcmc growth by {grown} rows", flush=True)
    widths = {"mean3d": 3, "rotation": 4, "logscale": 3, "opacity": 1, "sh0": 3, "sh3": 21}
    d = {k: torch.empty((cap, w) if w > 1 else (cap,), device="cuda") for k, w in widths.items()}
    for k, v in d.items():
        v[:n] = torch.randn(v[:n].shape, device="cuda")
        v[n:] = -77.0
    d["sh0"][:n, 0] = torch.arange(n, dtype=torch.float32, device="cuda")
    control = DensityControl(dict(algorithm=2, pruning_opacity_threshold=0.005, opacity_clamp_value=0.3, refine_every=100,
                                  start_refine=0, end_refine=1000, max_num_gaussians=cap, grow_ratio=1e6,
                                  noise_strength=0.0), seed=21)
    count, in_out, _ = control.step(100, n, 3, d, None, cap, {}, None)
    torch.cuda.synchronize()
    assert count == cap and not in_out
    # floats 2^32 - 256 on of the appended rows' sh3 lie in the last 8000 rows
    for rows in (slice(n, n + 5000), slice(cap - 9000, cap)):
        source = d["sh0"][rows, 0].long()
        assert int(source.min()) >= 0 and int(source.max()) < n
        for k in ("sh3", "mean3d", "rotation"):
            assert torch.equal(d[k][rows], d[k][source]), (k, rows)
