"""What the library's host code asks of HIP, on a stand-in for the runtime (fake_hip.c) in a process of its
own: no GPU is needed or touched, and kernels are counted, not run."""
import os
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes, os, sys
sys.path.insert(0, {root!r})
from gsx_amd import _lib
fake = ctypes.CDLL({fake!r})
fake.fake_threads_of.restype = ctypes.c_uint64
lib = _lib.load(require_device=False)
P = 0x7000000000  # an address on the device
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    """Runs a piece of Python against the library on the stand-in runtime."""
    fake = str(tmp_path_factory.mktemp("fake") / "libfakehip.so")
    subprocess.run(["gcc", "-std=c11", "-O1", "-fPIC", "-shared", "-Wall", "-o", fake,
                    os.path.join(ROOT, "tests", "fake_hip.c")], check=True)
    preload = ":".join([fake] + ([os.environ["LD_PRELOAD"]] if os.environ.get("LD_PRELOAD") else []))

    def run(code):
        text = PRELUDE.format(root=ROOT, fake=fake) + textwrap.dedent(code)
        res = subprocess.run([sys.executable, "-c", text], env={**os.environ, "LD_PRELOAD": preload},
                             capture_output=True, text=True, timeout=120)
        assert res.returncode == 0, res.stdout + res.stderr
    return run


ROWS = """
def rows(count):
    r = _lib.GsRows()
    r.count, r.sh_degree = count, 0
    for f in ("mean3d", "rotation", "logscale", "opacity", "sh0", "grad_acc"):
        setattr(r, f, P)
    return r

def step(handle, algorithm, count, capacity, stream=None, out=None, **more):
    p = _lib.AdcParams()
    p.algorithm, p.scene_scale, p.refine_every, p.end_refine = algorithm, 1.0, 100, 1000
    p.max_num_gaussians = capacity
    for k, v in more.items():
        setattr(p, k, v)
    r, o = rows(count), out if out is not None else rows(count)
    in_out, counts = ctypes.c_int32(0), (ctypes.c_int64 * 4)()
    _lib.check(lib.gsx_hip_adc_step(handle, ctypes.byref(p), 100, ctypes.byref(r), capacity, ctypes.byref(o),
                                    ctypes.byref(in_out), counts, stream), "adc step")
    return r.count, list(counts)

def context():
    h = ctypes.c_void_p()
    _lib.check(lib.gsx_hip_adc_context_create(ctypes.byref(h), 3), "create")
    return h
"""


@pytest.mark.parametrize("algorithm", [0, 2])
def test_a_density_control_steps_on_another_device(host, algorithm):
    """Made while device 0 is current and stepped on a stream and the null stream of device 1."""
    host(ROWS + f"""
h = context()
fake.fake_set_totals(1, 1)
fake.hipSetDevice(1)
stream = ctypes.c_void_p()
fake.hipStreamCreateWithFlags(ctypes.byref(stream), 0)
step(h, {algorithm}, 1000, 1000, stream)
step(h, {algorithm}, 1000, 1000, None)
_lib.check(lib.gsx_hip_adc_context_destroy(h), "destroy")
""")


RENDER = """
def camera():
    c = _lib.Camera()
    c.width, c.height, c.fx, c.fy, c.near_plane, c.far_plane = 64, 48, 50.0, 50.0, 0.1, 100.0
    c.rot[3] = 1.0
    return c

def gaussians(count):
    g = _lib.Gaussians()
    g.count, g.sh_degree = count, 0
    for f in ("mean3d", "rotation", "logscale", "opacity", "sh0"):
        setattr(g, f, P)
    return g

def forward(handle, count, instances):
    fake.fake_set_kept(instances)
    return lib.gsx_hip_render_forward(handle, ctypes.byref(camera()), ctypes.byref(gaussians(count)), 0, P, None, None)

def look(handle):
    b = _lib.RenderBuffers()
    _lib.check(lib.gsx_hip_render_context_get_buffers(handle, ctypes.byref(b)), "get buffers")
    return b.sorted_tiles

h = ctypes.c_void_p()
_lib.check(lib.gsx_hip_render_context_create(ctypes.byref(h)), "create")
_lib.check(forward(h, 100, 500), "forward")
"""


def test_a_look_at_the_buffers_allocates_nothing(host):
    host(RENDER + """
before = fake.fake_allocations()
assert look(h) and look(h) == look(h)
assert fake.fake_allocations() == before
assert fake.fake_launches_of(b"widen_tiles") == 1
_lib.check(forward(h, 100, 400), "forward")
assert look(h) and fake.fake_launches_of(b"widen_tiles") == 2
""")


def test_threads_look_at_the_buffers_at_the_same_time(host):
    host(RENDER + """
import threading
seen = []
threads = [threading.Thread(target=lambda: seen.append(look(h))) for _ in range(4)]
[t.start() for t in threads], [t.join() for t in threads]
assert len(set(seen)) == 1 and seen[0]
assert fake.fake_launches_of(b"widen_tiles") == 1
""")


def test_a_look_at_the_buffers_from_another_device(host):
    host(RENDER + """
fake.hipSetDevice(1)
assert look(h)
device = ctypes.c_int()
fake.hipGetDevice(ctypes.byref(device))
assert device.value == 1
""")


def test_no_sorted_tiles_of_an_earlier_forward(host):
    """A forward that runs out of memory behind its count leaves no sorted tiles, rather than the last one's."""
    host(RENDER + """
assert look(h)
fake.fake_set_no_memory(1)
assert forward(h, 100, 1 << 30) == _lib.ERROR_OUT_OF_MEMORY
assert not look(h)
fake.fake_set_no_memory(0)
_lib.check(forward(h, 100, 500), "forward")
assert look(h)
""")


@pytest.mark.parametrize("categories", [1000, 1_000_000])  # many samples a thread, and one
@pytest.mark.parametrize("samples", [1, 2**32 - 256, 2**32 - 255, 2**32, 2**34])
def test_multinomial_of_more_samples_than_threads(host, samples, categories):
    """A launch of 2^32 threads is refused: beyond that a thread draws several samples."""
    host(f"""
_lib.check(lib.gsx_hip_multinomial_i32(P, {samples}, P, {categories}, 1, 3, None), "multinomial")
assert fake.fake_launches_of(b"multinomial") == 1 and 0 < fake.fake_threads_of(b"multinomial") < 2**32
""")


@pytest.mark.parametrize("dead", [1000, 204_522_240, 250_000_000])  # 21 floats a row: the second fills a launch
def test_relocation_of_more_floats_than_threads(host, dead):
    host(ROWS + f"""
def rows(count, few=rows):
    r = few(count)
    r.sh_degree = 3
    r.sh1 = r.sh2 = r.sh3 = P
    return r

fake.fake_set_totals({dead}, 1)
_, counts = step(context(), 2, 400_000_000, 400_000_000)
assert counts[0] == counts[2] == {dead}
assert fake.fake_launches_of(b"mcmc_copy") == 1 and fake.fake_threads_of(b"mcmc_copy") >= min({dead} * 21, 2**32 - 256)
""")


@pytest.mark.parametrize("change", ["o.sh1, o.absgrad_acc = None, P", "o.sh1, o.sh2 = None, P",
                                    "o.first_moment[0], o.second_moment[0] = None, P"])
def test_out_rows_of_other_fields_are_not_written(host, change):
    """As many fields, but other ones: no compaction into them is queued, and the refine says so."""
    host(ROWS + f"""
def rows(count, few=rows):
    r = few(count)
    r.sh_degree, r.sh1 = 2, P
    r.first_moment[0] = P
    return r

fake.fake_set_totals(5, 0)  # rows kept
step(context(), 0, 1000, 1000)
assert fake.fake_launches_of(b"adc_compact") == 1
o = rows(1000)
{change}
try:
    step(context(), 0, 1000, 1000, out=o)
except _lib.GsxHipError as e:
    assert "the same fields" in str(e)
else:
    raise AssertionError("accepted")
assert fake.fake_launches_of(b"adc_compact") == 1
""")
