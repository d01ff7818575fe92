"""Host code of the library without a GPU: libsfx.so on the runtime of fake_hip.cpp, which runs no
kernel but keeps what was issued on which stream, what the host waited for, and what is allocated.
Each case runs in a process of its own, where the fake runtime comes before the real one."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C, os, sys
F = C.CDLL(sys.argv[1], mode=os.RTLD_GLOBAL | os.RTLD_NOW)
import numpy as np
from sfincs_amd import _lib
from sfincs_amd import workloads as W
F.fake_live.restype = F.fake_launches.restype = F.fake_stale.restype = F.fake_bytes.restype = F.fake_operations.restype = C.c_long
F.fake_fail.argtypes = [C.c_long]

def busy():
    b = C.create_string_buffer(4000)
    F.fake_busy(b, 4000)
    F.fake_settle()
    return b.value.decode()

def regular(n=30, m=41, **kw):
    return W.regular_case(n, m, seed=1, t_end=4.0e3, **kw).build_model()

def subgrid(n=30, m=41):
    return W.subgrid_case(n, m, seed=1, t_end=4.0e3, nsrc=2).build_model()
"""


@pytest.fixture(scope="session")
def fake(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           "-o", out, os.path.join(HERE, "fake_hip.cpp")])
    return out


def run(fake, body):
    p = subprocess.run([sys.executable, "-c", PRELUDE + body, fake], cwd=ROOT, capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, (p.returncode, p.stdout[-1500:], p.stderr[-1500:])
    return p.stdout


CALLS = ["x.profile(1)", "x.profile(2)", "x.set('zs', x.get('zs'))", "x.set('z_volume', x.get('z_volume'))",
         "x.set('zsderv', x.get('zsderv'))",
         "x.set('q', x.get('q'))", "x.set('kfuv', x.get('kfuv'))", "x.set_counting(True)", "x.set_counting(False)",
         "x.compute_fluxes(1.0)", "x.autotune(1)", "b.add(x, 50.0)", "b.advance(3)", "b.done(x)",
         "b.remove(x)", "F.fake_ones(1); x.update(50.0); F.fake_ones(0)", "x.set_tuning(-1, (32, 8), (64, 4))"]


def test_nothing_is_in_flight_on_return(fake):
    """A handle may be in a batch, which runs on another stream: what a call issued is finished when
    it returns, on the handle's stream and on the null stream, for which no stream waits."""
    left = run(fake, f"""
x, b = _lib.Instance(subgrid()), _lib.Batch()
for call in {CALLS!r}:
    if not x._nbatch: x.update(0.0)
    assert busy() == ''
    exec(call)
    left = busy()
    if left: print(call, '|', left)
assert F.fake_launches(b'k_step_scalars') > 0      # an odd number of steps was profiled
""")
    assert left == "", left


def test_autotune_moves_between_kernels_on_the_chosen_shapes(fake):
    """Sweeps that autotune completes are completed with the tiles they ran on: the handle's own
    descriptor is the one its trials were launched with."""
    run(fake, """
x = _lib.Instance(subgrid(130, 70))
x.update(0.0)
n = F.fake_launches(b'k_give_scalars')
x.autotune(1)
assert F.fake_launches(b'k_step') > 0 and F.fake_launches(b'k_give_scalars') > n
assert F.fake_stale() == 0, F.fake_stale()
""")


def test_autotune_while_counting_keeps_the_choice_of_kernel(fake):
    """With counting on, steps run on the separate kernels only, so no trial of theirs decides against
    the step kernel (the fake clock calls every later trial slower)."""
    run(fake, """
for pin in (-8, -1):
    x = _lib.Instance(subgrid())
    x.set_tuning(pin, (32, 8), (64, 4))
    x.set_counting(True)
    assert x.autotune(1)['momentum_kernel'] == -8 if pin == -8 else x.autotune(1)['momentum_kernel'] != -8
x = _lib.Instance(subgrid())
assert x.autotune(1)['momentum_kernel'] != -8
""")


def test_reads_go_on_without_helper_threads(fake):
    """A read of 8 MB takes helper threads; where none can be started (here: no address space for
    their stacks) the calling thread moves the pieces alone."""
    run(fake, """
import resource
x = _lib.Instance(regular(1000, 1050))
zs = np.arange(1050000, dtype=np.float64)
x.set('zs', zs)
out = [np.zeros_like(zs), np.zeros_like(zs)]
def read(a):
    return _lib.lib().sfx_get_state(x.h, b'zs', a.ctypes.data_as(C.c_void_p), C.c_size_t(a.nbytes))
size = int(open('/proc/self/statm').read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (size + (4 << 20), -1))     # a stack takes 8 MB
assert read(out[0]) == 0 and np.array_equal(out[0], zs)
resource.setrlimit(resource.RLIMIT_AS, (-1, -1))
assert read(out[1]) == 0 and np.array_equal(out[1], zs)
""")


def test_a_failed_create_keeps_nothing(fake):
    """Whichever allocation fails, device or pinned, the call says so and gives back what it had; the
    buffers that handles share are given back with the last of them, failed ones not counted."""
    run(fake, """
m = subgrid()
_lib.Instance(m).close()                 # the tables that stay
live = lambda: (F.fake_live(0), F.fake_live(1))
base = live()
x = _lib.Instance(m)
n = sum(live()) - sum(base)
x.close()
assert live() == base and n > 40
for k in range(1, n + 1):
    F.fake_fail(k)
    try:
        _lib.Instance(m)
        raise SystemExit('allocation %d: no error' % k)
    except _lib.SfxError as e:
        assert 'hipMalloc failed' in str(e), (k, e)
    assert live() == base, (k, live(), base)
F.fake_fail(0)
x = _lib.Instance(m)
x.get('zs')
assert F.fake_live(1) > base[1] + 1      # the shared buffers are there
x.close()
assert live() == base, (live(), base)
""")


def test_reads_and_writes_without_pinned_memory(fake):
    """Where the shared pinned buffers cannot be had, state is copied directly, and the failed
    allocation is no error of this call or of the next."""
    run(fake, """
x = _lib.Instance(regular())
zs = np.linspace(0.0, 1.0, x.sizes['np'])
F.fake_fail(1)
x.set('zs', zs)
x.update_forcing(1.0, 1.0)
F.fake_fail(1)
assert np.array_equal(x.get('zs'), zs)
x.update_forcing(2.0, 1.0)
pins = F.fake_live(1)
x.get('zs')
assert F.fake_live(1) == pins + 1        # tried again
""")


def test_a_tuning_can_be_pinned_on_any_run_of_the_mesh(fake):
    """What tuning() reports for a default run (the step kernel) is accepted by the same mesh with
    wind, by its FP64 twin and by an indexed mesh, which keep a kernel of their own; other unknown
    numbers are refused as ever."""
    run(fake, """
d = _lib.Instance(regular()).tuning()
assert d['momentum_kernel'] == -8
two = np.array([0.0, 1.0e5], np.float32)
wind = regular(wind=(two, np.full(2, 12.0, np.float32), np.full(2, 200.0, np.float32)))
for x in (_lib.Instance(wind), _lib.Instance(regular(), fp64=True), _lib.Instance(W.quadtree_case(5, 5, nlev=2).build_model())):
    own = x.tuning()['momentum_kernel']
    assert own != -8
    x.pin_tuning(d)
    assert x.tuning()['momentum_kernel'] == own
    for bad in (-3, -7, -9, 257):
        try:
            x.set_tuning(bad, (32, 8), (64, 4))
            raise SystemExit('accepted %d' % bad)
        except _lib.SfxError as e:
            assert '-8' in str(e)
x = _lib.Instance(regular())
x.set_tuning(-1, (32, 8), (64, 4))
assert x.tuning()['momentum_kernel'] == -1
x.pin_tuning(d)
assert x.tuning()['momentum_kernel'] == -8
""")


def test_footprint_counts_the_second_side_where_there_is_one(fake):
    """Admission by footprint: scenarios outside the step kernel's rule hold one side of the levels, and
    those inside it allocate no more than the footprint says."""
    run(fake, """
two = np.array([0.0, 1.0e5], np.float32)
wind = regular(300, 301, wind=(two, np.full(2, 12.0, np.float32), np.full(2, 200.0, np.float32)))
step = regular(300, 301)
np_ = 300 * 301
assert step.footprint() - wind.footprint() == np_ * 8 + 2 * np_          # levels, kfuv of 2 np slots
_lib.Instance(regular()).close()                                        # the tables that stay
base = F.fake_bytes()
for m in (step, wind, subgrid(), W.quadtree_case(5, 5, nlev=2).build_model()):
    x = _lib.Instance(m)
    assert F.fake_bytes() - base <= m.footprint(), (F.fake_bytes(), m.footprint())
    x.close()
""")


def test_a_move_between_the_kernels_is_one_launch(fake):
    """A host that alternates whole steps and a standalone call on a scenario of the step kernel: beside
    the two moves, a round takes the launches of the step and of the call (scalars written, the work,
    scalars handed over) and builds no lists anew."""
    run(fake, """
x = _lib.Instance(regular())
for k in range(3):
    n = F.fake_operations()
    x.update(0.0)
    x.compute_fluxes(0.5)
    n = F.fake_operations() - n
assert n <= 2 + 3 + 3, n
assert F.fake_launches(b'k_enter_step') == 3 and F.fake_launches(b'k_enter_general') == 3
""")


def test_large_subgrid_meshes_under_rain_start_on_the_separate_kernels(fake):
    """The default by size, mesh and forcing: the step kernel up to 750000 cells, on regular meshes and
    without rain or sources in every cell beyond; it can be pinned where it is not the default."""
    run(fake, """
import torch
torch.cuda.is_available = lambda: False          # terrain is made on the host
torch.set_num_threads(1)
def kernel(make, n, m, pin=False, **kw):
    if make is sub: kw.update(refi=2, nl=2, nsrc=0)
    x = _lib.Instance(make(n, m, seed=1, t_end=4.0e3, **kw).build_model())
    if pin: x.set_tuning(-8, (32, 8), (64, 4))
    return x.tuning()['momentum_kernel']
sub, reg = W.subgrid_case, W.regular_case
assert kernel(sub, 750, 1000, rain_mmh=20.0) == -8
assert kernel(sub, 751, 1000, rain_mmh=20.0) == -1
assert kernel(sub, 751, 1000, rain_mmh=0.0, use_qext=1) == -1
assert kernel(sub, 751, 1000, rain_mmh=0.0) == -8
assert kernel(sub, 751, 1000, rain_mmh=20.0, pin=True) == -8
assert kernel(reg, 1000, 1000, rain_mmh=20.0) == -8
""")
