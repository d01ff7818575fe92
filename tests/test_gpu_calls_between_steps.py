"""Calls between the steps of a scenario that the step kernel runs: what they change, and that the
steps after them are those of a scenario on the separate kernels, bit for bit."""
import numpy as np
import pytest

from sfincs_amd import _lib
from sfincs_amd import workloads as W

pytestmark = pytest.mark.gpu


def _fields(m):
    s = m.sizes()
    return (["zs", "q", "uv", "kfuv", "zsmax", "qtsrc", "uvmean"] +
            (["z_volume", "zs0", "zsderv"] if s["subgrid"] else []))


def _same(x, y, m, where):
    for f in _fields(m):
        assert x.get(f).tobytes() == y.get(f).tobytes(), (where, f)
    assert x.time() == y.time(), where


def _pair():
    sc = W.subgrid_case(66, 70, seed=5, t_end=4.0e3, nsrc=2)
    sc.params["t1"] = 1.0e7
    m = sc.build_model()
    x, y = _lib.Instance(m), _lib.Instance(m)
    y.set_tuning(-1, (32, 8), (64, 4))
    return m, x, y


@pytest.mark.parametrize("steps", [1, 2, 5])
def test_profiled_steps_of_a_batch_member(steps):
    """Profiled steps, odd numbers of them too, then steps of the batch on its own stream."""
    m, x, y = _pair()
    b = _lib.Batch()
    b.add(x, 1.0e9)
    y.update_to(1.0e-9)
    b.advance(1)
    for _ in range(3):
        x.profile(steps)
        b.advance(4)
        for _ in range(steps + 4):
            y.update(0.0)
    b.close()
    _same(x, y, m, steps)


def _rising():
    """Discharges that rise by 40 m3/s up to 290 s, the end of the simulation (a series that ends before
    is stretched to it); steps beyond are taken by running to a later time."""
    sc = W.subgrid_case(66, 70, seed=5, t_end=4.0e3, nsrc=2)
    sc.params["t1"] = 290.0
    px, py, _, q = sc.src
    sc.src = (px, py, np.array([0.0, 290.0], np.float32), np.stack([q[0], q[0] + 40.0]).astype(np.float32))
    return sc.build_model(), q[0]


@pytest.mark.parametrize("at", [150.0, 400.0])
def test_autotune_leaves_the_scenario_as_it_was(at):
    """Every field and the sums of the volume balance are the bits from before, the discharges too, inside
    their series and past its end, where the next steps keep them; the steps after are those of a
    scenario that was not tuned. (The balance's volume is no state: each call adds it up anew, in an
    order that is not fixed.)"""
    m, q = _rising()
    x, y = _lib.Instance(m), _lib.Instance(m)
    for i in (x, y):
        i.update_to(at)
    before = {f: x.get(f).tobytes() for f in _fields(m)}
    sums = ("boundary", "sources", "rain", "qext")
    balance = [x.balance()[k] for k in sums]
    x.autotune(2)
    assert [f for f in before if x.get(f).tobytes() != before[f]] == []
    assert [x.balance()[k] for k in sums] == balance
    for i in (x, y):
        i.update_to(at + 60.0)
    _same(x, y, m, at)


def test_discharges_past_their_series_stay_through_a_move_between_kernels():
    """Past the end of the series the last discharges stay in force, whichever kernels took the step
    that worked them out: the step kernel, standalone forcing, and the staged steps of the separate
    kernels in turn."""
    m, q = _rising()
    whole, moved = _lib.Instance(m), _lib.Instance(m)
    for i in (whole, moved):
        i.update_to(320.0)                       # on the step kernel
    last = whole.get("qtsrc")
    assert np.all(last > q + 35.0)
    moved.set_counting(True)                     # on the separate kernels
    for i in (whole, moved):
        i.update_to(400.0)
    assert np.array_equal(moved.get("qtsrc"), last)
    _same(whole, moved, m, "counted")
    apart = _lib.Instance(m)
    apart.set_tuning(-1, (32, 8), (64, 4))
    apart.update_to(100.0)                       # staged steps, then forcing of its own just before the end
    assert apart.time()[1] > 0.2
    apart.update_forcing(289.9, 1.0)
    want = apart.get("qtsrc")
    assert np.all(want > q + 39.0)
    apart.update_to(350.0)
    assert np.array_equal(apart.get("qtsrc"), want)


@pytest.mark.parametrize("steps", [3, 4])
def test_a_write_of_kfuv_holds_on_either_side(steps):
    """kfuv written after an odd and an even number of steps, closed points included."""
    m, x, y = _pair()
    for i in (x, y):
        for _ in range(steps):
            i.update(0.0)
        k = i.get("kfuv")
        k[::5] = 0
        k[3::7] = 1
        i.set("kfuv", k)
        assert np.array_equal(i.get("kfuv"), k)
        for _ in range(3):
            i.update(0.0)
    _same(x, y, m, steps)
