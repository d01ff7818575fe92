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
