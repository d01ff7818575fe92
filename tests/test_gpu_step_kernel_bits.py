"""The step kernel against the separate kernels byte for byte (the sign of a zero too: dry points and
sleeping tiles rest on exact zeros), on the scenarios of test_gpu_step_kernel.py, and on subgrid sizes
for every number of rows a tile can have and for both register budgets: launches of more than 1792
blocks take eight waves a SIMD, smaller ones seven."""
import numpy as np
import pytest

import test_gpu_step_kernel as T
from sfincs_amd import workloads as W

pytestmark = pytest.mark.gpu


def _same_bytes(a, b, fields, where):
    for f in fields:
        x, y = a.get(f), b.get(f)
        u = {1: np.uint8, 4: np.uint32, 8: np.uint64}[x.itemsize]
        bad = np.flatnonzero(x.view(u) != y.view(u))
        assert bad.size == 0, (where, f, bad.size, bad[:5], x[bad[:5]], y[bad[:5]])
    assert a.time() == b.time(), where


@pytest.fixture(autouse=True)
def _bytes(monkeypatch):
    monkeypatch.setattr(T, "_same", _same_bytes)


# rows a tile, blocks: (1, 1054) (1, 2223) (3, 832) (3, 2229) (5, 2858) (7, 4581)
@pytest.mark.parametrize("n,m", [(166, 400), (350, 400), (400, 393), (600, 700), (900, 1000), (1450, 1391)])
def test_subgrid_rows_and_register_budgets(n, m):
    sc = W.subgrid_case(n, m, seed=n + m, t_end=4.0e3, nsrc=3)
    mod, a, b = T._pair(sc)
    T._run(mod, a, b, (1, 2, 61), where=(n, m))


@pytest.mark.parametrize("n,m", [(63, 9), (2, 130), (127, 31), (301, 499), (870, 880), (1449, 1401)])
def test_regular_sizes(n, m):
    T.test_regular_sizes(n, m)


@pytest.mark.parametrize("kind", ["ring", "outflow", "river", "sources", "qext", "two_points", "dry_walls"])
def test_boundaries_and_sources(kind):
    T.test_boundaries_and_sources(kind, 70, 41)


def test_tiles_sleep_and_wake():
    T.test_tiles_sleep_and_wake()


def test_moves_between_the_paths():
    T.test_moves_between_the_paths()


def test_mixed_batch():
    T.test_mixed_batch()
