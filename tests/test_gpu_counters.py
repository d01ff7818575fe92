"""Branch counters of a momentum sweep: every uv slot of the mesh in one class, as many wet points as the
sweep left with kfuv set, and the same wet and partly wet points on every kernel."""
import numpy as np
import pytest

from sfincs_amd import _lib
from sfincs_amd import workloads as W

pytestmark = pytest.mark.gpu

KERNELS = [(-1, (32, 8)), (-1, (256, 1)), (-2, (64, 4)), (-4, (16, 16)), (0, (64, 4)), (8, (64, 4))]


@pytest.mark.parametrize("n,m", [(63, 41), (130, 97)])
@pytest.mark.parametrize("subgrid", [False, True])
def test_counters_add_up(n, m, subgrid):
    if subgrid:
        sc = W.subgrid_case(n, m, seed=11, t_end=4.0e3, nsrc=2)
    else:
        sc = W.regular_case(n, m, seed=11, t_end=4.0e3, dx=20.0)
        sc.zb_grid = (sc.zb_grid - sc.zb_grid.mean() + np.linspace(-3.0, 1.5, m)[:, None]).astype(np.float32)
    mod = sc.build_model()
    seen = None
    for kernel, tile in KERNELS:
        x = _lib.Instance(mod)
        x.set_tuning(kernel, tile, (64, 4))
        x.update(60.0)
        x.set_counting(True)
        last, rows = np.zeros(6, np.int64), []
        for _ in range(4):
            x.update(0.0)
            now = np.array(x.counters())
            rows.append((now - last).tolist())
            last = now
            c = rows[-1]
            assert sum(c) == 2 * n * m, (kernel, tile, c)
            assert c[2] + c[3] == int(x.get("kfuv").sum()), (kernel, tile, c)
        wet = [c[2:4] for c in rows]
        seen = seen or wet
        assert wet == seen and (not subgrid or any(w[1] for w in wet)), (kernel, tile, wet, seen)
