"""Whole steps on quadtrees, whose continuity makes the combined points at refinement transitions,
against the same steps as separate calls (forcing, fluxes, water levels), which make them in a launch
of their own: every state field is the same bits. Sizes give combined points around a block's edge
and none at all; weirs (whose discharge of the last step enters the mean) lie on transitions."""
import numpy as np
import pytest

from sfincs_amd import _lib
from sfincs_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,mb,nlev,weirs", [(3, 4, 2, False), (6, 6, 3, False), (10, 14, 3, True), (12, 16, 4, False),
                                              (5, 5, 1, False)])
def test_whole_steps_and_separate_calls_agree(nb, mb, nlev, weirs):
    sc = W.quadtree_case(nb, mb, nlev=nlev, dx0=100.0, seed=29, t_end=4.0e3, surge_amp=3.0, zsini=0.2 if weirs else 0.0,
                         store_velmax=1, store_fluxmax=1)
    if weirs:
        sc = W.beach_structures(sc, crest=(-0.5, 0.5), extent=(100.0 * mb, 100.0 * nb), cell=25.0, weir_x=0.09,
                                dam_x=(0.75, 0.85, 0.95))
    m = sc.build_model()
    whole, apart = _lib.Instance(m), _lib.Instance(m)
    ncuv = m.sizes()["ncuv"]
    assert ncuv > 0 or nlev == 1
    for step in range(40):
        whole.update(0.0)
        t, dt, _ = whole.time()
        apart.update_forcing(t, dt)
        apart.compute_fluxes(dt)
        apart.compute_water_levels(t, dt)
        for f in ("zs", "q", "uv", "kfuv", "zsmax", "vmax", "qmax"):
            assert np.array_equal(whole.get(f), apart.get(f)), (step, f)
    assert ncuv == 0 or np.any(whole.get("q")[m.sizes()["npuv"]:] != 0.0)
