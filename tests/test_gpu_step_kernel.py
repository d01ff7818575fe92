"""The step kernel (one launch per step on dense default-physics meshes) against the separate
forcing, momentum and continuity kernels on the same scenario: every state field is the same
bits after the same steps. Sizes lie at the edges of its tiles (63 columns by 1, 3, 5 or 7 rows)
and of its size rule; scenarios cover what the rule accepts (water-level, outflow and river
boundaries on any side, discharges, external sources, rain that starts and stops, tiles that fall
asleep and wake), host writes between steps, and moves between the two paths."""
import numpy as np
import pytest

from sfincs_amd import _lib
from sfincs_amd import workloads as W

pytestmark = pytest.mark.gpu

STEP = -8


def _same(a, b, fields, where):
    for f in fields:
        x, y = a.get(f), b.get(f)
        bad = np.flatnonzero(x.view(np.uint8).reshape(x.size, -1).any(1) != y.view(np.uint8).reshape(y.size, -1).any(1)) \
            if x.dtype == np.int8 else np.flatnonzero(x != y)
        assert bad.size == 0, (where, f, bad[:5], x[bad[:5]], y[bad[:5]])
    assert a.time() == b.time(), where


def _fields(m):
    s = m.sizes()
    out = ["zs", "q", "uv", "kfuv", "zsmax"] + (["z_volume", "zs0", "zsderv"] if s["subgrid"] else [])
    return out + (["uvmean"] if s["nkcuv2"] else []) + (["qtsrc"] if s["nsrc"] else [])


def _pair(sc):
    sc.params["t1"] = 1.0e7
    m = sc.build_model()
    a, b = _lib.Instance(m), _lib.Instance(m)
    assert a.tuning()["momentum_kernel"] == STEP
    b.set_tuning(-1, (32, 8), (64, 4))
    assert b.tuning()["momentum_kernel"] == -1
    return m, a, b


def _run(m, a, b, rounds=(1, 2, 37, 64, 5), where=""):
    ba, bb = _lib.Batch(), _lib.Batch()
    ba.add(a, 1.0e9)
    bb.add(b, 1.0e9)
    for k in rounds:
        ba.advance(k)
        bb.advance(k)
        _same(a, b, _fields(m), (where, k))
    ba.close()
    bb.close()


def _regular(n, m, **kw):
    kw.setdefault("rain_until", 60.0)
    return W.regular_case(n, m, seed=n * 1000 + m, t_end=4.0e3, dx=20.0, **kw)


@pytest.mark.parametrize("n,m", [(63, 9), (64, 7), (65, 3), (62, 64), (2, 130), (126, 2), (127, 31), (5, 301),
                                 (301, 499), (499, 303), (870, 880), (1449, 1401)])
def test_regular_sizes(n, m):
    sc = _regular(n, m, nbumps=6)
    zb = sc.zb_grid
    # tide, flat and dry parts on small meshes too: a bed from -3 m to +1.5 m along the mesh
    sc.zb_grid = (zb - zb.mean() + np.linspace(-3.0, 1.5, m)[:, None]).astype(np.float32)
    mod, a, b = _pair(sc)
    _run(mod, a, b, where=(n, m))


@pytest.mark.parametrize("n,m", [(17, 63), (64, 21), (66, 130), (400, 390)])
def test_subgrid_sizes(n, m):
    sc = W.subgrid_case(n, m, seed=n + m, t_end=4.0e3, nsrc=3)
    mod, a, b = _pair(sc)
    _run(mod, a, b, where=(n, m))
    va, vb = a.balance(), b.balance()
    for k in va:
        assert abs(va[k] - vb[k]) <= 1e-9 * max(1.0, abs(va["volume"])), (k, va, vb)


def _edges(sc, kind):
    msk = sc.msk.reshape(sc.mmax, sc.nmax).copy()
    msk[:, 0] = msk[:, -1] = msk[0, :] = msk[-1, :] = 2
    if kind == "outflow":
        msk[-1, :] = 3
        msk[:, -1] = 1
    sc.msk = msk.reshape(-1)
    return sc


@pytest.mark.parametrize("kind", ["ring", "outflow", "river", "sources", "qext", "two_points", "dry_walls"])
@pytest.mark.parametrize("n,m", [(70, 41), (63, 64)])
def test_boundaries_and_sources(kind, n, m):
    sc = _regular(n, m, rain_mmh=0.0 if kind in ("ring", "dry_walls") else 30.0, use_qext=1 if kind == "qext" else 0)
    lo, hi = (-9.0, 5.0) if kind == "sources" else (-2.0, 2.0)     # the source recipe wants deep water and high land
    sc.zb_grid = (sc.zb_grid - sc.zb_grid.mean() + np.linspace(lo, hi, m)[:, None]).astype(np.float32)
    if kind in ("ring", "outflow"):
        sc = _edges(sc, kind)
    if kind == "river":
        sc = W.with_river(sc)
    if kind == "sources":
        sc = W.regular_sources(sc)
    if kind == "two_points":
        x, y, t, z = sc.bnd
        sc.bnd = (np.repeat(x, 2), np.array([0.0, n * 20.0], np.float32), t, np.concatenate([z, 0.5 * z], 1))
    if kind == "dry_walls":     # the boundary column stands dry, so its points take the no-flow branch
        sc.zb_grid[0, :] = 3.0
    mod, a, b = _pair(sc)
    if kind == "qext":
        q = np.zeros(mod.sizes()["np"], np.float32)
        q[::17] = 1.0e-4
        for i in (a, b):
            i.set("qext", q)
    _run(mod, a, b, where=kind)


def test_tiles_sleep_and_wake():
    """A steep tide over dry land with no rain: tiles fall asleep, the flood and a host write wake
    them, and a long run ends with the same bits."""
    sc = _regular(130, 70, rain_mmh=0.0, tide_amp=2.5)
    sc.zb_grid = np.linspace(-4.0, 4.0, 70)[:, None].repeat(130, 1).astype(np.float32)
    t = np.arange(0.0, 4.1e3, 20.0)
    sc.bnd = (*sc.bnd[:2], t.astype(np.float32), (2.5 * np.sin(2 * np.pi * t / 1500.0)).astype(np.float32)[:, None])
    mod, a, b = _pair(sc)
    _run(mod, a, b, (200, 301, 300), "tide")
    zs = a.get("zs")
    zs[5 + 130 * 60] += 1.5
    for i in (a, b):
        i.set("zs", zs)
    _run(mod, a, b, (1, 2, 30, 500), "after a write")
    q = a.get("q")
    q[::7] *= 0.5
    for i in (a, b):
        i.set("q", q)
    _run(mod, a, b, (1, 1, 40), "after a write of q")


def test_moves_between_the_paths():
    """Whole steps, single steps, the standalone entry points, counting and pinned shapes in turn."""
    sc = W.subgrid_case(66, 70, seed=5, t_end=4.0e3, nsrc=2)
    mod, a, b = _pair(sc)
    f = _fields(mod)
    for i in (a, b):
        i.update(40.0)
    _same(a, b, f, "update")
    for i in (a, b):
        for _ in range(3):
            i.update(0.0)
    _same(a, b, f, "single steps")
    for i in (a, b):
        t, dt, _ = i.time()
        i.update_forcing(t + 1.0, 1.0)
        i.compute_fluxes(1.0)
        i.compute_water_levels(t + 1.0, 1.0)
    _same(a, b, f, "standalone")
    for i in (a, b):
        i.update(30.0)
    _same(a, b, f, "update again")
    assert a.total_volume() == pytest.approx(b.total_volume(), rel=1e-14)
    a.set_counting(True)
    for i in (a, b):
        i.update(20.0)
    a.set_counting(False)
    for i in (a, b):
        i.update(20.0)
    _same(a, b, f, "counted")
    a.set_tuning(-2, (64, 4), (64, 4))
    b.set_tuning(STEP, (64, 4), (64, 4))
    for i in (a, b):
        i.update(50.0)
    _same(a, b, f, "swapped")


def test_mixed_batch():
    """Members on the step kernel and on the separate kernels (masked, wind, pinned) in one batch
    end as they do alone."""
    def scs():
        s1 = _regular(70, 40)
        s2 = W.subgrid_case(40, 66, seed=3, t_end=4.0e3, nsrc=2)
        s3 = _regular(30, 33, wind=(np.array([0.0, 1.0e5], np.float32), np.full(2, 12.0, np.float32),
                                    np.full(2, 200.0, np.float32)))
        s4 = _regular(64, 65)
        return [s1, s2, s3, s4]
    models = [s.build_model() for s in scs()]
    together, alone = [_lib.Instance(m) for m in models], [_lib.Instance(m) for m in models]
    together[3].set_tuning(-4, (64, 4), (64, 4))
    batch = _lib.Batch()
    ends = [150.0, 90.0, 120.0, 200.0]
    for i, e in zip(together, ends):
        batch.add(i, e)
    while batch.advance(33):
        pass
    batch.close()
    for k, (m, x, y, e) in enumerate(zip(models, together, alone, ends)):
        y.update_to(e)
        _same(x, y, _fields(m), k)
