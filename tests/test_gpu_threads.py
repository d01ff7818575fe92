"""Scenarios driven by threads of their own on one GPU: the pinned buffers through which state passes
are shared, and every read and write is that of the scenario run alone."""
import threading

import numpy as np
import pytest

from sfincs_amd import _lib
from sfincs_amd import workloads as W

pytestmark = pytest.mark.gpu


def _drive(inst, out, rounds):
    try:
        for _ in range(rounds):
            inst.update(20.0)
            out.append({f: inst.get(f) for f in ("zs", "q", "zsmax")})
            zs = out[-1]["zs"].copy()
            zs[:: 97] += 0.01
            inst.set("zs", zs)
            assert np.array_equal(inst.get("zs"), zs)
    except Exception as e:      # shown by the main thread
        out.append(e)


def test_reads_and_writes_of_several_threads():
    """One piece (24 KB), several (3.9 MB) and several with helper threads (8.4 MB), on the step kernel
    and (pinned) on the separate ones."""
    models = [W.regular_case(n, m, seed=n, t_end=4.0e3).build_model() for n, m in ((48, 64), (700, 697), (1024, 1027))]
    rounds = 6
    alone = []
    for k, mod in enumerate(models + models[:1]):
        x = _lib.Instance(mod)
        if k == len(models):
            x.set_tuning(-1, (32, 8), (64, 4))
        alone.append([])
        _drive(x, alone[-1], rounds)
        x.close()
    insts = [_lib.Instance(m) for m in models + models[:1]]
    insts[-1].set_tuning(-1, (32, 8), (64, 4))
    outs = [[] for _ in insts]
    threads = [threading.Thread(target=_drive, args=(i, o, rounds)) for i, o in zip(insts, outs)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not any(t.is_alive() for t in threads)
    for k, (a, b) in enumerate(zip(alone, outs)):
        assert len(a) == len(b) == rounds, (k, b[-1:])
        for r in range(rounds):
            for f in a[r]:
                assert a[r][f].tobytes() == b[r][f].tobytes(), (k, r, f)
