"""Sphere tagging (tagType 0) on several streams: it reads the centre of mass,
which the geometry refresh writes last, so the tags of a substep queued ahead must
be those of one stream, bit for bit, eager and replayed as a graph."""
import numpy as np
import pytest

from melt_ibm_amd.api import MeltContext
from melt_ibm_amd.inputs import inqpr_temperature
from tests.helpers import load_state, make_cfg, melt_case, with_body

pytestmark = pytest.mark.gpu


def match_one_stream(gpu_lib, cfg, tunes, level=3, rad=1.2, steps=5, hit=False):
    """Steps of a moving body under each tuning (graph=1: replayed) equal those on one stream."""
    st, dt = melt_case(make_cfg(cfg.n1m, cfg.n3m), level, rad, seed=23)
    ctxs = {}
    for tune in (dict(streams=1), *tunes):
        c = ctxs[str(tune)] = MeltContext(cfg, lib=gpu_lib)
        c.set_tuning(**{k: v for k, v in tune.items() if k != "graph"})
        load_state(c, st)
        with_body(c, level, rad)
        c.upload("temp", inqpr_temperature(cfg, c.body().pos_cm[:], rad))
        c.set_dt(dt)
        c.tagCells()
        if hit:
            c.hit_init(0.5, 0.05, 2.5, seed=7)
        c.graph("graph" in tune)
    one = next(iter(ctxs.values()))
    fields = ("vx", "vy", "vz", "temp", "pr", "VOFp", "VOFx", "VOFy", "VOFz")
    for step in range(steps):
        print(f"# tagType {cfg.tagtype} precision {cfg.precision} step {step}", flush=True)
        for c in ctxs.values():
            if hit:
                c.hit_force()
            c.tschem()
        want = {q: one.download(q) for q in fields}
        xyz = one.lag("xyzv")
        assert np.isfinite(xyz).all()
        for tune, c in ctxs.items():
            for q, a in want.items():
                same = np.array_equal(c.download(q), a)
                assert same, (step, tune, q)
            same = np.array_equal(c.lag("xyzv"), xyz)
            assert same, (step, tune)
    for c in ctxs.values():
        c.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,n3", [(64, 64), (32, 24)])
def test_sphere_tagging_queued_ahead(gpu_lib, n, n3, precision):
    cfg = make_cfg(n, n3, tagtype=0, imelt=0, precision=precision)
    match_one_stream(gpu_lib, cfg, (dict(streams=2), dict(streams=2, graph=1), dict(streams=2, coef=2)), level=3 if n == 64 else 2)
