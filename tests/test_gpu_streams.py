"""One stream or several: a step's results do not depend on it.  A small grid
takes one by itself; replaying some of the steps as graphs keeps the bits as
well."""
import numpy as np
import pytest

from melt_ibm_amd.api import MeltContext
from melt_ibm_amd.inputs import inqpr_temperature
from tests.helpers import load_state, make_cfg, melt_case, with_body

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,level", [(32, 2), (64, 3)])
def test_streams_do_not_change_a_step(gpu_lib, n, level, precision):
    cfg = make_cfg(n, precision=precision)
    st, dt = melt_case(make_cfg(n), level, 1.2, seed=5)
    ctxs = {}
    for streams in (0, 1, 2, "toggled"):
        c = ctxs[streams] = MeltContext(cfg, lib=gpu_lib)
        if streams in (1, 2):
            c.set_tuning(streams=streams)
        load_state(c, st)
        with_body(c, level, 1.2)
        c.upload("temp", inqpr_temperature(cfg, c.body().pos_cm[:], 1.2))
        c.set_dt(dt)
        c.tagCells()
    for step in range(5):
        print(f"# streams {n}^3 precision {precision} step {step}", flush=True)
        ctxs["toggled"].graph(step in (1, 2, 4))
        for c in ctxs.values():
            c.tschem()
        for q in ("vx", "vy", "vz", "temp", "pr", "VOFp"):
            want = ctxs[2].download(q)
            for streams, c in ctxs.items():
                same = np.array_equal(c.download(q), want)
                assert same, (step, streams, q)
        want = ctxs[2].lag("xyzv")
        assert np.isfinite(want).all()
        for streams, c in ctxs.items():
            same = np.array_equal(c.lag("xyzv"), want)
            assert same, (step, streams)
    for c in ctxs.values():
        c.close()
