"""The y and z line solves of the fused substep over the shapes at which their
rules change: the one-thread-per-run filters (any grid), the fused pass with its
segment lengths, and the cyclic reduction.  The forms of the filter compute the
same expressions (bit-identical); the cyclic reduction is another exact route
to the same solution."""
import numpy as np
import pytest

from melt_ibm_amd.api import MeltContext
from tests.helpers import load_state, make_cfg, random_state, rel_err

pytestmark = pytest.mark.gpu

FIELDS = ("vx", "vy", "vz", "temp", "pr")


def step(gpu_lib, monkeypatch, cfg, st, tune):
    monkeypatch.setenv("MELT_TUNE", tune)
    c = MeltContext(cfg, lib=gpu_lib)
    load_state(c, st)
    c.set_dt(2e-3)
    c.tschem()
    c.sync()
    out = {q: c.download(q) for q in FIELDS}
    c.close()
    return out


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,n3", [(24, 24), (32, 48), (48, 24), (64, 24), (64, 64), (96, 32), (128, 24), (128, 96), (192, 32)])
def test_filter_forms_and_cyclic_reduction_agree(gpu_lib, monkeypatch, n, n3, precision):
    cfg = make_cfg(n, n3, imlsfor=0, imlsstr=0, imelt=0, precision=precision)
    st = random_state(make_cfg(n, n3), seed=n + n3)
    ref = step(gpu_lib, monkeypatch, cfg, st, "")
    for tune in ("yz_jb=1", "yz_jb=8", "yz_jb=16"):
        got = step(gpu_lib, monkeypatch, cfg, st, tune)
        for q in FIELDS:
            assert np.array_equal(got[q], ref[q]), (tune, q)
    pcr = step(gpu_lib, monkeypatch, cfg, st, "green=0")
    # FP64: round-off of three substeps; FP32: the filters' truncation (1e-8) and a
    # few roundings of 6e-8 of the solution per solve, on u, v, w, T; the pressure
    # takes the divergence's differences over dt, scaled by its own size
    for q in FIELDS:
        bar = 1e-12 if precision == 0 else (1e-4 if q == "pr" else 2e-6)
        assert rel_err(ref[q], pcr[q]) < bar, q
