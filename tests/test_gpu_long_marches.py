"""Marches of many planes: the explicit pass with as many planes per block as
the larger grids take (two rows per block in FP64 at 384 cells, two cells per
thread in FP32 from 256), on grids short enough for a test by asking for the
planes (xf_z), against line tiles (xf_w=1); and the fused y/z pass with segments
of 64 and 128 planes against two passes (yz_jb=1).  Bit for bit."""
import numpy as np
import pytest

from melt_ibm_amd.api import MeltContext
from tests.helpers import make_cfg

pytestmark = pytest.mark.gpu

FIELDS = ("vx", "vy", "vz", "temp", "pr")


def fields(cfg, names, seed):
    rng = np.random.default_rng(seed)
    return {q: rng.standard_normal(cfg.shape, dtype=np.float32).astype(np.float64) * 0.1 for q in names}


def substeps(gpu_lib, monkeypatch, cfg, st, tune, stages, out):
    monkeypatch.setenv("MELT_TUNE", tune)
    c = MeltContext(cfg, lib=gpu_lib)
    for q, a in st.items():
        c.upload(q, a)
    c.set_dt(1e-3)
    for ns in stages:
        c.substep(ns)
    c.sync()
    got = {q: c.download(q) for q in out}
    c.close()
    return got


@pytest.mark.parametrize("n,n3,precision,tunes", [
    (384, 48, 0, ("xf_z=12", "xf_z=24", "xf_z=48")),          # two rows per block
    (384, 16, 1, ("xf_z=4", "xf_z=8", "xf_z=16", "xf_one=1,xf_z=8")),
    (256, 16, 1, ("xf_z=4", "xf_z=8", "xf_one=1,xf_z=8")),    # two cells per thread, or one
    (256, 16, 0, ("xf_z=4", "xf_z=8")),
    (192, 16, 0, ("xf_z=8", "xf_z=16")),
])
def test_explicit_pass(gpu_lib, monkeypatch, n, n3, precision, tunes):
    cfg = make_cfg(n, n3, imlsfor=0, imlsstr=0, imelt=0, precision=precision)
    st = fields(cfg, (*FIELDS, "ru1", "ru2", "ru3", "rut", "forcx", "forcy", "forcz", "VOFp"), seed=n + n3)
    out = (*FIELDS, "ru1", "ru2", "ru3", "rut")
    ref = substeps(gpu_lib, monkeypatch, cfg, st, "xf_w=1", (1, 2), out)
    for tune in tunes:
        got = substeps(gpu_lib, monkeypatch, cfg, st, tune, (1, 2), out)
        for q in out:
            assert np.array_equal(got[q], ref[q]), (tune, q)


@pytest.mark.parametrize("n,n3,precision", [(256, 128, 1), (128, 256, 0), (128, 512, 0), (128, 512, 1), (128, 1024, 1)])
def test_yz_segments(gpu_lib, monkeypatch, n, n3, precision):
    """Segments of 64, 64, 128, 64 and 128 planes."""
    cfg = make_cfg(n, n3, imlsfor=0, imlsstr=0, imelt=0, precision=precision)
    st = fields(cfg, ("vx", "vy", "vz", "temp"), seed=n + n3)
    ref = substeps(gpu_lib, monkeypatch, cfg, st, "yz_jb=1", (1,), FIELDS)
    got = substeps(gpu_lib, monkeypatch, cfg, st, "", (1,), FIELDS)
    for q in FIELDS:
        assert np.array_equal(got[q], ref[q]), q
