"""The explicit pass's default launch shapes where their rule changes (line tiles,
z-march with 2 to 8 planes, two rows per block, one or two cells per thread)
against one x-line tiles (xf_w=1): the same values, bit for bit."""
import numpy as np
import pytest

from melt_ibm_amd.api import MeltContext
from tests.helpers import load_state, make_cfg, random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,n3", [(24, 8), (32, 24), (48, 16), (64, 16), (96, 8), (128, 8), (128, 16), (192, 8), (256, 8), (384, 8), (384, 12)])
def test_default_shape_matches_line_tiles(gpu_lib, monkeypatch, n, n3, precision):
    cfg = make_cfg(n, n3, imlsfor=0, imlsstr=0, imelt=0, precision=precision)
    st = random_state(make_cfg(n, n3), seed=n * n3)
    out = []
    for tune in ("", "xf_w=1"):
        monkeypatch.setenv("MELT_TUNE", tune)
        c = MeltContext(cfg, lib=gpu_lib)
        load_state(c, st)
        c.set_dt(1e-3)
        c.substep(1)
        c.substep(2)
        c.sync()
        out.append({q: c.download(q) for q in ("vx", "vy", "vz", "temp", "pr", "ru1", "ru2", "ru3", "rut")})
        c.close()
    for q in out[0]:
        assert np.array_equal(out[0][q], out[1][q]), q
