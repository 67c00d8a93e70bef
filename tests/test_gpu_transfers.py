"""Field transfers of the precision form: the conversion on the device rounds a
double as the host does (to nearest), keeps infinities and NaN, and widens
exactly; odd-shaped layouts and ghost planes included."""
import ctypes as C

import numpy as np
import pytest

from melt_ibm_amd.api import FIELD_ID, MeltContext, _Layout
from tests.helpers import make_cfg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n3", [(8, 8), (24, 8), (48, 32), (64, 96)])
def test_fp32_round_trip(gpu_lib, n, n3):
    cfg = make_cfg(n, n3, precision=1)
    c = MeltContext(cfg, lib=gpu_lib)
    rng = np.random.default_rng(n)
    a = rng.normal(size=cfg.shape) * 10.0 ** rng.integers(-30, 30, cfg.shape)
    a.flat[:4] = (np.inf, -np.inf, np.nan, -0.0)
    a.flat[-1] = 1e300   # overflows to infinity
    c.upload("temp", a)
    with np.errstate(over="ignore"):
        ref = a.astype(np.float32).astype(np.float64)
    got = c.download("temp")
    assert np.array_equal(got.view(np.int64), ref.view(np.int64)) or np.array_equal(got, ref, equal_nan=True)
    assert np.array_equal(c.download_with_ghosts("temp")[1:-1], ref, equal_nan=True)
    # the reference's padded arrays: one more column and row, ghost planes
    pad = np.full((n3 + 2, n + 1, n + 1), 7.0)
    lay = _Layout(n + 1, n + 1, 1, 0)
    assert gpu_lib.melt_download_field(c._ctx, FIELD_ID["temp"], pad.ctypes.data, C.byref(lay)) == 0
    assert np.array_equal(pad[1:-1, :n, :n], ref, equal_nan=True)
    assert np.all(pad[:, n, :] == 7.0) and np.all(pad[:, :, n] == 7.0)
    assert gpu_lib.melt_upload_field(c._ctx, FIELD_ID["pr"], pad.ctypes.data, C.byref(lay)) == 0
    assert np.array_equal(c.download("pr"), ref, equal_nan=True)
    c.close()
