"""Field transfers of the precision form on both sides of the sizes at which the
conversion moves between the calling thread and the device, from and into
pinned and pageable arrays: the same values, rounded to nearest, as numpy's."""
import ctypes as C

import numpy as np
import pytest

from melt_ibm_amd.api import FIELD_ID, MeltContext
from tests.helpers import make_cfg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n3", [(64, 48), (64, 64), (128, 64), (128, 96), (128, 128), (128, 192)])
def test_conversion_places_agree(gpu_lib, n, n3):
    import torch
    cfg = make_cfg(n, n3, precision=1)
    rng = np.random.default_rng(n3)
    a = rng.standard_normal(cfg.shape) * 10.0 ** rng.integers(-45, 38, cfg.shape)   # down to subnormal floats
    a.flat[:6] = (np.inf, -np.inf, np.nan, -0.0, 1e300, 1.0 + 2.0 ** -24)             # the last a tie
    with np.errstate(over="ignore"):
        want = a.astype(np.float32).astype(np.float64)
    c = MeltContext(cfg, lib=gpu_lib)
    fid = FIELD_ID["temp"]
    for up_pinned in (False, True):
        src = torch.empty(cfg.shape, dtype=torch.float64, pin_memory=up_pinned)
        src.numpy()[:] = a
        c.fill("temp", 7.0)
        assert gpu_lib.melt_upload_field(c._ctx, fid, C.c_void_p(src.data_ptr()), None) == 0
        for down_pinned in (False, True):
            dst = torch.full(cfg.shape, 5.0, dtype=torch.float64, pin_memory=down_pinned)
            assert gpu_lib.melt_download_field(c._ctx, fid, C.c_void_p(dst.data_ptr()), None) == 0
            got = dst.numpy()
            assert np.array_equal(got, want, equal_nan=True), (up_pinned, down_pinned)
            assert np.array_equal(np.signbit(got), np.signbit(want)), (up_pinned, down_pinned)
    c.close()
