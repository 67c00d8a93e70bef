"""The Poisson solve at every transform length of the register FFTs, as x and y
lines (n) and as z lines (n3), and at lengths of the staged transforms beside
them, against numpy's FFT in float64; and the fused substep's form (divergence
formed in the x pass), whose projected field is free of divergence."""
import numpy as np
import pytest

from melt_ibm_amd.api import MeltContext
from tests.helpers import make_cfg, random_state, load_state

pytestmark = pytest.mark.gpu

SHAPES = [(32, 24), (48, 8), (64, 48), (96, 8), (128, 32), (192, 8), (256, 8), (384, 8), (512, 8), (24, 96), (16, 128), (16, 192), (24, 256), (16, 384),
          (16, 512)]


def poisson(cfg, rhs):
    d = (cfg.n3m / cfg.zlen, cfg.n2m / cfg.ylen, cfg.n1m / cfg.xlen)
    lam = [2.0 * (1.0 - np.cos(2.0 * np.pi * np.arange(n) / n)) * w * w for n, w in zip(cfg.shape, d)]
    ev = -(lam[0][:, None, None] + lam[1][None, :, None] + lam[2][None, None, : cfg.n1m // 2 + 1])
    ev[0, 0, 0] = 1.0
    s = np.fft.rfftn(rhs) / ev
    s[0, 0, 0] = 0.0
    return np.fft.irfftn(s, s=cfg.shape, axes=(0, 1, 2))


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,n3", SHAPES)
def test_poisson_solve(gpu_lib, n, n3, precision):
    cfg = make_cfg(n, n3, imlsfor=0, imlsstr=0, imelt=0, precision=precision)
    c = MeltContext(cfg, lib=gpu_lib)
    rhs = np.random.default_rng(n + n3).normal(size=cfg.shape).astype(np.float32).astype(np.float64)
    c.upload("dph", rhs)
    c.phcalc()
    got, ref = c.download("dph"), poisson(cfg, rhs)
    c.close()
    # round-off of three transforms each way, against the largest value
    bar = 1e-13 if precision == 0 else 2e-6
    assert np.max(np.abs(got - ref)) < bar * np.max(np.abs(ref))


@pytest.mark.parametrize("n,n3", [(48, 8), (96, 24), (128, 16), (192, 8), (384, 8), (512, 8)])
def test_fused_step_is_divergence_free(gpu_lib, n, n3):
    cfg = make_cfg(n, n3, imlsfor=0, imlsstr=0, imelt=0)
    c = MeltContext(cfg, lib=gpu_lib)
    load_state(c, random_state(cfg, seed=n))
    c.set_dt(1e-3)
    c.tschem()
    c.sync()
    u = max(np.max(np.abs(c.download(q))) for q in ("vx", "vy", "vz"))
    assert c.divgck() < 1e-12 * u * n   # round-off of u over the cell width
    c.close()
