"""The precision form's refinement gate compares the FP64 divergence of the
projected field with that of the provisional one, whose maximum the forward x
pass of the Poisson solve takes along: at every line length of that pass, with
the largest value in lines that different waves of a block hold."""
import numpy as np
import pytest

from melt_ibm_amd.api import MeltContext
from tests.helpers import make_cfg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [24, 32, 48, 64, 96, 128, 192, 256, 384])
def test_gate_measures_the_largest_divergence(gpu_lib, n):
    n3 = 8
    cfg = make_cfg(n, n3, imlsfor=0, imlsstr=0, imelt=0, forcing=0, betagz=0.0, precision=1)
    rng = np.random.default_rng(n)
    d = (cfg.n1m / cfg.xlen, cfg.n2m / cfg.ylen, cfg.n3m / cfg.zlen)
    c = MeltContext(cfg, lib=gpu_lib)
    # so short a step that the provisional field is the uploaded one: the step moves it
    # by dt |u| (|u| d + d^2 / Re), below 1e-10 of the largest value on these grids
    c.set_dt(1e-12)
    c.set_refinement(1, 1e30)   # measure, never refine
    for spike, (j, i) in enumerate([(0, 0), (7, n // 2 + 1), (n // 3 * 2 + 1, n // 3), (11, 1), (n - 1, n - 1)]):
        u = [rng.normal(0.0, 1e-2, cfg.shape).astype(np.float32).astype(np.float64) for _ in range(3)]
        u[0][spike, j, i] = 1.0 + spike
        for q, a in zip(("vx", "vy", "vz"), u):
            c.upload(q, a)
        for q in ("pr", "temp", "ru1", "ru2", "ru3", "rut"):
            c.fill(q, 0.0)
        c.substep(1)
        c.sync()
        ratio = c.refinement_stats()[2]
        want = np.abs((np.roll(u[0], -1, 2) - u[0]) * d[0] + (np.roll(u[1], -1, 1) - u[1]) * d[1] + (np.roll(u[2], -1, 0) - u[2]) * d[2]).max()
        before = c.divgck() / ratio
        assert abs(before - want) <= 1e-9 * want, (n, spike, before, want)
    c.close()
