"""The block shapes of the diagnostics' reductions: fewer tiles than blocks,
a remainder, and more tiles than blocks, where each block walks several.
The maxima are exact in any order, so they equal the host's bit for bit (the
same operations in the same order, no contraction).  The sums of the
dissipation are of positive terms; a column of k planes, a tree and 16 partials
a lane round below 100 times, 1e-13 relative with the host's own sum: 1e-12."""
import ctypes as C

import numpy as np
import pytest

from melt_ibm_amd.api import MeltContext
from tests.helpers import make_cfg

pytestmark = pytest.mark.gpu


def _up(a, ax):
    return np.roll(a, -1, ax)


def _max_div(u, h):
    vx, vy, vz = (a.astype(np.float64) for a in u)          # [k, j, i]
    return np.abs((_up(vx, 2) - vx) * h[0] + (_up(vy, 1) - vy) * h[1] + (_up(vz, 0) - vz) * h[2]).max()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_max_divergence_over_block_shapes(gpu_lib, dtype):
    """From large to small, so a slot that an earlier, larger grid filled
    must not reach a later maximum."""
    import torch
    f = gpu_lib.melt_divgck_noalloc
    f.restype = C.c_int
    rng = np.random.default_rng(7)
    box = 2.0
    for n1, n2, n3 in ((1024, 1024, 5), (640, 640, 4), (128, 72, 33), (36, 31, 7), (4, 2, 2)):
        u = [rng.standard_normal((n3, n2, n1)).astype(dtype) * n1 for _ in range(3)]
        dev = [torch.from_numpy(a).cuda() for a in u]
        q = torch.full((1,), -1.0, dtype=torch.float64, device="cuda")
        print(f"# divgck_noalloc {n1}x{n2}x{n3} {np.dtype(dtype).name}", flush=True)
        for _ in range(2):
            rc = f(*(C.c_void_p(t.data_ptr()) for t in dev), n1, n2, n3, C.c_double(box), C.c_double(box), C.c_double(box),
                   u[0].itemsize, C.c_void_p(torch.cuda.current_stream().cuda_stream), C.c_void_p(q.data_ptr()))
            assert rc == 0
            assert q.item() == _max_div(u, (n1 / box, n2 / box, n3 / box))


@pytest.mark.parametrize("n,n3", [(8, 8), (12, 24), (48, 12), (768, 8)])
def test_dissipation_over_tile_shapes(gpu_lib, n, n3):
    cfg = make_cfg(n, n3, prandtl=0.7)
    rng = np.random.default_rng(n)
    c = MeltContext(cfg, lib=gpu_lib)
    f = {k: rng.standard_normal(cfg.shape) for k in ("vx", "vy", "vz", "temp")}      # [k, j, i]
    f["VOFp"] = rng.choice([0.0, 0.5, 1.0, 1.0], cfg.shape)
    for k, v in f.items():
        c.upload(k, v)
    got = c.dissipation()
    c.close()
    u, t, vof = [f[k].transpose(2, 1, 0) for k in ("vx", "vy", "vz")], f["temp"].transpose(2, 1, 0), f["VOFp"].transpose(2, 1, 0)
    d = (cfg.n1m / cfg.xlen, cfg.n2m / cfg.ylen, cfg.n3m / cfg.zlen)

    def mid(a, ax):
        return np.roll(a, -1, ax) - np.roll(a, 1, ax)
    g = [[mid(u[q] + _up(u[q], q), a) * 0.25 * d[a] for a in range(3)] for q in range(3)]
    for q in range(3):
        g[q][q] = (_up(u[q], q) - u[q]) * d[q]
    m = vof == 1.0
    s = m.sum()
    tke = sum(u[q] ** 2 + _up(u[q], q) ** 2 for q in range(3))[m].sum() * 0.25 / s
    dis = sum(g[q][q] ** 2 for q in range(3)) + 0.5 * sum((g[b][a] + g[a][b]) ** 2 for a, b in ((0, 1), (0, 2), (1, 2)))
    dis = dis[m].sum() * 2.0 / cfg.ren / s
    chi = sum((0.5 * d[q] * mid(t, q)) ** 2 for q in range(3))[m].sum() / (cfg.ren * cfg.prandtl) / s
    assert got["sumvof"] == s
    for k, want in (("kenerg", tke), ("diss", dis), ("chi", chi)):
        assert abs(got[k] - want) <= 1e-12 * want, (k, got[k], want)
