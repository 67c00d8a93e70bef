"""The HIT synthesis at grids whose blocks take 32 and 64 planes (with a
remainder) per column, against the oracle's direct sum: round-off of the field
scale, as for the small grids' 8 planes."""
import pytest

import oracle
from melt_ibm_amd.api import MeltContext
from tests.helpers import make_cfg, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n3", [(192, 128), (256, 96)])
def test_hit_segments_match_oracle(gpu_lib, n, n3):
    cfg = make_cfg(n, n3, imlsfor=0)
    g, o = MeltContext(cfg, lib=gpu_lib), oracle.context(cfg)
    print(f"# hit_force {n}x{n}x{n3}", flush=True)
    for c in (g, o):
        c.set_dt(0.013)
        c.hit_init(0.5, 0.05, 1.5, seed=9)
        c.hit_force()
    for q in ("forcx", "forcy", "forcz"):
        assert rel_err(g.download(q), o.download(q)) < 1e-13, q
    g.close()
    o.close()
