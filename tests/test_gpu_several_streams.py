"""Steps on several streams (tuning key streams = 2) on grids that take one by
themselves: what is queued ahead across substeps and calls, its cancelling, graph
replay, snapshots, remeshing and sphere tagging, as the checks of those parts do
them; and replayed graphs, both places of the probes' geometry stage, the HIT
forcing and remeshing against one stream, bit for bit."""
import numpy as np
import pytest

from melt_ibm_amd.api import MeltContext
from melt_ibm_amd.inputs import inqpr_temperature
from tests import test_gpu_graph, test_gpu_parity, test_gpu_remesh, test_gpu_snapshot
from tests.helpers import load_state, make_cfg, melt_case, with_body
from tests.test_gpu_sphere_streams import match_one_stream

pytestmark = pytest.mark.gpu


@pytest.fixture
def several(monkeypatch):
    monkeypatch.setenv("MELT_TUNE", "streams=2")


@pytest.mark.parametrize("precision", [0, 1])
def test_graph_replay(gpu_lib, several, precision):
    test_gpu_graph.test_graph_replay_matches_eager(gpu_lib, precision)


@pytest.mark.parametrize("use_graph", [False, True])
def test_queued_probe_geometry(gpu_lib, several, use_graph):
    test_gpu_graph.test_queued_probe_geometry_matches_recomputed(gpu_lib, use_graph)


def test_substeps_between_graph_replays(gpu_lib, several):
    test_gpu_graph.test_substeps_between_graph_replays_match_eager(gpu_lib)


@pytest.mark.parametrize("precision,graph", [(0, False), (1, False), (0, True)])
def test_resume(gpu_lib, several, tmp_path, precision, graph):
    test_gpu_snapshot.test_resume_continues_bit_for_bit(gpu_lib, tmp_path, precision, graph)


def test_remeshing_follows_the_oracle(gpu_lib, several):
    test_gpu_remesh.test_tschem_remeshes_like_the_oracle(gpu_lib, 0)


def test_snapshot_after_remeshing(gpu_lib, several):
    test_gpu_remesh.test_snapshot_after_remeshing_resumes(gpu_lib)


@pytest.mark.parametrize("precision", [0, 1])
def test_sphere_tagging(gpu_lib, several, precision):
    test_gpu_parity.test_sphere_tagging_and_step(gpu_lib, precision)


TUNES = (dict(streams=2), dict(streams=2, graph=1), dict(streams=2, coef=2), dict(streams=2, coef=2, graph=1))


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kw", [{}, dict(imelt=0), dict(imlsstr=0)], ids=["melt+move", "move", "melt"])
def test_graphs_and_coefficient_places_match_one_stream(gpu_lib, kw, precision):
    match_one_stream(gpu_lib, make_cfg(64, precision=precision, **kw), TUNES)


@pytest.mark.parametrize("precision", [0, 1])
def test_forcing_beside_the_step_matches_one_stream(gpu_lib, precision):
    match_one_stream(gpu_lib, make_cfg(64, precision=precision), (dict(streams=2), dict(streams=2, graph=1)), hit=True)


@pytest.mark.parametrize("precision", [0, 1])
def test_remeshing_matches_one_stream(gpu_lib, precision):
    cfg = test_gpu_remesh.remesh_cfg()
    cfg.precision = precision
    match_one_stream(gpu_lib, cfg, (dict(streams=2), dict(streams=2, coef=2)), level=test_gpu_remesh.LEVEL, rad=test_gpu_remesh.RAD, steps=3)


@pytest.mark.parametrize("precision", [0, 1])
def test_launch_shapes_on_a_marching_grid(gpu_lib, monkeypatch, precision):
    """128 x 128 x 32, above the one-stream size: a marching explicit pass, the
    fused y/z pass and several streams are the defaults here."""
    n, n3, level = 128, 32, 3
    cfg = make_cfg(n, n3, precision=precision)
    st, dt = melt_case(make_cfg(n, n3), level, 1.0, seed=29)
    outs = {}
    for tune in ("", "streams=1", "coef=2", "xf_w=1", "xf_z=1", "xf_z=8", "yz_jb=1", "yz_jb=16"):
        monkeypatch.setenv("MELT_TUNE", tune)
        c = MeltContext(cfg, lib=gpu_lib)
        load_state(c, st)
        with_body(c, level, 1.0)
        c.upload("temp", inqpr_temperature(cfg, c.body().pos_cm[:], 1.0))
        c.set_dt(dt)
        c.tagCells()
        c.tschem()
        c.tschem()
        c.sync()
        outs[tune] = [c.download(q) for q in ("vx", "vy", "vz", "temp", "pr", "VOFp")] + [c.lag("xyzv")]
        c.close()
    for tune, out in outs.items():
        assert all(np.array_equal(a, b) for a, b in zip(outs[""], out)), tune
