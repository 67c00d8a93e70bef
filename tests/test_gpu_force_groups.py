"""The tagging's and the MLS forcing's groups of faces (their size by
the face count, with remainders) against the oracle, and the same body with its faces in
random order, whose groups touch more cells than a block's table holds.  The
spread forces are exact integer sums, so the order of the faces changes no bit.
The oracle adds the same contributions in double precision, a few hundred per
cell: below 1e-13 of the sum of their magnitudes, 1e-12 of the largest force.
The distances and volume fractions are the oracle's bit for bit, the lowest
face among equals included."""
import numpy as np
import pytest

import oracle
from melt_ibm_amd import geometry
from melt_ibm_amd.api import MeltContext
from tests.helpers import load_state, make_cfg, random_state, rel_err

pytestmark = pytest.mark.gpu

FORCES = ("for_xc", "for_yc", "for_zc", "for_temp")


def _forces(cfg, st, mesh, order, lib=None):
    c = MeltContext(cfg, lib=lib) if lib is not None else oracle.context(cfg)
    c.set_geometry(mesh.xyz, mesh.vert_of_edge, np.ascontiguousarray(mesh.edge_of_face[order]), 1.1)
    load_state(c, st)
    c.set_dt(0.004)
    c.findCentroidIndices()
    c.mlsWeight()
    c.mlsForce()
    out = [c.download(f) for f in FORCES]
    c.close()
    return out


@pytest.mark.parametrize("freq", [3, 11, 13, 22])   # 180, 2420, 3380, 9680 faces
def test_forces_over_group_sizes_and_orders(gpu_lib, freq):
    cfg = make_cfg(64)
    st = random_state(cfg, 5)
    mesh = geometry.icosphere(freq)
    nf = mesh.edge_of_face.shape[0]
    plain, mixed = np.arange(nf), np.random.default_rng(freq).permutation(nf)
    want = _forces(cfg, st, mesh, plain)
    print(f"# mlsForce {nf} faces, as built and shuffled", flush=True)
    got, again = _forces(cfg, st, mesh, plain, gpu_lib), _forces(cfg, st, mesh, mixed, gpu_lib)
    for name, a, b, w in zip(FORCES, got, again, want):
        assert np.array_equal(a, b), (name, np.abs(a - b).max())
        assert np.abs(w).max() > 0 and np.abs(a - w).max() <= 1e-12 * np.abs(w).max(), name


@pytest.mark.parametrize("freq", [3, 11, 13, 22])
@pytest.mark.parametrize("order", ["as built", "shuffled"])
def test_tags_over_group_sizes_and_orders(gpu_lib, freq, order):
    cfg = make_cfg(96)
    mesh = geometry.icosphere(freq)
    nf = mesh.edge_of_face.shape[0]
    perm = np.arange(nf) if order == "as built" else np.random.default_rng(freq).permutation(nf)
    print(f"# tagCells {nf} faces, {order}", flush=True)
    out = []
    for c in (MeltContext(cfg, lib=gpu_lib), oracle.context(cfg)):
        c.set_geometry(mesh.xyz, mesh.vert_of_edge, np.ascontiguousarray(mesh.edge_of_face[perm]), 1.9)
        for _ in range(2):   # the second call resets what the first one tagged
            c.tagCells()
        out.append([c.download(f) for f in ("sdf", "VOFp")])
        c.close()
    for name, a, b in zip(("sdf", "VOFp"), *out):
        assert np.array_equal(a, b), (name, int((a != b).sum()))


def test_probes_of_a_body_across_the_corner(gpu_lib):
    """180 faces (a last, incomplete group of 64 probes) around the corner of the
    periodic box, where the stencils wrap in all three directions: heat fluxes
    and loads of one particle call.  The probes keep the oracle's order of
    operations on fields whose forces were added in another order (1e-16); a
    gradient over cells and a cancelling sum over faces take that to 1e-13 or
    so: 1e-10, as for the whole particle step."""
    cfg = make_cfg(32)
    st = random_state(cfg, 8)
    mesh = geometry.icosphere(3)
    out = []
    for c in (MeltContext(cfg, lib=gpu_lib), oracle.context(cfg)):
        c.set_geometry(mesh.xyz, mesh.vert_of_edge, mesh.edge_of_face, 1.2)
        centre = np.array(c.body().pos_cm[:])
        for q in ("xyzv", "tri_bar"):
            c.set_lag(q, c.lag(q) - centre)
        load_state(c, st)
        c.set_dt(0.002)
        c.set_stage(1)
        c.particle()
        b = c.body().as_dict()
        out.append({**{q: c.lag(q) for q in ("qw_oVert", "qw_iVert")}, **{q: np.atleast_1d(b[q]) for q in ("int_prn_dA", "int_tau_dA")}})
        c.close()
    for q, w in out[1].items():
        assert np.abs(w).max() > 0 and rel_err(out[0][q], w) <= 1e-10, q
