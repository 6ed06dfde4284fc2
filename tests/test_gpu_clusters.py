"""The stencil passes over cell clusters (records staged in LDS) against the
gathering passes: the same terms in the same order, so the same bits.

Which of the two a pass was shows in its bytes: a cluster pass also reads the
clusters' lists."""
import numpy as np
import pytest

from semo_mesh_amd.cases import dam_break_case
from semo_mesh_amd.mesh import hex_mesh, prism_stack_mesh, rotated, tet_mesh

pytestmark = pytest.mark.gpu

MESHES = {
    # 255 to 257 cells, the last a cluster of one cell, and several clusters
    "hex255": lambda: hex_mesh(5, 3, 17, jitter=0.1, seed=3, ref_face=False),
    "hex256": lambda: hex_mesh(4, 4, 16, jitter=0.1, seed=3, ref_face=False),
    "hex257": lambda: hex_mesh(257, 1, 1, jitter=0.1, seed=3, ref_face=False),
    "hex513": lambda: hex_mesh(3, 9, 19, jitter=0.1, seed=3, ref_face=False),
    "tet252": lambda: tet_mesh(7, 2, 3, jitter=0.1, seed=3),
    "tet2310": lambda: tet_mesh(11, 5, 7, hi=(2.0, 1.0, 1.0), jitter=0.1, seed=3),
    "tet_turned": lambda: rotated(tet_mesh(9, 8, 7, jitter=0.1, seed=3), 5),
    "prisms": lambda: prism_stack_mesh(9, 4, jitter=0.05, seed=3),
    # thin layers, so that a cluster is a column through all of them: lists
    # whose records of five fields pass the LDS limit, and lists past CL_LIST
    "tet_thin12": lambda: tet_mesh(8, 8, 12, hi=(1.0, 1.0, 1e-2), jitter=0.1, seed=3),
    "tet_thin24": lambda: tet_mesh(8, 8, 24, hi=(1.0, 1.0, 1e-2), jitter=0.1, seed=3),
}
PASSES = {"lsq1", "grad_minmax", "grad_minmax_uvw", "curv_kappa"}
GATHERED = {"tet_thin12": {"grad_minmax"}, "tet_thin24": PASSES}


@pytest.mark.parametrize("name", list(MESHES))
def test_same_bits_as_the_gathering_passes(name, monkeypatch):
    from semo_mesh_amd.solver import GpuSolver
    mesh = MESHES[name]()
    rng = np.random.default_rng(7)
    phi, fr = rng.standard_normal(mesh.n_cells), rng.standard_normal(mesh.n_faces)
    vf = rng.random(mesh.n_cells)
    out, nbytes = [], []
    for lanes in ("0", "1"):
        monkeypatch.setenv("SEMO_GPU_LSQ_LANES", lanes)
        g = GpuSolver(0)
        g.upload_mesh(mesh, reorder=True)
        g.profile(True)
        r = {"lsq": g.calcLeastSquare(phi, fr)}
        if set(mesh.patch_names) >= {"xmin", "zmax"}:
            case = dam_break_case(dt=1e-5)
            case.sigma = 0.07
            g.set_case(case)
            # cells 12 to 25 times as wide as high: solves end near 1e-9
            tol = 1e-8 if "thin" in name else 1e-10
            g.set_solver("fp64", tol_p=tol, tol_u=tol)
            g.set_field("VF", vf)
            g.incompressiblePressureBased(2)
            for f in ("gradP", "gradU", "gradV", "gradW", "gradVF", "maxP", "minP", "maxU", "minU", "maxV", "minV",
                      "maxW", "minW", "kappa", "P", "U"):
                r[f] = g.get_field(f)
        nbytes.append({k: v["bytes"] / v["count"] for k, v in g.profile_stats().items() if k in PASSES})
        g.close()
        out.append(r)
    print(name, nbytes)
    assert set(nbytes[0]) == (PASSES if len(out[0]) > 1 else {"lsq1"})
    for k, v in nbytes[0].items():
        assert (v == nbytes[1][k]) == (k in GATHERED.get(name, ())), k
    for f in out[0]:
        assert np.array_equal(out[0][f], out[1][f]), f
