"""The stencil passes over cell clusters (records staged in LDS) against the
gathering passes: the same terms in the same order, so the same bits."""
import numpy as np
import pytest

from semo_mesh_amd.cases import dam_break_case
from semo_mesh_amd.mesh import hex_mesh, prism_stack_mesh, rotated, tet_mesh

pytestmark = pytest.mark.gpu

MESHES = {
    # one cluster with 255, 256 and 257 of its 256 cells wanted, several, and
    # a last cluster of one cell
    "hex255": lambda: hex_mesh(5, 3, 17, jitter=0.1, seed=3, ref_face=False),
    "hex256": lambda: hex_mesh(4, 4, 16, jitter=0.1, seed=3, ref_face=False),
    "hex513": lambda: hex_mesh(3, 9, 19, jitter=0.1, seed=3, ref_face=False),
    "tet252": lambda: tet_mesh(7, 2, 3, jitter=0.1, seed=3),
    "tet2310": lambda: tet_mesh(11, 5, 7, hi=(2.0, 1.0, 1.0), jitter=0.1, seed=3),
    "tet_turned": lambda: rotated(tet_mesh(9, 8, 7, jitter=0.1, seed=3), 5),
    "prisms": lambda: prism_stack_mesh(9, 4, jitter=0.05, seed=3),
}


@pytest.mark.parametrize("name", list(MESHES))
def test_same_bits_as_the_gathering_passes(name, monkeypatch):
    from semo_mesh_amd.solver import GpuSolver
    mesh = MESHES[name]()
    rng = np.random.default_rng(7)
    phi, fr = rng.standard_normal(mesh.n_cells), rng.standard_normal(mesh.n_faces)
    vf = rng.random(mesh.n_cells)
    out = []
    for lanes in ("0", "1"):
        monkeypatch.setenv("SEMO_GPU_LSQ_LANES", lanes)
        g = GpuSolver(0)
        g.upload_mesh(mesh, reorder=True)
        r = {"lsq": g.calcLeastSquare(phi, fr)}
        if set(mesh.patch_names) >= {"xmin", "zmax"}:
            case = dam_break_case(dt=1e-5)
            case.sigma = 0.07
            g.set_case(case)
            g.set_solver("fp64", tol_p=1e-10, tol_u=1e-10)
            g.set_field("VF", vf)
            g.incompressiblePressureBased(2)
            for f in ("gradP", "gradU", "gradV", "gradW", "gradVF", "maxP", "minP", "maxU", "minU", "maxV", "minV",
                      "maxW", "minW", "kappa", "P", "U"):
                r[f] = g.get_field(f)
        g.close()
        out.append(r)
    for f in out[0]:
        assert np.array_equal(out[0][f], out[1][f]), f
