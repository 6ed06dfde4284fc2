"""HIP path (libsemo_gpu.so, called through its C ABI) against the CPU
oracle and the reference's golden vectors.

Bars: on a mesh uploaded without renumbering the FP64 assembly reproduces the
oracle bit for bit (both follow the reference's per-cell summation order;
the library is built with -ffp-contract=off); with RCM renumbering the
per-cell order of the sums changes, so results agree to round-off
(relative 1e-12).  Solved fields agree with the oracle to relative L2 1e-10
(FP64 path) / 1e-6 (mixed path) at tight solver tolerances.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from conftest import GOLDEN_CASES, golden_case, load_golden
from semo_mesh_amd.cases import cavity_case, dam_break_case
from semo_mesh_amd.mesh import cavity_mesh, hex_mesh, tet_mesh

pytestmark = pytest.mark.gpu

GEOM = ["face_area", "face_normal", "face_xyz", "face_wC", "face_magPN", "face_alphaF",
        "face_ePN", "face_skew", "cell_volume", "cell_xyz", "cell_lsq"]


def _gpu(mesh, case, reorder):
    from semo_mesh_amd.solver import GpuSolver
    g = GpuSolver(0)
    g.upload_mesh(mesh, reorder=reorder)
    g.set_case(case)
    return g


def _rel(a, b):
    a = np.asarray(a, dtype=np.float64).ravel(); b = np.asarray(b, dtype=np.float64).ravel()
    nb = np.linalg.norm(b)
    return np.linalg.norm(a - b) / (nb if nb > 0 else 1.0)


@pytest.mark.parametrize("name", GOLDEN_CASES)
@pytest.mark.parametrize("reorder", [False, True])
def test_geometry_vs_reference(name, reorder):
    d, mesh = load_golden(name)
    g = _gpu(mesh, golden_case(d), reorder)
    scale = np.abs(d["cell_xyz"]).max()
    for k in GEOM:
        a = g.get_field(k).ravel()
        if reorder:
            # renumbering changes summation orders: round-off level, measured
            # against each array's magnitude (skew is zero up to round-off on
            # a uniform mesh, so it is measured against the domain size)
            ref = scale if k == "face_skew" else np.abs(d[k]).max()
            assert np.abs(a - d[k]).max() <= 1e-13 * ref, k
        else:
            assert np.array_equal(a, d[k]), k
    g.close()


@pytest.mark.parametrize("name", GOLDEN_CASES)
def test_rcm_permutation_and_connectivity_bit_exact(name):
    d, mesh = load_golden(name)
    g = _gpu(mesh, golden_case(d), True)
    perm, inv = g.permutation()
    assert np.array_equal(perm, d["rcm_perm"]) and np.array_equal(inv, d["rcm_inv"])
    # device connectivity is the original one renumbered
    own, nbr = g.connectivity()
    fmap, flip = g.face_map()
    nif = mesh.n_internal_faces
    o0 = mesh.owner[fmap]; n0 = np.full(mesh.n_faces, -1); n0[:nif] = mesh.neighbour[fmap[:nif]]
    a = np.where(flip[:nif] == 1, n0[:nif], o0[:nif]); b = np.where(flip[:nif] == 1, o0[:nif], n0[:nif])
    assert np.array_equal(perm[own[:nif]], a) and np.array_equal(perm[nbr], b)
    assert np.array_equal(perm[own[nif:]], o0[nif:])
    assert np.all(own[:nif] < nbr)
    assert sorted(fmap) == list(range(mesh.n_faces))
    g.close()


def _state(o, g, seed, nc, vf=None):
    rng = np.random.default_rng(seed)
    f = dict(P=rng.normal(size=nc) * 10.0, U=rng.normal(size=nc), V=rng.normal(size=nc),
             W=rng.normal(size=nc))
    f["VF"] = np.ones(nc) if vf is None else vf
    for k, v in f.items():
        o.set(k, v)
    o.eos()
    for k in ("U", "V", "W"):
        o.set("old" + k, o.get(k))
        o.set("Qm" + "UVW".index(k).__str__(), o.get(k))
    for k in ("P", "U", "V", "W", "VF", "Rho", "mu"):
        g.set_field(k, o.get(k))
    for k in ("U", "V", "W"):
        g.set_field("old" + k, o.get(k))
        g.set_field("Qm" + str("UVW".index(k)), o.get(k))


def _csr(r, c, v, n):
    return sp.coo_matrix((v, (r, c)), shape=(n, n)).tocsr()


@pytest.mark.parametrize("reorder", [False, True])
@pytest.mark.parametrize("eq", ["momentum", "pressure"])
def test_assembly_vs_oracle(oracle_lib, eq, reorder):
    mesh = hex_mesh(7, 6, 5, jitter=0.1, seed=21)
    case = cavity_case(); case.mu = (0.05, 0.05)
    o = oracle_lib.Oracle(mesh, case)
    g = _gpu(mesh, case, reorder)
    _state(o, g, 5, mesh.n_cells)
    o.recon(); o.gravity()
    (o.assemble_momentum if eq == "momentum" else o.assemble_pressure)()
    g.assemble(eq)
    r, c, v = o.coo()
    A0 = _csr(r, c, v, mesh.n_cells)
    gr, gc, gv, gb = g.matrix(eq)
    A1 = _csr(gr, gc, gv, mesh.n_cells)
    nb = 3 if eq == "momentum" else 1
    for f in ("gradP", "gradU", "gradV", "gradW"):
        a, b = g.get_field(f), o.get(f).reshape(-1, 3)
        assert (np.array_equal(a, b) if not reorder else _rel(a, b) < 1e-12), f
    if not reorder:
        assert (A1 != A0).nnz == 0
        for k in range(nb):
            assert np.array_equal(gb[k], o.get(f"b{k}")), k
    else:
        assert abs(A1 - A0).max() <= 1e-12 * abs(A0).max()
        for k in range(nb):
            assert _rel(gb[k], o.get(f"b{k}")) < 1e-12
    g.close()


def _eq_of_call(d, k):
    for eq in ("momentum", "pressure", "volume_fraction"):
        if f"call{k}_{eq}_rows" in d:
            return eq
    return None


@pytest.mark.parametrize("name", ["cavity4_jitter_random", "box654_jitter_2x2", "orifice_lid",
                                  "vof_box654_2x2", "vof_tet433_2x1", "sigma_box766_2x1",
                                  "bc_open_box654_2x2", "bc_vof_box654_2x1"])
def test_assembly_replay_vs_reference(name):
    """The reference's own COO systems, replayed from its call-time fields.
    Momentum and pressure systems are bit-exact.  Volume-fraction systems
    depend on MSTACS's blend weight pow(cos(theta), 4): the reference's libm
    pow is not correctly rounded in ~0.1% of cases and the device pow
    differs from it there in the last bit, so MSTACS face values and the VOF
    system are compared at 1e-14 relative (all other entries exactly)."""
    d, mesh = load_golden(name)
    case = golden_case(d)
    g = _gpu(mesh, case, False)
    k = 0
    while _eq_of_call(d, k):
        eq = _eq_of_call(d, k)
        p = f"call{k}_{eq}_"
        for f in ("P", "U", "V", "W", "VF", "Rho", "mu", "oldU", "oldV", "oldW", "Qm0", "Qm1", "Qm2",
                  "Qm3", "oldVF"):
            if p + f in d:
                g.set_field(f, d[p + f])
        if p + "dt" in d:
            if case.adjust_dt and (k == 0 or _eq_of_call(d, k - 1) == "pressure"):
                # first call of a time step: the adjusted time step (timestep.cpp:260-330)
                dt, _ = g.calcTimeStep(True)
                assert dt == d[p + "dt"][0], p + "dt"
            case.dt = float(d[p + "dt"][0])
            g.set_case(case)
        if any(case.g):
            for q in range(3):
                g.set_field(f"srcG{q}", d[p + f"srcG{q}"])
        if case.sigma:
            # curvature and surface tension, once per time step after the VOF
            # loop (pressureBased.cpp:130); the reference inverts the level-set
            # least-squares matrices by SVD, the device by cofactors: round-off
            if eq == "momentum" and _eq_of_call(d, k - 1) == "volume_fraction":
                g.calcSourceSurfaceTension()
                for f in ("kappa", "srcS0", "srcS1", "srcS2"):
                    assert _rel(g.get_field(f), d[p + f]) <= 1e-12, p + f
            for f in ("kappa", "srcS0", "srcS1", "srcS2"):
                g.set_field(f, d[p + f])
        g.assemble(eq)
        gr, gc, gv, gb = g.matrix(eq)
        n = mesh.n_cells
        A1 = _csr(gr, gc, gv, n)
        A0 = _csr(d[p + "rows"], d[p + "cols"], d[p + "vals"], n)
        if eq == "volume_fraction":
            for f in ("faceLVF", "faceRVF"):
                a, b = g.get_field(f), d[p + f]
                assert np.abs(a - b).max() <= 1e-14, (p, f)
            assert (A1 != A0).nnz == 0 or abs(A1 - A0).max() <= 1e-14 * abs(A0).max(), p
            assert _rel(gb[0], d[p + "b0"]) <= 1e-14, p
        else:
            assert (A1 != A0).nnz == 0, p
            for q in range(3 if eq == "momentum" else 1):
                assert np.array_equal(gb[q], d[p + f"b{q}"]), p
        k += 1
    assert k == len([x for x in d if x.endswith("_rows")])
    g.close()


@pytest.mark.parametrize("name", ["box654_jitter_2x2", "vof_tet433_2x1", "bc_open_box654_2x2",
                                  "bc_vof_box654_2x1"])
def test_assembly_replay_renumbered(name):
    """The same replay on an RCM-renumbered upload, where faces whose owner
    changes are flipped: every system agrees to round-off (summation orders
    change).  The tetrahedral mesh flips many faces, which pins the
    orientation-dependent terms (the pressure matrix's rho* and the float
    rounding of wC are defined in the mesh's own orientation)."""
    d, mesh = load_golden(name)
    case = golden_case(d)
    g = _gpu(mesh, case, True)
    _, flip = g.face_map()
    k = 0
    while _eq_of_call(d, k):
        eq = _eq_of_call(d, k)
        p = f"call{k}_{eq}_"
        for f in ("P", "U", "V", "W", "VF", "Rho", "mu", "oldU", "oldV", "oldW", "Qm0", "Qm1", "Qm2",
                  "Qm3", "oldVF"):
            if p + f in d:
                g.set_field(f, d[p + f])
        if p + "dt" in d:
            case.dt = float(d[p + "dt"][0])
            g.set_case(case)
        if any(case.g):
            for q in range(3):
                g.set_field(f"srcG{q}", d[p + f"srcG{q}"])
        g.assemble(eq)
        gr, gc, gv, gb = g.matrix(eq)
        n = mesh.n_cells
        A1 = _csr(gr, gc, gv, n)
        A0 = _csr(d[p + "rows"], d[p + "cols"], d[p + "vals"], n)
        assert abs(A1 - A0).max() <= 1e-12 * abs(A0).max(), p
        for q in range(3 if eq == "momentum" else 1):
            assert _rel(gb[q], d[p + f"b{q}"]) <= 1e-12, p
        k += 1
    if name.startswith("vof_tet"):
        assert flip.sum() > 0
    g.close()


def test_lsq_and_minmax_vs_oracle(oracle_lib):
    mesh = hex_mesh(9, 7, 6, jitter=0.1, seed=3)
    case = cavity_case()
    o = oracle_lib.Oracle(mesh, case)
    for reorder in (False, True):
        g = _gpu(mesh, case, reorder)
        rng = np.random.default_rng(1)
        phi = rng.normal(size=mesh.n_cells); fr = rng.normal(size=mesh.n_faces)
        a = g.calcLeastSquare(phi, fr); b = o.lsq(phi, fr)
        assert (np.array_equal(a, b) if not reorder else _rel(a, b) < 1e-12)
        mx, mn = g.setCellVarMinMax(phi); mx0, mn0 = o.minmax(phi)
        assert np.array_equal(mx, mx0) and np.array_equal(mn, mn0)
        g.close()


@pytest.mark.parametrize("lanes", ["2", "4"])
def test_lsq_lanes_same_bits(oracle_lib, monkeypatch, lanes):
    """The one-field LSQ pass with 2 or 4 lanes per cell (the group spreads a
    cell's stencil gathers, then adds the terms in stencil order on every
    lane) gives the bits of the one-lane pass, and the oracle's on the
    un-renumbered mesh: a jittered tet mesh, whose vertex stencils hold up to
    about 70 cells in counts that are not multiples of the group."""
    mesh = tet_mesh(5, 4, 4, jitter=0.1, seed=2)
    case = dam_break_case(dt=1e-4, n_vof=1, urf_vf=1.0)
    o = oracle_lib.Oracle(mesh, case)
    rng = np.random.default_rng(7)
    phi = rng.normal(size=mesh.n_cells); fr = rng.normal(size=mesh.n_faces)
    ref = o.lsq(phi, fr)
    for reorder in (False, True):
        out = {}
        for lv in ("1", lanes):
            monkeypatch.setenv("SEMO_GPU_LSQ_LANES", lv)
            g = _gpu(mesh, case, reorder)
            try:
                out[lv] = g.calcLeastSquare(phi, fr)
            finally:
                g.close()
        assert np.array_equal(out[lanes], out["1"]), reorder
        if not reorder:
            assert np.array_equal(out[lanes], ref)


@pytest.mark.parametrize("name", GOLDEN_CASES)
def test_simple_run_vs_reference(name):
    """Full SIMPLE run on the device against the reference's final fields (the
    reference solves to AMGCL's 1e-9, so 1e-7 relative)."""
    d, mesh = load_golden(name)
    g = _gpu(mesh, golden_case(d), True)
    g.set_solver("fp64", tol_p=1e-13, tol_u=1e-13, maxit_p=2000, maxit_u=2000)
    nc = mesh.n_cells
    if "init" in d:
        for k, f in enumerate(("P", "U", "V", "W", "VF")):
            g.set_field(f, d["init"][k * nc:(k + 1) * nc])
    for _ in range(int(d["steps"])):
        g.incompressiblePressureBased(int(d["correctors"]))
    vel = np.sqrt(sum(np.linalg.norm(d["final_" + f]) ** 2 for f in "UVW"))
    for f in ("P", "U", "V", "W", "VF"):
        a, b = g.get_field(f), d["final_" + f]
        scale = np.linalg.norm(b) if f in ("P", "VF") else vel
        assert np.linalg.norm(a - b) <= 1e-7 * scale, f
    g.close()


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-10), ("mixed", 1e-6)])
def test_simple_iterations_vs_oracle(oracle_lib, precision, tol):
    """Three SIMPLE iterations on a jittered 12^3 cavity: every field within
    relative L2 1e-10 (FP64) / 1e-6 (mixed) of the oracle, both solved to a
    relative residual of 1e-13 (FP64) / 1e-10 (mixed)."""
    mesh = cavity_mesh(12, jitter=0.1)
    case = cavity_case(); case.mu = (0.01, 0.01)
    o = oracle_lib.Oracle(mesh, case)
    o.set_solver(1e-14, 10000)
    g = _gpu(mesh, case, True)
    g.set_solver(precision, tol_p=1e-13 if precision == "fp64" else 1e-10, tol_u=1e-13,
                 maxit_p=3000, maxit_u=3000)
    for _ in range(3):
        o.step(1)
        g.incompressiblePressureBased(1)
    vel = np.sqrt(sum(np.linalg.norm(o.get(f)) ** 2 for f in "UVW"))
    for f in ("P", "U", "V", "W"):
        a, b = g.get_field(f), o.get(f)
        scale = np.linalg.norm(b) if f == "P" else vel
        assert np.linalg.norm(a - b) <= tol * scale, (f, np.linalg.norm(a - b) / scale)
    g.close()


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-10), ("mixed", 1e-6)])
def test_vof_steps_vs_oracle(oracle_lib, precision, tol):
    """Two two-phase time steps (MSTACS + VOF equation, gravity, open top) on a
    jittered 10x8x8 box: every field, alpha included, within relative L2
    1e-10 (FP64) / 1e-6 (mixed) of the oracle."""
    from semo_mesh_amd.cases import dam_break_case
    mesh = hex_mesh(10, 8, 8, jitter=0.1, seed=5, ref_face=False)
    case = dam_break_case(dt=2e-3, n_vof=2, urf_vf=0.9)
    nc = mesh.n_cells
    cen = np.stack([mesh.points[mesh.cell_pts[mesh.cell_ptr[i]:mesh.cell_ptr[i + 1]]].mean(0)
                    for i in range(nc)])
    vf = ((cen[:, 0] < 0.45) & (cen[:, 2] < 0.55)).astype(float)
    rng = np.random.default_rng(9)
    init = {"P": rng.normal(size=nc), "U": 0.2 * rng.normal(size=nc), "V": 0.2 * rng.normal(size=nc),
            "W": 0.2 * rng.normal(size=nc), "VF": vf}
    o = oracle_lib.Oracle(mesh, case)
    o.set_solver(1e-14, 10000)
    g = _gpu(mesh, case, True)
    g.set_solver(precision, tol_p=1e-13 if precision == "fp64" else 1e-10, tol_u=1e-13,
                 maxit_p=3000, maxit_u=3000)
    for f, v in init.items():
        o.set(f, v); g.set_field(f, v)
    for _ in range(2):
        o.step(2)
        g.incompressiblePressureBased(2)
    vel = np.sqrt(sum(np.linalg.norm(o.get(f)) ** 2 for f in "UVW"))
    for f in ("P", "U", "V", "W", "VF"):
        a, b = g.get_field(f), o.get(f)
        scale = np.linalg.norm(b) if f in ("P", "VF") else vel
        assert np.linalg.norm(a - b) <= tol * scale, (f, np.linalg.norm(a - b) / scale)
    assert 0.0 < o.get("VF").mean() < 1.0
    g.close()


def _droplet(mesh, centre, radius, width):
    nc = mesh.n_cells
    ptr, pts = mesh.cell_ptr, mesh.cell_pts
    cen = np.stack([mesh.points[pts[ptr[i]:ptr[i + 1]]].mean(0) for i in range(nc)])
    r = np.linalg.norm(cen - np.asarray(centre), axis=1)
    return np.clip((radius - r) / width + 0.5, 0.0, 1.0)


@pytest.mark.parametrize("kind", ["hex", "tet"])
@pytest.mark.parametrize("reorder", [False, True])
def test_surface_tension_vs_oracle(oracle_lib, kind, reorder):
    """Curvature (level-set reinitialisation + normal divergence) and the
    surface-tension source of a smeared droplet, against the oracle.  Both
    use the same cofactor inverses; they differ in libm (pow(V, 0.3),
    pow(V, 0.333)), so the bar is round-off: 1e-12 relative.  A renumbered
    upload changes every summation order, and kappa is a second derivative
    of the reinitialised level set, which amplifies round-off: 1e-9 there."""
    from semo_mesh_amd.cases import dam_break_case
    from semo_mesh_amd.mesh import tet_mesh
    mesh = (hex_mesh(9, 8, 7, jitter=0.1, seed=13, ref_face=False) if kind == "hex"
            else tet_mesh(5, 4, 4, jitter=0.1, seed=13))
    case = dam_break_case(dt=1e-3); case.sigma = 0.07
    vf = _droplet(mesh, (0.5, 0.5, 0.45), 0.3, 0.15)
    rng = np.random.default_rng(4)
    nc = mesh.n_cells
    o = oracle_lib.Oracle(mesh, case)
    g = _gpu(mesh, case, reorder)
    for f, v in (("VF", vf), ("U", 0.1 * rng.normal(size=nc)), ("V", 0.1 * rng.normal(size=nc)),
                 ("W", 0.1 * rng.normal(size=nc))):
        o.set(f, v); g.set_field(f, v)
    o.eos(); o.recon(); o.surface_tension()
    g.calcSourceSurfaceTension()
    tol = 1e-9 if reorder else 1e-12
    for f in ("kappa", "srcS0", "srcS1", "srcS2"):
        a, b = g.get_field(f), o.get(f)
        assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b), (f, _rel(a, b))
    assert np.abs(o.get("kappa")).max() > 1.0
    g.close()


def test_solve_coo_seam():
    """solveAMGCL seam: a jittered-mesh pressure system and a momentum system
    solved from COO, checked by their FP64 residuals."""
    from semo_mesh_amd.solver import GpuSolver
    d, mesh = load_golden("box654_jitter_2x2")
    g = GpuSolver(0)
    g.set_solver("fp64", tol_p=1e-12, tol_u=1e-12)
    for eq in ("pressure", "momentum"):
        p = "call1_pressure_" if eq == "pressure" else "call0_momentum_"
        n = mesh.n_cells
        A = _csr(d[p + "rows"], d[p + "cols"], d[p + "vals"], n)
        nb = 1 if eq == "pressure" else 3
        b = np.stack([d[p + f"b{k}"] for k in range(nb)])
        x = np.atleast_2d(g.solveAMGCL(eq, d[p + "rows"], d[p + "cols"], d[p + "vals"], b))
        for k in range(nb):
            assert np.linalg.norm(b[k] - A @ x[k]) <= 1e-11 * np.linalg.norm(b[k])
            xr = d[p + f"x{k}"]
            assert np.linalg.norm(x[k] - xr) <= 1e-7 * np.linalg.norm(xr)
    g.close()


def test_error_paths():
    from semo_mesh_amd.solver import GpuSolver
    from semo_mesh_amd._lib import SemoError
    mesh = cavity_mesh(3)
    g = GpuSolver(0)
    with pytest.raises(SemoError):
        g.calcMomentumEqs()                        # no mesh yet
    g.upload_mesh(mesh)
    case = cavity_case()
    case.bcs["xmin"].u_type = 99                   # unknown boundary type
    with pytest.raises(SemoError) as e:
        g.set_case(case)
    assert e.value.code == 2
    g.close()


@pytest.mark.parametrize("reorder", [False, True])
@pytest.mark.parametrize("name", ["bc_open_box654_2x2", "bc_vof_box654_2x1"])
def test_gauss_green_vs_reference(name, reorder):
    """semo_gauss_green (calcGaussGreen, gradient.cpp:1778-1985) for every
    field against the reference's own call on the fixture's final state:
    bit-exact on the un-renumbered mesh, round-off after RCM renumbering."""
    d, mesh = load_golden(name)
    g = _gpu(mesh, golden_case(d), reorder)
    for f in ("P", "U", "V", "W", "VF"):
        a = g.calcGaussGreen(f, d["final_" + f], d["gg_faceR_" + f], d["gg_in_" + f]).ravel()
        b = d["gg_out_" + f]
        if reorder:
            # round-off of sums of terms of size |phi| A / V ~ |phi| / h, h ~ 0.1 (a
            # constant field has a zero gradient made of round-off)
            scale = np.abs(b).max() + np.abs(d["final_" + f]).max() * 10.0
            assert np.abs(a - b).max() <= 1e-12 * scale, f
        else:
            assert np.array_equal(a, b), f
    g.close()


@pytest.mark.parametrize("reorder", [False, True])
@pytest.mark.parametrize("size", [(2, 1, 1), (16, 16, 1), (257, 1, 1), (19, 9, 3)])
def test_fields_keep_the_callers_order(size, reorder):
    """A field set and read back is the caller's, bit for bit; three
    components of a cell (centres, which the mesh orders itself) come back
    with their cell."""
    from semo_mesh_amd.mesh import hex_mesh
    from semo_mesh_amd.solver import GpuSolver
    m = hex_mesh(*size)
    g = GpuSolver(0)
    g.upload_mesh(m, reorder=reorder)
    a = np.random.default_rng(5).standard_normal(m.n_cells)
    a[0] = -0.0
    g.set_field("P", a); g.set_field("U", -a)
    assert g.get_field("P").tobytes() == a.tobytes() and g.get_field("U").tobytes() == (-a).tobytes()
    perm, inv = g.permutation()
    assert reorder or np.array_equal(perm, np.arange(m.n_cells))
    x = g.get_field("cell_xyz")
    i = np.arange(m.n_cells)
    ref = (np.stack([i % size[0], i // size[0] % size[1], i // (size[0] * size[1])], 1) + 0.5) / np.array(size)
    g.close()
    np.testing.assert_allclose(x, ref, rtol=0, atol=1e-12)
