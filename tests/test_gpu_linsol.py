"""semo_linear_solver on the GPU: SEMO's density-based implicit updates
(src/solvers/linearSolver.cpp) against the compiled reference and the oracle.

* tests/golden/linsol_*.npz hold the reference's calcLinearSolver,
  calcSingleLinearSolver and calcLinearSolverLUSGS on seeded states (one,
  two and three species, hex and tet boxes).  On the mesh as given the
  device's updates equal them bit for bit (the same arithmetic in the same
  order; LU-SGS level-scheduled over lib_RCM's order, which reproduces the
  sequential sweeps exactly).  RCM-renumbered, the cells' faces are summed
  in another order: within 1e-11 of each equation's largest magnitude.
* Larger meshes against the oracle's sequential sweeps: a jittered 20^3
  hex box, a 8x8x6 tet box and a jittered 96^3 hex box (884,736 cells,
  hundreds of sweep levels): bit for bit on the mesh as given; renumbered,
  relative L2 per equation 1e-11 (measured 1.6e-12 at 96^3, the size of the
  change that reversing each cell's face order makes in the oracle itself).
* The device-array entry point equals the host one bit for bit."""
import ctypes as C

import numpy as np
import pytest

from conftest import load_golden
from golden.make_golden import linsol_residuals, linsol_states
from semo_mesh_amd.cases import cavity_case
from semo_mesh_amd.mesh import hex_mesh, tet_mesh

pytestmark = pytest.mark.gpu

CASES = ("linsol_box654", "linsol_tet433", "linsol_box543_nsp1", "linsol_tet322_nsp3")
METHODS = ("point", "single", "lusgs")


def _gpu(m, reorder):
    from semo_mesh_amd.solver import GpuSolver
    g = GpuSolver(0)
    g.upload_mesh(m, reorder=reorder)
    return g


def _run(g, method, dt, st, r0):
    if method == "point":
        return g.calcLinearSolver(dt, st, r0)
    if method == "single":
        return g.calcSingleLinearSolver(st, r0)
    return g.calcLinearSolverLUSGS(dt, st, r0)


def _close(a, ref, tol):
    scale = np.abs(ref).max(axis=0)
    err = (np.abs(a - ref) / scale).max()
    print("rel err", err)
    assert err <= tol, err


@pytest.mark.parametrize("reorder", [False, True])
@pytest.mark.parametrize("name", CASES)
def test_linsol_vs_reference(name, reorder):
    d, m = load_golden(name)
    st, r0, dt = d["linsol_state"], d["linsol_res0"], float(d["linsol_dt"])
    g = _gpu(m, reorder)
    try:
        for method in METHODS:
            out = _run(g, method, dt, st, r0)
            ref = d["linsol_" + method].reshape(r0.shape)
            print(name, method, reorder)
            if reorder and method == "lusgs":
                _close(out, ref, 1e-11)
            else:   # point and single updates are per cell: no order changes
                assert np.array_equal(out, ref), (method, np.abs(out - ref).max())
    finally:
        g.close()


@pytest.mark.parametrize("nsp", [1, 2, 3, 4])
def test_point_blocks_outside_the_shared_reciprocals(oracle_lib, nsp):
    """Blocks whose pivots are zero, overflow or lie outside [2^-900, 2^900]
    take plain divisions, among cells that do not: the oracle's results,
    infinities and NaN included."""
    m = hex_mesh(13, 5, 4, jitter=0.1, seed=5)
    o = oracle_lib.Oracle(m, cavity_case())
    st = linsol_states(m, nsp, 11, vol=o.get("cell_volume"))
    r0 = linsol_residuals(m.n_cells, nsp, 12)
    st[::7, 8] = 0.0; st[::7, 10] = 0.0          # no compressibility: singular blocks
    st[1::7, 5] *= 1e-290                        # density below the range
    st[2::7, 5] *= 1e290
    st[3::7, 7] = np.inf
    g = _gpu(m, False)
    try:
        for method in ("point", "single"):
            with np.errstate(all="ignore"):
                ref = o.linear_solver(method, nsp, 1e-3, st, r0)
            out = _run(g, method, 1e-3, st, r0)
            assert not np.isfinite(ref).all() and np.isfinite(ref[4::7]).all()
            assert np.array_equal(out, ref, equal_nan=True), method
    finally:
        g.close()


@pytest.mark.parametrize("kind", ["hex20", "tet886"])
def test_lusgs_vs_oracle(oracle_lib, kind):
    m = hex_mesh(20, 20, 20, jitter=0.1, seed=5) if kind == "hex20" else \
        tet_mesh(8, 8, 6, jitter=0.1, seed=6)
    o = oracle_lib.Oracle(m, cavity_case())
    st = linsol_states(m, 2, 11, vol=o.get("cell_volume"))
    r0 = linsol_residuals(m.n_cells, 2, 12)
    ref = o.linear_solver("lusgs", 2, 1e-3, st, r0)
    for reorder in (False, True):
        g = _gpu(m, reorder)
        try:
            out = g.calcLinearSolverLUSGS(1e-3, st, r0)
        finally:
            g.close()
        print(kind, reorder)
        if reorder:
            _close(out, ref, 1e-11)
        else:
            assert np.array_equal(out, ref)


@pytest.mark.parametrize("nsp", [1, 2, 3, 4])
@pytest.mark.parametrize("size", [(2, 1, 1), (2, 2, 2), (5, 5, 1), (13, 2, 1), (17, 3, 1), (13, 2, 2)])
def test_lusgs_of_a_few_cells(oracle_lib, size, nsp):
    """2 to 52 cells, fewer result values than the sweeps have control words:
    every call on a context starts from cleared tickets, other states in the
    middle one."""
    m = hex_mesh(*size, jitter=0.1, seed=5)
    o = oracle_lib.Oracle(m, cavity_case())
    vol = o.get("cell_volume")
    g = _gpu(m, False)
    try:
        for seed in (11, 13, 11):
            st, r0 = linsol_states(m, nsp, seed, vol=vol), linsol_residuals(m.n_cells, nsp, seed + 1)
            ref = o.linear_solver("lusgs", nsp, 1e-3, st, r0)
            assert np.array_equal(g.calcLinearSolverLUSGS(1e-3, st, r0), ref)
    finally:
        g.close()


def test_lusgs_large_vs_oracle(oracle_lib):
    """96^3 jittered hex (884,736 cells), both storage orders against the
    oracle's sequential sweeps."""
    m = hex_mesh(96, 96, 96, jitter=0.1, seed=21)
    o = oracle_lib.Oracle(m, cavity_case())
    st = linsol_states(m, 2, 31, vol=o.get("cell_volume"))
    r0 = linsol_residuals(m.n_cells, 2, 32)
    ref = o.linear_solver("lusgs", 2, 1e-3, st, r0)
    assert np.isfinite(ref).all()
    res = {}
    for reorder in (False, True):
        g = _gpu(m, reorder)
        try:
            res[reorder] = g.calcLinearSolverLUSGS(1e-3, st, r0)
        finally:
            g.close()
        a = res[reorder]
        l2 = np.linalg.norm(a - ref, axis=0) / np.linalg.norm(ref, axis=0)
        worst = np.abs(a - ref) / np.abs(ref).max(axis=0)
        k = np.unravel_index(np.argmax(worst), worst.shape)
        print("reorder", reorder, "rel L2 per equation", l2, "worst", worst.max(), "at", k, flush=True)
    assert np.array_equal(res[False], ref)
    l2 = np.linalg.norm(res[True] - ref, axis=0) / np.linalg.norm(ref, axis=0)
    assert l2.max() <= 1e-11


class _Dev:
    """Device buffers through the HIP runtime libsemo_gpu.so itself uses
    (torch carries a runtime of its own)."""

    def __init__(self):
        self.hip = C.CDLL("libamdhip64.so.7")
        self.bufs = []

    def put(self, a):
        a = np.ascontiguousarray(a, dtype=np.float64)
        p = C.c_void_p()
        assert self.hip.hipMalloc(C.byref(p), C.c_size_t(max(a.nbytes, 8))) == 0
        self.bufs.append(p)
        assert self.hip.hipMemcpy(p, a.ctypes.data_as(C.c_void_p), C.c_size_t(a.nbytes), 1) == 0
        return p.value

    def get(self, ptr, shape):
        out = np.empty(shape, dtype=np.float64)
        assert self.hip.hipDeviceSynchronize() == 0
        assert self.hip.hipMemcpy(out.ctypes.data_as(C.c_void_p), C.c_void_p(ptr), C.c_size_t(out.nbytes), 2) == 0
        return out

    def free(self):
        for p in self.bufs:
            self.hip.hipFree(p)
        self.bufs = []


def test_device_entry_matches_host_entry():
    d, m = load_golden("linsol_tet433")
    st, r0, dt = d["linsol_state"], d["linsol_res0"], float(d["linsol_dt"])
    g = _gpu(m, True)
    dv = _Dev()
    try:
        host = g.calcLinearSolverLUSGS(dt, st, r0)
        perm, _ = g.permutation()                 # device cell k = caller cell perm[k]
        ds, dr = dv.put(st[perm]), dv.put(r0[perm])
        g._ok(g._L.semo_linear_solver_device(g._h, 2, 2, dt, C.c_void_p(ds), C.c_void_p(dr)))
        dev = np.empty_like(host)
        dev[perm] = dv.get(dr, r0.shape)
        assert np.array_equal(dev, host)
    finally:
        dv.free()
        g.close()


def test_bad_arguments_refused():
    d, m = load_golden("linsol_box543_nsp1")
    g = _gpu(m, False)
    try:
        st, r0 = d["linsol_state"], d["linsol_res0"]
        with pytest.raises(Exception):
            g.calcLinearSolverLUSGS(0.0, st, r0)
        with pytest.raises(Exception):
            g.calcLinearSolver(1e-3, np.zeros((m.n_cells, 12 + 15)), np.zeros((m.n_cells, 9)))
    finally:
        g.close()
