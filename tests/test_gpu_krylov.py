"""The pressure solver's flexible CG at the sizes where its scalars change
hands, and the host's ring of residuals past its end."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(n, width, seed):
    """Five-point Laplacian plus 1e-2 on n cells in rows of `width`."""
    rng = np.random.default_rng(seed)
    r, c, v = [], [], []
    diag = np.full(n, 1e-2)
    for off in (1, width):
        i = np.arange(n - off)
        if off == 1:
            i = i[(i + 1) % width != 0]
        w = 1.0 + 0.2 * rng.random(i.size)
        for a, b in ((i, i + off), (i + off, i)):
            r.append(a); c.append(b); v.append(-w)
        diag += np.bincount(i, w, n) + np.bincount(i + off, w, n)
    r.append(np.arange(n)); c.append(np.arange(n)); v.append(diag)
    return np.concatenate(r), np.concatenate(c), np.concatenate(v), rng.standard_normal(n)


def _solver(precision):
    from semo_mesh_amd.cases import cavity_case
    from semo_mesh_amd.mesh import hex_mesh
    from semo_mesh_amd.solver import GpuSolver
    g = GpuSolver(0)
    g.upload_mesh(hex_mesh(2, 2, 2))
    g.set_case(cavity_case())
    g.set_solver(precision, tol_p=1e-9, tol_u=1e-9, maxit_p=200, maxit_u=200)
    return g


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [262079, 262144, 262145, 262401])
def test_totals_on_both_sides_of_the_block_limit(n, precision):
    """Up to 1024 blocks of 256 rows each block sums the partials itself,
    beyond a kernel does.  The recurrence stops at 1e-9; its distance from the
    true residual is round-off of the iterates, far below a factor of 2."""
    r, c, v, b = _system(n, 509, 3)
    g = _solver(precision)
    x = g.solveAMGCL("pressure", r, c, v, b)
    its = g.last_stats.iters[0]
    g.close()
    res = np.linalg.norm(b - np.bincount(r, v * x[c], n)) / np.linalg.norm(b)
    print(n, precision, its, res)
    assert 2 < its < 60 and res <= 2e-9


def _dense_stencil(m, ragged):
    """Every cell of an m^3 grid coupled to its 26 neighbours or, ragged, to
    its six and every 64th cell also to 24 further ones."""
    rng = np.random.default_rng(11)
    n = m ** 3
    idx = np.arange(n).reshape(m, m, m)
    pairs = []
    for dz, dy, dx in np.ndindex(3, 3, 3):
        d = np.array([dz, dy, dx]) - 1
        if tuple(d) <= (0, 0, 0) or (ragged and np.abs(d).sum() > 1):
            continue
        lo, hi = np.maximum(-d, 0), m - np.maximum(d, 0)
        i = idx[lo[0]:hi[0], lo[1]:hi[1], lo[2]:hi[2]].ravel()
        pairs.append((i, i + d @ (m * m, m, 1), 1.0 / (d @ d)))
    if ragged:
        i = np.repeat(np.arange(0, n, 64), 24)
        j = (i + 2 + np.arange(i.size) % 24) % n
        pairs.append((i, j, 0.01))
    r, c, v = [np.arange(n)], [np.arange(n)], [np.full(n, 1e-2)]
    for i, j, w in pairs:
        w = w * (1.0 + 0.2 * rng.random(i.size))
        r += [i, j, i, j]; c += [j, i, i, j]; v += [-w, -w, w, w]
    return np.concatenate(r), np.concatenate(c), np.concatenate(v), rng.standard_normal(n)


@pytest.mark.parametrize("ragged", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_finest_level_with_long_or_unequal_rows(precision, ragged):
    """Rows of 26 neighbours, and slices with one long row among short ones:
    the hierarchy keeps its finest operator in CSR, the Krylov product in
    sliced ELL.  Smoothed aggregation takes 13 iterations."""
    r, c, v, b = _dense_stencil(12, ragged)
    g = _solver(precision)
    x = g.solveAMGCL("pressure", r, c, v, b)
    its, levels = g.last_stats.iters[0], g.last_stats.n_levels
    g.close()
    res = np.linalg.norm(b - np.bincount(r, v * x[c], b.size)) / np.linalg.norm(b)
    print(precision, ragged, its, levels, res)
    assert levels >= 2 and its <= 20 and res <= 2e-9


def test_ring_of_residuals_wraps():
    """Solves until well over 1024 residuals have passed through the ring:
    each gives the first one's bits."""
    r, c, v, b = _system(3001, 53, 5)
    g = _solver("fp64")
    first, total = None, 0
    for _ in range(400):
        x = g.solveAMGCL("pressure", r, c, v, b)
        total += g.last_stats.iters[0]
        first = x if first is None else first
        assert np.array_equal(x, first)
        if total > 2500:
            break
    g.close()
    assert total > 1100


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_smoother_degree_changed_between_solves(precision):
    """Iterations are kept as graphs that hand the next V-cycle its start, and
    degree-2 smoothing swaps the buffers it lies in.  Whatever was solved
    before, with one or two iterations (not every graph captured) or more, a
    solve from the same state gives the first one's bits."""
    from semo_mesh_amd.cases import cavity_case
    from semo_mesh_amd.mesh import cavity_mesh
    from semo_mesh_amd.solver import GpuSolver
    m = cavity_mesh(16, jitter=0.1, seed=29)
    rng = np.random.default_rng(3)
    state = {f: 1e-2 * rng.standard_normal(m.n_cells) for f in "PUVW"}

    def solve(g, degree, tol=1e-10):
        for f, v in state.items():
            g.set_field(f, v)
        g.set_solver(precision, tol_p=tol, tol_u=1e-10, maxit_p=200, maxit_u=200, cheb_degree=degree)
        g.calcPressureEq()
        assert g.last_stats.n_levels >= 2
        return g.last_stats.iters[0], g.get_field("P")

    def fresh(history, degree):
        g = GpuSolver(0)
        g.upload_mesh(m, reorder=True)
        g.set_case(cavity_case())
        g.set_solver(precision, tol_p=1e-10, tol_u=1e-10, cheb_degree=5)
        g.incompressiblePressureBased(1)
        for d, tol in history:
            its, _ = solve(g, d, tol)
            print(d, tol, its)
        out = solve(g, degree)
        g.close()
        return out

    for history in ([(1, 0.09), (2, 0.09)], [(1, 0.3), (2, 0.3)], [(1, 0.3), (2, 1e-10)],
                    [(2, 0.3), (1, 0.09), (3, 0.09)], [(d, t) for t in (0.3, 1e-10) for d in (1, 2, 3, 4, 1)]):
        for degree in (1, 2):
            its, p = fresh([], degree)
            got, q = fresh(history, degree)
            assert 3 < its < 60 and got == its and np.array_equal(p, q), (history, degree, its, got)


@pytest.mark.parametrize("equation, precision, scale", [
    ("pressure", "fp64", 1.0), ("pressure", "mixed", 1.0), ("pressure", "mixed", 1e40),
    ("momentum", "fp64", 1.0), ("momentum", "fp64", 1e-311)])
def test_zero_right_side_gives_zero(equation, precision, scale):
    """Also where the preconditioner overflows its type (entries above FP32's
    range, diagonals whose reciprocal is infinite) and no residual says so."""
    r, c, v, _ = _system(3001, 53, 5)
    g = _solver(precision)
    x = g.solveAMGCL(equation, r, c, v * scale, np.zeros(3001))
    g.close()
    assert not x.any() and not np.isnan(x).any()


def test_momentum_residuals_past_the_rings_end():
    """A diffusion-dominated momentum system of a long column of cells, more
    than 1024 lockstep iterations: the relative residuals are those of the
    exported system, of which summing in another order changes 2e-10
    (measured; bar 1e-3)."""
    from semo_mesh_amd.cases import BC_FIXED_VALUE, BC_ZERO_GRADIENT, PatchBC, cavity_case
    from semo_mesh_amd.mesh import hex_mesh
    from semo_mesh_amd.solver import GpuSolver
    m = hex_mesh(5000, 1, 1)
    case = cavity_case(dt=1e-3)
    free = PatchBC(u_type=BC_ZERO_GRADIENT)
    case.bcs = {k: free for k in case.bcs}
    case.bcs["pref"] = PatchBC(p_type=BC_FIXED_VALUE, u_type=BC_ZERO_GRADIENT)
    case.bcs["xmin"] = PatchBC(u_type=BC_FIXED_VALUE, u_value=(1.0, 0.5, 0.2))
    case.bcs["xmax"] = PatchBC(u_type=BC_FIXED_VALUE)
    g = GpuSolver(0)
    g.upload_mesh(m)
    g.set_case(case)
    g.set_momentum_solver("jacobi")
    g.set_solver("mixed", tol_p=1e-2, tol_u=1e-8)
    g.incompressiblePressureBased(1)
    case.dt, case.mu = 1e6, (1e3, 1e3)
    g.set_case(case)
    g.set_solver("fp64", tol_u=1e-8, maxit_u=20000)
    rng = np.random.default_rng(3)
    for f in "UVW":
        g.set_field(f, rng.standard_normal(m.n_cells))
    g.calcMomentumEqs()
    st = g.last_stats
    r, c, v, b = g.matrix("momentum")
    x = [g.get_field(f) for f in ("x0", "x1", "x2")]
    g.close()
    print(st.iters[0], list(st.rel_res))
    assert st.iters[0] > 1100
    for k in range(3):
        rel = np.linalg.norm(b[k] - np.bincount(r, v * x[k][c], m.n_cells)) / np.linalg.norm(b[k])
        assert abs(st.rel_res[k] - rel) <= 1e-3 * rel
