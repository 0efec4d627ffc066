"""Kernels at the sizes where they can go wrong: remainders of their row and
column groups, the smallest and the largest of their ranges."""
import numpy as np
import pytest

from gds2para_amd import _capi as capi
from gds2para_amd import mesh as M
from gds2para_amd.layout import Layout

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [capi.GP_PREC_FP64, capi.GP_PREC_MIXED])
@pytest.mark.parametrize("cells,slots", [((2, 2, 6), 1), ((4, 3, 6), 4), ((4, 4, 6), 16), ((3, 3, 7), 64)])
def test_coarsest_solve_alone(cells, slots, prec):
    """A grid of at most 400 edges has no coarser level: the dense coarsest
    solve of the whole system is the preconditioner.  Its error is the
    rounding of its inverses and of FP32 vectors, amplified by the 1e9 between
    the curl-curl and the mass terms, so a few steps reach 1e-8; a coarsest
    solve that skips or mixes rows or columns leaves an indefinite system of
    126 to 390 unknowns to plain GMRES.  Every column must end inside its
    first restart cycle."""
    m = M.Mesh(M.plate_spec(cells=cells, f=1e9))
    lay = Layout(m)
    lay.prepare(prec)
    edges = [e[0] for e in lay.hierarchy_info()["edge"]]
    print(f"[kernels] coarsest {cells}: {edges} edges, {slots} slots, precision {prec}", flush=True)
    assert len(edges) == 1 and edges[0] <= 400
    fs = np.geomspace(1e9, 1e10, slots)
    Z, st, _ = lay.solve(fs, precision=prec, rtol=1e-8, batch=slots, restart=16)
    print(f"[kernels]   iterations {max(st['iters'])}", flush=True)
    assert st["status"] == capi.GP_OK and st["converged"] == slots
    assert max(st["iters"]) <= 16
    lay.close()


@pytest.mark.parametrize("prec,slots", [(capi.GP_PREC_MIXED, 1), (capi.GP_PREC_MIXED, 2), (capi.GP_PREC_MIXED, 4),
                                        (capi.GP_PREC_MIXED, 8), (capi.GP_PREC_MIXED, 16), (capi.GP_PREC_MIXED, 32),
                                        (capi.GP_PREC_MIXED, 64), (capi.GP_PREC_FP64, 1), (capi.GP_PREC_FP64, 4)])
def test_aux_products_match_csr_kernels(prec, slots):
    """The auxiliary products of listed rows (a wavefront per chunk of 256
    entries, the longest rows in several) and short rows against the (row,
    slot) CSR kernels: 48x48x12 has rows of 1 to 11,924 entries on its finest
    auxiliary level.  The two differ by rounding only, which moves an
    application by 1e-7 (FP32) or 1e-16 of itself: the iteration counts agree
    to one step in ten, and Z to 100 times the residual."""
    m = M.Mesh(M.WORKLOADS["manhattan_48x48x12"]())
    lay = Layout(m)
    fs = np.geomspace(2e8, 4e9, max(1, slots // 4))
    kw = dict(ports=list(range(min(slots, 4))), precision=prec, rtol=1e-10, batch=slots, max_iters=400)
    Za, sa, _ = lay.solve(fs, **kw)
    Zb, sb, _ = lay.solve(fs, sell_min_rows=1 << 40, **kw)
    print(f"[kernels] aux products, {slots} slots, precision {prec}: iterations {max(sa['iters'])} / {max(sb['iters'])}, "
          f"dZ {np.abs(Za - Zb).max() / np.abs(Zb).max():.2e}", flush=True)
    assert sa["status"] == sb["status"] == capi.GP_OK
    assert all(abs(a - b) <= 1 + b // 10 for a, b in zip(sa["iters"], sb["iters"]))
    assert np.abs(Za - Zb).max() <= 1e-8 * np.abs(Zb).max()
    lay.close()


@pytest.mark.parametrize("prec", [capi.GP_PREC_FP64, capi.GP_PREC_MIXED])
@pytest.mark.parametrize("sweeps", [1, 2])
@pytest.mark.parametrize("slots", [1, 2, 3, 6, 12, 32, 64])
def test_fused_transfers_match_csr_kernels(slots, sweeps, prec):
    """Restrictions with the next level's first sweep, G^T products with the nodal
    one (which keeps its right-hand side only for a second sweep) and both
    prolongations in a launch, at every slots-per-lane and lanes-per-row shape,
    against the separate (row, slot) CSR kernels: the same Z to 100 times the
    residual.  A converged solve hides what the preconditioner does; its kernels
    themselves are compared in test_one_preconditioner_application."""
    m = M.Mesh(M.manhattan_spec((24, 20, 10), n_ports=3, nfreq=3, f_range=(2e8, 4e9), seed=11))
    lay = Layout(m)
    fs = np.geomspace(2e8, 4e9, -(-slots // 3))
    kw = dict(ports=list(range(min(slots, 3))), precision=prec, rtol=1e-10, batch=slots, max_iters=400,
              smooth_edge=sweeps)
    Za, sa, _ = lay.solve(fs, **kw)
    Zb, sb, _ = lay.solve(fs, sell_min_rows=1 << 40, **kw)
    print(f"[kernels] fused transfers, {slots} slots, {sweeps} sweeps, precision {prec}: iterations {max(sa['iters'])} / "
          f"{max(sb['iters'])}, dZ {np.abs(Za - Zb).max() / np.abs(Zb).max():.2e}", flush=True)
    assert sa["status"] == sb["status"] == capi.GP_OK
    assert np.abs(Za - Zb).max() <= 1e-8 * np.abs(Zb).max()
    lay.close()


@pytest.mark.parametrize("prec", [capi.GP_PREC_FP64, capi.GP_PREC_MIXED])
@pytest.mark.parametrize("sweeps", [1, 2])
@pytest.mark.parametrize("cells,slots", [((24, 20, 10), k) for k in (1, 2, 3, 6, 12, 32, 64)] +
                         [((48, 48, 12), k) for k in (1, 4, 16)])
def test_one_preconditioner_application(cells, slots, sweeps, prec):
    """One FGMRES step from zero returns a multiple of the preconditioner's
    application to the right-hand side, so its kernels are compared without the
    solver around them: the fused ones against the separate (row, slot) CSR
    kernels, at every slots-per-lane and lanes-per-row shape (48x48x12: rows of
    several chunks in the auxiliary products too).

    In FP64 the two differ by rounding, amplified by at most the 1e9 between
    the curl-curl and the mass terms: 1e-16 x 1e9 x some tens of products,
    under 1e-5.  In FP32 both are compared with the FP64 application, and the
    fused kernels may be off by ten times what the separate ones are (1e-5 at
    least, some hundred products' rounding).  A sweep left out, a wrong
    diagonal or a row skipped changes it by percents."""
    m = M.Mesh(M.manhattan_spec(cells, n_ports=3, nfreq=3, f_range=(2e8, 4e9), seed=11))
    lay = Layout(m)
    fs = np.geomspace(2e8, 4e9, -(-slots // 3))
    kw = dict(ports=list(range(min(slots, 3))), batch=slots, max_iters=1, rtol=1e-10, smooth_edge=sweeps, want_x=True)
    X = lay.solve(fs, precision=prec, **kw)[2]
    Xc = lay.solve(fs, precision=prec, sell_min_rows=1 << 40, **kw)[2]
    X64 = lay.solve(fs, precision=capi.GP_PREC_FP64, sell_min_rows=1 << 40, **kw)[2]
    lay.close()
    off = lambda a: (np.linalg.norm(a - X64, axis=1) / np.linalg.norm(X64, axis=1)).max()  # noqa: E731
    print(f"[kernels] one application, {cells}, {slots} slots, {sweeps} sweeps, precision {prec}: fused off by {off(X):.2e}, "
          f"separate by {off(Xc):.2e}", flush=True)
    assert np.all(np.isfinite(X))
    assert off(X) <= (1e-5 if prec == capi.GP_PREC_FP64 else max(1e-5, 10 * off(Xc)))


def _dense_coo(A):
    r, c = np.nonzero(np.ones_like(A))
    return r.astype(np.int64), c.astype(np.int64), A.ravel()


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 63, 64, 65, 250, 257, 511, 512])
def test_dense_inverse_small(n):
    """A real system of at most 512 unknowns is its own coarsest level: the
    preconditioner is the dense inverse.  Random matrices whose diagonal is
    zero, so that every step needs its pivot; partial pivoting's growth and a
    condition number c leave an error of at most about n c eps per
    application, and FGMRES takes two steps to 1e-12 at the most."""
    from gds2para_amd.layout import solve_real
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n))
    if n > 1:
        np.fill_diagonal(A, 0.0)
    A += 3.0 * np.sqrt(n) * np.eye(n)[rng.permutation(n)] * (1.0 if n > 2 else 0.0)
    c = np.linalg.cond(A)
    b = rng.standard_normal(n)
    x, it, rr = solve_real(*_dense_coo(A), n, b, rtol=1e-12)
    ref = np.linalg.solve(A, b)
    print(f"[kernels] dense inverse n={n}: cond {c:.1e}, {it} steps, error {np.linalg.norm(x - ref) / np.linalg.norm(ref):.1e}",
          flush=True)
    assert c < 1e6 and it <= 2
    assert np.linalg.norm(x - ref) <= 1e-11 * c * np.linalg.norm(ref)


@pytest.mark.parametrize("n", [1000, 1900, 2500, 3800])
def test_dense_inverse_of_stalled_coarsening(n):
    """Rows coupled in pairs across the matrix with a zero diagonal: nothing
    aggregates, so the dense inverse takes all n unknowns (narrower panels, and
    above ~3700 rows a launch per step).  The inverse of each 2 x 2 pair is
    exact to rounding: one step to 1e-12."""
    from gds2para_amd.layout import solve_real
    rng = np.random.default_rng(n)
    i = np.arange(n, dtype=np.int64)
    v = rng.uniform(0.5, 2.0, n)
    b = rng.standard_normal(n)
    print(f"[kernels] dense inverse of {n} unknowns", flush=True)
    x, it, rr = solve_real(i, n - 1 - i, v, n, b, rtol=1e-12)
    assert it <= 1
    ref = np.empty(n)
    ref[n - 1 - i] = b / v
    assert np.linalg.norm(x - ref) <= 1e-12 * np.linalg.norm(ref)


def _solve_singular(row, col, val, n):
    from gds2para_amd.layout import solve_real
    with pytest.raises(capi.GpError, match="singular"):
        solve_real(row, col, val, n, np.ones(n), rtol=1e-12)


@pytest.mark.parametrize("n,col", [(1, 0), (2, 1), (64, 0), (64, 63), (250, 100), (512, 0), (512, 255), (512, 511)])
def test_dense_inverse_singular(n, col):
    """A zero column leaves the elimination without a pivot in that column's
    step, in the first launch or a later one: the call reports the singular
    matrix, and the next one is solved."""
    from gds2para_amd.layout import solve_real
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n)) + 2.0 * n * np.eye(n)
    good = A.copy()
    A[:, col] = 0.0
    print(f"[kernels] singular matrix n={n}, column {col}", flush=True)
    _solve_singular(*_dense_coo(A), n)
    x, it, rr = solve_real(*_dense_coo(good), n, good @ np.ones(n), rtol=1e-12)
    assert it <= 2 and np.abs(x - 1.0).max() <= 1e-10


@pytest.mark.parametrize("n", [1000, 1900, 2500, 3800])
def test_dense_inverse_singular_of_stalled_coarsening(n):
    """The same with narrower panels and a launch per step (pairs across the
    matrix, see above, one of them without its coupling)."""
    i = np.arange(n, dtype=np.int64)
    v = np.random.default_rng(n).uniform(0.5, 2.0, n)
    v[n // 3] = 0.0
    print(f"[kernels] singular matrix of {n} unknowns", flush=True)
    _solve_singular(i, n - 1 - i, v, n)


@pytest.mark.parametrize("runs", [(1, 47, 48, 49), (1023, 1024, 1025, 5), (2047, 2049, 3500, 2)])
def test_duplicate_sums(runs):
    """Triplets of equal (row, column) are summed by one thread up to 48 of
    them and by a workgroup, 1024 at a time, above: a diagonal matrix given as
    runs of such triplets.  A sum of m terms of one sign is off by m eps at
    most."""
    from gds2para_amd.layout import solve_real
    rng = np.random.default_rng(sum(runs))
    n = len(runs)
    row = np.repeat(np.arange(n, dtype=np.int64), runs)
    val = rng.uniform(0.5, 1.5, len(row))
    b = rng.standard_normal(n)
    print(f"[kernels] sums of {runs} triplets", flush=True)
    x, it, rr = solve_real(row, row, val, n, b, rtol=1e-10)
    d = np.array([float(np.sum(val[row == i].astype(np.longdouble))) for i in range(n)])
    assert np.all(np.abs(x - b / d) <= 4 * max(runs) * 2.3e-16 * np.abs(b / d))


def test_ad_sums_in_order():
    """Ad of 48x48x12, whose conductor aggregates sum up to 12,000 terms into
    one entry: the same bits as the oracle's sums in the reference's order."""
    import oracle
    m = M.Mesh(M.WORKLOADS["manhattan_48x48x12"]())
    lay = Layout(m)
    lay.build_v0()
    print("[kernels] Ad sums of 48x48x12", flush=True)
    got, ref = lay.v0d(), oracle.v0d(m)
    for k in ("ad_row", "ad_col", "ad_val"):
        assert np.array_equal(got[k], ref[k]), k
    lay.close()


def _z_from_yd(m, yd, src):
    """Construct_Z_V0's column of source port src from the field yd."""
    c, n = m.c, m.num_ports
    psp = np.ctypeslib.as_array(c.port_side_ptr, shape=(n + 1,))
    sep = np.ctypeslib.as_array(c.side_edge_ptr, shape=(int(psp[-1]) + 1,))
    edges = np.ctypeslib.as_array(c.side_edges, shape=(int(sep[-1]),))
    area = np.ctypeslib.as_array(c.side_area, shape=(int(psp[-1]),))
    sdir = np.ctypeslib.as_array(c.side_dir, shape=(int(psp[-1]),))
    zn = np.ctypeslib.as_array(c.zn, shape=(c.nz,))
    es, ev = int(m.sizes.n_edge_s), int(m.sizes.n_edge_v)
    z = np.zeros(n, complex)
    for p in range(n):
        s0 = psp[p]
        e = edges[sep[s0]:sep[s0 + 1]]
        iz = e // (es + ev)
        z[p] = -np.sum(yd[e] * (zn[iz + 1] - zn[iz])) * sdir[s0]
    return z / area[psp[src]:psp[src + 1]].sum()


@pytest.mark.parametrize("smoother", [capi.GP_SMOOTH_CHEBYSHEV, capi.GP_SMOOTH_L1_JACOBI])
@pytest.mark.parametrize("ports", [1, 2, 3, 8, 9])
def test_v0_ports_side_by_side(ports, smoother):
    """Z0 with the ports solved side by side (1, 2, 4 or 8 columns, the last
    group partly empty) against each port's field solved alone.  Both reach a
    relative residual of 1e-10, which leaves the responses alike to 1e-8 of the
    column's largest."""
    m = M.Mesh(M.manhattan_spec((30, 26, 11), n_ports=ports, nfreq=2, f_range=(1e8, 1e10), seed=21))
    lay = Layout(m)
    lay.set_v0_smoother(smoother)
    Z0, _, st = lay.solve_v0(1e-10)
    print(f"[kernels] V0 with {ports} ports, smoother {smoother}: {st['solves']} solves, {st['max_iters']} iterations", flush=True)
    assert st["solves"] == 3 * ports and st["max_rel_residual"] <= 1e-10
    Z0 = Z0.reshape(ports, ports)
    for src in range(ports):
        ref = _z_from_yd(m, lay.v0_vh_inputs(src, 1e-10)[2], src)
        assert np.abs(Z0[src] - ref).max() <= 1e-8 * np.abs(ref).max(), src
    lay.close()
