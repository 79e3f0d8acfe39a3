"""The subspace eigenkernel (stda_hip_sym_lowest) against numpy's eigh."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


@pytest.fixture(scope="module")
def h():
    from stda_amd.core import StdaHip
    with StdaHip(0) as ctx:
        yield ctx


def matrix(kind, n, rng):
    G = rng.standard_normal((n, n))
    if kind == "dense":
        return G + G.T
    if kind == "davidson":      # a subspace matrix: rising diagonal, weak couplings
        return np.diag(np.sort(rng.uniform(0.15, 0.5, n))) + 2e-3 * (G + G.T)
    if kind == "ritz":          # after a restart: diagonal head, coupled tail
        A = np.diag(np.sort(rng.uniform(0.15, 0.5, n)))
        b = max(1, n // 4)
        A[:, n - b:] += 1e-3 * G[:, n - b:]
        A[n - b:, :] = A[:, n - b:].T
        return 0.5 * (A + A.T)
    Q = np.linalg.qr(G)[0]      # "close": pairs 1e-9 apart, orthogonal to 1e-7 only as they come
    w = np.sort(rng.uniform(0.1, 1.0, n))
    w[1::2] = w[:-1:2][:len(w[1::2])] + 1e-9
    return (Q * w) @ Q.T


@pytest.mark.parametrize("kind", ["dense", "davidson", "ritz", "close"])
@pytest.mark.parametrize("n", [1, 2, 3, 8, 15, 16, 17, 32, 33, 63, 64, 65, 95, 96, 97, 120, 128,
                               129, 160, 191, 192])
def test_lowest_pairs(h, kind, n):
    rng = np.random.default_rng(1000 * n + len(kind))
    A = matrix(kind, n, rng)
    A = 0.5 * (A + A.T)
    norm = np.linalg.norm(A, 2)
    for k in sorted({1, min(n, 20), min(n, 32)}):
        out = h.sym_lowest(A, k)
        assert out is not None
        w, Z = out
        # backward stable reduction: n eps |A| with a small constant
        assert np.abs(w - np.linalg.eigvalsh(A)[:k]).max() <= 4 * n * EPS * norm
        assert np.abs(Z.T @ Z - np.eye(k)).max() <= 8 * n * EPS
        # an orthonormalisation of vectors with overlaps up to 1e-6 mixes values 1e-9 apart
        assert np.linalg.norm(A @ Z - Z * w, axis=0).max() <= 8 * n * EPS * norm + 1e-14


@pytest.mark.parametrize("n", [3, 20, 70, 130, 192])
def test_scaled_matrices(h, n):
    """A matrix times a power of two, down to where its elements' squares underflow: the same
    vectors and the scaled values, bit for bit."""
    A = matrix("dense", n, np.random.default_rng(n))
    k = min(n, 20)
    w, Z = h.sym_lowest(A, k)
    for e in (-1000, -700, -540, -100, 100, 540, 1000):
        out = h.sym_lowest(np.ldexp(A, e), k)
        assert out is not None
        np.testing.assert_array_equal(out[0], np.ldexp(w, e))
        np.testing.assert_array_equal(out[1], Z)


@pytest.mark.parametrize("n", [4, 40, 100])
def test_repeated_and_nonfinite(h, n):
    """Repeated eigenvalues and NaN: pairs that hold, or None, and always an end."""
    for A in (np.eye(n), np.zeros((n, n)), np.diag(np.r_[np.ones(n // 2), 2 * np.ones(n - n // 2)])):
        out = h.sym_lowest(A, min(n, 20))
        if out is not None:
            w, Z = out
            assert np.abs(A @ Z - Z * w).max() <= 8 * n * EPS
            assert np.abs(Z.T @ Z - np.eye(len(w))).max() <= 8 * n * EPS
    A = np.eye(n)
    A[0, n - 1] = A[n - 1, 0] = np.nan
    assert h.sym_lowest(A, 2) is None


@pytest.mark.parametrize("k", [1, 3, 10, 16, 17, 20, 24, 25, 32, 33, 48, 49, 64])
def test_root_counts(h, k):
    """The k lowest roots for block widths on both sides of every kernel size (block
    orthonormalisation, subspace step) against the dense eigenvalues of the explicit A."""
    from stda_amd.prep import prepare
    from stda_amd.synth import cluster
    if not hasattr(test_root_counts, "ref"):
        mol, ints = cluster(24, seed=11, basis="minimal")
        ci = prepare(mol, 7.0, 0.25, ints)
        h.setup(ci, 7.0, 0.25)
        test_root_counts.ref = ci, np.linalg.eigvalsh(h.build_a())
    ci, w = test_root_counts.ref
    h.setup(ci, 7.0, 0.25)
    sol = h.solve_tda(k)
    assert len(sol.omega) == k
    # residual norms of 1e-8 bound the roots by 1e-8, and squared over the gap in practice
    assert np.abs(sol.omega - w[:k]).max() <= 1e-10
    assert np.abs(sol.X.T @ sol.X - np.eye(k)).max() <= 1e-11


def dense_rpa(apb, amb, n):
    """All RPA roots from the packed A+B and A-B: L^T (A+B) L with A-B = L L^T."""
    full = []
    for p in (apb, amb):
        M = np.zeros((n, n))
        M[np.tril_indices(n)] = p          # element lin(i, j), j <= i
        full.append(M + np.tril(M, -1).T)
    L = np.linalg.cholesky(full[1])
    return np.sqrt(np.linalg.eigvalsh(L.T @ full[0] @ L)), full


@pytest.mark.parametrize("k", [1, 10, 21, 22, 32, 33])
def test_rpa_root_counts(h, k):
    """RPA roots with reduced problems on the device (21 roots with their restart pairs) and on
    the host, blocks orthonormalised on the device (32) and by the host's path (33)."""
    from stda_amd.prep import prepare
    from stda_amd.synth import cluster
    if not hasattr(test_rpa_root_counts, "ref"):
        mol, ints = cluster(20, seed=12, basis="minimal")
        ci = prepare(mol, 7.0, 0.25, ints)
        h.setup(ci, 7.0, 0.25)
        test_rpa_root_counts.ref = ci, dense_rpa(*h.build_apb_amb(), h.nci)[0]
    ci, w = test_rpa_root_counts.ref
    h.setup(ci, 7.0, 0.25)
    sol = h.solve_rpa(k)
    assert np.abs(sol.omega - w[:k]).max() <= 1e-10
    xpy, xmy = sol.X + sol.Y, sol.X - sol.Y
    assert np.abs(np.einsum("ij,ij->j", xpy, xmy) - 1.0).max() <= 1e-10


@pytest.mark.parametrize("seed", [1, 2, 3, 4])
@pytest.mark.parametrize("rpa", [False, True])
def test_window_finds_every_root(h, seed, rpa):
    """Every root up to the threshold, also where more of them lie there than the CSF
    energies promise, against the dense eigenvalues."""
    from stda_amd.prep import prepare
    from stda_amd.synth import cluster
    mol, ints = cluster(14, seed=seed, basis="minimal")
    ci = prepare(mol, 8.0, 0.5, ints)
    h.setup(ci, 8.0, 0.5)
    w = dense_rpa(*h.build_apb_amb(), h.nci)[0] if rpa else np.linalg.eigvalsh(h.build_a())
    w = w[w <= h.thr]
    sol = h.solve_rpa(None) if rpa else h.solve_tda(None)
    assert len(sol.omega) == len(w)
    assert np.abs(sol.omega - w).max() <= 1e-10


@pytest.mark.parametrize("edge", [None, 0, 4])
@pytest.mark.parametrize("na,seed,thr,ax,triplet,rpa", [(24, 5, 4.0, 2.0, True, False),
                                                        (24, 5, 5.0, 2.0, False, False),
                                                        (24, 2, 6.0, 1.5, False, False),
                                                        (20, 3, 8.0, 1.0, False, True),
                                                        (24, 4, 6.0, 0.5, False, True)])
def test_window_enlarged(h, na, seed, thr, ax, triplet, rpa, edge):
    """Windows that hold up to 40 roots more than CSF energies: solved again until 8 roots
    lie beyond, also for a threshold 1e-6 eV below a root (the highest one, the fifth one)."""
    from stda_amd.constants import HARTREE_EV
    from stda_amd.prep import prepare
    from stda_amd.synth import cluster
    mol, ints = cluster(na, seed=seed, basis="minimal")

    def dense(thr):
        h.setup(prepare(mol, thr, ax, ints), thr, ax, triplet=triplet)
        return (dense_rpa(*h.build_apb_amb(), h.nci)[0] if rpa else np.linalg.eigvalsh(h.build_a()))
    w = dense(thr)
    if edge is not None:
        thr = w[w <= h.thr][-1 - edge] * HARTREE_EV - 1e-6
        w = dense(thr)
    roots = int((w <= h.thr).sum())
    k, solves = int((h.csf()[1] <= h.thr).sum()) + 8, 1
    while w[k - (1 if solves == 1 else 8)] <= h.thr:
        k, solves = k + max(16, k // 4), solves + 1
    assert solves > 1
    sol = h.solve_rpa(None) if rpa else h.solve_tda(None)
    w = w[:roots]
    w = w[w > 0.0]
    assert len(sol.omega) == len(w)
    assert np.abs(sol.omega - w).max() <= 1e-10
    assert h.kernel_stats("window_solve")["launches"] == solves


@pytest.mark.parametrize("na,seed,thr,ax,tol,k", [(20, 3, 8.0, 1.0, 1e-12, 0), (24, 4, 6.0, 0.5, 1e-12, 0),
                                                  (24, 11, 7.0, 0.25, 2e-15, 10),
                                                  (24, 11, 7.0, 0.25, 2e-15, 19)])
def test_tolerance_near_rounding(h, na, seed, thr, ax, tol, k):
    """Tolerances that the iteration just reaches: windows of RPA roots that start too small
    (k = 0) and fewer than 20 TDA roots, which ask for more than the caller's tolerance."""
    from stda_amd.prep import prepare
    from stda_amd.synth import cluster
    mol, ints = cluster(na, seed=seed, basis="minimal")
    h.setup(prepare(mol, thr, ax, ints), thr, ax)
    if k:
        w = np.linalg.eigvalsh(h.build_a())[:k]
        sol = h.solve_tda(k, tol=tol)
    else:
        w = dense_rpa(*h.build_apb_amb(), h.nci)[0]
        w = w[w <= h.thr]
        assert len(w) > (h.csf()[1] <= h.thr).sum() + 8
        sol = h.solve_rpa(None, tol=tol)
    assert len(sol.omega) == len(w)
    assert np.abs(sol.omega - w).max() <= 1e-10


@pytest.mark.parametrize("omegas", [(0.0,), (0.0, 0.05, 0.1), (0.05, 0.05, 0.05 + 1e-9), (0.0, 0.3)])
def test_response_reduced_problem(h, omegas):
    """alpha(w) below and above poles, and with dependent residuals (equal frequencies: the
    new block's dead columns leave the space), against a dense solve."""
    from stda_amd.prep import prepare
    from stda_amd.synth import cluster
    mol, ints = cluster(14, seed=3, basis="minimal")
    ci = prepare(mol, 7.0, 0.25, ints)
    h.setup(ci, 7.0, 0.25)
    P, M = dense_rpa(*h.build_apb_amb(), h.nci)[1]
    csf = h.csf()[0].astype(int) - 1
    hi, lo = csf.max(axis=1), csf.min(axis=1)
    mu = ci.moments[:3, lo + hi * (hi + 1) // 2].T
    inv = np.linalg.inv(M)
    for w, a in h.lresp(omegas):
        ref = 4.0 * mu.T @ np.linalg.solve(P - w * w * inv, mu)
        # residuals of 1e-10 of norm-1 right-hand sides, amplified by 1 / |w_n - w| at a pole
        assert np.abs(a - ref).max() <= 1e-6 * np.abs(ref).max()


@pytest.mark.parametrize("na,seed,below,above,spectral", [(14, 3, 40, 0, True), (24, 11, 20, 20, True),
                                                          (14, 3, 0, 14, True), (14, 3, 12, 4, False),
                                                          (14, 3, 20, 0, False)])
def test_response_many_frequencies(h, na, seed, below, above, spectral):
    """alpha(w) at many frequencies below the first pole and midway between poles, each but
    static ones twice with either sign: few are solved one by one (a repeated w^2 once), many
    through one eigenproblem an iteration."""
    from stda_amd.prep import prepare
    from stda_amd.synth import cluster
    mol, ints = cluster(na, seed=seed, basis="minimal")
    ci = prepare(mol, 7.0, 0.25, ints)
    h.setup(ci, 7.0, 0.25)
    poles, (P, M) = dense_rpa(*h.build_apb_amb(), h.nci)
    gaps = np.flatnonzero(np.diff(poles) > 2e-3)[:above]
    w = np.r_[np.linspace(0.0, 0.9, below) * poles[0], 0.5 * (poles[gaps] + poles[gaps + 1])]
    assert len(w) == below + above
    w = np.r_[w, -w[::-1]]
    out = h.lresp(w)
    factored = h.kernel_stats("lresp_factor")["launches"]
    if spectral:         # but for iterations before the frequencies are known to lie above poles
        assert factored <= 2 * (below + above) < 2 * len(w)
        assert h.kernel_stats("lresp_spectrum")["launches"] > 0
    else:                # each w^2 once an iteration
        assert factored > 0 and factored % (below + above) == 0
    csf = h.csf()[0].astype(int) - 1
    hi, lo = csf.max(axis=1), csf.min(axis=1)
    mu = ci.moments[:3, lo + hi * (hi + 1) // 2].T
    inv = np.linalg.inv(M)
    for x, a in out:
        ref = 4.0 * mu.T @ np.linalg.solve(P - x * x * inv, mu)
        # as in test_response_reduced_problem, half a gap of at least 1e-3 from a pole
        assert np.abs(a - ref).max() <= 1e-6 * np.abs(ref).max()


@pytest.mark.parametrize("mode,unit", [("fp64", EPS), ("fp32", 2.0 ** -24)])
@pytest.mark.parametrize("m,n,kk", [(33, 31, 50), (320, 330, 37), (1030, 1050, 37), (2950, 2890, 19)])
def test_gemm_tile_sizes(h, mode, unit, m, n, kk):
    """Shapes of each tile size of the matrix-core GEMM (32, 32, 64, 128), ragged edges."""
    rng = np.random.default_rng(m)
    A, B = rng.standard_normal((m, kk)), rng.standard_normal((kk, n))
    if mode == "fp32":
        A, B = A.astype(np.float32).astype(float), B.astype(np.float32).astype(float)
    for ta in (False, True):
        for tb in (False, True):
            C = h.gemm(A.T if ta else A, B.T if tb else B, ta=ta, tb=tb, mode=mode)
            bound = (kk + 2) * unit * (np.abs(A) @ np.abs(B))
            assert (np.abs(C - A @ B) <= bound + kk * EPS).all()


@pytest.mark.parametrize("k", [20, 40, 70])
@pytest.mark.parametrize("precision", ["fp64", "mixed", "bf16"])
def test_nonfinite_orbital_is_an_error(h, precision, k):
    """A NaN in an orbital of no selected CSF (0 times it enters every product) ends in an
    error, also where a phase starts from the vectors of an earlier one and no column of its
    start block lives, and the context goes on to the next molecule."""
    from stda_amd.core import StdaHipError
    from stda_amd.prep import prepare
    from stda_amd.synth import cluster
    mol, ints = cluster(24, seed=11, basis="minimal")
    ci = prepare(mol, 7.0, 0.25, ints)
    good = ci.clow.copy()
    print(f"non-finite orbital, {precision}, {k} roots", flush=True)
    try:
        ci.clow[0, -1] = np.nan
        h.setup(ci, 7.0, 0.25)
        h.set_precision(precision)
        # one phase finds no new directions, a second one no start vectors
        with pytest.raises(StdaHipError, match="no finite vectors" if precision == "bf16"
                           else "no new directions") as e:
            h.solve_tda(k)
        assert e.value.status == 6       # STDA_HIP_ERR_NOT_CONVERGED
        ci.clow[:] = good
        h.setup(ci, 7.0, 0.25)
        assert np.isfinite(h.solve_tda(k).omega).all()
    finally:
        ci.clow[:] = good
        h.set_precision("fp64")


@pytest.mark.parametrize("mode,unit", [("fp64", EPS), ("fp32", 2.0 ** -24)])
def test_gemm_tuned_small_tiles(h, mode, unit):
    """A product large enough to be tuned (2.1 GFLOP) whose 64-tiles are fewer than the compute
    units: the tuning call and the calls after it, which use the tile it chose."""
    rng = np.random.default_rng(5)
    m, n, kk = 650, 610, 2700
    A, B = rng.standard_normal((m, kk)), rng.standard_normal((kk, n))
    if mode == "fp32":
        A, B = A.astype(np.float32).astype(float), B.astype(np.float32).astype(float)
    bound = (kk + 2) * unit * (np.abs(A) @ np.abs(B)) + kk * EPS
    for _ in range(3):
        assert (np.abs(h.gemm(A, B, mode=mode) - A @ B) <= bound).all()
