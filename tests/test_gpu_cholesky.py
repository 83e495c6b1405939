"""The blocked Cholesky solve of (S + shift) x = F at the edges of its blocks: one block and
less, a ragged last block, a last block of one column, and both sides of the size from which
the factorisation works in outer panels (with full and ragged panels).

A matrix that is not positive definite is refused, wherever in its blocks the first bad pivot
stands; the padding of a ragged block is none.

Tolerance: the backward error of a Cholesky solve, |(S + shift) x - F| <= c P eps |S + shift| |x|
with a small constant c (here 4, Frobenius norm)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,M", [(1, 1), (7, 9), (8, 8), (5, 13), (8, 24), (3, 43), (23, 89), (8, 256), (3, 683),
                                 (16, 145)])
def test_cholesky_backward_error(N, M):
    import annongpu_amd as A
    rng = np.random.default_rng(N * 1000 + M)
    W = 0.2 * (rng.standard_normal((N, M)) + 1j * rng.standard_normal((N, M)))
    psi = A.PsiRBM(W, final_weight=1.0)
    H = sum((A.sigma_x(i) for i in range(1, N)), 1.0 * A.sigma_x(0))
    confs = rng.integers(0, 2 ** N, size=257, dtype=np.uint64)[:, None]
    t = A.TDVP(N * M)
    t.eval(A.Operator(H), psi, A.SampleList(N, confs))
    shift = 1e-2
    x = t.solve(shift, "cholesky")
    S = t.S_matrix + shift * np.eye(N * M)
    r = np.linalg.norm(S @ x - t.F_vector)
    assert r <= 4 * N * M * np.finfo(float).eps * np.linalg.norm(S) * np.linalg.norm(x)
    assert t.last_solve["residual"] < 1e-9



@pytest.mark.parametrize("N,M,C,n", [(8, 1, 6, 256), (17, 8, 5, 1024), (23, 15, 6, 2048), (24, 15, 6, 2048),
                                     (64, 62, 31, 4096), (64, 397, 4, 8192)])
@pytest.mark.parametrize("at", ["last", "second to last row", "first"])
def test_indefinite_matrix_is_refused(N, M, C, n, at):
    """P = 15, 65, 128, 129, 2,048 and 2,049.  A unit that reads one site twice has two equal O, so S is
    singular in exactly one direction (the smallest other eigenvalue of the scaled matrix is 3e-5 or
    more): with the shift -1e-8 the pivot of the second of the two, and no other, is negative.  "first":
    -10, where the first pivot is."""
    import annongpu_amd as A
    rng = np.random.default_rng(N * 1000 + M)
    conn = np.stack([rng.permutation(N)[:C] for _ in range(M)], axis=1)
    row = C - 1 if at != "second to last row" else C - 2
    conn[row, M - 1] = conn[0, M - 1]

    def gauss(shape, sigma):
        return sigma * (rng.standard_normal(shape) + 1j * rng.standard_normal(shape))

    psi = A.PsiDeep(N, np.zeros(N), [gauss(M, 0.3)], [conn], [gauss((C, M), 0.6 / np.sqrt(C))], np.ones(M))
    bits = rng.random((n, N)) < 0.5
    confs = np.packbits(np.pad(bits, ((0, 0), (0, 64 - N))), axis=1, bitorder="little").view(np.uint64)
    t = A.TDVP(psi.num_params)
    t.eval(A.Operator(sum((A.sigma_x(i) for i in range(1, N)), 1.0 * A.sigma_x(0))), psi,
           A.SampleList(N, np.ascontiguousarray(confs)))
    x = t.solve(1e-3, "cholesky")
    assert np.all(np.isfinite(x)) and t.last_solve["residual"] < 1e-9
    with pytest.raises(Exception, match="not positive definite"):
        t.solve(-10.0 if at == "first" else -1e-8, "cholesky")
    assert np.array_equal(t.solve(1e-3, "cholesky"), x)
