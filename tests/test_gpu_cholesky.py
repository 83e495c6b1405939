"""The blocked Cholesky solve of (S + shift) x = F at the edges of its blocks: one block and
less, a ragged last block, a last block of one column, and both sides of the size from which
the factorisation works in outer panels (with full and ragged panels).

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
