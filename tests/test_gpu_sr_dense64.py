"""The fp64 statistics, S.v and CG solve of a one-layer net against numpy on its O_k samples, at the
edges of the kernels' tiles (16 samples, 16 rows and units, 64-site words, 64-sample chunks) and over
the layouts that reach them.

O_k is materialised by a kernel of its own, exactly from the same g and spins, so both sides are fp64
sums of the same products.  A sum over n samples of products of sums over k = N + M + P terms differs by
at most 4 (n + k) eps times the same sum over absolute values."""
import numpy as np
import pytest

from test_gpu_dense_gram import net

pytestmark = pytest.mark.gpu

CASES = [("rbm", 1, 1, 1), ("rbm", 15, 17, 16), ("circulant", 16, 64, 17), ("rbm", 64, 65, 63), ("shuffled", 63, 9, 65),
         ("circulant", 65, 100, 130), ("repeated", 16, 5, 300), ("rbm", 129, 130, 64), ("circulant", 23, 500, 33),
         ("rbm", 256, 3, 70)]


def evaluated(kind, N, M, n):
    import annongpu_amd as A
    rng = np.random.default_rng(1000 * N + M)
    psi = net(kind, N, M, rng)
    psi.precision = "fp64"
    confs = rng.integers(0, 2 ** 63, size=(n, (N + 63) // 64), dtype=np.uint64)
    if N % 64:
        confs[:, -1] &= np.uint64(2 ** (N % 64) - 1)
    w = rng.random(n) / n
    op = A.Operator(sum((A.sigma_z(i) * A.sigma_z((i + 1) % N) for i in range(1, N)), 1.0 * A.sigma_z(0)))
    t = A.TDVP(psi.num_params)
    t.eval_F(op, psi, A.SampleList(N, confs, w))
    return t, t.O_k_samples, w, rng


@pytest.mark.parametrize("kind,N,M,n", CASES)
def test_S_dot_vector(kind, N, M, n):
    t, O, w, rng = evaluated(kind, N, M, n)
    P = O.shape[1]
    v = rng.standard_normal(P) + 1j * rng.standard_normal(P)
    mean = w @ O
    u = w * (O @ v - mean @ v)
    bound = 4 * (n + N + M + P) * np.finfo(float).eps
    scale = np.abs(O).T @ (w * (np.abs(O) @ np.abs(v) + np.abs(mean) @ np.abs(v)))
    assert (np.abs(t.S_dot_vector(v) - O.conj().T @ u) <= bound * scale).all()
    assert (np.abs(t.O_k_vector - mean) <= bound * (w @ np.abs(O))).all()


@pytest.mark.parametrize("kind,N,M,n,method", [("circulant", 65, 100, 130, "cg"), ("rbm", 15, 17, 16, "cg"),
                                               ("repeated", 16, 5, 300, "cg"), ("rbm", 129, 512, 24, "cg"),
                                               ("circulant", 65, 100, 130, "cg_kfac")])
def test_cg_directions(kind, N, M, n, method):
    """The direction formed inside the product, up to and beyond 65,536 parameters (where p^H Ap has a
    kernel of its own): after 20 iterations the recursion's residual is the one of the returned x.  Each
    iteration rounds r by at most 4 eps |S + shift| |x|."""
    t, O, w, _ = evaluated(kind, N, M, n)
    mean = w @ O
    F = t.F_vector
    x = t.solve(shift=0.05, method=method, rtol=1e-15, max_iter=20, raise_on_failure=False)
    r = O.conj().T @ (w * (O @ x - mean @ x)) + 0.05 * x - F
    assert t.last_solve["iterations"] == 20
    S_norm = (w @ np.abs(O) ** 2).sum() + 0.05
    assert abs(np.linalg.norm(r) - t.last_solve["residual"] * np.linalg.norm(F)) <= \
        4 * 20 * np.finfo(float).eps * S_norm * np.linalg.norm(x)
    assert t.last_solve["residual"] < 0.5
