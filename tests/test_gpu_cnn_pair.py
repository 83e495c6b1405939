"""The kernels of two-layer PsiCNNs of one symmetry class against the general ones.  The same network
written with two symmetry classes that hold the same weights takes the general path, so every form
is compared on the device: chains step for step (every decision takes its sums in the same order:
identical configurations in both precisions), log psi, E_loc and O_k (summed over the classes).

Shapes: kernels of 1 to 9 sites in one to three dimensions, kernels as wide as the lattice (a site
read twice), a lattice of one site, 256 sites, odd channel numbers and channel blocks of 2, 4 and 8,
flips that reach more and fewer than 32 sites, exchange moves, operators of one and two flips.

Tolerances: a pre-activation is a sum of K <= C0 v1 products of size below 1, log psi one of N C1
outputs, O_k one of N products: 8 eps per sum's square root of terms, relative to the largest value
(ratios: to the largest ratio)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [([1, 4, 4], (3, [1, 2, 2]), (5, [1, 3, 3])), ([1, 6, 6], (8, [1, 3, 3]), (8, [1, 3, 3])),
          ([1, 1, 13], (2, [1, 1, 3]), (1, [1, 1, 5])), ([1, 3, 3], (9, [1, 3, 3]), (3, [1, 2, 2])),
          ([2, 2, 2], (4, [2, 2, 2]), (2, [2, 2, 2])), ([1, 16, 16], (2, [1, 3, 3]), (9, [1, 3, 3])),
          ([1, 2, 2], (1, [1, 2, 2]), (1, [1, 1, 1])), ([3, 4, 3], (2, [2, 2, 2]), (3, [2, 2, 2])),
          ([1, 1, 1], (2, [1, 1, 1]), (2, [1, 1, 1])), ([1, 9, 9], (4, [1, 3, 3]), (4, [1, 3, 3]))]


def nets(extent, layers, precision, seed):
    import annongpu_amd as A
    rng = np.random.default_rng(seed)
    N = int(np.prod(extent))
    one, two, prev = [], [], 1
    for ch, conn in layers:
        v = int(np.prod(conn))
        w = 0.25 / np.sqrt(prev * v) * (rng.standard_normal((prev * ch, v)) + 1j * rng.standard_normal((prev * ch, v)))
        one.append(w.ravel())
        two.append(np.repeat(w[:, None], 2, axis=1).ravel())
        prev = ch
    chs, conns = [l[0] for l in layers], [l[1] for l in layers]
    classes = np.arange(N) % 2 if N > 1 else np.zeros(1)
    psi = [A.PsiCNN(extent, chs, conns, np.zeros(N), np.concatenate(one), 1.5),
           A.PsiCNN(extent, chs, conns, classes, np.concatenate(two if N > 1 else one), 1.5)]
    for p in psi:
        p.precision = precision
    return N, psi


def words(N, n, rng):
    confs = rng.integers(0, 2 ** 63, size=(n, (N + 63) // 64), dtype=np.uint64) * np.uint64(2) + \
        rng.integers(0, 2, size=(n, (N + 63) // 64), dtype=np.uint64)
    if N % 64:
        confs[:, -1] &= np.uint64(2 ** (N % 64) - 1)
    return confs


def operators(A, N):
    flips, bonds = 0.7 * A.sigma_z(0), 0.3 * A.sigma_z(0)
    for i in range(N):
        flips = flips + (0.5 + 0.01 * i) * A.sigma_x(i) + 0.2 * A.sigma_y(i)
        if i:
            flips = flips + A.sigma_z(i - 1) * A.sigma_z(i)
            bonds = bonds + A.sigma_x(i - 1) * A.sigma_x(i) + 0.5 * A.sigma_y(i - 1) * A.sigma_y(i) + 0.1 * A.sigma_x(i)
    return [A.Operator(flips), A.Operator(bonds)]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("case", range(len(SHAPES)))
def test_values(case, precision):
    import annongpu_amd as A
    extent, *layers = SHAPES[case]
    N, (fast, general) = nets(extent, layers, precision, case)
    rng = np.random.default_rng(case)
    eps = np.finfo(np.float64 if precision == "fp64" else np.float32).eps
    n = 37
    confs = words(N, n, rng)
    ens = A.SampleList(N, confs)
    ch = [l[0] for l in layers]
    terms = N * ch[1] + ch[0] * int(np.prod(layers[1][1]))
    a, b = A.log_psi_vector(fast, ens), A.log_psi_vector(general, ens)
    assert np.abs(a - b).max() <= 8 * eps * np.sqrt(terms) * max(1.0, np.abs(b).max())
    for op in operators(A, N):
        a, b = A.local_energies(op, fast, ens), A.local_energies(op, general, ens)
        assert np.abs(a - b).max() <= 8 * eps * terms * np.abs(b).max()
    t, u = A.TDVP(fast.num_params), A.TDVP(general.num_params)
    t.eval_F(operators(A, N)[0], fast, ens)
    u.eval_F(operators(A, N)[0], general, ens)
    a, b = t.O_k_samples, u.O_k_samples
    prev, oa, ob = 1, 0, 0
    for c, conn in layers:
        v = int(np.prod(conn))
        classes = 2 if N > 1 else 1
        x = a[:, oa:oa + prev * c * v].reshape(n, prev * c, v)
        y = b[:, ob:ob + prev * c * classes * v].reshape(n, prev * c, classes, v).sum(2)
        assert np.abs(x - y).max() <= 8 * eps * np.sqrt(terms) * np.abs(y).max()
        oa, ob, prev = oa + prev * c * v, ob + prev * c * classes * v, c


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("move", ["flip", "exchange"])
@pytest.mark.parametrize("case,chains", [(0, 1), (1, 67), (2, 33), (3, 16), (4, 40), (5, 9), (6, 17), (7, 31), (8, 5), (9, 66)])
def test_chains_step_alike(case, chains, move, precision):
    import annongpu_amd as A
    extent, *layers = SHAPES[case]
    N, psi = nets(extent, layers, precision, 50 + case)
    got = []
    for p in psi:
        ens = A.MonteCarloSpins(3 * chains, 2, 3, chains, move=move, total_z=N % 2, seed=case, persistent=True)
        A.log_psi(p, ens)
        A.log_psi(p, ens)
        got.append((ens.last_samples(), ens.acceptance_rate))
    assert np.array_equal(got[0][0], got[1][0]) and got[0][1] == got[1][1]
