"""The kernels of two-layer PsiCNNs of one symmetry class against the general ones.  The same network
written with two symmetry classes that hold the same weights takes the general path, so every form
is compared on the device: chains step for step (every decision takes its sums in the same order:
identical configurations in both precisions), log psi, E_loc and O_k (summed over the classes).  The
profiler's counts say that the first net took these kernels and the second did not.

Shapes: kernels of 1 to 9 sites in one to three dimensions, kernels as wide as the lattice (a site
read twice), 256 sites, odd channel numbers and channel blocks of 2, 4 and 8, flips that reach more
and fewer than 32 sites, exchange moves, operators of one and two flips.  The last shape's flips reach
45 sites: one flip is served, two are not (more than 64).  A lattice of one site has one class only and
is compared with the oracle.  Which kernels take a call may depend on the number of chains or samples;
both give a chain the same configurations and a sample the same values.

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
          ([1, 1, 1], (2, [1, 1, 1]), (2, [1, 1, 1])), ([1, 9, 9], (4, [1, 3, 3]), (4, [1, 3, 3])),
          ([4, 5, 4], (2, [3, 3, 1]), (2, [1, 3, 3]))]


def served(kind, psi, call, times=1):
    """call()'s result; asserts that psi[0] alone takes the kernel `kind`"""
    import annongpu_amd as A
    out = []
    for i, p in enumerate(psi):
        A.profiler_reset()
        A.start_profiling()
        out.append(call(p))
        A.stop_profiling()
        assert A.profiler_query("cnn_pair_" + kind)[1] == (times if i == 0 else 0)
    return out


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
    psi = [A.PsiCNN(extent, chs, conns, np.zeros(N), np.concatenate(one), 1.5)]
    if N > 1:
        psi.append(A.PsiCNN(extent, chs, conns, np.arange(N) % 2, np.concatenate(two), 1.5))
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
@pytest.mark.parametrize("case", [c for c in range(len(SHAPES)) if c != 8])
def test_values(case, precision):
    import annongpu_amd as A
    extent, *layers = SHAPES[case]
    N, psi = nets(extent, layers, precision, case)
    rng = np.random.default_rng(case)
    eps = np.finfo(np.float64 if precision == "fp64" else np.float32).eps
    n = 37
    confs = words(N, n, rng)
    ens = A.SampleList(N, confs)
    ch = [l[0] for l in layers]
    terms = N * ch[1] + ch[0] * int(np.prod(layers[1][1]))
    a, b = served("log_psi", psi, lambda p: A.log_psi_vector(p, ens))
    assert np.abs(a - b).max() <= 8 * eps * np.sqrt(terms) * max(1.0, np.abs(b).max())
    for i, op in enumerate(operators(A, N)):
        a, b = served("local_energy", psi, lambda p: A.local_energies(op, p, ens), 0 if case == 10 and i else 1)
        assert np.abs(a - b).max() <= 8 * eps * terms * np.abs(b).max()

    def samples(p):
        t = A.TDVP(p.num_params)
        t.eval_F(operators(A, N)[0], p, ens)
        return t.O_k_samples

    a, b = served("ok", psi, samples)
    prev, oa, ob = 1, 0, 0
    for c, conn in layers:
        v = int(np.prod(conn))
        x = a[:, oa:oa + prev * c * v].reshape(n, prev * c, v)
        y = b[:, ob:ob + prev * c * 2 * v].reshape(n, prev * c, 2, v).sum(2)
        assert np.abs(x - y).max() <= 8 * eps * np.sqrt(terms) * np.abs(y).max()
        oa, ob, prev = oa + prev * c * v, ob + prev * c * 2 * v, c


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("move", ["flip", "exchange"])
@pytest.mark.parametrize("case,chains", [(0, 1), (1, 67), (2, 33), (3, 16), (4, 40), (5, 9), (6, 17), (7, 31), (9, 66),
                                         (10, 17)])
def test_chains_step_alike(case, chains, move, precision):
    import annongpu_amd as A
    extent, *layers = SHAPES[case]
    N, psi = nets(extent, layers, precision, 50 + case)
    # thermalisation and two more intervals, then three intervals
    times = 0 if case == 10 and move == "exchange" else 6

    def run(p):
        ens = A.MonteCarloSpins(3 * chains, 2, 3, chains, move=move, total_z=N % 2, seed=case, persistent=True)
        A.log_psi(p, ens)
        A.log_psi(p, ens)
        return ens.last_samples(), ens.acceptance_rate

    a, b = served("mc", psi, run, times)
    assert np.array_equal(a[0], b[0]) and a[1] == b[1]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_one_site(precision):
    import annongpu_amd as A
    import pyoracle as orc
    from helpers import oracle_operator
    extent, *layers = SHAPES[8]
    _, [psi] = nets(extent, layers, precision, 8)
    o = orc.cnn(extent, [2, 2], [[1, 1, 1]] * 2, np.zeros(1, np.uint32), psi.params, 1.5, 0.0)
    eps = np.finfo(np.float64 if precision == "fp64" else np.float32).eps
    confs = np.array([[0], [1], [1]], dtype=np.uint64)
    ens = A.SampleList(1, confs)
    ref = np.array([orc.log_psi_s(o, orc.conf_words(int(c), 4)) for c in confs[:, 0]])
    [got] = served("log_psi", [psi], lambda p: A.log_psi_vector(p, ens))
    assert np.abs(got - ref).max() <= 32 * eps
    H = 0.7 * A.sigma_z(0) + 0.5 * A.sigma_x(0) + 0.2 * A.sigma_y(0)
    op = oracle_operator(H, 1)
    ref = np.array([orc.local_energy(op, o, orc.conf_words(int(c), 4), l) for c, l in zip(confs[:, 0], ref)])
    [got] = served("local_energy", [psi], lambda p: A.local_energies(A.Operator(H), p, ens))
    assert np.abs(got - ref).max() <= 32 * eps
    t = A.TDVP(psi.num_params)
    served("ok", [psi], lambda p: t.eval_F(A.Operator(H), p, ens))
    ref = np.array([orc.psi_O_k(o, orc.conf_words(int(c), 4)) for c in confs[:, 0]])
    assert np.abs(t.O_k_samples - ref).max() <= 32 * eps
    mc = A.MonteCarloSpins(15, 2, 3, 5, seed=8)
    served("mc", [psi], lambda p: A.log_psi(p, mc), 3)
    if precision == "fp64":
        run = orc.mc_run(o, 5, 3, 2, 3, move=orc.MOVE_FLIP, seed=8)
        assert np.array_equal(mc.last_samples()[:, 0], run["samples"][:, 0])


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_few_and_many(precision):
    """sixteen channels at five sites: few chains and samples take the general kernels, many these; one
    channel: many samples' O_k take the general kernel"""
    import annongpu_amd as A
    N, [psi, _] = nets([1, 1, 20], [(16, [1, 1, 3]), (16, [1, 1, 3])], precision, 3)
    eps = np.finfo(np.float64 if precision == "fp64" else np.float32).eps
    few, many = 8, 5000

    def chains(p, n, move):
        ens = A.MonteCarloSpins(n, 1, 2, n, move=move, seed=5)
        A.log_psi(p, ens)
        return ens.last_samples()[:few]

    for move in ("flip", "exchange"):
        [a] = served("mc", [psi], lambda p: chains(p, few, move), 0)
        [b] = served("mc", [psi], lambda p: chains(p, many, move))
        assert np.array_equal(a, b)
    rng = np.random.default_rng(1)
    confs = words(N, many, rng)
    op = operators(A, N)[1]
    [a] = served("local_energy", [psi], lambda p: A.local_energies(op, p, A.SampleList(N, confs[:few])), 0)
    [b] = served("local_energy", [psi], lambda p: A.local_energies(op, p, A.SampleList(N, confs)))
    terms = N * 16 + 16 * 3
    assert np.abs(a - b[:few]).max() <= 8 * eps * terms * np.abs(a).max()
    N, [psi, _] = nets([1, 1, 20], [(1, [1, 1, 3]), (1, [1, 1, 3])], precision, 4)

    def samples(p, n):
        t = A.TDVP(p.num_params)
        t.eval_F(operators(A, N)[0], p, A.SampleList(N, confs[:n]))
        return t.O_k_samples[:few]

    [a] = served("ok", [psi], lambda p: samples(p, few))
    [b] = served("ok", [psi], lambda p: samples(p, many), 0)
    assert np.abs(a - b).max() <= 8 * eps * np.sqrt(N + 3) * np.abs(a).max()
