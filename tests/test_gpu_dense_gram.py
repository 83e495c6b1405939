"""S of a one-layer net from pairs of sites and units against the Gram of its O_k samples, at the
edges of the kernel's tiles (64 site pairs a wave, 32 unit pairs, 16 samples a stage, 64-sample
words) and over the layouts that reach it, sample counts and weights that do not sum to one.

The O_k samples are exact copies of what S is built from, so both sides are fp64 sums of the
same products: |S - S_ref| <= 4 n eps max|sum w |O_k|^2| entrywise (n summands).

The pairs serve while no parameter's squared mean exceeds twice its variance (fp32: 1,024 times it); where
one does, S comes from the centred O_k and its error stays within the rounding of the n products and
of the centring, relative to the two parameters' spreads."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def net(kind, N, M, rng):
    import annongpu_amd as A

    def gauss(shape, sigma):
        return sigma * (rng.standard_normal(shape) + 1j * rng.standard_normal(shape))

    if kind == "rbm":
        return A.PsiRBM(gauss((N, M), 0.2), final_weight=1.5 - 0.5j)
    if kind == "circulant":
        conn = (np.arange(M)[None, :] + np.arange(N)[:, None]) % N
    elif kind == "shuffled":
        conn = np.stack([rng.permutation(N) for _ in range(M)], axis=1)
    else:   # repeated: every unit reads one of its sites twice
        conn = np.stack([np.concatenate([rng.permutation(N), rng.integers(0, N, 1)]) for _ in range(M)], axis=1)
    return A.PsiDeep(N, gauss(N, 0.1), [gauss(M, 0.1)], [conn], [gauss(conn.shape, 0.2)], 1.0 + rng.random(M))


def evaluate(A, psi, op, ens):
    """the TDVP object and whether its S came from pairs"""
    t = A.TDVP(psi.num_params)
    A.profiler_reset()
    A.start_profiling()
    t.eval(op, psi, ens)
    A.stop_profiling()
    assert A.profiler_query("gram")[1] == 1
    return t, A.profiler_query("gram_pairs")[1] == 1


def dominance(O, w):
    """largest ratio of a squared mean to the variance (inf where there is no variance)"""
    m = np.abs(w @ O) ** 2
    d = w @ np.abs(O) ** 2 - m
    return np.where(d > 0, m / np.where(d > 0, d, 1), np.inf).max()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind,N,M,n", [("circulant", 1, 1, 1), ("circulant", 11, 6, 65), ("rbm", 11, 7, 64),
                                        ("rbm", 12, 24, 1000), ("shuffled", 23, 9, 129), ("circulant", 22, 8, 15),
                                        ("repeated", 16, 5, 300), ("circulant", 70, 3, 63)])
def test_dense_gram(kind, N, M, n, precision):
    import annongpu_amd as A
    rng = np.random.default_rng(100 * N + M)
    psi = net(kind, N, M, rng)
    psi.precision = precision
    words = (N + 63) // 64
    confs = rng.integers(0, 2 ** 63, size=(n, words), dtype=np.uint64)
    if N % 64:
        confs[:, -1] &= np.uint64(2 ** (N % 64) - 1)
    w = rng.random(n) / n
    t, pairs = evaluate(A, psi, A.Operator(1.0 * A.sigma_z(0)), A.SampleList(N, confs, w))
    O = t.O_k_samples
    if n > 1:
        assert pairs == (dominance(O, w) <= (2 if precision == "fp64" else 1024))
    mean = w @ O
    S = (O.conj() * w[:, None]).T @ O - np.outer(mean.conj(), mean)
    assert np.abs(t.S_matrix - S).max() <= 4 * max(n, 8) * np.finfo(float).eps * (w @ np.abs(O) ** 2).max()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("bias,flips", [(0.0, 0.5), (0.0, 0.02), (0.8, 0.5), (0.8, 0.02)])
def test_dominating_means(bias, flips, precision):
    """hidden biases far above the spread of the angles and polarised spins; n a power of two, so that
    the weights sum to one exactly.  Per entry, in units of the two spreads: n products and sums of
    eps (8 for the complex parts), the centring's eps |O| and, in fp32, its rounding of the centred O.
    (From uncentred sums the error is eps |O|^2, 1e5 to 1e6 in these units.)"""
    import annongpu_amd as A
    N, M, n = 12, 24, 512
    rng = np.random.default_rng(3)
    conn = (np.arange(M)[None, :] + np.arange(N)[:, None]) % N
    W = 1e-3 * (rng.standard_normal((N, M)) + 1j * rng.standard_normal((N, M)))
    psi = A.PsiDeep(N, np.zeros(N), [bias * (1 + 0.1 * rng.random(M))], [conn], [W], np.ones(M))
    psi.precision = precision
    bits = rng.random((n, N)) >= flips
    confs = (bits.astype(np.uint64) << np.arange(N, dtype=np.uint64)).sum(1, dtype=np.uint64)[:, None]
    t, pairs = evaluate(A, psi, A.Operator(1.0 * A.sigma_z(0)), A.SampleList(N, confs))
    O = t.O_k_samples.astype(np.clongdouble)
    w = np.full(n, 1 / n)
    ratio = dominance(O.astype(complex), w)
    assert pairs == (ratio <= (2 if precision == "fp64" else 1024))
    x = O - O.mean(0)
    S = (x.conj().T @ x) / n
    spread = np.sqrt(np.diag(S).real)
    size = np.sqrt((np.abs(O) ** 2).mean(0)) / spread
    eps = np.finfo(float).eps
    bound = 8 * (n + 3) * eps + 4 * eps * (size[:, None] + size[None, :])
    if pairs:
        bound = bound + 8 * (n + 3) * eps * size[:, None] * size[None, :]
    elif precision == "fp32":
        bound = bound + 4 * np.finfo(np.float32).eps
    assert np.all(np.abs(t.S_matrix - S) <= bound * spread[:, None] * spread[None, :])


def ring(N, M, n):
    import annongpu_amd as A
    rng = np.random.default_rng(5)
    psi = net("circulant", N, M, rng)
    psi.precision = "fp32"
    confs = rng.integers(0, 2 ** 63, size=(n, 1), dtype=np.uint64) >> np.uint64(max(0, 63 - N))
    return A, psi, A.Operator(1.0 * A.sigma_z(0)), A.SampleList(N, confs)


def free_memory(A):
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert A._lib.lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("n,expected", [(64, False), (512, True)])
def test_few_samples_of_many_parameters(n, expected):
    """few samples do not pay for the pairs' table of 12,662 parameters; bound as above"""
    A, psi, op, ens = ring(62, 200, n)
    t, pairs = evaluate(A, psi, op, ens)
    assert pairs == expected
    O = t.O_k_samples
    x = O - O.mean(0)
    rows = np.r_[0:3, 61, 62, 261, 262, 5000, 12661]
    S = x[:, rows].conj().T @ x / n
    eps = np.finfo(float).eps if expected else np.finfo(np.float32).eps   # (the centred O is rounded)
    assert np.abs(t.S_matrix[rows] - S).max() <= 4 * max(n, 8) * eps * (np.abs(O) ** 2).mean(0).max()


def test_memory_held():
    """after an evaluation and a solve the object holds S and the factor, and no third buffer of their
    size class: the workspace of S is the factor's (72 MB of pairs here)"""
    A, psi, op, ens = ring(4, 3, 8)
    evaluate(A, psi, op, ens)[0].solve(1e-2, "cholesky")   # streams, code and their memory
    A, psi, op, ens = ring(32, 128, 256)
    P = psi.num_params
    A.log_psi(psi, ens)
    before = free_memory(A)
    t, pairs = evaluate(A, psi, op, ens)
    t.solve(1e-2, "cholesky")
    held = before - free_memory(A)
    assert held <= 2 * 16 * P * P + 48 * 2 ** 20
    assert pairs


def test_pairs_do_not_fit():
    """S next to the samples' O fits the card, S next to the pairs' table does not: the evaluation
    still answers"""
    A, psi, op, ens = ring(62, 200, 512)   # S 2.6 GB, the table 0.64 GB, O 52 MB
    P = psi.num_params
    t, pairs = evaluate(A, psi, op, ens)
    assert pairs
    want = t.S_matrix[:100].copy()
    diag = np.diag(t.S_matrix).real.copy()
    del t
    hip = A._lib.lib

    def allocate(size):
        p = ctypes.c_void_p()
        return p if hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size)) == 0 else None

    room = allocate(16 * P * P + 350 * 2 ** 20)
    size, held = 2 ** 36, []
    while size >= 2 ** 24:
        p = allocate(size)
        if p:
            held.append(p)
        else:
            size //= 2
    hip.hipGetLastError()
    assert hip.hipFree(room) == 0
    try:
        t, pairs = evaluate(A, psi, op, ens)
    finally:
        for p in held:
            assert hip.hipFree(p) == 0
    assert not pairs
    d = np.sqrt(diag)
    assert np.abs((t.S_matrix[:100] - want) / d / d[:100, None]).max() <= 1e-5


@pytest.mark.parametrize("bias", [0.1, 0.8])
def test_next_calls_leave_S_alone(bias):
    """an evaluation may return with S still queued (a few ms of work here): the same wave function and
    ensemble changed, evaluated elsewhere and destroyed meanwhile do not reach it"""
    A, psi, op, _ = ring(62, 200, 512)
    psi.precision = "fp64"
    if bias > 0.5:   # the means dominate: S from the centred samples
        psi.params = np.concatenate([np.zeros(62), np.full(200, bias), 1e-3 * psi.params[262:]])
    first = psi.params

    def chains():
        ens = A.MonteCarloSpins(512, 2, 3, 512, seed=4, persistent=True)
        A.log_psi(psi, ens)
        return ens

    t, pairs = evaluate(A, psi, op, chains())
    assert pairs == (bias < 0.5)
    want = t.S_matrix[:300].copy()
    for _ in range(2):
        psi.params = first
        ens = chains()
        t.eval(op, psi, ens)
        psi.params = 0.5 * first
        A.TDVP(psi.num_params).eval_F(op, psi, ens)
        del ens
        assert np.array_equal(t.S_matrix[:300], want)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [1, 127, 129, 300, 1025])
def test_gram_of_materialised_samples(n, precision):
    """S of a PsiCNN (no pair structure) at the edges of the Gram's sample chunks: the fp64 rank-one
    term and n summands, entrywise as above."""
    import annongpu_amd as A
    rng = np.random.default_rng(n)
    psi = A.seeded_cnn([1, 3, 4], [(3, [1, 2, 2]), (2, [1, 3, 2])], seed=n, sigma=0.2)
    psi.precision = precision
    confs = rng.integers(0, 2 ** 12, size=(n, 1), dtype=np.uint64)
    w = rng.random(n) / n
    t = A.TDVP(psi.num_params)
    t.eval(A.Operator(1.0 * A.sigma_z(0)), psi, A.SampleList(12, confs, w))
    O = t.O_k_samples
    mean = w @ O
    S = (O.conj() * w[:, None]).T @ O - np.outer(mean.conj(), mean)
    assert np.abs(t.S_matrix - S).max() <= 4 * max(n, 8) * np.finfo(float).eps * (w @ np.abs(O) ** 2).max()
