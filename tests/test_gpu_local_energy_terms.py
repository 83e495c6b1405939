"""Local energies of a dense net where a lane takes a term, at the edges of that kernel: units that
do not fill a tile, terms with equal spins and strings that read other sites, more terms than a
tile of 32 units holds, one to four configuration words, sample counts around a workgroup's, and
operators with a string of three flips, which take the general kernel.  So do operators with few
terms for the units; the profiler's counts say which kernel served a shape.

Reference: the sum over the strings in numpy (complex128).  fp64: rounding of a sum of M polynomial
terms and of the strings, 1e-12 of sum |c psi'/psi|.  fp32: a unit's angle is rounded to eps |theta|
and its term to a few eps of its value, both below eps here (|theta| < 1), 8 roundings a unit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def operator(A, kind, N, rng):
    x, y, z = A.sigma_x, A.sigma_y, A.sigma_z
    H = 0.3 * z(0)
    if kind == "xx":        # equal and opposite spins alike
        for i in range(N - 1):
            H = H + (0.5 + 0.1 * i) * x(i) * x(i + 1)
    elif kind == "dressed":   # two flips whose coefficient reads a third site, imaginary parts, single flips
        for i in range(N - 2):
            H = H + (1.0 + 0.05 * i) * x(i) * z(i + 1) * y(i + 2) + 0.2 * y(i)
    elif kind == "bonds":
        for i in range(N - 1):
            H = H + (x(i) * x(i + 1) + y(i) * y(i + 1) + z(i) * z(i + 1))
    elif kind == "all pairs":
        for i in range(N):
            for j in range(i):
                H = H + rng.random() * (x(i) * x(j) + y(i) * y(j)) + rng.random() * z(i) * z(j)
    else:                   # three flips
        for i in range(N - 2):
            H = H + 0.3 * x(i) * x(i + 1) * x(i + 2) + 0.1 * x(i)
    return H


def reference(H, theta, W, f, spins):
    def lc(t):
        u = t * t
        return u * (0.5 + u * (-1 / 12 + u / 45))

    base = lc(theta)
    out, size = np.zeros(len(spins), complex), np.zeros(len(spins))
    for (a, b), c in H:
        flip = [i for i in range(spins.shape[1]) if ((a ^ b) >> i) & 1]
        zy = [i for i in range(spins.shape[1]) if (b >> i) & 1]
        ny = bin(~a & b).count("1")
        coef = c * (-1j) ** ny * np.prod(spins[:, zy], axis=1)   # -1 for Z or Y on a down spin
        t = theta - 2 * spins[:, flip] @ W[flip]
        v = coef * np.exp(((lc(t) - base) * f).sum(1))
        out += v
        size += np.abs(v)
    return out, size


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind,N,M,n", [("xx", 6, 1, 1), ("xx", 9, 33, 511), ("dressed", 8, 70, 513),
                                        ("dressed", 70, 5, 1030), ("bonds", 130, 7, 40), ("bonds", 12, 64, 8200),
                                        ("all pairs", 30, 37, 65), ("all pairs", 40, 3, 5),
                                        ("bonds", 200, 36, 33), ("three", 10, 20, 100), ("xx", 20, 1, 1),
                                        ("xx", 40, 33, 511), ("dressed", 40, 70, 513), ("bonds", 60, 64, 8200),
                                        ("bonds", 26, 100, 20), ("bonds", 9, 600, 20), ("bonds", 60, 600, 20)])
@pytest.mark.parametrize("real_f", [True, False])
def test_local_energy_terms(kind, N, M, n, real_f, precision):
    import annongpu_amd as A
    rng = np.random.default_rng(N * 100 + M)
    sigma = 0.15 / np.sqrt(N)
    W = sigma * (rng.standard_normal((N, M)) + 1j * rng.standard_normal((N, M)))
    b = 0.05 * (rng.standard_normal(M) + 1j * rng.standard_normal(M))
    f = rng.random(M) + (0 if real_f else 0.3j * rng.standard_normal(M))
    conn = np.repeat(np.arange(N)[:, None], M, axis=1)
    psi = A.PsiDeep(N, np.zeros(N), [b], [conn], [W], f)
    psi.precision = precision
    spins = np.where(rng.random((n, N)) < 0.5, 1, -1)
    bits = np.zeros((n, (N + 63) // 64 * 64), np.uint8)
    bits[:, :N] = spins > 0
    confs = np.ascontiguousarray(np.packbits(bits, axis=1, bitorder="little")).view(np.uint64)
    H = operator(A, kind, N, rng)
    A.profiler_reset()
    A.start_profiling()
    e = A.local_energies(A.Operator(H), psi, A.SampleList(N, confs))
    A.stop_profiling()
    few = [("xx", 6), ("xx", 9), ("dressed", 8), ("bonds", 12), ("bonds", 26), ("bonds", 9)]
    served = precision == "fp32" and kind != "three" and (kind, N) not in few
    assert A.profiler_query("local_energy_terms")[1] == served
    ref, size = reference(H, spins @ W + b, W, f, spins)
    tol = 1e-12 if precision == "fp64" else 8 * np.finfo(np.float32).eps * (M + 1)
    assert np.all(np.abs(e - ref) <= tol * size)
