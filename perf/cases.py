"""Cases for timing the framework's main path through its public entry points.

A case is one call (or the few calls that a program makes together) of a variational
Monte Carlo run: sampling, TDVP statistics, stochastic-reconfiguration solves, for the
dense nets (PsiRBM, PsiDeep), PsiCNN and multi-layer PsiDeep, in both precisions (fp64
is the default of every wave function, fp32 what large runs choose).

    exact    exact summation: normalise, TDVP.eval, Cholesky solve (a small system studied
             with exact sums, one right-hand side of its time evolution)
    eval     TDVP.eval_F of a dense net on given configurations: E_loc samples, F, <O_k>
    sr       parameters set, TDVP.eval_F, CG solve with a fixed iteration budget
    vmc      the same with Monte Carlo sampling inside: a whole optimisation step
    dense    TDVP.eval with the S matrix and the Cholesky solve
    sample   one sampling interval of persistent Markov chains of a dense net
    block    the same with the learned block proposal attached
    cnn      TDVP.eval and Cholesky solve of a PsiCNN on given configurations
    cnnmc    one sampling interval of persistent chains of a PsiCNN
    deepmc   sampling and local energies of a two-layer PsiDeep
"""
import math

import numpy as np
import torch

import annongpu_amd as A


def listed():
    return [
        # smallest: 12-site transverse-field Ising ring with exact sums; latency and launches
        dict(name="exact_ring12", kind="exact", model="ising", Lx=1, Ly=12, M=24, precision="fp64"),
        # ordinary: 6x6 Heisenberg, RBM with two hidden units per site, default precision, a
        # ragged number of samples
        dict(name="eval_6x6_fp64", kind="eval", model="heisenberg", net="rbm", Lx=6, Ly=6, M=72, samples=1000,
             precision="fp64"),
        # the benchmark's workload: 10x10 Heisenberg, 400 hidden units, 16,384 samples; its
        # statistics alone and with the preconditioned solve
        dict(name="eval_10x10_fp32", kind="eval", model="heisenberg", net="deep", Lx=10, Ly=10, M=400, samples=16384,
             precision="fp32"),
        dict(name="sr_10x10_fp32", kind="sr", model="heisenberg", net="deep", Lx=10, Ly=10, M=400, samples=16384,
             precision="fp32", method="cg_kfac", iters=40),
        # a whole optimisation step in the default precision on the 64-site ring
        dict(name="vmc_ring64_fp64", kind="vmc", model="heisenberg", net="deep", Lx=1, Ly=64, M=128, samples=4096,
             sweeps=2, move="exchange", precision="fp64", method="cg", iters=40),
        # sampling: the benchmark's exchange chains, odd-sized single-flip chains in fp64, and
        # the learned block proposal
        dict(name="sample_10x10_fp32", kind="sample", net="deep", Lx=10, Ly=10, M=400, samples=16384, sweeps=2,
             move="exchange", precision="fp32"),
        dict(name="sample_ring45_fp64", kind="sample", net="rbm", Lx=1, Ly=45, M=90, samples=1000, sweeps=10,
             move="flip", precision="fp64"),
        dict(name="block_10x10_fp32", kind="block", net="deep", Lx=10, Ly=10, M=400, samples=16384, sweeps=2,
             move="exchange", precision="fp32"),
        # largest: the dense S matrix of the 64-site ring with 16,704 parameters and its solve
        dict(name="dense_ring64_fp32", kind="dense", model="heisenberg", net="deep", Lx=1, Ly=64, M=256, samples=8192,
             precision="fp32"),
        # the quench workload: 12x12 transverse-field Ising, PsiCNN of two 3x3 layers
        dict(name="cnnmc_12x12_fp32", kind="cnnmc", Lx=12, Ly=12, channels=8, kernel=3, samples=16384, sweeps=1,
             move="flip", precision="fp32"),
        dict(name="cnn_12x12_fp32", kind="cnn", Lx=12, Ly=12, channels=8, kernel=3, samples=4096, precision="fp32"),
        # two hidden layers
        dict(name="deepmc_ring32_fp64", kind="deepmc", model="ising", Lx=1, Ly=32, M=64, M2=32, samples=2048, sweeps=1,
             move="flip", precision="fp64"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["exact", "eval", "eval", "sr", "vmc", "dense", "sample", "sample", "block", "cnn", "cnnmc",
                       "deepmc"])
    precision = rng.choice(["fp32", "fp64"])
    net = rng.choice(["deep", "rbm"])
    lattice = rng.choice([(1, rng.randint(8, 30) * 2), (4, 4), (6, 5), (6, 6), (8, 7), (8, 8), (10, 9), (10, 10)])
    Lx, Ly = lattice
    N = Lx * Ly
    if kind == "exact":
        n = rng.randint(8, 13)
        return dict(kind=kind, model="ising", Lx=1, Ly=n, M=rng.randint(n, 2 * n), precision=precision)
    if kind == "eval":
        return dict(kind=kind, model=rng.choice(["heisenberg", "ising"]), net=net, Lx=Lx, Ly=Ly,
                    M=min(400, _log_int(rng, N, 4 * N)), samples=_log_int(rng, 200, 16384), precision=precision)
    if kind == "sr":
        return dict(kind=kind, model="heisenberg", net="deep", Lx=Lx, Ly=Ly, M=min(400, _log_int(rng, N, 4 * N)),
                    samples=_log_int(rng, 500, 16384), precision=precision, method=rng.choice(["cg", "cg_kfac"]),
                    iters=rng.randint(8, 40))
    if kind == "vmc":
        return dict(kind=kind, model="heisenberg", net="deep", Lx=Lx, Ly=Ly, M=_log_int(rng, N, 3 * N),
                    samples=_log_int(rng, 256, 4096), sweeps=rng.randint(1, 4), move="exchange", precision="fp64",
                    method=rng.choice(["cg", "cg_kfac"]), iters=rng.randint(8, 40))
    if kind == "dense":
        Lx, Ly = rng.choice([(1, 24), (5, 6), (6, 6), (1, 50)])
        return dict(kind=kind, model="heisenberg", net="deep", Lx=Lx, Ly=Ly, M=_log_int(rng, 20, 100),
                    samples=_log_int(rng, 500, 8192), precision=precision)
    if kind in ("sample", "block"):
        c = dict(kind=kind, net=net, Lx=Lx, Ly=Ly, M=min(400, _log_int(rng, N, 4 * N)),
                 samples=_log_int(rng, 200, 16384), sweeps=rng.randint(1, 4), move=rng.choice(["flip", "exchange"]),
                 precision=precision)
        if kind == "block":
            c.update(net="deep", move="exchange")
        return c
    if kind in ("cnn", "cnnmc"):
        L = rng.randint(5, 12)
        c = dict(kind=kind, Lx=L, Ly=L, channels=rng.choice([2, 4, 5, 6, 8]), kernel=rng.choice([2, 3, 3, 4]),
                 precision=precision)
        if kind == "cnn":
            c["samples"] = _log_int(rng, 200, 4096)
        else:
            c.update(samples=_log_int(rng, 200, 16384), sweeps=1,
                     move=rng.choice(["flip", "exchange"]) if L % 2 == 0 else "flip")
        return c
    n = rng.randint(6, 20) * 2
    return dict(kind=kind, model=rng.choice(["heisenberg", "ising"]), Lx=1, Ly=n, M=2 * n, M2=n,
                samples=_log_int(rng, 200, 2048), sweeps=1, move="flip", precision="fp64")


# --------------------------------------------------------------- inputs from the seed

SHIFT = 1e-3


def _bonds(case):
    Lx, Ly = case["Lx"], case["Ly"]
    out = []
    for r in range(Lx):
        for c in range(Ly):
            if c + 1 < Ly or Ly > 2:
                out.append((r * Ly + c, r * Ly + (c + 1) % Ly))
            if Lx > 1 and (r + 1 < Lx or Lx > 2):
                out.append((r * Ly + c, ((r + 1) % Lx) * Ly + c))
    return out


def _gauss(rng, shape, sigma):
    return sigma * (rng.standard_normal(shape) + 1j * rng.standard_normal(shape))


def _dense_weights(case, seed):
    """weights of a partly optimised net: angles of a few tenths"""
    N, M = case["Lx"] * case["Ly"], case["M"]
    rng = np.random.default_rng([11, seed])
    sigma = 0.3 / math.sqrt(2 * N)
    if case.get("net", "deep") == "rbm":
        return dict(W=_gauss(rng, (N, M), sigma))
    d = N // M if N >= M and N % M == 0 else 1 if M > N else N
    conn = (np.arange(M)[None, :] * d + np.arange(N)[:, None]) % N
    return dict(a=_gauss(rng, N, 0.05), b=_gauss(rng, M, 0.05), W=_gauss(rng, (N, M), sigma), conn=conn)


def _spins(case, seed, sector):
    """configurations as +-1, at zero magnetisation when `sector`"""
    N, n = case["Lx"] * case["Ly"], case["samples"]
    rng = np.random.default_rng([12, seed])
    if not sector:
        return np.where(rng.random((n, N)) < 0.5, 1, -1).astype(np.int8)
    order = np.argsort(rng.random((n, N)), axis=1)
    return np.where(order < N // 2, 1, -1).astype(np.int8)


def _words(spins):
    n, N = spins.shape
    W = (N + 63) // 64
    bits = np.zeros((n, 64 * W), dtype=np.uint8)
    bits[:, :N] = spins > 0
    return np.ascontiguousarray(np.packbits(bits, axis=1, bitorder="little")).view(np.uint64)


def _cnn_params(case, seed):
    rng = np.random.default_rng([13, seed])
    C, v = case["channels"], case["kernel"] ** 2
    return np.concatenate([_gauss(rng, C * v, 0.1), _gauss(rng, C * C * v, 0.05)])


def _dense_net(case, seed):
    p = _dense_weights(case, seed)
    N, M = case["Lx"] * case["Ly"], case["M"]
    if "conn" in p:
        psi = A.PsiDeep(N, p["a"], [p["b"]], [p["conn"]], [p["W"]], np.ones(M))
    else:
        psi = A.PsiRBM(p["W"], final_weight=1.0)
    psi.precision = case["precision"]
    return psi


def _operator(case):
    bonds = _bonds(case)
    if case.get("model", "ising") == "heisenberg":
        return A.Operator(A.hamiltonians.heisenberg(bonds))
    return A.Operator(A.hamiltonians.transverse_ising(bonds, case["Lx"] * case["Ly"], 1.0, _field(case)))


def _field(case):
    return 1.0 if case["Lx"] == 1 else 3.04


def _cnn(case, seed):
    L, C, k = [1, case["Lx"], case["Ly"]], case["channels"], case["kernel"]
    psi = A.PsiCNN(L, [C, C], [[1, k, k]] * 2, np.zeros(case["Lx"] * case["Ly"], dtype=np.uint32),
                   _cnn_params(case, seed), 1.0)
    psi.precision = case["precision"]
    return psi


# ------------------------------------------------------------------------ the cases

def prepare(case, seed):
    kind = case["kind"]
    N = case["Lx"] * case["Ly"]
    s = dict(kind=kind, case=case)
    if kind in ("cnn", "cnnmc"):
        s["psi"] = psi = _cnn(case, seed)
    elif kind == "deepmc":
        rng = np.random.default_rng([14, seed])
        M, M2 = case["M"], case["M2"]
        conn1 = (np.arange(M)[None, :] + np.arange(N)[:, None]) % N
        conn2 = (2 * np.arange(M2)[None, :] + np.arange(8)[:, None]) % M
        s["psi"] = psi = A.PsiDeep(N, _gauss(rng, N, 0.05), [_gauss(rng, M, 0.05), _gauss(rng, M2, 0.05)],
                                   [conn1, conn2], [_gauss(rng, (N, M), 0.3 / math.sqrt(2 * N)),
                                                    _gauss(rng, (8, M2), 0.3)], np.ones(M2))
        psi.precision = case["precision"]
    else:
        s["psi"] = psi = _dense_net(case, seed)
    if kind not in ("sample", "block", "cnnmc"):
        s["op"] = _operator(case)
    if kind in ("eval", "sr", "dense", "cnn"):
        sector = case.get("model") == "heisenberg"
        s["ens"] = A.SampleList(N, _words(_spins(case, seed, sector)))
    elif kind == "exact":
        s["ens"] = A.ExactSummationSpins(N)
    else:
        s["ens"] = A.MonteCarloSpins(case["samples"], case["sweeps"], 5, case["samples"], move=case["move"],
                                     total_z=N % 2, seed=seed, persistent=True)
        if kind == "block":
            blocks = A.chain_blocks(N, 8) if case["Lx"] == 1 else A.rect_blocks((case["Lx"], case["Ly"]), (2, 4))
            s["ens"].set_proposal(A.BlockProposal(N, blocks, hidden=256, seed=seed), plain_sweeps=1,
                                  exclude_current=True)
        A.log_psi(psi, s["ens"])   # thermalises the persistent chains
    if kind in ("exact", "eval", "sr", "vmc", "dense", "cnn"):
        s["tdvp"] = A.TDVP(psi.num_params)
        s["params"] = psi.params
    return s


def run(s):
    kind, case, psi, ens = s["kind"], s["case"], s["psi"], s["ens"]
    if kind in ("sample", "block", "cnnmc"):
        A.log_psi(psi, ens)
        return dict(samples=ens.last_samples().view(np.int64), acceptance=ens.acceptance_rate)
    if kind == "deepmc":
        e = A.local_energies(s["op"], psi, ens)
        return dict(E=e, samples=ens.last_samples().view(np.int64))
    t = s["tdvp"]
    if kind == "eval":
        t.eval_F(s["op"], psi, ens)
        return dict(E_samples=t.E_local_samples, F=t.F_vector, O=t.O_k_vector)
    psi.params = s["params"]
    if kind in ("sr", "vmc"):
        t.eval_F(s["op"], psi, ens)
        x = t.solve(SHIFT, case["method"], rtol=0.0, max_iter=case["iters"], raise_on_failure=False)
    else:
        if kind == "exact":
            psi.normalize(ens)
        t.eval(s["op"], psi, ens)
        x = t.solve(SHIFT, "cholesky")
    return dict(E_samples=t.E_local_samples, F=t.F_vector, x=x)


def work(case):
    """what a pass cannot do without: real flops of the formulas, inputs read and results
    written once"""
    kind = case["kind"]
    N = case["Lx"] * case["Ly"]
    n = 2 ** N if kind == "exact" else case["samples"]
    cb = 8 if case["precision"] == "fp32" else 16
    words = 8 * ((N + 63) // 64)
    if kind in ("cnn", "cnnmc"):
        C, v = case["channels"], case["kernel"] ** 2
        P = C * v + C * C * v
        f1, f2 = min(v, N), min((2 * case["kernel"] - 1) ** 2, N)   # sites a flip reaches
        flip = 8.0 * (C * f1 + v * f1 * C * C) + 20.0 * C * (f1 + f2)   # only changed inputs
        if kind == "cnnmc":
            moves = 2 if case["move"] == "exchange" else 1
            return dict(bytes=2.0 * n * words + cb * P, flops=n * case["sweeps"] * N * moves * flip)
        forward = 8.0 * N * (C * v + C * C * v)
        gram = 4.0 * n * P * P
        return dict(bytes=float(n * words + 16 * n + cb * P + 32 * P),
                    flops=n * (3 * forward + N * flip) + gram + 4.0 / 3.0 * P ** 3)
    M = case["M"]
    bonds = len(_bonds(case))
    if kind == "deepmc":
        per = 4.0 * M + 20.0 * M + 8.0 * 8 * case["M2"] + 20.0 * case["M2"]
        flips = 0.5 * bonds if case["model"] == "heisenberg" else N
        return dict(bytes=float(n * (2 * words + 16)), flops=n * (case["sweeps"] * N + flips) * per)
    P = N * M if case.get("net", "deep") == "rbm" else N + M + N * M
    theta = 4.0 * N * M
    move = 26.0 * M + (8.0 if case.get("move") == "exchange" else 4.0) * M
    if kind == "sample":
        return dict(bytes=float(2 * n * words + cb * N * M), flops=n * (theta + case["sweeps"] * N * move))
    if kind == "block":
        k = case["sweeps"] * math.ceil(N / 8)
        per = 26.0 * M + 4 * 4.0 * M + 2 * 8 * 256 + 8 * 256
        return dict(bytes=float(2 * n * words + cb * N * M), flops=n * (theta + N * move + k * per))
    flips = 0.5 * bonds * (34.0 * M) if case["model"] == "heisenberg" else N * 30.0 * M
    flops = n * (theta + flips + 10.0 * M + 2 * 4.0 * N * M)   # E_loc, <O> and F
    byts = float(n * words + 16 * n + 3 * 16 * P + 16 * P)
    if kind in ("sr", "vmc"):
        flops += case["iters"] * n * 2 * 4.0 * N * M
        byts += case["iters"] * (cb * n * M)   # g streamed once per iteration
    if kind == "vmc":
        flops += n * case["sweeps"] * N * move
    if kind in ("dense", "exact"):
        flops += 4.0 * n * P * P + 4.0 / 3.0 * P ** 3
        byts += 16.0 * P * P
    return dict(bytes=byts, flops=flops)


# -------------------------------------------------- the same in plain torch, 64 bits

def _lc(z):
    u = z * z
    return u * (0.5 + u * (-1.0 / 12.0 + u / 45.0))


def _th(z):
    u = z * z
    return z * (1.0 + u * (-1.0 / 3.0 + u * (2.0 / 15.0)))


def _dth(z):
    u = z * z
    return 1.0 + u * (-1.0 + u * (2.0 / 3.0))


def _c(x):
    return torch.as_tensor(np.asarray(x), dtype=torch.complex128, device="cuda")


class _Dense:
    def __init__(self, case, seed, spins):
        p = _dense_weights(case, seed)
        self.N, self.M = case["Lx"] * case["Ly"], case["M"]
        self.deep = "conn" in p
        Wd = np.zeros((self.N, self.M), dtype=complex)
        if self.deep:
            np.add.at(Wd, (p["conn"], np.arange(self.M)[None, :]), p["W"])
            self.b = _c(p["b"])
            self.conn = torch.as_tensor(p["conn"], device="cuda")
        else:
            Wd = p["W"]
            self.b = _c(np.zeros(self.M))
        self.W = _c(Wd)
        self.S = _c(spins)
        self.theta = self.S @ self.W + self.b
        self.g = _th(self.theta)

    def local_energy(self, case):
        s, diag = self.S.real, 0
        out = torch.zeros(s.shape[0], dtype=torch.complex128, device="cuda")
        base = _lc(self.theta)
        if case["model"] == "heisenberg":
            for i, j in _bonds(case):
                diag = diag + s[:, i] * s[:, j]
                k = torch.nonzero(s[:, i] != s[:, j])[:, 0]
                t = self.theta[k] - 2 * s[k, i, None] * self.W[i] - 2 * s[k, j, None] * self.W[j]
                out[k] += 2 * torch.exp((_lc(t) - base[k]).sum(1))
            return out + diag
        for i, j in _bonds(case):
            diag = diag - s[:, i] * s[:, j]
        for i in range(self.N):
            t = self.theta - 2 * s[:, i, None] * self.W[i]
            out -= _field(case) * torch.exp((_lc(t) - base).sum(1))
        return out + diag

    def pack(self, a, b, w):
        """parameter order from the (site) a, (unit) b and (site, unit) W parts"""
        if not self.deep:
            return w.reshape(-1)
        return torch.cat([a, b, torch.gather(w, 0, self.conn).reshape(-1)])

    def sums(self, coef, conj):
        """sum_s coef_s O_s (or conj O_s)"""
        x = coef[:, None] * (self.g.conj() if conj else self.g)
        return self.pack(self.S.T @ coef, x.sum(0), self.S.T @ x)

    def split(self, v):
        if not self.deep:
            return None, None, v.reshape(self.N, self.M)
        w = torch.zeros((self.N, self.M), dtype=v.dtype, device=v.device)
        w.scatter_(0, self.conn, v[self.N + self.M:].reshape(self.N, self.M))
        return v[:self.N], v[self.N:self.N + self.M], w

    def dot(self, v):
        a, b, w = self.split(v)
        u = (self.g * (self.S @ w + (0 if b is None else b))).sum(1)
        return u if a is None else u + self.S @ a

    def rows(self):
        w = self.S[:, :, None] * self.g[:, None, :]
        if not self.deep:
            return w.reshape(w.shape[0], -1)
        w = torch.gather(w, 1, self.conn[None].expand(w.shape[0], -1, -1))
        return torch.cat([self.S, self.g, w.reshape(w.shape[0], -1)], 1)


def _cg(net, F, w, O, method, iters):
    n = net.S.shape[0]

    def S_dot(v):
        return net.sums(w * (net.dot(v) - (O * v).sum()), True) + SHIFT * v

    ones = torch.full((n,), 1.0 / n, dtype=torch.complex128, device="cuda")
    g2 = ((net.g.abs() ** 2).sum(0) / n).to(torch.complex128)
    sq = net.pack(torch.ones(net.N, dtype=torch.complex128, device="cuda"), g2, g2.expand(net.N, -1).contiguous())
    diag = sq.real - O.abs() ** 2

    def jacobi(r):
        return r / (diag + SHIFT)

    if method == "cg_kfac":
        s = net.S.real
        C = s.T @ s / n - torch.outer(s.mean(0), s.mean(0))
        m = (ones[:, None] * net.g).sum(0)
        D = net.g.conj().T @ net.g / n - torch.outer(m.conj(), m)
        pi = torch.sqrt((torch.trace(C) / net.N) / (torch.trace(D).real / net.M))
        Ci = torch.linalg.inv(C + 0.3 * math.sqrt(SHIFT) * pi * torch.eye(net.N, device="cuda", dtype=C.dtype))
        Di = torch.zeros_like(D)
        for k in range(0, net.M, 64):
            e = min(k + 64, net.M)
            blk = D[k:e, k:e] + 0.3 * math.sqrt(SHIFT) / pi * torch.eye(e - k, device="cuda", dtype=D.dtype)
            Di[k:e, k:e] = torch.linalg.inv(blk)

    def precondition(r):
        if method != "cg_kfac":
            return jacobi(r)
        z = jacobi(r)
        a, b, w_ = net.split(r)
        w_ = (Ci.to(torch.complex128) @ w_) @ Di.T
        packed = net.pack(z[:net.N], z[net.N:net.N + net.M], w_)
        return packed

    x = torch.zeros_like(F)
    r = F.clone()
    z = precondition(r)
    p = z.clone()
    rz = (r.conj() * z).sum().real
    for _ in range(iters):
        Ap = S_dot(p)
        alpha = rz / (p.conj() * Ap).sum().real
        x = x + alpha * p
        r = r - alpha * Ap
        z = precondition(r)
        new = (r.conj() * z).sum().real
        p = z + (new / rz) * p
        rz = new
    return x


def _neighbours(case):
    Lx, Ly, k = case["Lx"], case["Ly"], case["kernel"]
    x = np.arange(Lx * Ly)
    out = [((x // Ly + i) % Lx) * Ly + (x % Ly + j) % Ly for i in range(k) for j in range(k)]
    return torch.as_tensor(np.stack(out, 1), device="cuda")   # [N][vol]


def _cnn_exact(case, seed):
    spins = _spins(case, seed, False)
    n, N, C, v = len(spins), case["Lx"] * case["Ly"], case["channels"], case["kernel"] ** 2
    p = _c(_cnn_params(case, seed))
    w0, w1 = p[:C * v].reshape(C, v), p[C * v:].reshape(C, C, v)   # [c][o], [ci][cj][o]
    nb = _neighbours(case)

    def forward(s):
        a0 = s[:, nb]                                           # [n][N][vol]
        z0 = a0 @ w0.T                                          # [n][N][C]
        h = _lc(z0)
        a1 = h[:, nb]                                           # [n][N][vol][ci]
        z1 = a1.reshape(len(s), N, v * C) @ w1.permute(2, 0, 1).reshape(v * C, C)
        return a0, z0, a1, z1

    def log_psi(s):
        out = []
        for q in torch.split(s, 2048):
            out.append(_th(forward(q)[3]).sum((1, 2)))
        return torch.cat(out)

    S = _c(spins)
    base = log_psi(S)
    e = torch.zeros(n, dtype=torch.complex128, device="cuda")
    s = S.real
    for i, j in _bonds(case):
        e -= s[:, i] * s[:, j]
    for i in range(N):
        q = S.clone()
        q[:, i] *= -1
        e -= _field(case) * torch.exp(log_psi(q) - base)
    rows = []
    for q in torch.split(S, 1024):
        a0, z0, a1, z1 = forward(q)
        d1 = _dth(z1)                                           # [n][N][cj]
        m = len(q)
        g1 = torch.bmm(a1.reshape(m, N, v * C).transpose(1, 2).contiguous(), d1).reshape(m, v, C, C)
        back = (d1 @ w1.permute(1, 2, 0).reshape(C, v * C)).reshape(m, N, v, C)   # [n][x][o][ci]
        g0h = torch.zeros((m, N, C), dtype=torch.complex128, device="cuda")
        for o in range(v):
            g0h.index_add_(1, nb[:, o], back[:, :, o].contiguous())
        d0 = g0h * _th(z0)
        g0 = torch.bmm(a0.transpose(1, 2).contiguous(), d0)     # [n][vol][C]
        rows.append(torch.cat([g0.permute(0, 2, 1).reshape(m, -1), g1.permute(0, 2, 3, 1).reshape(m, -1)], 1))
    return e, torch.cat(rows)


def _dense_solution(e, O, w):
    E = (w * e).sum()
    Ob = (w[:, None] * O).sum(0)
    F = (O.conj() * (w * e)[:, None]).sum(0) - E * Ob.conj()
    S = O.conj().T @ (w[:, None] * O) - torch.outer(Ob.conj(), Ob)
    S.diagonal().add_(SHIFT)
    d = torch.rsqrt(S.diagonal().real)
    S *= d[:, None]
    S *= d
    L = torch.linalg.cholesky(S)
    x = d * torch.cholesky_solve((d * F)[:, None], L)[:, 0]
    return dict(E_samples=e.cpu().numpy(), F=F.cpu().numpy(), x=x.cpu().numpy())


def exact(case, seed):
    kind = case["kind"]
    N = case["Lx"] * case["Ly"]
    if kind in ("sample", "block", "cnnmc", "deepmc", "vmc"):
        return None
    if kind == "cnn":
        e, O = _cnn_exact(case, seed)
        return _dense_solution(e, O, torch.full((len(e),), 1.0 / len(e), dtype=torch.complex128, device="cuda"))
    if kind == "exact":
        spins = np.where((np.arange(2 ** N)[:, None] >> np.arange(N)) & 1, 1, -1)
        net = _Dense(case, seed, spins)
        lp = _lc(net.theta).sum(1)
        w = torch.exp(2 * lp.real)
        w = (w / w.sum()).to(torch.complex128)
        return _dense_solution(net.local_energy(case), net.rows(), w)
    net = _Dense(case, seed, _spins(case, seed, case["model"] == "heisenberg"))
    n = net.S.shape[0]
    w = torch.full((n,), 1.0 / n, dtype=torch.complex128, device="cuda")
    e = net.local_energy(case)
    if kind == "dense":
        return _dense_solution(e, net.rows(), w)
    E = (w * e).sum()
    O = net.sums(w, False)
    F = net.sums(w * (e - E), True)
    if kind == "eval":
        return dict(E_samples=e.cpu().numpy(), F=F.cpu().numpy(), O=O.cpu().numpy())
    x = _cg(net, F, w, O, case["method"], case["iters"])
    return dict(E_samples=e.cpu().numpy(), F=F.cpu().numpy(), x=x.cpu().numpy())
