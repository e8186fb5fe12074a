"""Performance cases of the BLD solvers: what a user's program has bnmf_hip do.

A case is one use of the package through its public entry points, on inputs
drawn from the allocation model the solvers assume (Poisson counts of a
nonnegative low-rank mean, bnmf_priors / sample_S). `mean` is the average
count of an entry of X: a corpus of word counts or any large count matrix has
far fewer counts than entries (the sizes of the benchmark configurations with
a = 40 give 0.02 to 0.4), a spectrogram or a small table several per entry.

  call    bld_mult / bld_add / bld_appr on host arrays, as the reference's
          templates are called
  batch   a Batch / ApprBatch held by the program, solved from its resident
          starting point, its results fetched
  score   a Batch solved with the log-marginal convergence check, then its
          S and the factors of its first instance
  server  a burst of requests into a running solve server, collected as they
          finish
"""
import math
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bnmf-algs_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import bnmf_hip as hip  # noqa: E402

EPS = 1e-50


def _case(name, use, algo, dtype, iters, x, y, z, mean, n=0, appr=False, start="seed", shapes=0):
    c = {"name": name, "use": use, "algo": algo, "dtype": dtype, "iters": iters, "x": x, "y": y, "z": z,
         "mean": mean, "n": n, "appr": appr, "start": start, "shapes": shapes}
    if name is None:
        del c["name"]
    return c


def listed():
    return [
        # the reference's own unit-test problem: a table of 8 x 10 counts,
        # 2000 iterations, where an iteration is all launches
        _case("fixture_f64", "call", "mult", "f64", 2000, 8, 10, 3, 5.0),
        # the reference's CPU configuration: 100 x 100, 17 sources, 1000 iterations
        _case("single_f64", "call", "mult", "f64", 1000, 100, 100, 17, 0.4),
        # the FP64 drop-in configuration: 1024 x 1024, 32 sources, 500 iterations
        _case("large_f64", "call", "mult", "f64", 500, 1024, 1024, 32, 40 / 1024),
        # the FP32 configuration: 2048 x 2048, 64 sources, 300 iterations
        _case("large_f32", "call", "mult", "f32", 300, 2048, 2048, 64, 40 / 2048, appr=True),
        # a magnitude spectrogram (513 bins), dense counts, through the plain call
        _case("spectrogram_f32", "call", "mult", "f32", 200, 513, 861, 24, 6.0, appr=True),
        # the batched workload: independent instances of uneven shapes with
        # their own starting tensors, FP32, 200 iterations
        _case("batch_f32", "batch", "mult", "f32", 200, 512, 512, 32, 0.0, n=60, appr=True, start="given", shapes=1),
        # model comparison in double: dense small tables solved to a
        # tolerance on the log-marginal, scored, factors of the first
        _case("score_f64", "score", "mult", "f64", 100, 384, 384, 32, 4.0, n=16, start="given", shapes=2),
        # the additive solver over a batch of the same kind
        _case("batch_add_f32", "batch", "add", "f32", 200, 512, 512, 32, 0.0, n=32, appr=True, start="given", shapes=3),
        # the approximate solver on one large count matrix
        _case("appr_f32", "call", "appr", "f32", 200, 1024, 1024, 32, 40 / 1024, start="given"),
        # and over a batch in double
        _case("batch_appr_f64", "batch", "appr", "f64", 100, 384, 384, 32, 0.0, n=16, start="given", shapes=4),
        # serving: a burst of requests of log-uniform sizes, S0 drawn on the GPU
        _case("server_f32", "server", "mult", "f32", 200, 1024, 1024, 64, 0.0, n=16, appr=True, shapes=5),
        # more sources than the usual few dozen (z > 64), dense counts
        _case("deep_f32", "batch", "mult", "f32", 100, 320, 448, 100, 3.0, n=1, appr=True, start="given"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _log(rng, lo, hi):
    return round(math.exp(rng.uniform(math.log(lo), math.log(hi))), 4)


def draw(rng):
    use = rng.choice(["call", "call", "call", "batch", "batch", "score", "server", "appr", "deep"])
    dtype = rng.choice(["f32", "f64"])
    shapes = rng.randrange(1, 1 << 30)
    if use == "call" or use == "appr":
        algo = "appr" if use == "appr" else rng.choice(["mult", "mult", "mult", "add"])
        while True:
            x, y, z = _log_int(rng, 8, 2048), _log_int(rng, 8, 2048), _log_int(rng, 2, 64)
            if x * y * z <= (1 << 25):
                break
        # the usual mean counts: a = 40 over the rows, or a dense table (the
        # additive solver's step grows with X: it is for small counts)
        mean = rng.choice([round(40 / x, 4), _log(rng, 0.02, 20.0)]) if algo != "add" else _log(rng, 0.02, 0.5)
        iters = rng.randrange(100, 301) if x * y * z > (1 << 18) else rng.randrange(300, 1001)
        return _case(None, "call", algo, dtype, iters, x, y, z, mean, appr=dtype == "f32" or rng.random() < 0.3,
                     start="given" if algo == "appr" else "seed", shapes=shapes)
    if use == "deep":
        x, y, z = _log_int(rng, 32, 512), _log_int(rng, 32, 512), _log_int(rng, 65, 200)
        return _case(None, "batch", "mult", "f32", rng.randrange(50, 101), x, y, z, _log(rng, 0.05, 5.0), n=1,
                     appr=True, start="given", shapes=shapes)
    if use == "server":
        return _case(None, "server", "mult", "f32", rng.randrange(100, 201), 1024, 1024, 64, 0.0,
                     n=rng.randrange(3, 17), appr=True, shapes=shapes)
    algo = "mult" if use == "score" else rng.choice(["mult", "mult", "add", "appr"])
    big = rng.randrange(128, 513) if dtype == "f32" else rng.randrange(96, 385)
    mean = _log(rng, 0.2, 8.0) if use == "score" else rng.choice([0.0, 0.0, _log(rng, 0.05, 0.5 if algo == "add" else 8.0)])
    return _case(None, use, algo, dtype, rng.randrange(50, 201), big, big, 32, mean,
                 n=rng.randrange(2, 41 if dtype == "f32" else 17), appr=dtype == "f32" or rng.random() < 0.3,
                 start="given", shapes=shapes)


def _problems(case):
    """(x, y, z, a) of every instance: a = the mean column total of X."""
    if not case["n"] or case["n"] == 1:
        return [(case["x"], case["y"], case["z"], case["mean"] * case["x"])]
    rng, out = random.Random(case["shapes"]), []
    for _ in range(case["n"]):
        if case["use"] == "server":
            x, y, z = _log_int(rng, 64, case["x"]), _log_int(rng, 64, case["y"]), _log_int(rng, 8, case["z"])
            a = 40.0
        else:
            x, y, z = rng.randint(32, case["x"]), rng.randint(32, case["y"]), rng.randint(4, case["z"])
            a = rng.uniform(10, 80)
        out.append((x, y, z, case["mean"] * x if case["mean"] else a))
    return out


def _sample(gen, x, y, z, a, dtype, start, appr_factors):
    """X of the allocation model with alpha = beta = 1 and, if given, the
    starting point: S0 with X split over Dirichlet(1) weights, or nu0, mu0."""
    def dirichlet(*shape, dim):
        e = torch.empty(shape, dtype=torch.float64, device="cuda").exponential_(generator=gen)
        return e / e.sum(dim, keepdim=True)

    W, H = dirichlet(x, z, dim=0), dirichlet(z, y, dim=0)
    L = torch.empty((40, y), dtype=torch.float64, device="cuda").exponential_(generator=gen).mean(0) * a
    X = torch.poisson((W @ H) * L, generator=gen).to(dtype)
    if start != "given":
        return X, None, None
    if appr_factors:
        return X, dirichlet(x, z, dim=1).to(dtype), dirichlet(z, y, dim=0).to(dtype)
    return X, (X[:, :, None].double() * dirichlet(x, y, z, dim=2)).to(dtype), None


def _inputs(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    dt = torch.float32 if case["dtype"] == "f32" else torch.float64
    for n, (x, y, z, a) in enumerate(_problems(case)):
        X, s, m = _sample(gen, x, y, z, a, dt, case["start"], case["algo"] == "appr")
        yield n, x, y, z, a, X, s, m


class _Instance:
    pass


def _instance(case, seed, n, x, y, z, a, X, s, m):
    i = _Instance()
    i.X, i.z, i.params, i.seed = X.cpu().numpy(), z, hip.Params(a, 1.0, [1.0] * x, [1.0] * z), int(seed) * 1009 + n
    i.S0 = i.nu0 = i.mu0 = None
    if m is not None:
        i.nu0, i.mu0 = s.cpu().numpy(), m.cpu().numpy()
    elif s is not None:
        i.S0 = s.cpu().numpy()
    return i


def prepare(case, seed):
    hip.init(0)
    insts = [_instance(case, seed, *p) for p in _inputs(case, seed)]
    dt = np.float32 if case["dtype"] == "f32" else np.float64
    state = {"case": case, "insts": insts, "dtype": dt}
    if case["use"] in ("batch", "score"):
        if case["algo"] == "appr":
            state["batch"] = hip.ApprBatch(insts, dtype=dt)
        else:
            state["batch"] = hip.Batch(insts, dtype=dt, use_psi_appr=case["appr"],
                                       algo=hip.ALGO_ADD if case["algo"] == "add" else hip.ALGO_MULT)
    elif case["use"] == "server":
        state["server"] = hip.Server(3 << 30, dtype=dt, use_psi_appr=case["appr"])
    return state


def run(state):
    case, insts, dt = state["case"], state["insts"], state["dtype"]
    iters = case["iters"]
    if case["use"] == "call":
        i = insts[0]
        if case["algo"] == "appr":
            return hip.bld_appr(i.X, i.z, i.params, iters, nu0=i.nu0, mu0=i.mu0, seed=i.seed, dtype=dt)
        if case["algo"] == "add":
            return hip.bld_add(i.X, i.z, i.params, iters, seed=i.seed, dtype=dt)
        return hip.bld_mult(i.X, i.z, i.params, iters, case["appr"], seed=i.seed, dtype=dt)
    if case["use"] == "server":
        srv = state["server"]
        tickets = [srv.submit(i, iters) for i in insts]
        out = []
        for t in tickets:
            srv.wait(t)
            out.append(srv.collect(t)[0])
        return out
    b = state["batch"]
    if case["use"] == "score":
        ran, lm = b.solve_tol(iters, 1e-7, 20)
        return [ran, lm, b.fact(0)] + [b.S(n) for n in range(len(insts))]
    b.solve(iters)
    if case["algo"] == "appr":
        return [b.get(n) for n in range(len(insts))]
    return [b.S(n) for n in range(len(insts))]


def work(case):
    """X and the given start read once, the results written once; 30
    operations (a digamma, the fiber sums, the update) for each element of a
    nonempty fiber and iteration."""
    es, nbytes, flops = (4 if case["dtype"] == "f32" else 8), 0.0, 0.0
    for x, y, z, a in _problems(case):
        live = x * y * (1.0 - math.exp(-a / x))
        nbytes += es * (x * y + x * y * z)
        if case["start"] == "given":
            nbytes += es * ((x + y) * z if case["algo"] == "appr" else x * y * z)
        flops += 30.0 * live * z * case["iters"] * (2 if case["algo"] == "appr" else 1)
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------------ 64-bit results
def _philox_uniform(seed, fibers, n):
    """The first n uniforms of the init_S stream of every fiber (Philox4x32-10
    keyed by seed, counter (block, 6, fiber), 53 bits), in torch int64."""
    lo32 = 0xFFFFFFFF
    blocks = []
    for b in range((n + 1) // 2):
        c = [torch.full_like(fibers, b), torch.full_like(fibers, 6), fibers & lo32, fibers >> 32]
        k0, k1 = seed & lo32, (seed >> 32) & lo32
        for _ in range(10):
            p0, p1 = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57
            c = [((p1 >> 32) & lo32) ^ c[1] ^ k0, p1 & lo32, ((p0 >> 32) & lo32) ^ c[3] ^ k1, p0 & lo32]
            k0, k1 = (k0 + 0x9E3779B9) & lo32, (k1 + 0xBB67AE85) & lo32
        for hi, lo in ((c[0], c[1]), (c[2], c[3])):
            m = ((hi << 21) ^ (lo >> 11)) & ((1 << 53) - 1)
            blocks.append((m.double() + 0.5) * 2.0 ** -53)
    return torch.stack(blocks[:n], 1)


class _Fibers:
    """The fibers with X > 0 in double; the others are zero in every solver."""

    def __init__(self, X, z):
        self.shape, self.z = X.shape, z
        self.i, self.j = torch.nonzero(X > 0, as_tuple=True)
        self.X = X[self.i, self.j].double()[:, None]

    def over_rows(self, v):  # sum over axis 0: (y, z)
        return torch.zeros((self.shape[1], self.z), dtype=torch.float64, device="cuda").index_add_(0, self.j, v)

    def over_cols(self, v):  # sum over axis 1: (x, z)
        return torch.zeros((self.shape[0], self.z), dtype=torch.float64, device="cuda").index_add_(0, self.i, v)

    def grads(self, S):
        """grad_plus of the fibers and grad_minus (x, z), alpha = beta = 1."""
        beta_eph, alpha_eph = self.over_rows(S) + 1.0, self.over_cols(S) + 1.0
        gp = torch.digamma(beta_eph)[self.j] - torch.digamma(S + 1.0)
        return gp, torch.digamma(alpha_eph.sum(0)) - torch.digamma(alpha_eph)

    def dense(self, S):
        out = torch.zeros((*self.shape, self.z), dtype=torch.float64, device="cuda")
        out[self.i, self.j] = S
        return out


def _solve(case, f, S, iters):
    for t in range(iters):
        gp, gm = f.grads(S)
        g = gm[f.i]
        if case["algo"] == "add":
            grad = gp - g
            Z = torch.log(S) + EPS + 0.1 / (t + 1) ** 0.55 * S * (f.X * grad - (S * grad).sum(1, keepdim=True))
            E = torch.exp(Z)
            S = f.X * (E / (E.sum(1, keepdim=True) + EPS))
        else:
            xr = 1.0 / (f.X + EPS)
            nom, den = (S * xr * g).sum(1, keepdim=True), (S * xr * gp).sum(1, keepdim=True)
            S = S * ((gp + nom) * (f.X / (S.sum(1, keepdim=True) + EPS)) / (g + den + EPS))
    return S


def _solve_appr(f, nu, mu, iters):
    def fiber_S():
        v = nu[f.i] * mu.T[f.j]
        h = v.sum(1, keepdim=True)
        return f.X / (h + EPS), f.X / (h * h + EPS), v

    for _ in range(iters):
        for half in range(2):
            oa, oa2, v = fiber_S()
            gp, gm = f.grads(oa * v)
            g = gm[f.i]
            A, B = (v * g).sum(1, keepdim=True), (v * gp).sum(1, keepdim=True)
            other = mu.T[f.j] if half == 0 else nu[f.i]
            n, d = other * (oa * gp + oa2 * A), other * (oa * g + oa2 * B)
            if half == 0:
                nu = nu * (f.over_cols(n) / (f.over_cols(d) + EPS))
                nu = nu / (nu.sum(1, keepdim=True) + EPS)
            else:
                mu = mu * (f.over_rows(n) / (f.over_rows(d) + EPS)).T
                mu = mu / (mu.sum(0, keepdim=True) + EPS)
    oa, _, v = fiber_S()
    return f.dense(oa * v), nu, mu


def exact(case, seed):
    if case["use"] == "score":
        return None  # the number of iterations run follows from the solve itself
    out = []
    for n, x, y, z, a, X, s, m in _inputs(case, seed):
        f = _Fibers(X, z)
        if case["algo"] == "appr":
            out.append(_solve_appr(f, s.double(), m.double(), case["iters"]))
            continue
        if s is None:
            e = -torch.log(_philox_uniform(int(seed) * 1009 + n, f.i * y + f.j, z))
            S = f.X * (e / e.sum(1, keepdim=True))
            S = S.float().double() if case["dtype"] == "f32" else S
        else:
            S = s[f.i, f.j].double()
        S = f.dense(_solve(case, f, S, case["iters"]))
        out.append(S)
    return out[0] if case["use"] == "call" else out
