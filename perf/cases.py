"""The work that users of this framework have it do, as cases that can be timed.

Five kinds, each through the public binding (rbmgpu.Model / rbmgpu.Gpu):

  epoch      one SR training epoch from given weights (train_epoch, replayed
             from its graph): sample, local energies, moments, solve, update
  learned    one sampling epoch with the learned proposal and its moments
  enumerate  one exact epoch over all 2^N states (sampler.type = full): new
             weights, enumeration, moments, and the SR solve
  stored     an SR step on a stored sample set: local energies (read back),
             O, moments and the solve on states that are in hand (replayed
             samples, a sampler of the user's own)
  logpsi     log psi of given states (overlaps, state export)

Models are the Kitaev honeycomb and the toric code with the basic and the
symmetric RBM, with and without the Pfaffian factor, as in the examples,
tests and benchmark.  FP32 contexts compute in single precision and return
doubles; their results are handed on in single precision here.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "rbm-nqs_amd", "python"))

import rbmgpu  # noqa: E402

CHECKPOINT = os.path.join(ROOT, "rbm-nqs_amd", "examples", "kitaev6_sym.rbm")
CHECKPOINT_ED2 = os.path.join(ROOT, "rbm-nqs_amd", "examples", "kitaev2_sym_ed.rbm")


def case(kind, model, n, rbm, alpha, precision, weights, **kw):
    c = {"kind": kind, "model": model, "n": n, "rbm": rbm, "alpha": alpha, "precision": precision, "weights": weights}
    c.update(kw)
    return c


def listed():
    def one(name, *a, **kw):
        return dict(case(*a, **kw), name=name)

    return [
        # the benchmark's headline: a converged 6x6 Kitaev state, trained on
        one("epoch_kitaev6_sym_fp32", "epoch", "kitaev", 6, "symmetry", 4, 32, "kitaev6_sym", chains=16384,
            per_chain=8, warmup=100, step=1, bonds=0.5, age=15),
        # the benchmark's toric side lines: many samples of a basic RBM, in
        # the default precision and in that of the reference
        one("epoch_toric4_basic_fp32", "epoch", "toric", 4, "basic", 2, 32, "0.05", chains=4096, per_chain=64,
            warmup=100, step=1, bonds=0.5, age=15),
        one("epoch_toric4_basic_fp64", "epoch", "toric", 4, "basic", 2, 64, "0.05", chains=4096, per_chain=64,
            warmup=100, step=1, bonds=0.5, age=15),
        # the benchmark's Pfaffian line
        one("epoch_kitaev4_pfaffian_fp32", "epoch", "kitaev", 4, "pfaffian", 2, 32, "0.05", chains=8192, per_chain=8,
            warmup=100, step=1, bonds=0.5, age=15),
        # examples/toric4.ini as it stands, in the reference's precision: few
        # chains, where latency counts
        one("epoch_toric4_sym_small_fp64", "epoch", "toric", 4, "symmetry", 1, 64, "0.01", chains=64, per_chain=50,
            warmup=200, step=5, bonds=0.2, age=15),
        # examples/kitaev2_full.ini: the smallest whole step, an exact epoch
        # with the direct solver
        one("enumerate_kitaev2_sym_direct_fp64", "enumerate", "kitaev", 2, "symmetry", 4, 64, "0.05", solver="direct",
            age=15),
        # the largest lattice that the reference's tests diagonalise, exactly
        one("enumerate_kitaev3_basic_fp64", "enumerate", "kitaev", 3, "basic", 1, 64, "0.05", solver="cg", age=15),
        # an SR step on stored samples, symmetric on the explicit S and basic
        # matrix-free
        one("stored_kitaev6_sym_fp32", "stored", "kitaev", 6, "symmetry", 4, 32, "kitaev6_sym", samples=65536,
            solver="cg-single", age=15),
        one("stored_toric4_basic_fp64", "stored", "toric", 4, "basic", 2, 64, "0.05", samples=20000, solver="cg",
            age=15),
        # overlaps over many states, and a single batch of a few
        one("logpsi_kitaev6_sym_fp64", "logpsi", "kitaev", 6, "symmetry", 4, 64, "0.03", samples=65536),
        one("logpsi_kitaev4_basic_few_fp32", "logpsi", "kitaev", 4, "basic", 2, 32, "0.05", samples=37),
        # the benchmark's learned proposal on the reference's 2x2 example
        one("learned_kitaev2_sym_fp32", "learned", "kitaev", 2, "symmetry", 4, 32, "kitaev2_sym_ed", chains=256,
            per_chain=256, warmup=100, step=1, bonds=0.2, hidden=32, fraction=0.5),
    ]


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["epoch", "epoch", "epoch", "enumerate", "stored", "stored", "logpsi", "learned"])
    std = "%.3f" % math.exp(rng.uniform(math.log(0.01), math.log(0.06)))
    prec = rng.choice([32, 64])
    age = rng.randint(0, 20)
    model = rng.choice(["kitaev", "toric"])
    n = rng.randint(3, 6) if model == "kitaev" else rng.randint(3, 5)
    rbm = rng.choice(["basic", "symmetry"])
    alpha = rng.randint(1, 4) if rbm == "symmetry" else rng.randint(1, 2)
    if rbm == "basic":  # up to about 3000 parameters
        n = min(n, 5 if alpha == 1 else 4)
    if kind == "epoch":
        if rng.random() < 0.25:
            return case(kind, "kitaev", rng.choice([2, 3, 4]), "pfaffian", rng.randint(1, 2), prec, std,
                        chains=log_int(rng, 32, 2000), per_chain=rng.randint(2, 9), warmup=rng.randint(20, 100),
                        step=1, bonds=round(rng.uniform(0.0, 0.7), 2), age=age)
        if rbm == "symmetry" and alpha == 3 and prec == 32:
            alpha = 4
        chains = log_int(rng, 16, 4096)
        # the O matrix of a basic RBM in FP64 bounds the samples of a draw
        most = 60000 if rbm == "basic" else 120000
        per = max(1, min(rng.randint(2, 60), most // chains))
        return case(kind, model, n, rbm, alpha, prec, std, chains=chains, per_chain=per, warmup=rng.randint(20, 150),
                    step=rng.choice([1, 1, 2, 5]), bonds=round(rng.uniform(0.0, 0.7), 2), age=age)
    if kind == "enumerate":
        model, n = rng.choice([("kitaev", 2), ("kitaev", 3), ("toric", 2), ("toric", 3)])
        return case(kind, model, n, rbm, alpha, rng.choice([32, 64, 64]), std,
                    solver=rng.choice(["direct", "cg", "cg-single"]) if rbm == "symmetry" else "cg", age=age)
    if kind == "stored":
        return case(kind, model, n, rbm, alpha, prec, std, samples=log_int(rng, 200, 40000 if rbm == "symmetry" else 20000),
                    solver=rng.choice(["cg", "cg-single"]) if rbm == "symmetry" else "cg", age=age)
    if kind == "logpsi":
        return case(kind, model, n, rbm, alpha, prec, "%.3f" % min(float(std), 0.03 if n > 4 else 0.05),
                    samples=log_int(rng, 1, 100000))
    return case(kind, "kitaev", rng.choice([2, 3, 4]), rng.choice(["basic", "symmetry"]), rng.choice([1, 2, 4]), 32, std,
                chains=log_int(rng, 16, 512), per_chain=rng.randint(4, 64), warmup=rng.randint(20, 100), step=1,
                bonds=round(rng.uniform(0.0, 0.5), 2), hidden=rng.choice([16, 32, 64]),
                fraction=round(rng.uniform(0.1, 0.6), 2))


# ---------------------------------------------------------------- inputs
def symmetry(c):
    return 0.5 if c["model"] == "kitaev" else 1


def spec(c, seed):
    rbm = "basic" if c["rbm"] == "pfaffian" else c["rbm"]
    s = f"seed = {421390484 + seed}\n[model]\ntype = {c['model']}\nn_cells = {c['n']}\nJ = -1\n"
    s += f"symmetry = {symmetry(c)}\n[rbm]\ntype = {rbm}\nalpha = {c['alpha']}\n"
    if c["rbm"] == "pfaffian":
        s += "pfaffian = true\n"
    s += "[sampler]\n"
    if c["kind"] in ("epoch", "learned"):
        s += f"n_samples = {c['chains'] * c['per_chain']}\nmetropolis.n_chains = {c['chains']}\n"
        s += f"metropolis.n_warmup_steps = {c['warmup']}\nmetropolis.n_steps_per_sample = {c['step']}\n"
        s += f"metropolis.bond_flips = {c['bonds']}\npfaffian_refresh = 64\n"
    if c["kind"] == "enumerate":
        s += "type = full\n"
    if c.get("solver") == "cg-single":
        s += "[optimizer]\nsr.method = cg-single\n"
    if c["kind"] == "learned":
        s += f"[learn]\nhidden = {c['hidden']}\nfraction = {c['fraction']}\n"
    return s


def checkpoint(path):
    """a .rbm file's [v | h | W column-major]"""
    data = open(path, "rb").read()
    off, mats = 0, []
    for _ in range(3):
        r, k = np.frombuffer(data, dtype=np.uint64, count=2, offset=off)
        off += 16
        mats.append(np.frombuffer(data, dtype=np.complex128, count=int(r * k), offset=off))
        off += 16 * int(r * k)
    return np.concatenate([mats[2], mats[1], mats[0]])


def parameters(c, P, n_neural, seed):
    """N(0, std^2) weights as after initialisation, or a trained state's with
    a little noise; the Pfaffian weights as initialised (0.01 around 1 is
    what normalises a state, here N(0, 0.3^2))"""
    rng = np.random.default_rng([seed, 1])
    z = rng.normal(size=P) + 1j * rng.normal(size=P)
    if c["weights"] == "kitaev6_sym":
        return checkpoint(CHECKPOINT) + 1e-3 * z
    if c["weights"] == "kitaev2_sym_ed":
        return checkpoint(CHECKPOINT_ED2) + 1e-4 * z
    p = float(c["weights"]) * z
    p[n_neural:] = 0.3 * z[n_neural:]
    return p


def states_of(c, N, seed):
    n, words = c["samples"], (N + 63) // 64
    s = np.random.default_rng([seed, 2]).integers(0, 1 << 64, size=(n, words), dtype=np.uint64, endpoint=False)
    if N % 64:
        s[:, -1] &= np.uint64((1 << (N % 64)) - 1)
    return s


def regularisation(c):
    """reg1, reg2, their Pfaffian offset after `age` epochs of the defaults' decay"""
    return max(0.9 ** c["age"], 1e-4), max(1e-3 * 0.9 ** c["age"], 1e-6), 1e-2


def prepare(c, seed):
    m = rbmgpu.Model(spec(c, seed))
    # FP32 chains follow the launch shape's rounding: one chain per wavefront,
    # the sampler that the autotuner settles on, is asked for by name
    lanes = -1 if c["kind"] == "epoch" and c["precision"] == 32 and c["rbm"] != "pfaffian" else 0
    g = m.gpu(precision=c["precision"], lanes=lanes)
    p = parameters(c, m.P, m.n_neural, seed)
    g.set_params(p)
    s = {"case": c, "model": m, "gpu": g, "params": p, "epoch": 0}
    if c["kind"] == "epoch":  # a run that is under way: launch shape tuned, graph captured
        for _ in range(2):
            run(s)
    if c["kind"] in ("stored", "logpsi"):
        s["states"] = states_of(c, m.N, seed)
    if c["kind"] in ("stored", "enumerate"):
        s["x0"] = np.zeros(m.P, dtype=np.complex128)
    return s


# ---------------------------------------------------------------- one pass
def typed(c, v):
    """results in the precision that the context computes in"""
    if c["precision"] == 64:
        return v
    return {k: x.astype(np.complex64 if np.iscomplexobj(x) else np.float32) for k, x in v.items()}


def statistics(r):
    return np.array([r["mean"].real, r["mean"].imag, r["var"]]), np.array([r["var_binned"], r["tau"], r["std"]])


def solve(s, r):
    c, g = s["case"], s["gpu"]
    b = r["eo"] - r["mean"] * np.conj(r["o_mean"])
    method = {"cg": 0, "cg-single": 1, "direct": 2}[c["solver"]]
    return g.sr_solve_ex(method, b, s["x0"], *regularisation(c), max_iter=100)[0]


def run(s):
    c, g = s["case"], s["gpu"]
    s["epoch"] += 1
    if c["kind"] == "epoch":
        g.set_params(s["params"])
        r = g.train_epoch(s["epoch"], 1e-2, *regularisation(c), max_iter=100)
        energy, binned = statistics(r)
        return typed(c, {"energy": energy, "binned": binned, "acceptance": np.array([r["acc"]]),
                         "weights": g.get_params()})
    if c["kind"] == "logpsi":
        return typed(c, {"logpsi": g.eval_logpsi(s["states"])})
    if c["kind"] == "learned":
        g.sample_epoch(s["epoch"])
    elif c["kind"] == "enumerate":
        g.set_params(s["params"])
        g.full_epoch()
    else:
        g.load_samples(s["states"])
    r = g.reduce()
    energy, binned = statistics(r)
    out = {"energy": energy, "binned": binned, "o_mean": r["o_mean"], "o_var": r["o_var"], "eo": r["eo"]}
    if c["kind"] != "learned":
        out["x"] = solve(s, r)
    if c["kind"] == "stored":
        out["eloc"] = g.get_samples(states=False)[1][:, 0]
    return typed(c, out)


# ---------------------------------------------------------------- work
def sizes(c):
    """N, hidden units, parameters, |symmetry group|"""
    N = 2 * c["n"] ** 2
    if c["rbm"] == "symmetry":
        g = N if c["model"] == "kitaev" else N // 2
        na = c["alpha"] * (N // g)
        return N, na * g, N // g + na + na * N, g
    H = c["alpha"] * N
    P = N + H + H * N
    if c["rbm"] == "pfaffian":
        P += 4 * (N // 2 + N // 4 + 1)  # about one row of weights per translation class of site pairs
    return N, H, P, 1


def work(c):
    N, H, P, _ = sizes(c)
    real = 4 if c["precision"] == 32 else 8
    words = (N + 63) // 64
    if c["kind"] == "logpsi":
        # theta: a complex N x H product with +-1; ~40 operations of an ln cosh
        return {"bytes": c["samples"] * (8 * words + 16) + 16 * P, "flops": c["samples"] * H * (4 * N + 40)}
    if c["kind"] == "enumerate":
        S = 1 << N
    elif c["kind"] == "stored":
        S = c["samples"]
    else:
        S = c["chains"] * c["per_chain"]
    terms = N  # off-diagonal terms: 2 N / 2 bonds of x and y type, or N / 2 vertices of 4 flips
    flops = S * (terms * 16 * H)  # the local energies' ratios
    flops += 24 * S * P  # the moments and one product with S
    if c["kind"] in ("epoch", "learned"):
        b = c["bonds"]
        sweeps = c["chains"] * (c["warmup"] + c["per_chain"] * c["step"])
        flops += sweeps * N / (1 + b) * (24 * (1 - b) + 40 * b) * H
    else:
        flops += S * H * (4 * N + 40)
    # states in or out, the tanh rows that the SR products read, the parameters
    return {"bytes": S * (8 * words + 2 * real * H) + 32 * P, "flops": flops}


# ------------------------------------------------ the same in 64 bits, in torch
def lattice(c):
    """bonds (a, b, type) or plaquettes, and the symmetry permutations"""
    n = c["n"]

    def idx(i, j, b):
        return 2 * ((i % n) + n * (j % n)) + b

    cells = [(i, j) for j in range(n) for i in range(n)]
    if c["model"] == "kitaev":
        terms = []
        for i, j in cells:
            a = idx(i, j, 0)
            terms += [((a, idx(i, j, 1)), "x"), ((a, idx(i - 1, j, 1)), "y"), ((a, idx(i, j - 1, 1)), "z")]
    else:
        terms = []
        for i, j in cells:
            terms.append(((idx(i, j, 0), idx(i, j, 1), idx(i, j + 1, 0), idx(i + 1, j, 1)), "z"))
            terms.append(((idx(i, j, 0), idx(i, j, 1), idx(i - 1, j, 0), idx(i, j - 1, 1)), "x"))
    N = 2 * n * n
    if c["rbm"] != "symmetry":
        return terms, np.arange(N)[None, :], np.arange(N)
    perms = []
    for dj in range(n):
        for di in range(n):
            p = np.array([idx(i + di, j + dj, b) for i, j in cells for b in (0, 1)])
            perms.append(p)
            if c["model"] == "kitaev":
                perms.append(N - 1 - p)
    return terms, np.array(perms), np.array([0] if c["model"] == "kitaev" else [0, 1])


class Exact:
    """theta, local energies and O of the RBM for given spins, in 64 bits"""

    def __init__(self, c, seed):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        N, H, P, _ = sizes(c)
        self.c, self.N = c, N
        p = torch.from_numpy(np.ascontiguousarray(parameters(c, P, P, seed))).to(self.dev)
        self.terms, perms, basis = lattice(c)
        self.perm = torch.from_numpy(perms).to(self.dev)
        self.nsym, self.nvb = len(perms), len(basis)
        self.na = H // self.nsym
        self.v, self.h = p[: self.nvb], p[self.nvb: self.nvb + self.na]
        self.W = p[self.nvb + self.na:].reshape(self.na, N).T  # W[k, a]
        # units ordered (s, a): theta_{s,a} = h_a + sum_f sigma_f W[perm_s(f), a]
        self.Wf = self.W[self.perm]  # (s, f, a)
        self.images = self.perm[:, torch.from_numpy(basis).to(self.dev)]  # (s, i)
        self.lb = torch.zeros(N, dtype=torch.complex128, device=self.dev)
        for i in range(self.nvb):
            self.lb.index_add_(0, self.images[:, i], self.v[i].expand(self.nsym).contiguous())

    def theta(self, spins):
        A = self.Wf.permute(1, 0, 2).reshape(self.N, -1)
        return torch.complex(spins @ A.real.contiguous(), spins @ A.imag.contiguous()) + self.h.repeat(self.nsym)

    def logpsi(self, spins):
        th = self.theta(spins)
        return torch.complex(spins @ self.lb.real, spins @ self.lb.imag) + torch.log(torch.cosh(th)).sum(1)

    def energy(self, spins, th):
        t = torch.tanh(th)
        out = torch.zeros(len(spins), dtype=torch.complex128, device=self.dev)
        for sites, kind in self.terms:
            sg = spins[:, list(sites)]
            sign = sg.prod(1)
            if kind == "z":
                out -= sign
                continue
            d = torch.zeros_like(th)
            for q, f in enumerate(sites):
                d -= 2 * sg[:, q: q + 1] * self.Wf[:, f, :].reshape(1, -1)
            r = (torch.cosh(d) + t * torch.sinh(d)).prod(1)
            r = r * torch.exp(-2 * (sg.to(torch.complex128) @ self.lb[list(sites)]))
            out -= r * (-sign if kind == "y" else 1.0)
        return out

    def O(self, spins, th):
        t = torch.tanh(th).reshape(len(spins), self.nsym, self.na)
        sv = torch.stack([spins[:, self.images[:, i]].sum(1) for i in range(self.nvb)], 1).to(torch.complex128)
        w = torch.zeros(len(spins), self.na, self.N, dtype=torch.complex128, device=self.dev)
        for s in range(self.nsym):
            moved = torch.zeros_like(spins)
            moved[:, self.perm[s]] = spins  # (P_s sigma)_j
            w += t[:, s, :, None] * moved[:, None, :]
        return torch.cat([sv, t.sum(1), w.reshape(len(spins), -1)], 1)


def bits(words, N, dev):
    w = torch.from_numpy(words.astype(np.int64)).to(dev)
    s = torch.stack([(w[:, f // 64] >> (f % 64)) & 1 for f in range(N)], 1)
    return 1.0 - 2.0 * s.to(torch.float64)


def exact(c, seed):
    if c["kind"] in ("epoch", "learned"):
        return None  # random numbers of the sampler's own
    N, _, P, _ = sizes(c)
    e = Exact(c, seed)
    if c["kind"] == "logpsi":
        spins = bits(states_of(c, N, seed), N, e.dev)
        return {"logpsi": torch.cat([e.logpsi(x) for x in spins.split(8192)]).cpu().numpy()}
    if c["kind"] == "enumerate":
        spins = bits(np.arange(1 << N, dtype=np.uint64)[:, None], N, e.dev)
        lp = torch.cat([e.logpsi(x) for x in spins.split(8192)]).real
        w = torch.exp(2 * (lp - lp.max()))
    else:
        spins = bits(states_of(c, N, seed), N, e.dev)
        w = torch.ones(len(spins), dtype=torch.float64, device=e.dev)
    Ws, block = w.sum(), max(256, min(8192, (1 << 24) // P))
    E, mean, eo = [], 0, 0
    for x, wx in zip(spins.split(block), w.split(block)):
        th = e.theta(x)
        E.append(e.energy(x, th))
        O = e.O(x, th)
        mean = mean + (wx[:, None] * O).sum(0)
        eo = eo + ((wx * E[-1])[:, None] * O.conj()).sum(0)
    E, mean, eo = torch.cat(E), mean / Ws, eo / Ws
    em = (w * E).sum() / Ws
    den = Ws - (w * w).sum() / Ws
    var = (w * (E - em).abs() ** 2).sum() / den
    S = torch.zeros(P, P, dtype=torch.complex128, device=e.dev)
    for x, wx in zip(spins.split(block), w.split(block)):
        D = e.O(x, e.theta(x)) - mean
        S += D.conj().T.contiguous() @ (wx[:, None] * D)
    o_var = S.diagonal().real / den
    S = S / Ws
    r1, r2, _ = regularisation(c)
    if c["solver"] == "direct":
        A = S + torch.diag(r1 * S.diagonal() + r2 * o_var.max())
    else:
        A = S + torch.diag((r1 * o_var + r2 * o_var.max()).to(torch.complex128))
    b = eo - em * mean.conj()
    x = torch.linalg.solve(A.cpu(), b.cpu()).numpy()
    out = {"energy": np.array([em.real.item(), em.imag.item(), var.item()]), "binned": None,
           "o_mean": mean.cpu().numpy(), "o_var": o_var.cpu().numpy(), "eo": eo.cpu().numpy(), "x": x}
    if c["kind"] == "stored":
        out["eloc"] = E.cpu().numpy()
    return out
