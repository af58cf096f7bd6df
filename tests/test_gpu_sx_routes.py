"""S.x of basic RBMs over the O matrix and with O's entries formed from the tanh
rows (k_sx_partial, k_sx_ofree): the same products and sums in the same order,
so the same bits -- an ill-conditioned solve amplifies a change of rounding.

The product is taken before and after O is read; on sets as small as these the
second product goes over O.  Spin counts that divide 128 and that do not, 4- and
16-wave blocks, one to several pairs per lane, the Pfaffian block, sets around
the rows that a wave takes together, and weighted sets.  Solves and training
epochs run over O on such sets: against the same solve on the explicit S."""
import numpy as np
import pytest

import pyoracle as po
import rbmgpu
from helpers import ini, random_params

pytestmark = pytest.mark.gpu

SHAPES = [("kitaev", 2, 1, ""), ("kitaev", 2, 3, ""), ("kitaev", 2, 13, ""), ("kitaev", 3, 1, ""), ("toric", 3, 4, ""),
          ("kitaev", 5, 1, ""), ("kitaev", 2, 1, "pfaffian = true\n"), ("kitaev", 2, 4, "pfaffian = true\n"),
          ("kitaev", 3, 2, "pfaffian = true\n"), ("kitaev", 4, 2, "pfaffian = true\n"),
          ("kitaev", 2, 1, "[model]\nn_cells_b = 3\n")]


def setup(model, n, alpha, extra, prec, rest=""):
    rng = np.random.default_rng(n * 100 + alpha)
    m = rbmgpu.Model(ini(model, n, alpha=alpha, extra=extra) + "[gpu]\nkeep_o = true\n" + rest)
    p = random_params(rng, m.P, 0.1)
    p[m.n_neural:] = random_params(rng, m.P - m.n_neural, 0.5)
    g = m.gpu(precision=prec)
    g.set_params(p)
    return m, g, rng, p


@pytest.mark.parametrize("model,n,alpha,extra", SHAPES)
@pytest.mark.parametrize("prec", [64, 32])
def test_same_bits(model, n, alpha, extra, prec):
    print(f"[gpu-test] sx routes {model} {n} alpha={alpha} {extra.strip()} prec={prec}", flush=True)
    m, g, rng, _ = setup(model, n, alpha, extra, prec)
    x = random_params(rng, m.P, 1.0)
    for S in (1, 3, 33, 700, 1501):
        g.load_samples(po.random_states(rng, S, m.N))
        formed = g.apply_S(x, 0.9, 9e-4, 1e-2)
        g.get_samples(O=True)
        assert np.array_equal(g.apply_S(x, 0.9, 9e-4, 1e-2), formed), S
    if m.N <= 8:
        g.full_epoch()
        formed = g.apply_S(x, 0.9, 9e-4, 1e-2)
        g.get_samples(O=True)
        assert np.array_equal(g.apply_S(x, 0.9, 9e-4, 1e-2), formed)


@pytest.mark.parametrize("model,n,alpha,extra", [("kitaev", 2, 2, ""), ("kitaev", 3, 1, ""), ("kitaev", 2, 1, "pfaffian = true\n"),
                                                 ("kitaev", 3, 2, "pfaffian = true\n")])
@pytest.mark.parametrize("prec", [64, 32])
def test_solve_over_O(model, n, alpha, extra, prec):
    """one CG step on a set that grows and shrinks, matrix-free against the
    explicit S: 1e-9 (FP64) and 1e-3 (FP32) of the largest entry"""
    print(f"[gpu-test] solve over O {model} {n} alpha={alpha} {extra.strip()} prec={prec}", flush=True)
    m, g, rng, _ = setup(model, n, alpha, extra, prec)
    b, x0 = random_params(rng, m.P, 1.0), np.zeros(m.P, dtype=complex)
    for S in (40, 900, 40):
        g.load_samples(po.random_states(rng, S, m.N))
        free = g.sr_solve_ex(0, b, x0, 0.9, 9e-4, 1e-2, max_iter=3)[0]
        dense = g.sr_solve_ex(1, b, x0, 0.9, 9e-4, 1e-2, max_iter=3)[0]
        assert np.max(np.abs(free - dense)) <= (1e-9 if prec == 64 else 1e-3) * np.abs(dense).max(), S


@pytest.mark.parametrize("model,n,alpha,extra", [("kitaev", 2, 2, ""), ("kitaev", 3, 1, "pfaffian = true\n")])
@pytest.mark.parametrize("prec", [64, 32])
def test_graph_over_O(model, n, alpha, extra, prec):
    """captured epochs hold O: a larger set in between moves it, and the epochs
    that follow are those of an eager context, bit for bit"""
    print(f"[gpu-test] graph over O {model} {n} alpha={alpha} {extra.strip()} prec={prec}", flush=True)
    rest = "explicit_s = false\n[sampler]\nn_samples = 640\nmetropolis.n_chains = 64\nmetropolis.n_warmup_steps = 10\n"
    out = []
    for graph in (True, False):
        m, g, rng, p = setup(model, n, alpha, extra, prec, rest)
        big = po.random_states(rng, 3000, m.N)
        for e in range(1, 7):
            r = g.train_epoch(e, 1e-2, 0.1, 1e-4, 0.0, max_iter=20, graph=graph)
            if e == 3:
                g.load_samples(big)
                g.get_samples(O=True)
            if e == 5:
                g.load_samples(big[:100])
                g.sr_solve_ex(0, p, np.zeros(m.P, dtype=complex), 0.1, 1e-4, 0.0, max_iter=5)
        out.append((g.get_params(), r["mean"], g.get_samples(O=True)[2]))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
