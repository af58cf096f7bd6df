"""Moments and S.x of basic RBMs whose O entries are formed from the tanh rows
and the state bits (k_sx_ofree, k_o_partial) against the oracle, through the
C ABI: spin counts that divide 128 and that do not, one and several pairs per
lane, 4- and 16-wave blocks, the Pfaffian block, sample counts around the rows
that a wave takes together.  The O matrix is built when it is read.

Bounds as in test_gpu_parity.py: 1e-10 of the largest entry in FP64 (sums of
at most 1500 terms of order 1), 1e-4 / 5e-4 in FP32."""
import numpy as np
import pytest

import pyoracle as po
import rbmgpu
from helpers import ini, random_params

pytestmark = pytest.mark.gpu

# (model, n_cells, alpha, extra): N = 2 n^2 spins, M = alpha N hidden units
SHAPES = [("kitaev", 2, 1, ""), ("kitaev", 2, 13, ""), ("kitaev", 3, 1, ""), ("toric", 3, 4, ""), ("toric", 4, 1, ""),
          ("toric", 4, 2, ""), ("kitaev", 5, 1, ""), ("kitaev", 2, 1, "pfaffian = true\n"),
          ("kitaev", 3, 2, "pfaffian = true\n"), ("kitaev", 4, 2, "pfaffian = true\n")]


@pytest.mark.parametrize("model,n,alpha,extra", SHAPES)
@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("S", [2, 33, 1500])
def test_ofree_moments_and_product(model, n, alpha, extra, prec, S):
    print(f"[gpu-test] ofree {model} {n} alpha={alpha} {extra.strip()} prec={prec} S={S}", flush=True)
    rng = np.random.default_rng(n * 100 + alpha)
    spec = ini(model, n, alpha=alpha, extra=extra)
    m, o = rbmgpu.Model(spec + "[gpu]\nkeep_o = true\n"), po.Oracle(spec)
    p = random_params(rng, m.P, 0.1)
    p[m.n_neural:] = random_params(rng, m.P - m.n_neural, 0.5)
    o.set_params(p)
    g = m.gpu(precision=prec)
    g.set_params(p)
    st = po.random_states(rng, S, m.N)
    g.load_samples(st)
    e, O = o.eloc(st), o.derivative(st)
    ref, got = o.aggregate(e, O), g.reduce()
    tol = 1e-10 if prec == 64 else 1e-4
    for k in ("o_mean", "o_var", "eo"):
        assert np.max(np.abs(got[k] - ref[k])) <= 10 * tol * (1 + np.abs(ref[k]).max()), k
    x = rng.normal(size=m.P) + 1j * rng.normal(size=m.P)
    y = g.apply_S(x, 0.9, 9e-4, 1e-2)
    want = po.apply_S(O, ref["o_mean"], ref["o_var"], 0.9, 9e-4, 1e-2, m.n_neural, x)
    assert np.max(np.abs(y - want)) <= (1e-10 if prec == 64 else 5e-4) * np.abs(want).max()
    assert np.max(np.abs(g.get_samples(O=True)[2] - O)) <= tol * np.abs(O).max()
    g.load_samples(st[: S // 2])  # a smaller set: O follows it
    assert np.max(np.abs(g.get_samples(O=True)[2] - O[:, : S // 2])) <= tol * np.abs(O).max()


# machines whose last pair of entries reaches past the last unit (N = 8 with 8,
# 16 and 24 units, 2 x 3 cells with 12), through more than one step of a block's waves
SMALL = [("toric", 2, 1, ""), ("kitaev", 2, 2, ""), ("toric", 2, 2, ""), ("kitaev", 2, 3, ""),
         ("kitaev", 2, 1, "[model]\nn_cells_b = 3\n")]


@pytest.mark.parametrize("model,n,alpha,extra", SMALL)
@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("S", [3, 37, 1501])
def test_ofree_past_the_last_unit(model, n, alpha, extra, prec, S):
    test_ofree_moments_and_product(model, n, alpha, extra, prec, S)
