"""Stored FP32 sample sets through the wave sampler's tables (k_eval_wave)
against the oracle, through the C ABI: one unit per lane up to several, lanes
with padding units, two state words, basic (observables by k_eloc) and
symmetric RBMs, hexagon operators of six sites, and sample counts around one
block's wavefronts.  Bounds as in test_gpu_parity.py's FP32 cases: 1e-4 of the
largest local energy and O entry."""
import numpy as np
import pytest

import pyoracle as po
import rbmgpu
from helpers import ini, random_params

pytestmark = pytest.mark.gpu

MODELS = [("kitaev", 2, "symmetry", 1, ""), ("kitaev", 4, "symmetry", 4, ""), ("kitaev", 5, "symmetry", 2, ""),
          ("toric", 5, "symmetry", 4, ""), ("toric", 4, "basic", 3, ""), ("kitaev", 6, "basic", 1, ""),
          ("kitaev", 3, "symmetry", 4, "helper_strength = 0.2\n")]


@pytest.mark.parametrize("model,n,rbm,alpha,extra", MODELS)
@pytest.mark.parametrize("S", [1, 9, 700])
def test_eval_wave(model, n, rbm, alpha, extra, S):
    print(f"[gpu-test] eval_wave {model} {n} {rbm} alpha={alpha} {extra.strip()} S={S}", flush=True)
    rng = np.random.default_rng(n * 10 + alpha)
    spec = ini(model, n, rbm=rbm, alpha=alpha, extra="[model]\n" + extra if extra else "")
    m, o = rbmgpu.Model(spec), po.Oracle(spec)
    p = random_params(rng, m.P, 0.1)
    o.set_params(p)
    g = m.gpu(precision=32)
    g.set_params(p)
    st = po.random_states(rng, S, m.N)
    g.load_samples(st)
    e = o.eloc(st)
    got = g.get_samples(O=rbm == "symmetry")
    assert np.max(np.abs(got[1][:, 0] - e)) <= 1e-4 * (1 + np.abs(e).max())
    if rbm == "symmetry":
        O = o.derivative(st)
        assert np.max(np.abs(got[2] - O)) <= 1e-4 * np.abs(O).max()


# visible biases whose factor exp(-4 c) of a bond flip comes near FP32's limit
# (3.3e37 to 1.7e38): the energies, some 1e45, are within the doubles' range
@pytest.mark.parametrize("n,alpha", [(2, 4), (3, 2), (4, 2), (6, 1), (6, 4)])
@pytest.mark.parametrize("c", [21.8, -21.8, 22.0, -22.0, 22.15])
def test_eval_wave_large_visible_bias(n, alpha, c):
    print(f"[gpu-test] eval_wave kitaev {n} alpha={alpha} visible bias {c}", flush=True)
    rng = np.random.default_rng(3)
    spec = ini("kitaev", n, rbm="symmetry", alpha=alpha)
    m, o = rbmgpu.Model(spec), po.Oracle(spec)
    p = random_params(rng, m.P, 0.3)
    p[: m.n_vb] = c + 0.3j
    p = p.astype(np.complex64).astype(np.complex128)
    o.set_params(p)
    g = m.gpu(precision=32)
    g.set_params(p)
    st = po.random_states(np.random.default_rng(7), 64, m.N)
    g.load_samples(st)
    e, got = o.eloc(st), g.get_samples()[1][:, 0]
    assert np.all(np.isfinite(got))
    assert np.max(np.abs(got - e)) <= 1e-4 * np.abs(e).max()


# set sizes on both sides of the lines between the evaluations: groups of lanes
# below, the wave sampler's tables above
@pytest.mark.parametrize("model,n,rbm,alpha,extra,line",
                         [("toric", 3, "symmetry", 4, "", 16384), ("kitaev", 3, "symmetry", 2, "helper_strength = 0.2\n", 5120),
                          ("kitaev", 6, "symmetry", 1, "helper_strength = 0.2\n", 8192), ("toric", 4, "basic", 2, "", 5120),
                          ("kitaev", 4, "basic", 3, "", 4096), ("kitaev", 5, "basic", 2, "", 512),
                          ("kitaev", 4, "basic", 1, "helper_strength = 0.2\n", 8192)])
def test_eval_wave_lines(model, n, rbm, alpha, extra, line):
    print(f"[gpu-test] eval_wave line {model} {n} {rbm} alpha={alpha} {extra.strip()} {line}", flush=True)
    rng = np.random.default_rng(n * 10 + alpha)
    spec = ini(model, n, rbm=rbm, alpha=alpha, extra="[model]\n" + extra if extra else "")
    m, o = rbmgpu.Model(spec), po.Oracle(spec)
    p = random_params(rng, m.P, 0.1)
    o.set_params(p)
    g = m.gpu(precision=32)
    g.set_params(p)
    st = po.random_states(rng, 64, m.N)
    e = o.eloc(st)
    for S in (line - 1, line):
        g.load_samples(np.resize(st, (S, st.shape[1])))
        got = g.get_samples()[1][:, 0]
        assert np.max(np.abs(got - np.resize(e, S))) <= 1e-4 * (1 + np.abs(e).max()), S
