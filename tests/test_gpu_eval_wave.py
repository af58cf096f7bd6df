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
