"""Given states with the Pfaffian factor: log psi (without the inverse), local
energies and the Pfaffian part of O, on both sides of the line between the FP64
instances with one and with two wavefronts per SIMD (more than 1024 states and
LDS for them), with one to eight units per lane.

Bounds as in test_gpu_pfaffian.py: 1e-9 (energies and O, which go through the
inverse) and 1e-10 (log psi) of the largest in FP64, 2e-3 and 1e-4 in FP32."""
import numpy as np
import pytest

import pyoracle as po
import rbmgpu
from helpers import ini, random_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model,n,alpha", [("kitaev", 2, 1), ("toric", 3, 1), ("kitaev", 3, 3), ("kitaev", 2, 16),
                                           ("kitaev", 2, 32), ("kitaev", 2, 64), ("kitaev", 4, 1)])
@pytest.mark.parametrize("prec", [64, 32])
def test_pf_eval(model, n, alpha, prec):
    print(f"[gpu-test] pf eval {model} {n} alpha={alpha} prec={prec}", flush=True)
    rng = np.random.default_rng(n * 100 + alpha)
    spec = ini(model, n, alpha=alpha, extra="pfaffian = true\n")
    m, o = rbmgpu.Model(spec), po.Oracle(spec)
    p = random_params(rng, m.P, 0.1)
    p[m.n_neural:] = random_params(rng, m.P - m.n_neural, 0.5)
    o.set_params(p)
    g = m.gpu(precision=prec)
    g.set_params(p)
    st = po.random_states(rng, 40, m.N)
    e, O, lp = o.eloc(st), o.derivative(st), o.logpsi(st)
    tol, ltol = (1e-9, 1e-10) if prec == 64 else (2e-3, 1e-4)
    for S in (40, 1024, 1025):
        sets = np.resize(st, (S, st.shape[1]))
        got = g.eval_logpsi(sets)
        d = got - np.resize(lp, S)
        d = d.real + 1j * ((d.imag + np.pi) % (2 * np.pi) - np.pi)
        assert np.max(np.abs(d)) <= ltol * (1 + np.abs(lp).max()), S
        g.load_samples(sets)
        obs = g.get_samples()[1][:, 0]
        assert np.max(np.abs(obs - np.resize(e, S))) <= tol * (1 + np.abs(e).max()), S
        if g.structured():
            continue
        got_O = np.asarray(g.get_samples(O=True)[2])[:, :40]
        assert np.max(np.abs(got_O - O)) <= tol * np.abs(O).max(), S
