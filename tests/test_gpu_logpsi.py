"""log psi of given states on matrix tiles (k_logpsi) against the oracle,
through the C ABI: state counts around the 16 rows of a tile, sites that fill
the K steps of 4 or not, units that fill their tiles or not, weights in LDS and
in memory, two state words, and arguments that wrap many times (the sum of
principal arguments is returned, as the reference's sum of ln cosh).

Bounds as test_gpu_parity.py's: FP64 1e-10, FP32 2e-5, times (1 + |log psi|)."""
import numpy as np
import pytest

import pyoracle as po
import rbmgpu
from helpers import ini, random_params

pytestmark = pytest.mark.gpu

MODELS = [("kitaev", 2, "basic", 1), ("kitaev", 3, "basic", 1), ("kitaev", 3, "symmetry", 3), ("toric", 5, "symmetry", 2),
          ("kitaev", 6, "symmetry", 4), ("kitaev", 6, "basic", 2)]


@pytest.mark.parametrize("model,n,rbm,alpha", MODELS)
@pytest.mark.parametrize("prec,std", [(64, 0.1), (64, 0.7), (32, 0.05)])
def test_logpsi_tiles(model, n, rbm, alpha, prec, std):
    print(f"[gpu-test] logpsi {model} {n} {rbm} alpha={alpha} prec={prec} std={std}", flush=True)
    rng = np.random.default_rng(n * 10 + alpha)
    spec = ini(model, n, rbm=rbm, alpha=alpha)
    m, o = rbmgpu.Model(spec), po.Oracle(spec)
    p = random_params(rng, m.P, std)
    o.set_params(p)
    g = m.gpu(precision=prec)
    g.set_params(p)
    st = po.random_states(rng, 50, m.N)
    want = o.logpsi(st)
    tol = 1e-10 if prec == 64 else 2e-5
    for S in (1, 15, 16, 17, 50):
        got = g.eval_logpsi(st[:S])
        err = np.abs(got - want[:S])
        assert np.all(err <= tol * (1 + np.abs(want[:S]))), (S, err.max())


# 32 x 128 complex weights in FP64, 32 x 256 in FP32: 64 KiB, which with the
# kernel's own sums do not fit the 64 KiB of a launch without opting in
@pytest.mark.parametrize("alpha,prec", [(4, 64), (8, 32)])
def test_logpsi_tables_of_64_kib(alpha, prec):
    test_logpsi_tiles("toric", 4, "basic", alpha, prec, 0.05)
