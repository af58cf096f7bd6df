"""The FP64 sampler's acceptance (u against the group product of the lanes'
|p|^2 as mantissa and exponent, visible bias on u's side) and its moves,
against the oracle state for state: every group width with one and with
several units per lane, padded lanes, two state words, symmetric RBMs, and
visible biases and weights whose ratios span hundreds of binary orders.  E_loc
of the kept samples to 1e-10 of the largest, as in test_gpu_parity.py: it is
formed from tanh(theta) itself."""
import numpy as np
import pytest

import pyoracle as po
import rbmgpu
from helpers import ini, random_params

pytestmark = pytest.mark.gpu

MODELS = [("kitaev", 2, "basic", 1), ("toric", 4, "symmetry", 1), ("toric", 4, "basic", 2), ("kitaev", 6, "symmetry", 2)]


# 72 units: two per lane of a wavefront (9, 5 and 3 per lane are no launch shapes)
@pytest.mark.parametrize("model,n,rbm,alpha,lanes",
                         [(*m, lanes) for m in MODELS for lanes in (8, 16, 32, 64) if m[1] < 6 or lanes == 64])
@pytest.mark.parametrize("big", [False, True])
def test_accept_fp64(model, n, rbm, alpha, lanes, big):
    print(f"[gpu-test] accept {model}{n} {rbm} lanes={lanes} big={big}", flush=True)
    spec = ini(model, n, rbm=rbm, alpha=alpha, extra="[sampler]\nn_samples = 40\nmetropolis.n_chains = 10\n"
               "metropolis.n_warmup_steps = 6\nmetropolis.n_steps_per_sample = 2\nmetropolis.bond_flips = 0.4\n")
    m, o = rbmgpu.Model(spec), po.Oracle(spec)
    p = random_params(np.random.default_rng(11), m.P, 0.1)
    if big:  # |psi'/psi|^2 down to 2^-300 and up to 2^300
        p[: m.n_vb] *= 250
    o.set_params(p)
    g = m.gpu(precision=64, lanes=lanes)
    g.set_params(p)
    g.sample_epoch(epoch=3)
    assert g.launch_shape()[0] == lanes
    st, obs, _, _ = g.get_samples(states=True, obs=True, O=False)
    st_o, e_o, _, _ = o.sample(seed=421390484, epoch=3, n_samples=m.n_samples, n_chains=m.n_chains)
    assert np.array_equal(st, st_o)
    assert np.max(np.abs(obs[:, 0] - e_o)) <= 1e-10 * (np.abs(e_o).max() + 1)


# weights at which an incremental tanh loses its digits within a sweep
@pytest.mark.parametrize("model,n,rbm,alpha,std", [("toric", 4, "basic", 2, 1.5), ("toric", 4, "symmetry", 1, 2.0),
                                                   ("kitaev", 6, "symmetry", 2, 1.5), ("kitaev", 6, "symmetry", 2, 2.0)])
def test_large_weights_fp64(model, n, rbm, alpha, std):
    print(f"[gpu-test] large weights {model}{n} {rbm} std={std}", flush=True)
    spec = ini(model, n, rbm=rbm, alpha=alpha, extra="[sampler]\nn_samples = 960\nmetropolis.n_chains = 48\n"
               "metropolis.n_warmup_steps = 20\nmetropolis.bond_flips = 0.4\n")
    m, o = rbmgpu.Model(spec), po.Oracle(spec)
    p = random_params(np.random.default_rng(1), m.P, std)
    o.set_params(p)
    g = m.gpu(precision=64)
    g.set_params(p)
    g.sample_epoch(epoch=3)
    st_o, _, _, _ = o.sample(seed=421390484, epoch=3, n_samples=m.n_samples, n_chains=m.n_chains)
    assert np.array_equal(g.get_samples()[0], st_o)
