"""The Pfaffian sampler's register updates over long runs between fresh
inverses, against the oracle, through the C ABI: single flips only, bonds only
and mixed, N = 8, 18 and 32 (rows that fill the 32 lanes and rows that do
not).

  * FP64: the chains follow the oracle's state for state; E_loc to 1e-9 of the
    largest (the bound of test_gpu_pfaffian.py for a fresh inverse).
  * FP32, with a block of 8 chains and a ragged last one: E_loc of the kept
    states to 2e-3 of the largest, the bound of a fresh FP32 inverse, for all
    but 1 % of the samples (an update's error is that of the inverse times
    the inverse of the ratio, so a chain that has just passed a small |psi| may
    exceed it until its next fresh inverse).
"""
import numpy as np
import pytest

import pyoracle as po
import rbmgpu
from helpers import ini, random_params

pytestmark = pytest.mark.gpu


def setup(model, n, bonds, chains, per_chain, refresh, prec, std):
    print(f"[gpu-test] pf chains {model}{n} bonds={bonds} prec={prec}", flush=True)
    spec = ini(model, n, alpha=2, extra="pfaffian = true\n[sampler]\n"
               f"n_samples = {chains * per_chain}\nmetropolis.n_chains = {chains}\n"
               f"metropolis.n_warmup_steps = 12\nmetropolis.bond_flips = {bonds}\npfaffian_refresh = {refresh}\n")
    m, o = rbmgpu.Model(spec), po.Oracle(spec)
    p = random_params(np.random.default_rng(7), m.P, std)
    o.set_params(p)
    g = m.gpu(precision=prec)
    g.set_params(p)
    g.sample_epoch(epoch=1)
    return m, o, g


@pytest.mark.parametrize("bonds", [0.0, 0.5, 1.0])
@pytest.mark.parametrize("model,n", [("kitaev", 2), ("toric", 3), ("kitaev", 4)])
def test_pf_chains_fp64(model, n, bonds):
    m, o, g = setup(model, n, bonds, 12, 6, 64, 64, 0.1)
    st, obs, _, _ = g.get_samples(states=True, obs=True, O=False)
    st_o, e_o, _, _ = o.sample(seed=421390484, epoch=1, n_samples=m.n_samples, n_chains=m.n_chains)
    assert np.array_equal(st, st_o)
    assert np.max(np.abs(obs[:, 0] - e_o)) <= 1e-9 * (np.abs(e_o).max() + 1)


@pytest.mark.parametrize("bonds", [0.0, 0.5, 1.0])
@pytest.mark.parametrize("model,n", [("kitaev", 2), ("toric", 3), ("kitaev", 4)])
def test_pf_chains_fp32(model, n, bonds):
    m, o, g = setup(model, n, bonds, 2051, 1, 16, 32, 0.1)
    assert g.launch_shape()[2] == 512
    st, obs, _, _ = g.get_samples(states=True, obs=True, O=False)
    e = o.eloc(st)
    far = np.abs(obs[:, 0] - e) > 2e-3 * (np.abs(e).max() + 1)
    assert far.mean() <= 0.01, far.mean()
