"""A sample set whose O matrix does not fit the card: the call that needs O
fails, and the context goes on.  A later, smaller set must get buffers of its
own (not the null pointers that the failed allocation left), and the error must
not be reported again by a later call.

12 million samples of toric 4x4 with 64 hidden units in FP64: 13 GB of states,
tanh rows and observables, 412 GB of O."""
import numpy as np
import pytest

import pyoracle as po
import rbmgpu
from helpers import ini, random_params

pytestmark = pytest.mark.gpu


def test_o_matrix_too_large():
    print("[gpu-test] O of 12 million samples refused", flush=True)
    rng = np.random.default_rng(4)
    spec = ini("toric", 4, alpha=2)
    m, o = rbmgpu.Model(spec), po.Oracle(spec)
    p = random_params(rng, m.P, 0.05)
    o.set_params(p)
    g = m.gpu(precision=64)
    g.set_params(p)
    few = po.random_states(rng, 20, m.N)
    g.load_samples(few)
    g.get_samples(O=True)
    g.load_samples(np.tile(few, (600000, 1)))
    g.reduce()
    with pytest.raises(RuntimeError, match="memory"):
        g.build_S(0.9, 9e-4, 1e-2)
    g.load_samples(few[:10])
    O = o.derivative(few[:10])
    assert np.max(np.abs(g.get_samples(O=True)[2] - O)) <= 1e-10 * np.abs(O).max()
    r = g.reduce()
    ref = o.aggregate(o.eloc(few[:10]), O)
    assert np.max(np.abs(r["o_mean"] - ref["o_mean"])) <= 1e-10 * (1 + np.abs(ref["o_mean"]).max())


def test_set_too_large_leaves_no_set():
    print("[gpu-test] 80 million samples refused", flush=True)
    # symmetric Kitaev 4x4 alpha = 4 in FP64: 164 GB of tanh rows, then 172 GB of O
    m = rbmgpu.Model(ini("kitaev", 4, rbm="symmetry", alpha=4))
    g = m.gpu(precision=64)
    g.set_params(random_params(np.random.default_rng(5), m.P, 0.05))
    few = po.random_states(np.random.default_rng(6), 16, m.N)
    g.load_samples(few)
    want = g.reduce()
    with pytest.raises(RuntimeError, match="memory"):
        g.load_samples(np.tile(few, (5000000, 1)))
    assert g.n_samples() == 0
    with pytest.raises(RuntimeError, match="no samples"):
        g.reduce()
    g.load_samples(few)
    got = g.reduce()
    assert got["mean"] == want["mean"] and np.array_equal(got["eo"], want["eo"])
