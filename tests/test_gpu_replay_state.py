"""Training epochs replayed from their graph after the context held another
sample set: what follows the replay (CG iterations past the captured count, the
moments, the sample set that can be read) has to be that of the epoch's samples,
as it is when every epoch runs eagerly.

Epochs 1 and 2 stop their CG at once (loose rtol), so the graph holds 8
iterations; epoch 3 needs more.  Between them a smaller set is loaded, or all
states are enumerated (a weighted set).  Both contexts run the same kernels on
the same inputs: equal bits."""
import numpy as np
import pytest

import pyoracle as po
import rbmgpu
from helpers import ini, random_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rbm,prec,explicit", [("basic", 64, "false"), ("basic", 64, "true"), ("basic", 32, "false"),
                                               ("symmetry", 64, "false"), ("symmetry", 32, "true")])
@pytest.mark.parametrize("between", ["load", "full"])
def test_replay_after_another_set(rbm, prec, explicit, between):
    print(f"[gpu-test] replay after {between}: {rbm} prec={prec} explicit={explicit}", flush=True)
    if between == "full" and rbm == "basic" and prec == 32:
        keep = "keep_o = true\n"
    else:
        keep = ""
    spec = ini("kitaev", 2, rbm=rbm, alpha=4, extra="[sampler]\nn_samples = 4096\nmetropolis.n_chains = 256\n"
               f"metropolis.n_warmup_steps = 10\n[gpu]\nexplicit_s = {explicit}\n{keep}")
    m = rbmgpu.Model(spec)
    p = random_params(np.random.default_rng(8), m.P, 0.1)
    few = po.random_states(np.random.default_rng(9), 37, m.N)
    out = []
    for graph in (True, False):
        g = m.gpu(precision=prec, lanes=64)
        g.set_params(p)

        def other():
            if between == "load":
                g.load_samples(few)
            else:
                g.full_epoch()
            g.apply_S(p, 0.1, 1e-4, 0.0)

        other()  # every buffer is there before the graph: it is not captured again
        for e in (1, 2):
            r = g.train_epoch(e, 1e-2, 0.1, 1e-4, 0.0, max_iter=100, rtol=1e6, graph=graph)
            assert r["itn"] < 6
        other()
        r = g.train_epoch(3, 1e-2, 0.1, 1e-4, 0.0, max_iter=100, graph=graph)
        assert r["itn"] > 8 and r["graph"] == graph
        assert g.n_samples() == 4096
        st, obs, _, acc = g.get_samples(chain_acc=True)
        q = g.reduce()
        y = g.apply_S(p, 0.1, 1e-4, 0.0)
        out.append((g.get_params(), r["mean"], r["n_bins"], st, obs, acc, q["mean"], q["o_mean"], y))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_reading_O_keeps_the_graph():
    """O of a basic FP64 machine is built when it is read.  Its buffer is not in
    the captured epoch, so reading it must not cost the graph: a replay records
    no timing events, and kernel_times shows those of the last eager epoch."""
    print("[gpu-test] reading O between replays", flush=True)
    m = rbmgpu.Model(ini("toric", 3, alpha=2, extra="[sampler]\nn_samples = 2000\nmetropolis.n_chains = 100\n"
                         "metropolis.n_warmup_steps = 10\n[gpu]\nexplicit_s = false\n"))
    g = m.gpu(precision=64, lanes=64)
    g.set_params(random_params(np.random.default_rng(8), m.P, 0.05))

    def epoch(e):
        g.train_epoch(e, 1e-3, 0.1, 1e-4, 0.0, max_iter=8)
        g.reduce()
        return g.kernel_times()

    epoch(1)
    before = epoch(2)
    O = g.get_samples(O=True)[2]
    assert np.abs(O).max() > 0
    after = epoch(3)
    # (the same two events: the conversion of their ticks drifts by some 1e-6)
    assert abs(after["sample"] - before["sample"]) <= 1e-5 * before["sample"]
