"""Training of the learned proposal (lceq_mlp_collect, lceq_mlp_train) against
the same records, normalisation, permutation, gradient and Adam steps in numpy
with 64 bits: mini-batches of one block, of a few, of a number of blocks that
is no multiple of the reduction's group, of more than one group, and of every
record (a new permutation each step).

Bounds: a loss is a mean of single-precision values (about 1e-6 each).  An
Adam step moves a parameter by lr g / |g| early on, so a parameter is off by
lr times the relative error of its gradient: a hundredth for all but those
whose gradient is a near cancellation, and never more than twice the step."""
import os
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))


@pytest.mark.parametrize("shape,stride,batch,steps", [
    ((16, 16, 16), 1, 32, 6), ((16, 16, 16), 1, 96, 6), ((16, 16, 16), 1, 4096, 4),
    ((18, 10, 14), 3, 832, 5), ((24, 24, 16), 2, 2080, 6), ((24, 24, 16), 2, 4128, 3)])
def test_training_steps(shape, stride, batch, steps):
    from perf import cases
    print("training steps", shape, stride, batch, steps, flush=True)
    case = {"kind": "train", "lx": shape[0], "ly": shape[1], "lz": shape[2], "stride": stride,
            "steps": steps, "batch": batch}
    ref = cases.exact(case, 9)
    state = cases.prepare(case, 9)
    got = cases.run(state)
    np.testing.assert_allclose(got["higgs"], ref["higgs"], rtol=0, atol=1e-12)
    np.testing.assert_allclose(got["loss"], ref["loss"], rtol=2e-5)
    np.testing.assert_allclose(got["state"][5254:], ref["state"][5254:], rtol=1e-6, atol=1e-7)
    off = np.abs(got["state"][:5254] - ref["state"][:5254]) / (2e-3 * steps)
    print("parameters off, in steps: median %.1e 99%% %.1e max %.1e"
          % (np.median(off), np.quantile(off, 0.99), off.max()), flush=True)
    assert np.quantile(off, 0.99) < 1e-2 and off.max() < 2.0
    # the same again from the same weights: bit for bit, also without losses
    again = cases.run(cases.prepare(case, 9))
    assert np.array_equal(again["state"], got["state"])
    assert np.array_equal(again["loss"], got["loss"])
    mlp = state["mlp"]
    mlp.set_state(state["weights"])
    assert mlp._lib.lceq_mlp_train(mlp.h, steps, batch, 2e-3, 1, 1, None) == 0
    assert np.array_equal(mlp.get_state(), got["state"])


def test_losses_of_more_steps_than_one_download():
    """600 steps: the losses come in two downloads, the same as in two calls."""
    from perf import cases
    print("training losses over two downloads", flush=True)
    case = {"kind": "train", "lx": 8, "ly": 8, "lz": 8, "stride": 1, "steps": 600, "batch": 512}
    state = cases.prepare(case, 4)
    got = cases.run(state)
    mlp = state["mlp"]
    mlp.set_state(state["weights"])
    # every batch is all records, so a call's permutations are new ones of the
    # same records: only the order of the sums differs from the one call's
    a = np.concatenate([mlp.train(512, batch=512, lr=2e-3, seed=1), ])
    assert np.array_equal(a.astype(np.float32), got["loss"][:512])
    assert np.isfinite(got["loss"]).all() and (got["loss"] != 0).all()


def test_each_loss_is_that_of_its_step():
    """Losses at the end of the first download (512 steps), in the second and at its
    end: with batches of all records a step's loss is the mean over the records at
    the parameters before it, so that a call of one step from these parameters
    gives it again, up to the order of 512 single-precision terms in blocks of 32
    (32 x 2^-24 of their size, which 2e-5 of 1 + |loss| covers tenfold)."""
    from perf import cases
    print("losses of their steps", flush=True)
    case = {"kind": "train", "lx": 8, "ly": 8, "lz": 8, "stride": 1, "steps": 600, "batch": 512}
    state = cases.prepare(case, 4)
    loss = cases.run(state)["loss"]
    mlp = state["mlp"]
    for step in (0, 1, 511, 512, 513, 555, 599):
        mlp.set_state(state["weights"])
        first = mlp.train(step, batch=512, lr=2e-3, seed=1)
        assert np.array_equal(first.astype(np.float32), loss[:step])
        again = mlp.train(1, batch=512, lr=2e-3, seed=1)[0]
        assert abs(again - loss[step]) <= 2e-5 * (1.0 + abs(again)), step
    # a loss of the first download in the place of one of the second would not pass
    assert np.abs(loss[512:] - loss[:88]).min() > 1e-3
