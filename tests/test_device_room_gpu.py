"""A model with little room on the device: what it can do without (the stored
dS of attention's backward, split-K partial sums) is not taken, or given back
when something else needs the room.  The room is limited by
NSHIP_MODEL_BUFFER_BYTES, which a model reads when it is made."""
import numpy as np
import pytest

import helpers
import oracle
from neuralscript_amd import runtime

pytestmark = pytest.mark.gpu

NAME, ROWS, SEED = "c5s", 500, 31   # 8 heads: dS is 8 x 500 x 512 floats
DS_BYTES = 8 * ROWS * 512 * 4
GRADS = {"g24": ROWS * 64, "g25": 4096, "g26": 4096, "g27": 4096, "g28": 4096}  # attention's x, wq, wk, wv, wo
STEP = 1 << 14                      # bytes to which a limit is searched


@pytest.fixture
def case(monkeypatch):
    net = oracle.Net(helpers.ir_text(NAME))
    w, plan = helpers.net_weights(NAME, SEED), runtime.Plan.load(NAME)
    x, y = helpers.net_inputs(net, NAME, SEED, ROWS), helpers.net_labels(net, SEED, ROWS)

    def step(limit):
        """A model after a step (lr 0) and its attention gradients; None without room for it."""
        if limit is None:
            monkeypatch.delenv("NSHIP_MODEL_BUFFER_BYTES", raising=False)
        else:
            monkeypatch.setenv("NSHIP_MODEL_BUFFER_BYTES", str(limit))
        m = runtime.Model(plan, w)
        try:
            m.train_step(x, y, 0.0)
        except runtime.NshipError as e:
            assert "out of memory" in str(e)
            m.free()
            return None
        return m, {g: m.read_value(g, n) for g, n in GRADS.items()}

    def least(ok):
        lo, hi = 0, 1 << 27
        while hi - lo > STEP:
            mid = (lo + hi) // 2
            lo, hi = (lo, mid) if ok(step(mid)) else (mid, hi)
        return hi

    return net, step, least


def same(a, b):
    return all(helpers.bitwise_equal(a[g], b[g]) for g in GRADS)


def test_training_with_room_for_less_and_less(case):
    net, step, least = case
    m, want = step(None)
    with_ds = least(lambda r: r is not None and same(r[1], want))
    without = least(lambda r: r is not None)
    print(f"room: {with_ds} with dS, {without} without", flush=True)
    assert with_ds - without > DS_BYTES / 2
    got = step(without)
    assert not same(got[1], want)  # (dQ from S and dP again, other roundings)
    for g in GRADS:
        helpers.assert_close(got[1][g], want[g], f"{g} without room for dS")
    # dS is held after a step that has just room for it; a longer call takes its place
    held, _ = step(with_ds)
    long = helpers.net_inputs(net, NAME, SEED + 1, 2 * ROWS)
    out = held.eval_infer(long)
    helpers.assert_close(out, m.eval_infer(long), "the longer call")
    # and the next step runs without it
    x, y = helpers.net_inputs(net, NAME, SEED, ROWS), helpers.net_labels(net, SEED, ROWS)
    held.train_step(x, y, 0.0)
    after = {g: held.read_value(g, n) for g, n in GRADS.items()}
    assert not same(after, want)
    for g in GRADS:
        helpers.assert_close(after[g], want[g], f"{g} after a longer call")
