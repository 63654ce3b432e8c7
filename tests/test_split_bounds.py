"""The bounds that the three-piece kernels' results are held to
(tests/split3_model.py) are tight enough to see a product of pieces that is
left out: a numpy model that leaves one out breaks each of them, and the whole
one stays far inside."""
import numpy as np
import pytest

import split3_model as sm
from neuralscript_amd import synth

LOST = sm.ALL[1:]


def normal(seed, *shape):
    return synth.normal(seed, int(np.prod(shape))).reshape(shape)


def without(lost):
    return tuple(p for p in sm.ALL if p != lost)


@pytest.mark.parametrize("K", [128, 512, 4096])
def test_normal_products(K):
    A, B = normal(K, 40, K), normal(K + 1, K, 40)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    assert sm.rel(sm.product(A, B), ref) < 0.2 * sm.normal_bound(K)
    for lost in LOST:
        assert sm.rel(sm.product(A, B, without(lost)), ref) > 2 * sm.normal_bound(K), lost


def test_one_term_products():
    rng = np.random.default_rng(1)
    a, b = ((1 + rng.random(4000)).astype(np.float32).reshape(-1, 1) for _ in range(2))
    a[0] = b[0] = float.fromhex("0x1.00ff8p+0")
    exact = a.astype(np.float64) * b

    def worst(keep):
        return max(abs(sm.product(x.reshape(1, 1), y.reshape(1, 1), keep)[0, 0] / e - 1)
                   for x, y, e in zip(a[:400], b[:400], exact[:400, 0]))
    assert 0.98 * sm.U < worst(sm.ALL) <= sm.U
    for lost in LOST:
        assert worst(without(lost)) > 2 * sm.one_term_bound(), lost


@pytest.mark.parametrize("dk", [32, 64, 128])
@pytest.mark.parametrize("lossy,outputs", [("s", (0, 1, 2, 3)), ("o", (0,)), ("dp", (1, 2)), ("dq", (1,)),
                                           ("dk", (2,)), ("dv", (3,))])
def test_attention(dk, lossy, outputs):
    arrs = [normal(dk + i, 130, dk) for i in range(4)]
    ref = sm.attention(*arrs)
    for lost in LOST:
        got = sm.attention(*arrs, lossy, without(lost))
        for i in outputs:
            assert sm.rel(got[i], ref[i]) > 1.5 * (sm.BACKWARD_BOUND if i else sm.FORWARD_BOUND), (lost, i)
