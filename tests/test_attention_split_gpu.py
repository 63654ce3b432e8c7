"""The attention core on three bf16 pieces: at the edges of its query and key
tiles against float64, and on the values the pieces cannot hold.

Bound: the core's results are averages (forward) or sums of S terms with
fp32-rounded probabilities; 2^-24 times a small multiple of sqrt(S) of the
largest value covers the roundings, where the tests above this file's allow
1e-5 + 1e-4 |ref|.
"""
import numpy as np
import pytest

from neuralscript_amd import runtime, synth
from neuralscript_amd.runtime import DeviceArray as DA

pytestmark = pytest.mark.gpu


def inputs(S, D, seed, n=3):
    return [synth.normal(seed + i, S * D).reshape(S, D) for i in range(n)]


def core(Q, K, V, H):
    S, D = Q.shape
    ctx, lse = DA(S * D), DA(S * H)
    runtime.op("attention_fwd", DA.from_host(Q), DA.from_host(K), DA.from_host(V), ctx, lse, S, D, H)
    return ctx.to_host().reshape(S, D), lse


def probabilities(Q, K, H, h):
    dk = Q.shape[1] // H
    c = slice(h * dk, (h + 1) * dk)
    with np.errstate(all="ignore"):
        s = Q[:, c].astype(np.float64) @ K[:, c].astype(np.float64).T / np.sqrt(np.float64(dk))
        p = np.exp(s - s.max(1, keepdims=True))
        return p / p.sum(1, keepdims=True), c


def reference(Q, K, V, H):
    out = np.zeros(Q.shape)
    for h in range(H):
        p, c = probabilities(Q, K, H, h)
        with np.errstate(all="ignore"):
            out[:, c] = p @ V[:, c].astype(np.float64)
    return out


def bar(S, ref):
    return 2.0 ** -24 * (16 + 2 * np.sqrt(S)) * np.max(np.abs(ref))


# one token, one short of and one past the key tile (32 or 64), the queries of
# a wave (32) and of a workgroup (256)
@pytest.mark.parametrize("S", [1, 31, 33, 63, 64, 65, 255, 257, 600])
@pytest.mark.parametrize("dk", [32, 64, 128])
def test_forward_tile_edges(S, dk):
    print(f"attention forward S={S} dk={dk}", flush=True)
    H = 2
    Q, K, V = inputs(S, H * dk, 31 * S + dk)
    got, _ = core(Q, K, V, H)
    ref = reference(Q, K, V, H)
    assert np.max(np.abs(got - ref)) <= bar(S, ref)


@pytest.mark.parametrize("dk", [32, 64, 128])
def test_forward_values_without_three_pieces(dk):
    """An infinite or NaN key, query or value reaches the rows it reaches in
    float64, and no other."""
    S, H = 300, 2
    base = inputs(S, H * dk, 5)
    for which, value in [(1, np.inf), (1, -np.inf), (1, np.nan), (0, np.inf), (2, np.inf), (2, np.nan), (2, 3.39e38)]:
        arrs = [a.copy() for a in base]
        arrs[which][7, 3] = value
        print(f"attention forward dk={dk} operand {which} = {value}", flush=True)
        got, _ = core(*arrs, H)
        ref = reference(*arrs, H)
        ok = np.isfinite(ref)
        assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isinf(got), np.isinf(ref))
        calm = ok & (np.abs(ref) < 1e3)
        assert np.max(np.abs(got[calm] - ref[calm])) <= bar(S, ref[calm])
        big = ok & ~calm
        assert np.all(np.abs(got[big] - ref[big]) <= 1e-5 * np.abs(ref[big]))


@pytest.mark.parametrize("scale", [2.0 ** -112, 2.0 ** -126, 2.0 ** 60])
def test_forward_values_of_any_magnitude(scale):
    S, H, dk = 100, 2, 64
    Q, K, V = inputs(S, H * dk, 9)
    V = (V * np.float32(scale)).astype(np.float32)
    got, _ = core(Q, K, V, H)
    ref = reference(Q, K, V, H)
    assert np.max(np.abs(got - ref)) <= bar(S, ref) + 2.0 ** -149 * S
