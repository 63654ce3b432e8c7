"""The attention core on three bf16 pieces: at the edges of its query and key
tiles against float64, and on the values the pieces cannot hold.

Bound: the core's results are averages (forward) or sums of S terms with
fp32-rounded probabilities; 2^-24 times a small multiple of sqrt(S) of the
largest value covers the roundings, where the tests above this file's allow
1e-5 + 1e-4 |ref|.
"""
import numpy as np
import pytest

import split3_model as sm
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


def gradients(Q, K, V, dO, H, store_ds=1):
    S, D = Q.shape
    gQ, gK, gV, gdO = (DA.from_host(a) for a in (Q, K, V, dO))
    ctx, lse = DA(S * D), DA(S * H)
    runtime.op("attention_fwd", gQ, gK, gV, ctx, lse, S, D, H)
    out = [DA(S * D) for _ in range(3)]
    nb = runtime.lib().nsh_op_attention_bwd_workspace(S, D, H, store_ds)
    ws = DA.from_host(np.full(nb // 4 + 1, np.nan, np.float32))  # what the pass leaves unwritten must not be read
    runtime.op("attention_bwd", gQ, gK, gV, ctx, gdO, lse, *out, S, D, H, store_ds, ws)
    return [o.to_host().reshape(S, D) for o in out]


def reference_gradients(Q, K, V, dO, H):
    Q, K, V, dO = (a.astype(np.float64) for a in (Q, K, V, dO))
    dQ, dK, dV = (np.zeros(Q.shape) for _ in range(3))
    sc = 1.0 / np.sqrt(np.float64(Q.shape[1] // H))
    for h in range(H):
        p, c = probabilities(Q, K, H, h)
        with np.errstate(all="ignore"):
            dV[:, c] = p.T @ dO[:, c]
            dp = dO[:, c] @ V[:, c].T
            ds = p * (dp - np.sum(p * dp, axis=1, keepdims=True))
            dQ[:, c], dK[:, c] = ds @ K[:, c] * sc, ds.T @ Q[:, c] * sc
    return dQ, dK, dV


def gradient_bounds(Q, K, V, dO, H):
    """The same sums over absolute values, dP - rowsum(P dP) as |dP| +
    rowsum(P |dP|) (it may cancel): a score's error is at most 2^-24 (6 dk / 16
    + 8) |q| |k| / sqrt(dk), which a probability takes over relatively, and
    every later sum adds less than that again."""
    Q, K, V, dO = (np.abs(a.astype(np.float64)) for a in (Q, K, V, dO))
    dk = Q.shape[1] // H
    return Q, K, V, dO, 2.0 ** -24 * (6 * dk / 16 + 8) * np.sqrt(dk), 1.0 / np.sqrt(np.float64(dk))


def assert_gradients(arrs, H, got):
    Qa, Ka, Va, dOa, unit, sc = gradient_bounds(*arrs, H)
    refs = reference_gradients(*arrs, H)
    for h in range(H):
        p, c = probabilities(arrs[0], arrs[1], H, h)
        dp = dOa[:, c] @ Va[:, c].T
        ds = p * (dp + np.sum(p * dp, axis=1, keepdims=True)) * sc
        for g, r, most in zip(got, refs, (ds @ Ka[:, c], ds.T @ Qa[:, c], p.T @ dOa[:, c])):
            assert np.all(np.abs(g[:, c] - r[:, c]) <= unit * most)


# one short of and one past the query tile (32), the dQ pass's key tile (64)
# and a workgroup's keys (128); with and without the stored dS
@pytest.mark.parametrize("S", [1, 31, 33, 63, 65, 127, 129, 300])
@pytest.mark.parametrize("dk", [32, 64, 128])
@pytest.mark.parametrize("store_ds", [0, 1])
def test_gradient_tile_edges(S, dk, store_ds):
    print(f"attention gradients S={S} dk={dk} store_ds={store_ds}", flush=True)
    H = 2
    arrs = inputs(S, H * dk, 17 * S + dk, 4)
    assert_gradients(arrs, H, gradients(*arrs, H, store_ds))


@pytest.mark.parametrize("S", [64, 130, 500])
@pytest.mark.parametrize("dk", [32, 64, 128])
@pytest.mark.parametrize("store_ds", [0, 1])
def test_every_piece_counts(S, dk, store_ds):
    """The bounds that a lost product of pieces breaks (test_split_bounds.py)."""
    print(f"precise attention S={S} dk={dk} store_ds={store_ds}", flush=True)
    arrs = inputs(S, dk, 7 * S + dk, 4)
    refs = sm.attention(*arrs)
    assert sm.rel(core(*arrs[:3], 1)[0], refs[0]) <= sm.FORWARD_BOUND
    for name, g, r in zip(("dQ", "dK", "dV"), gradients(*arrs, 1, store_ds), refs[1:]):
        assert sm.rel(g, r) <= sm.BACKWARD_BOUND, name


@pytest.mark.parametrize("dk", [32, 64])
def test_gradients_of_values_without_three_pieces(dk):
    """A value near fp32's largest, an infinite one or a NaN in one row: where
    float64's gradients are finite the results follow them, where they are
    not the results are not finite either."""
    S, H = 200, 2
    base = inputs(S, H * dk, 3, 4)
    for which, value in [(3, 3.39e38), (3, np.inf), (3, np.nan), (2, np.nan)]:
        arrs = [a.copy() for a in base]
        arrs[which][9, 2] = value
        print(f"attention gradients dk={dk} operand {which} = {value}", flush=True)
        got, ref = gradients(*arrs, H), reference_gradients(*arrs, H)
        other = slice(dk, 2 * dk)  # the second head holds no special value
        clean = reference_gradients(*base, H)
        for g, r, c in zip(got, ref, clean):
            assert np.max(np.abs(g[:, other] - c[:, other])) <= bar(S, c[:, other])
            assert not np.any(np.isfinite(g[:, :dk][~np.isfinite(r[:, :dk])]) &
                              (np.abs(g[:, :dk][~np.isfinite(r[:, :dk])]) < 1e30))


def error_norms(got, refs):
    return [np.linalg.norm(g.astype(np.float64) - r) for g, r in zip(got, refs)]


# from full-size gradients down to where the operand itself is subnormal
@pytest.mark.parametrize("exponent", [-90, -100, -108, -115, -126])
@pytest.mark.parametrize("dk", [32, 64, 128])
@pytest.mark.parametrize("store_ds", [0, 1])
@pytest.mark.parametrize("which", [2, 3])
def test_gradients_of_any_magnitude(exponent, dk, store_ds, which):
    """V or dO times a power of two, which is exact: the gradients it enters
    scale with it and their errors may only scale with them (a quarter is left
    to the other rounding of the fp32 loop, which one subnormal operand sends a
    workgroup to), besides what fp32 has no bits for: 2^-149 a product, over S
    products and the row of dS that each comes from."""
    print(f"attention gradients dk={dk} store_ds={store_ds} operand {which} * 2^{exponent}", flush=True)
    S, H = 200, 2
    arrs = inputs(S, H * dk, 41, 4)
    base = error_norms(gradients(*arrs, H, store_ds), reference_gradients(*arrs, H))
    f = 2.0 ** exponent
    arrs[which] = (arrs[which] * np.float32(f)).astype(np.float32)
    refs = reference_gradients(*arrs, H)
    errs = error_norms(gradients(*arrs, H, store_ds), refs)
    least = 2.0 ** -149 * 4 * S * np.sqrt(S * H * dk)
    for name, e, b, unscaled in zip(("dQ", "dK", "dV"), errs, base, (False, False, which == 2)):
        assert e <= 1.25 * b * (1.0 if unscaled else f) + least, name


@pytest.mark.parametrize("dk", [32, 64, 128])
def test_output_of_a_lone_small_probability(dk):
    """Only one key has a value, and its score lies 85 to 86 below the others':
    the output is that value times a probability of about 2^-123, of which
    unscaled bf16 pieces would keep 11 bits."""
    S, H = 130, 1
    rng = np.random.default_rng(dk)
    Q, K, V = (np.zeros((S, dk), np.float32) for _ in range(3))
    Q[:, 0] = np.sqrt(np.float32(dk)) * (8.5 + 0.1 * rng.random(S)).astype(np.float32)
    K[77, 0] = -10.0
    V[77] = 2.0 ** 30 * (1 + rng.random(dk)).astype(np.float32)
    got, _ = core(Q, K, V, H)
    ref = reference(Q, K, V, H)
    # the exponential's argument, 123 in log2 units, is rounded three times
    # (query, score, difference) to 2^-24 of itself; the sums as bar()
    bound = 3 * 124 * np.log(2) * 2.0 ** -24 + 2.0 ** -24 * (16 + 2 * np.sqrt(S))
    assert np.max(np.abs(got / ref - 1)) <= bound


def test_rows_too_wide_for_the_tile_offsets():
    """Rows of 2^24 floats and more: a tile's 32-bit offsets cannot reach its
    last row, so the heads run in groups on copies.  The columns repeat 1024
    heads 528 times; every repetition equals those 1024 heads alone."""
    S, dk, H, reps = 64, 32, 1024, 528
    D = H * dk
    assert (S - 1) * D * reps * 4 >= 2 ** 32
    print(f"attention of {reps * H} heads", flush=True)

    def run(Q, K, V, dO, heads, want=None):
        n = Q.shape[1]
        q, k, v, do = (DA.from_host(a) for a in (Q, K, V, dO))
        ctx, lse = DA(S * n), DA(S * heads)
        runtime.op("attention_fwd", q, k, v, ctx, lse, S, n, heads)
        grads = [DA(S * n) for _ in range(3)]
        ws = DA(runtime.lib().nsh_op_attention_bwd_workspace(S, n, heads, 1) // 4)
        runtime.op("attention_bwd", q, k, v, ctx, do, lse, *grads, S, n, heads, 1, ws)
        out = []
        for i, a in enumerate([ctx, *grads]):
            a = a.to_host().reshape(S, n)
            out.append(a if want is None else
                       all(np.array_equal(a[:, j:j + D], want[i]) for j in range(0, n, D)))
        for a in (q, k, v, do, ctx, lse, ws, *grads):
            a.free()
        return out

    base = inputs(S, D, 77, 4)
    want = run(*base, H)
    assert all(run(*(np.tile(a, (1, reps)) for a in base), reps * H, want))
