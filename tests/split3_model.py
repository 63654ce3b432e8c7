"""Three-piece bf16 products (neuralscript_amd/csrc/split3.h) in numpy: what
the kernels keep of a product, with sums in float64, and the bounds that their
results are held to.  A product left out breaks each bound (test_split_bounds.py)."""
import numpy as np

U = 2.0 ** -24
ALL = ((0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0))  # piece of A, piece of B


def bf16(x):
    """fp32 values rounded to nearest even bf16 (finite, no overflow)."""
    b = np.asarray(x, np.float32).view(np.uint32)
    return ((b + (0x7FFF + ((b >> 16) & 1)).astype(np.uint32)) & np.uint32(0xFFFF0000)).view(np.float32)


def pieces(x):
    x = np.ascontiguousarray(x, np.float32)
    a0 = bf16(x)
    a1 = bf16(x - a0)
    return a0, a1, (x - a0) - a1


def product(A, B, keep=ALL):
    """A . B of the piece products `keep`, in float64."""
    a, b = [p.astype(np.float64) for p in pieces(A)], [p.astype(np.float64) for p in pieces(B)]
    return sum(a[i] @ b[j] for i, j in keep)


def rel(got, ref):
    return np.linalg.norm(np.asarray(got, np.float64) - ref) / np.linalg.norm(ref)


def one_term_bound():
    """Relative, of a product with one nonzero term: the three products left out
    are at most 2^-24 |a b| (0.99 of it at a = b = 0x1.00ff8p+0), the two
    accumulators' sum rounds by at most as much again, and the smaller one's
    sums, of up to 2^-7 |a b|, by 5 x 2^-31.  (fp32's own product: 2^-24.)"""
    return (2 + 5 / 128) * U


def normal_bound(K):
    """Relative 2-norm of N(0, 1) products: at slab i the accumulator is about
    sqrt(16 i); truncation and rounding add an error of at most its last place
    (2^-23 of it) over sqrt(12) each, so after K / 16 slabs 2^-23 sqrt(K / 192),
    and the result rounds once more."""
    return 2 * U * np.sqrt(K / 192) + U / 2


# Attention on N(0, 1) operands of up to 500 tokens, relative 2-norms.  Measured
# 2.0 to 3.1 units of 2^-24 forward and 4.2 to 11.4 backward (the most where a
# sum is left to fp32 MFMA: dK and dV of heads of 128, dQ without a stored dS);
# without one of the six products of one contraction 37 and more, either way.
FORWARD_BOUND = 6 * U
BACKWARD_BOUND = 20 * U


def attention(Q, K, V, dO, lossy=None, keep=ALL):
    """ctx, dQ, dK, dV of one head in float64, the contraction `lossy` (s, o, dp,
    dq, dk, dv) by the piece products `keep`."""
    def dot(name, A, B):
        return product(A, B, keep) if name == lossy else A.astype(np.float64) @ B.astype(np.float64)
    scale = 1.0 / np.sqrt(np.float64(Q.shape[1]))
    s = dot("s", Q, K.T) * scale
    p = np.exp(s - s.max(1, keepdims=True))
    p /= p.sum(1, keepdims=True)
    dp = dot("dp", dO, V.T)
    ds = p * (dp - (p * dp).sum(1, keepdims=True))
    return dot("o", p, V), dot("dq", ds, K) * scale, dot("dk", ds.T, Q) * scale, dot("dv", p.T, dO)
