"""numpy model of the three-way bf16 split products (csrc/gemm_split.hip, csrc/attn.hip) and the
bounds on their error that tell six products from five.  All errors here are root mean squares, in
units of 2^-24 of the root sum of squares of the products that were added up."""
import numpy as np

PRODUCTS = [(2, 0), (0, 2), (1, 1), (1, 0), (0, 1), (0, 0)]  # planes of a and b, in the kernels' order


def bf16(x):
    u = np.ascontiguousarray(x, np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16 << 16).astype(np.uint32).view(np.float32)


def split(x):
    h = bf16(x)
    m = bf16(x - h)
    return h, m, bf16((x - h) - m)


def matmul(A, B, without=None, step=32):
    """A B by the split's products but the one named, each over `step` k at a time into an fp32 sum."""
    a, b = split(A), split(B)
    acc = np.zeros((A.shape[0], B.shape[1]), np.float32)
    for k in range(0, A.shape[1], step):
        for i, j in PRODUCTS:
            if (i, j) != without:
                acc = (acc + a[i][:, k:k + step].astype(np.float64) @ b[j][k:k + step].astype(np.float64)).astype(np.float32)
    return acc


def error(got, want, magnitude):
    return np.sqrt(np.mean(((got - want) / magnitude) ** 2)) * 2.0 ** 24


def gemm_bound(K):
    """Bound on `error` of K products of unit normal numbers (magnitude sqrt(K)).  The result's last
    rounding is 0.43 (its rms over a binade).  A matrix instruction adds 32 products; rounding the
    running sum after every four of them makes 6 K / 4 roundings of 0.43 of a sum that grows as
    sqrt(k): 0.43 sqrt(6 K / 4 / 2) = 0.37 sqrt(K).  A lost product of two planes is 33 or more."""
    return 1 + 0.5 * np.sqrt(K)


# the same for attention of unit normal inputs over up to 300 keys: its two products by the bound
# above are 1 + 0.5 sqrt(300) = 9.7 at most each, and the scores' and exponentials' own roundings
# (exponents of up to 8, 2^-24 of them each) add about 4
ATTENTION_BOUND = 20.0


def attention(Q, K, V, causal, without=(None, None), step=32):
    """One head; without: the product that Q K^T and P V leave out."""
    f32 = np.float32
    s = matmul(Q, np.ascontiguousarray(K.T), without[0], step)
    s = (s.astype(np.float64) * f32(np.log2(np.e) / np.sqrt(Q.shape[1]))).astype(f32)
    if causal:
        s = np.where(np.arange(len(K)) <= np.arange(len(Q))[:, None] + len(K) - len(Q), s, -np.inf).astype(f32)
    top = s.max(1, keepdims=True)
    p = np.exp2((s - np.where(top > 8, top, 0).astype(f32)).astype(np.float64)).astype(f32)
    return matmul(p, V, without[1], step) / p.sum(1, keepdims=True, dtype=f32)


def attention64(Q, K, V, causal):
    """One head in 64 bits, causal aligned to the last key: the result and its magnitude, the root sum
    of squares of the products of probabilities and V."""
    Q, K, V = (x.astype(np.float64) for x in (Q, K, V))
    s = Q @ K.T / np.sqrt(Q.shape[1])
    if causal:
        s = np.where(np.arange(len(K)) <= np.arange(len(Q))[:, None] + len(K) - len(Q), s, -np.inf)
    p = np.exp(s - s.max(1, keepdims=True))
    p /= p.sum(1, keepdims=True)
    return p @ V, np.sqrt(p ** 2 @ V ** 2)
