"""Large products whose k range is split (csrc/gemm_split.hpp, ksplit_wanted) against numpy: k a
multiple of nothing, odd sides and leading dimensions, alpha and beta, every mode, and a
product just below the k from which a split is considered.

Tolerances: FP64 2 eps sqrt(K) |A| |B| + eps |C|; FP32 and split-BF16x3 as for the unsplit
product, 2e-6 sqrt(K / 64) and 3e-5 of |A| |B| / sqrt(...) (relative to the result of
zero-mean operands)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SLICES = {  # M, N, K: the slices of each mode on 256 CUs (tests/test_gemm_split_host.py)
    (2804, 593, 2965): {"f64": 3, "f32": 4, "bf16x3": 4},
    (2048, 700, 2049): {"f64": 2, "f32": 4, "bf16x3": 4},
    (1100, 1283, 2500): {"f64": 2, "f32": 4, "bf16x3": 4},
    (1100, 1283, 2047): {"f64": 1, "f32": 1, "bf16x3": 1},
}


@pytest.mark.parametrize("prec", ["f64", "f32", "bf16x3"])
@pytest.mark.parametrize("ops", ["NN", "NT", "TN"])
@pytest.mark.parametrize("mnk", SLICES)
def test_split_product(ctx, rng, mnk, ops, prec):
    from tnhip import Tensor, ops as T

    M, N, K = mnk
    A = rng.standard_normal((K, M) if ops[0] == "T" else (M, K))
    B = rng.standard_normal((N, K) if ops[1] == "T" else (K, N))
    C = rng.standard_normal((M + 1, N))
    dt = np.float64 if prec == "f64" else np.float32
    dA, dB, dC = Tensor.from_numpy(A, dt, ctx=ctx), Tensor.from_numpy(B, dt, ctx=ctx), Tensor.from_numpy(C, ctx=ctx)
    T.gemm(ops[0], ops[1], M, N, K, 0.75, dA, A.shape[0], dB, B.shape[0], -0.5, dC, M + 1, prec)
    ref = C.copy()
    ref[:M] = 0.75 * ((A.T if ops[0] == "T" else A) @ (B.T if ops[1] == "T" else B)) - 0.5 * C[:M]
    out = dC.numpy()
    tol = {"f64": 1e-14, "f32": 2e-6 * np.sqrt(K / 64), "bf16x3": 3e-5}[prec]
    assert np.linalg.norm(out - ref) <= tol * np.linalg.norm(ref)
    assert np.array_equal(out[M:], C[M:])
