"""The 256 x 256 tiles (csrc/gemm_wide.hip, csrc/gemm_wide_bf16.hip) against numpy: sides one vector into a tile or
short of it, k below, at and above whole k-steps, strides, alpha and beta, both output types, k
slices; and, FP32 unsplit, bit for bit against the other tiles, which a product with an odd
leading dimension takes. tests/test_gemm_split_host.py holds the sizes to the kernels they are for.

Tolerance, of the result (zero-mean operands): FP32 sums 2e-6 sqrt(K / 64), split-BF16x3 3e-5."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [  # M, N, K of one slice, at least 0.9 of whole rounds of tiles on 256 CUs
    (4096, 4096, 256), (4092, 3844, 260), (3844, 4096, 287), (4096, 4088, 317),
]
# products in slices of k, with the kernel and the slices of each mode; the last two are on the
# other side of the line (the kernel of one 128 x 128 tile a workgroup)
SLICED = {
    (752, 6732, 8064): {"f32": ("wide", 3), "bf16x3": ("wide", 3)},
    (756, 6732, 8067): {"f32": ("wide", 3), "bf16x3": ("wide", 3)},
    (5116, 1276, 5132): {"f32": ("wide", 5), "bf16x3": ("tiles", 1)},
    (2048, 4096, 4100): {"f32": ("tiles", 1), "bf16x3": ("tiles", 1)},
    (3076, 4084, 2049): {"f32": ("tiles", 3), "bf16x3": ("wide", 1)},
}
SAME_BITS = [(4092, 3844, 300)]


@pytest.mark.parametrize("prec", ["f32", "bf16x3"])
@pytest.mark.parametrize("out", ["f32", "f64"])
@pytest.mark.parametrize("ops", ["NN", "NT", "TN"])
@pytest.mark.parametrize("mnk", SIZES + list(SLICED))
def test_wide_product(ctx, rng, mnk, ops, out, prec):
    from tnhip import Tensor, ops as T

    M, N, K = mnk
    if ops != "NT" and prec == "f32":
        K = (K + 3) // 4 * 4  # whole vectors along k
    A = rng.standard_normal((K, M) if ops[0] == "T" else (M, K), dtype=np.float32)
    B = rng.standard_normal((N, K) if ops[1] == "T" else (K, N), dtype=np.float32)
    C = rng.standard_normal((M + 4, N))
    C = C.astype(np.float32) if out == "f32" else C
    dA, dB = (Tensor.from_numpy(x, np.float32, ctx=ctx) for x in (A, B))
    dC = Tensor.from_numpy(C, C.dtype, ctx=ctx)
    T.gemm(ops[0], ops[1], M, N, K, 0.75, dA, A.shape[0], dB, B.shape[0], -0.5, dC, M + 4, prec)
    got = dC.numpy()
    tol = 2e-6 * np.sqrt(K / 64) if prec == "f32" else 3e-5
    rows = np.r_[0:8, 120:136, 250:262, M - 8:M]
    ref = 0.75 * ((A.T if ops[0] == "T" else A)[rows].astype(float) @ (B.T if ops[1] == "T" else B)) - 0.5 * C[rows]
    assert np.linalg.norm(got[rows] - ref) <= tol * np.linalg.norm(ref)
    assert np.array_equal(got[M:], C[M:])
    v = rng.standard_normal(N)
    full = 0.75 * ((A.T if ops[0] == "T" else A) @ ((B.T if ops[1] == "T" else B) @ v)) - 0.5 * C[:M] @ v
    assert np.linalg.norm(got[:M] @ v - full) <= tol * np.linalg.norm(full)


@pytest.mark.parametrize("ops", ["NN", "NT", "TN"])
def test_same_bits_as_other_tiles(ctx, rng, ops):
    from tnhip import Tensor, ops as T

    M, N, K = SAME_BITS[0]
    A = rng.standard_normal((K, M) if ops[0] == "T" else (M, K), dtype=np.float32)
    B = rng.standard_normal((N, K) if ops[1] == "T" else (K, N), dtype=np.float32)
    dA, dB = (Tensor.from_numpy(x, np.float32, ctx=ctx) for x in (A, B))
    pad = np.zeros((A.shape[0] + 1, A.shape[1]), np.float32)
    pad[:-1] = A
    dP = Tensor.from_numpy(pad, np.float32, ctx=ctx)  # an odd leading dimension: the other tiles
    res = []
    for a, ld in ((dA, A.shape[0]), (dP, A.shape[0] + 1)):
        dC = Tensor.from_numpy(np.zeros((M, N), np.float32), np.float32, ctx=ctx)
        T.gemm(ops[0], ops[1], M, N, K, 1.0, a, ld, dB, B.shape[0], 0.0, dC, M, "f32")
        res.append(dC.numpy())
    assert np.array_equal(res[0], res[1])
