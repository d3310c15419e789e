"""The MPO mixing kernel (csrc/contract.hip) inside the matvec and the environment updates, at
bonds around its vector width and its column split, odd ones among them, for the MPO bond
dimensions with and without a compile-time term count (d D and d^2 D of 6 .. 32 and others),
real and complex, in FP64 and FP32, against the oracle's contractions. Tolerances as for the
matvec: 1e-13 relative in FP64, 2e-6 sqrt(K / 64) in FP32 with K = D chi."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("D,cplx", [(3, False), (5, False), (8, False), (4, False), (10, False), (3, True), (5, True)])
@pytest.mark.parametrize("chi", [(1, 3), (2, 2), (5, 7), (24, 25), (61, 34), (130, 127)])
def test_mix_in_matvec(ctx, rng, chi, D, cplx, prec):
    from oracle.projmps import product_optimal
    from tnhip import Tensor, ops as T

    def rand(*s):
        a = rng.standard_normal(s)
        return np.asfortranarray(a + 1j * rng.standard_normal(s) if cplx else a)

    cl, cr = chi
    L, R, x = rand(cl, D, cl), rand(cr, D, cr), rand(cl, 2, 2, cr)
    for W in (np.asfortranarray(rng.standard_normal((D, 2, 2, D))), rand(D, 2, 2, D)):
        dt = {("f64", False): np.float64, ("f64", True): np.complex128, ("f32", False): np.float32,
              ("f32", True): np.complex64}[prec, cplx]
        out = T.heff_apply(Tensor.from_numpy(L, dt), Tensor.from_numpy(W), Tensor.from_numpy(W),
                           Tensor.from_numpy(R, dt), Tensor.from_numpy(x), precision=prec).numpy()
        ref = product_optimal(L, W, W, R, x)
        tol = 1e-13 if prec == "f64" else 2e-6 * max(1.0, np.sqrt(D * max(chi) / 64))
        assert np.linalg.norm(out - ref) <= tol * np.linalg.norm(ref)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("D", [3, 5, 8, 11])
@pytest.mark.parametrize("chi", [(1, 2), (7, 5), (33, 64), (90, 91)])
def test_mix_in_environments(ctx, rng, chi, D, cplx):
    from tnhip import Tensor, ops as T

    def rand(*s):
        a = rng.standard_normal(s)
        return np.asfortranarray(a + 1j * rng.standard_normal(s) if cplx else a)

    ca, cb = chi
    A, W = rand(ca, 2, cb), np.asfortranarray(rng.standard_normal((D, 2, 2, D)))
    L, R = rand(ca, D, ca), rand(cb, D, cb)
    left = T.env_left(Tensor.from_numpy(L), Tensor.from_numpy(A), Tensor.from_numpy(W)).numpy()
    ref = np.tensordot(np.tensordot(np.tensordot(L, A, (2, 0)), W, ((1, 2), (0, 2))), A.conj(), ((0, 2), (0, 1)))
    assert np.linalg.norm(left - ref.transpose(2, 1, 0)) <= 1e-13 * np.linalg.norm(ref)
    right = T.env_right(Tensor.from_numpy(R), Tensor.from_numpy(A), Tensor.from_numpy(W)).numpy()
    ref = np.tensordot(np.tensordot(np.tensordot(A, R, (2, 2)), W, ((1, 3), (2, 3))), A.conj(), ((3, 1), (1, 2)))
    assert np.linalg.norm(right - ref.transpose(2, 1, 0)) <= 1e-13 * np.linalg.norm(ref)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("D,d", [(1, 2), (1, 3), (2, 3), (3, 3), (7, 2)])
def test_mix_term_counts(ctx, rng, D, d, cplx):
    """Term counts d^2 D of every remainder modulo four (4, 9, 18, 27, 28), with a value of 1e300
    in the last term."""
    from oracle.projmps import product_optimal
    from tnhip import Tensor, ops as T

    def rand(*s):
        a = rng.standard_normal(s)
        return np.asfortranarray(a + 1j * rng.standard_normal(s) if cplx else a)

    L, R, x = rand(13, D, 13), rand(6, D, 6), rand(13, d, d, 6)
    x[5, -1, -1, 2] = 1e300
    for W in (np.asfortranarray(rng.standard_normal((D, d, d, D))), rand(D, d, d, D)):
        out = T.heff_apply(*(Tensor.from_numpy(a) for a in (L, W, W, R, x))).numpy()
        ref = product_optimal(L, W, W, R, x)
        assert np.linalg.norm(out / 1e300 - ref / 1e300) <= 1e-13 * np.linalg.norm(ref / 1e300)


@pytest.mark.parametrize("prec,cplx", [("f64", False), ("f64", True), ("f32", False)])
@pytest.mark.parametrize("chi", [(5, 7), (61, 34)])
def test_mix_profiled_work(ctx, rng, chi, prec, cplx):
    """The work the profile reports for one mixing pass of a matvec: cl cr (I + J) values moved
    and cl cr I J multiply-adds (twice that with a complex input), whatever a thread takes."""
    from tnhip import Tensor, ops as T

    def rand(*s):
        a = rng.standard_normal(s)
        return np.asfortranarray(a + 1j * rng.standard_normal(s) if cplx else a)

    (cl, cr), D, d = chi, 5, 2
    dt = np.float32 if prec == "f32" else None
    L, R = (Tensor.from_numpy(rand(c, D, c), dt, ctx=ctx) for c in chi)
    W = Tensor.from_numpy(rng.standard_normal((D, d, d, D)), ctx=ctx)
    x = Tensor.from_numpy(rand(cl, d, d, cr), ctx=ctx)
    T.heff_apply(L, W, W, R, x, precision=prec)
    ctx.profile_reset()
    ctx.profile(True)
    T.heff_apply(L, W, W, R, x, precision=prec)
    got = ctx.profile_read("mix")
    ctx.profile(False)
    n, ij = cl * cr * (2 if cplx else 1), D * d * d
    assert got["launches"] == 1
    assert got["flops"] == 2 * n * ij * ij
    assert got["bytes"] == n * 2 * ij * (4 if prec == "f32" else 8)
