"""The Lanczos step's forms (csrc/krylov.hip): one launch for short real vectors, subtraction
fused with the next dot products for complex or long ones and at most four vectors, separate
launches otherwise, at sizes on both sides of each line (16384 entries; 16384 entries times
vectors; four and eight vectors), real and complex, against the oracle's Lanczos on the same data: the Ritz value to 1e-11 of the largest
Krylov coefficient's scale and the Ritz vector up to a phase to 1e-9 (krylovdim 10 orthogonalises
nearly dependent vectors)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("kdim", [3, 10])
@pytest.mark.parametrize("chi", [(3, 2), (40, 50), (64, 64), (65, 64), (90, 97)])
def test_lanczos_forms(ctx, rng, chi, kdim, cplx):
    from oracle.krylov import eigsolve_ground
    from oracle.projmps import product_optimal
    from tnhip import Tensor, ops as T

    def env(c):
        a = rng.standard_normal((c, 3, c)) + (1j * rng.standard_normal((c, 3, c)) if cplx else 0)
        return np.asfortranarray((a + a.conj().transpose(2, 1, 0)) / np.sqrt(4 * c))

    cl, cr = chi
    sz, sx = np.diag([0.5, -0.5]), np.array([[0, 0.5], [0.5, 0]])
    W = np.zeros((3, 2, 2, 3))
    W[0, :, :, 0] = W[2, :, :, 2] = np.eye(2)
    W[0, :, :, 1], W[1, :, :, 2], W[0, :, :, 2] = sz, -sz, -sx
    L, R = env(cl), env(cr)
    x = rng.standard_normal((cl, 2, 2, cr)) + (1j * rng.standard_normal((cl, 2, 2, cr)) if cplx else 0)
    x = np.asfortranarray(x / np.linalg.norm(x))
    e0, y, nmv0 = eigsolve_ground(lambda v: product_optimal(L, W, W, R, v), x, krylovdim=kdim, maxiter=2)
    th = Tensor.from_numpy(x)
    e, nmv = T.eigsolve_ground(Tensor.from_numpy(L), Tensor.from_numpy(W), Tensor.from_numpy(W),
                               Tensor.from_numpy(R), th, krylovdim=kdim, maxiter=2)
    v = th.numpy()
    assert nmv == nmv0
    assert abs(e - e0) <= 1e-11 * max(1.0, abs(e0))
    assert abs(abs(np.vdot(v, y)) - 1) <= 1e-9
    assert abs(np.linalg.norm(v) - 1) <= 1e-12


@pytest.mark.parametrize("cr,kdim", [(32, 3), (16, 8), (31, 4)])
def test_step_forms_same_bits(ctx, rng, cr, kdim):
    """The one-launch step and the separate kernels on one input give the same bits. The input
    padded with zeros to 16384 entries takes the separate kernels from the second vector on (all
    its sums meet the same entries in the same order, then zeros). The operator is diagonal with
    powers of two, so that the products before a step are exact at either size."""
    from tnhip import Tensor, ops as T

    cl, wide = 32, 128  # 32 x 2 x 2 x 128 = 16384

    def diag(n, seed):
        g = np.random.default_rng(seed)
        a = np.zeros((n, 1, n))
        a[np.arange(n), 0, np.arange(n)] = g.choice([-1.0, 1.0], n) * 2.0 ** g.integers(-3, 3, n)
        return np.asfortranarray(a)

    W = np.zeros((1, 2, 2, 1))
    W[0, :, :, 0] = np.diag([1.0, 0.5])
    R = diag(wide, 1)
    x = np.zeros((cl, 2, 2, wide), order="F")
    x[..., :cr] = rng.standard_normal((cl, 2, 2, cr))
    got = []
    for c in (cr, wide):
        th = Tensor.from_numpy(np.asfortranarray(x[..., :c]))
        e, nmv = T.eigsolve_ground(Tensor.from_numpy(diag(cl, 0)), Tensor.from_numpy(W), Tensor.from_numpy(W),
                                   Tensor.from_numpy(np.asfortranarray(R[:c, :, :c])), th, krylovdim=kdim, maxiter=2)
        got.append((e, nmv, th.numpy()))
    assert got[0][:2] == got[1][:2] and got[0][1] >= 2 * kdim - 1
    assert np.array_equal(got[0][2], got[1][2][..., :cr]) and not got[1][2][..., cr:].any()
