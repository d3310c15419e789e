"""The whole-GPU eigensolver of the split's Gram matrix (csrc/tri_eig.hip) through
tnh_svd_trunc, against LAPACK: at the sides where a different kernel takes over (register
tiles 32, 64, 96, 128, 160, 192 of the last columns, 128 for complex matrices; real sides up
to 96 run the one-workgroup solver and are here as the other side of that line; one wave per
column or panels in the back-transformation at 1024) and on spectra that take every branch of
the divide and conquer (graded, repeated, rank-deficient, zero).

Tolerances as for every Gram path: s^2 to 1e-13 sqrt(n) s_max^2 (the backward error of the
Gram product and of the reduction, eps sqrt(n) |G| each, with room for the constants),
orthonormal bases to 1e-12 (one Newton-Schulz step leaves rounding), and the product of the
factors equal to M to 1e-12 where the rank is full."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def randn(rng, shape, cplx):
    a = rng.standard_normal(shape)
    return np.asfortranarray(a + 1j * rng.standard_normal(shape) if cplx else a)


def check(M, full_rank):
    from tnhip import Tensor, ops as T

    U, S, Vt, _, fb = T.svd_trunc(Tensor.from_numpy(M), 0.0, 0, 1)
    assert not fb
    u, s = U.numpy(), S.numpy()
    ref = np.linalg.svd(M, compute_uv=False)
    p = min(M.shape)
    top = max(ref[0], 1e-300)
    assert s.shape == ref.shape
    assert np.max(np.abs((s / top) ** 2 - (ref / top) ** 2)) <= 1e-13 * np.sqrt(max(M.shape))
    b = u if M.shape[0] <= M.shape[1] else Vt.numpy().conj().T
    assert np.abs(b.conj().T @ b - np.eye(p)).max() <= 1e-12
    if full_rank:
        assert np.linalg.norm((u * s) @ Vt.numpy() - M) <= 1e-12 * np.linalg.norm(M)
    else:  # the basis spans M's range up to the Gram path's resolution of it
        r = M - b @ (b.conj().T @ M) if M.shape[0] <= M.shape[1] else M - (M @ b) @ b.conj().T
        assert np.linalg.norm(r) <= 1e-12 * max(np.linalg.norm(M), 1e-300)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("p", [24, 31, 32, 33, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 257])
def test_tri_eig_sides(ctx, rng, cplx, p):
    check(randn(rng, (p, p + 3), cplx), True)
    check(randn(rng, (p + 2, p), cplx), True)


@pytest.mark.parametrize("cplx,p", [(False, 1024), (False, 1025), (True, 1025), (False, 1153)])
def test_tri_eig_panels(ctx, rng, cplx, p):
    check(randn(rng, (p, p), cplx), True)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("p", [40, 150, 530])
@pytest.mark.parametrize("kind", ["graded", "repeated", "rank1", "deficient", "diagonal", "zero"])
def test_tri_eig_spectra(ctx, rng, cplx, p, kind):
    if kind in ("graded", "repeated", "deficient"):
        q1, _ = np.linalg.qr(randn(rng, (p, p), cplx))
        q2, _ = np.linalg.qr(randn(rng, (p, p), cplx))
        s = {"graded": 10.0 ** np.linspace(0, -6, p), "repeated": np.repeat([3.0, 2.0, 1.0], p)[:: 3][:p],
             "deficient": np.where(np.arange(p) < p // 3, 1.0 + np.arange(p), 0.0)}[kind]
        M = (q1 * s) @ q2.conj().T
    elif kind == "rank1":
        M = randn(rng, (p, 1), cplx) @ randn(rng, (1, p), cplx)
    elif kind == "diagonal":
        M = np.diag(1.0 + np.arange(p) % 7).astype(complex if cplx else float)
    else:
        M = np.zeros((p, p), dtype=complex if cplx else float)
    check(np.asfortranarray(M), kind in ("graded", "repeated", "diagonal") and kind != "graded")


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("p", [160, 530])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_tri_eig_failure_is_reported(ctx, rng, cplx, p, value):
    """A non-finite entry: the solver reports failure, the paths behind it refuse the matrix too,
    the call ends with a status, and the next call on the same workspaces is right."""
    from tnhip import Tensor, TnhError, ops as T

    M = randn(rng, (p, p + 3), cplx)
    M[3, 7] = value
    with pytest.raises(TnhError) as e:
        T.svd_trunc(Tensor.from_numpy(M), 0.0, 0, 1)
    assert e.value.status in (-5, -6)
    check(randn(rng, (p, p + 3), cplx), True)


@pytest.mark.parametrize("cplx,p", [(True, 1850), (True, 3072), (False, 6144)])
def test_tri_eig_largest_sides(ctx, rng, cplx, p):
    """The complex column step in one 1024-thread workgroup a CU (sides above 1800), and the
    largest sides of either type, where the column step's vectors fill LDS. M = H1 H2 diag(s) H3
    H4 with Householder reflections H, so its singular values are known."""
    from tnhip import Tensor, ops as T

    s = 2.0 - np.arange(p) / p
    M = np.diag(s).astype(complex if cplx else float)
    for _ in range(2):
        v, w = randn(rng, (p, 1), cplx), randn(rng, (p, 1), cplx)
        M -= v @ ((2.0 / np.linalg.norm(v) ** 2) * (v.conj().T @ M))
        M -= (M @ w) @ ((2.0 / np.linalg.norm(w) ** 2) * w.conj().T)
    U, S, Vt, _, fb = T.svd_trunc(Tensor.from_numpy(np.asfortranarray(M)), 0.0, 0, 1)
    assert not fb
    u, got, vt = U.numpy(), S.numpy(), Vt.numpy()
    assert np.abs(got ** 2 - s ** 2).max() <= 1e-13 * np.sqrt(p) * s[0] ** 2
    assert np.abs(u.conj().T @ u - np.eye(p)).max() <= 1e-12
    assert np.linalg.norm((u * got) @ vt - M) <= 1e-12 * np.linalg.norm(M)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("p,top,solver", [(520, 36, "jacobi"), (520, 40, "tri_eig"), (1601, 194, "jacobi"),
                                          (1601, 199, "tri_eig")])
def test_solver_by_active_pairs(ctx, rng, cplx, p, top, solver):
    """Above side 512 a Gram matrix whose pairs lie mostly below the block Jacobi's floor (only
    `top` rows of M have weight, top^2 / p^2 of the pairs: 0.0048 and 0.0059 around the line 0.0052
    at side 520, 0.0147 and 0.0154 around 0.015 at 1601) is solved by it, others by the reduction;
    both to the same accuracy."""
    from tnhip import Tensor, ops as T

    w = np.where(np.arange(p) < top, 10.0 ** -(3.0 * np.arange(p) / top), 1e-15)
    q, _ = np.linalg.qr(randn(rng, (p, p), cplx))
    M = np.asfortranarray(rng.permutation(w)[:, None] * q)
    ctx.profile_reset()
    ctx.profile(True)
    U, S, Vt, _, fb = T.svd_trunc(Tensor.from_numpy(M), 0.0, 0, 1)
    ran = {f: int(ctx.profile_read(f)["launches"]) for f in ("jacobi", "tri_eig")}
    ctx.profile(False)
    assert ran == {"jacobi": int(solver == "jacobi"), "tri_eig": int(solver == "tri_eig")}
    assert not fb
    u, s = U.numpy(), S.numpy()
    assert np.abs(s ** 2 - w ** 2).max() <= 1e-13 * np.sqrt(p)
    assert np.abs(u.conj().T @ u - np.eye(p)).max() <= 1e-12
    assert np.linalg.norm(u @ (u.conj().T @ M) - M) <= 1e-12 * np.linalg.norm(M)


@pytest.mark.parametrize("cplx,p", [(True, 44), (True, 76), (True, 140), (False, 109), (False, 140), (False, 220)])
def test_graded_rows_keep_relative_accuracy(ctx, p, cplx):
    """M = D B with rows graded over five decades and B random: a solver that starts at the large
    end resolves each squared singular value relative to itself, to a few eps kappa(B)^2 sqrt(p)
    (the Gram matrix and the reduction are exact up to eps relative to their rows' and columns'
    scales). The sides leave the last block of the divide and conquer part padding."""
    from tnhip import Tensor, ops as T

    rng = np.random.default_rng(p)
    B = randn(rng, (p, p), cplx)
    M = np.asfortranarray(B * 10.0 ** np.linspace(0, -5, p)[:, None])
    _, S, _, _, fb = T.svd_trunc(Tensor.from_numpy(M), 0.0, 0, 1)
    assert not fb
    ref = np.linalg.svd(M, compute_uv=False)
    kappa = np.linalg.cond(B / np.linalg.norm(B, axis=1)[:, None])
    assert np.abs(S.numpy() / ref - 1).max() <= 16 * 2.3e-16 * np.sqrt(p) * kappa ** 2
