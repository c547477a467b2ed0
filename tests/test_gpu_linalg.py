"""GPU FP64 orthonormalisation and Cholesky solve against the oracle
(ortho_prim_mpi.c:198-284 layouts) and against the invariants they must meet."""
import numpy as np
import pytest

import modalcmb
import pyoracle as O
from modalcmb import workloads as W

pytestmark = pytest.mark.gpu


def spd(n, seed, cond=1e4):
    rng = np.random.default_rng(seed)
    Q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    ev = np.logspace(0, np.log10(cond), n)
    d = rng.uniform(0.5, 3.0, n)
    return (Q * ev) @ Q.T * np.outer(d, d)


@pytest.mark.parametrize("n", [1, 5, 31, 32, 33, 63, 64, 65, 100, 257, 700, 1030])
def test_orthonormalise_matches_oracle(ctx, n):
    G = spd(n, n)
    ortho, lam, norm = ctx.orthonormalise(G)
    st, o_ref, l_ref, n_ref = O.orthonormalise(G)
    assert st == 0
    assert np.allclose(norm, n_ref, rtol=1e-15, atol=0)
    assert np.allclose(ortho, o_ref, rtol=1e-12, atol=1e-12 * np.abs(o_ref).max())
    assert np.allclose(lam, l_ref, rtol=1e-9, atol=1e-11 * np.abs(l_ref).max())
    F, Lam = np.tril(ortho), np.tril(lam)
    assert np.allclose(F @ F.T, G, rtol=1e-11, atol=1e-12 * np.abs(G).max())
    assert np.abs(Lam @ G @ Lam.T - np.eye(n)).max() < 1e-9


def test_orthonormalise_not_spd_reports_pivot(ctx):
    G = spd(40, 1)
    G[17, :] = G[16, :]
    G[:, 17] = G[:, 16]
    with pytest.raises(modalcmb.NotSPDError) as e:
        ctx.orthonormalise(G)
    assert "pivot 17" in str(e.value)


@pytest.mark.parametrize("n,nrhs", [(300, 7), (300, 1), (611, 70), (129, 130)])
def test_cholesky_solve_many_rhs(ctx, n, nrhs):
    G = spd(n, 9, cond=1e3)
    ortho, _, _ = ctx.orthonormalise(G)
    rng = np.random.default_rng(2)
    C = rng.standard_normal((n, nrhs))
    A = G @ C
    B = ctx.cholesky_solve(ortho, A)
    assert np.allclose(B, C, rtol=1e-9, atol=1e-9)
    for j in range(0, nrhs, max(1, nrhs // 7)):
        assert np.allclose(B[:, j], O.cholesky_solve(ortho, A[:, j]), rtol=1e-10, atol=1e-10)


def test_orthonormalise_inverse_is_exact_triangle(ctx):
    """tril(lambda) is (D L)^-1: lower triangular with L^-1 D^-1 on it, so
    tril(lambda) @ tril(ortho) = I to rounding, on a size with ragged tiles."""
    n = 517
    G = spd(n, 5, cond=1e3)
    ortho, lam, _ = ctx.orthonormalise(G)
    P = np.tril(lam) @ np.tril(ortho)
    assert np.abs(P - np.eye(n)).max() < 1e-11


@pytest.mark.parametrize("n", [127, 128, 129, 191, 321, 2049, 2900])
def test_orthonormalise_block_edges(ctx, n):
    """Sizes around the 64-column blocks, the pairs that the inverse joins (a
    last pair without or with a short second block) and the 128-wide tiles:
    both triangles against the matrix itself.  1e-11: rounding of n-term sums at
    condition 1e3, as test_orthonormalise_inverse_is_exact_triangle."""
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n + 50)) * np.exp(-3.0 * np.arange(n + 50) / n)
    G = A @ A.T + 0.05 * n * np.eye(n)
    d = rng.uniform(0.5, 3.0, n)
    G = G * np.outer(d, d)
    ortho, lam, norm = ctx.orthonormalise(G)
    F, Lam = np.tril(ortho), np.tril(lam)
    assert np.array_equal(ortho, ortho.T) and np.array_equal(lam, lam.T)
    assert np.abs(F @ F.T - G).max() < 1e-13 * np.abs(G).max()
    assert np.abs(Lam @ F - np.eye(n)).max() < 1e-11
    C = rng.standard_normal((n, 5))
    assert np.abs(ctx.cholesky_solve(ortho, G @ C) - C).max() < 1e-10


@pytest.mark.parametrize("bad", [0, 15, 16, 63, 64, 127, 200, 255])
def test_not_spd_pivot_positions(ctx, bad):
    """A dependent row at every edge of the panels and blocks is reported at its
    own column, and a later call on a good matrix is not affected."""
    n = 256
    G = spd(n, 3, cond=10)
    H = G.copy()
    H[bad, bad] = -1.0 if bad == 0 else (H[bad, :bad] @ np.linalg.solve(H[:bad, :bad], H[:bad, bad])) * (1 - 1e-3)
    if bad == 0:
        with pytest.raises(modalcmb.ModalError):
            ctx.orthonormalise(H)
    else:
        with pytest.raises(modalcmb.NotSPDError) as e:
            ctx.orthonormalise(H)
        assert f"pivot {bad})" in str(e.value)
    ortho, _, _ = ctx.orthonormalise(G)
    assert np.abs(np.tril(ortho) @ np.tril(ortho).T - G).max() < 1e-13 * np.abs(G).max()


@pytest.mark.parametrize("n,nrhs", [(64, 1), (65, 4), (200, 5), (129, 128), (129, 129), (1000, 9)])
def test_cholesky_solve_block_steps(ctx, n, nrhs):
    """Few right-hand sides (a launch per block of 64, groups of four) and the
    first count past them, against the matrix."""
    G = spd(n, 4, cond=1e2)
    ortho, _, _ = ctx.orthonormalise(G)
    C = np.random.default_rng(n).standard_normal((n, nrhs))
    assert np.abs(ctx.cholesky_solve(ortho, G @ C) - C).max() < 1e-11


@pytest.mark.parametrize("nrhs", [1, 4, 128, 129])
def test_cholesky_solve_rounds_as_a_division(ctx, nrhs):
    """With a diagonal factor a solve is two quotients an entry, each rounded
    once however many right-hand sides there are, also at the ends of the
    exponent range."""
    n = 130
    rng = np.random.default_rng(nrhs)
    d = rng.uniform(0.5, 2.0, n)
    d[[3, 70, 100, 129]] = 4e-309, 1.3e-200, 6e307, 1.7e150
    C = rng.standard_normal((n, nrhs))
    C[[3, 70, 100, 129]] *= np.array([1e-310, 1e-200, 1e300, 1e120])[:, None]
    assert np.array_equal(ctx.cholesky_solve(np.diag(d), C), C / d[:, None] / d[:, None])


def test_lmax500_gram_orthonormalisation_status(ctx):
    # The lmax-500 Gram (r<=s<=t<10 Legendre modes, weight h^2/C^3) has
    # kappa(D^-1 G D^-1) ~ 1e17 > 1/eps: whether FP64 Cholesky meets a
    # non-positive pivot depends on summation order (the oracle passes, the GPU
    # order stops near column 174).  Either outcome must be clean: a NOT_SPD
    # status (the reference would abort inside GSL), or a factor that
    # reproduces the normalised Gram to FP64 accuracy.
    ws = W.lspace(500, 10)
    ctx.lspace_set(2, 500, ws["q"], ws["v"], ws["order"])
    G = ctx.gamma_tet(modalcmb.FP64)
    d = np.sqrt(np.diag(G))
    ev = np.linalg.eigvalsh(G / np.outer(d, d))
    assert ev.max() / max(ev.min(), 1e-300) > 1e15 or ev.min() <= 0
    try:
        ortho, lam, norm = ctx.orthonormalise(G)
    except modalcmb.NotSPDError as e:
        assert "pivot" in str(e)
    else:
        F = np.tril(ortho)
        assert np.abs(F @ F.T - G).max() < 1e-12 * np.abs(G).max()
