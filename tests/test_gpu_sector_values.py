"""Sector factorisations at the ends of the doubles' range: entries that are not
finite, sweeps that reach their limit, entries whose squares leave the range."""
import numpy as np
import pytest

import factorcase
from mpstools_amd import models, native, synth
from mpstools_amd.blocks import Blocks

pytestmark = pytest.mark.gpu

NAN, INF = float("nan"), float("inf")


def one_sector(M, s1=2, s2=2, l=0):
    """A two-site state whose only sector is M (rows by s1, columns by s2)."""
    m, n = M.shape[0] // s1, M.shape[1] // s2
    psi = Blocks(2)
    for a in range(s1):
        for b in range(s2):
            psi[(l, l, a, b)] = np.asfortranarray(M[a * m:(a + 1) * m, b * n:(b + 1) * n])
    return psi


def split(torch, psi, **kw):
    t = native.Table.from_blocks(psi)
    return native.split(t, torch.from_numpy(t.pack(psi)).cuda(), [0, 0], [0, 0], direction=1, chimax=10 ** 6, **kw)


# one singular value (both ways), two, a sector in one workgroup's LDS, one
# beyond it, two of several workgroups (the longest that they take)
SHAPES = [(1, 14), (14, 1), (2, 14), (30, 40), (30, 600), (64, 80), (40, 1024)]


@pytest.mark.parametrize("value", [NAN, INF, -INF])
@pytest.mark.parametrize("m,n", SHAPES)
@pytest.mark.parametrize("last", [False, True])
def test_split_refuses_what_is_not_finite(gpu, m, n, last, value):
    """One bad entry in the first or the last row and column of one of two
    sectors is an error, as a sector of rocSOLVER's that does not converge is."""
    print("[case] split", m, n, last, value, flush=True)
    rng = np.random.default_rng(5 * m + n)
    M = rng.standard_normal((m, n))
    at = (m - 1, n - 1) if last else (0, 0)
    s1, s2 = (1 if m % 2 else 2), (1 if n % 2 else 2)
    psi = one_sector(rng.standard_normal((6, 8)), 2, 2, l=4)
    for bad in (False, True):
        if bad:
            M[at] = value
        for k, b in one_sector(M, s1, s2).b.items():
            psi[k] = b
        if bad:
            with pytest.raises(native.MpsaError, match="did not converge"):
                split(gpu, psi)
        else:
            assert split(gpu, psi)["chi"] == min(m, n) + 6


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("blocked", [False, True])
def test_outputs_of_a_sector_that_is_not_finite(gpu, cplx, blocked):
    """NaN in every output of the SVD and in R of the QR (L of the LQ), for a
    bad entry at either end and of either plane; the sectors beside it keep
    their factors."""
    rng = np.random.default_rng(17)
    draw = lambda m, n: rng.standard_normal((m, n)) + (1j * rng.standard_normal((m, n)) if cplx else 0.0)  # noqa: E731
    shapes = [(40, 33), (33, 50)] if blocked else [(1, 9), (9, 1), (2, 2), (30, 12), (12, 31), (600, 7)]
    for m, n in shapes:
        for at in ((0, 0), (m - 1, n - 1)):
            for value in (NAN, INF) + ((1j * NAN, 1j * INF) if cplx else ()):
                bad = draw(m, n)
                bad[at] = value
                mats = [draw(m, n), bad, draw(n, m)]
                for right in (None, False, True):
                    print("[case]", m, n, at, value, right, flush=True)
                    case = factorcase.Case(gpu, mats, right)
                    got = case.blocked() if blocked else case.batched()
                    for i in (0, 2):
                        U, S, Vh = got[i]
                        assert np.max(np.abs((U * S) @ Vh - mats[i])) <= 1e-12
                    U, S, Vh = got[1]
                    if right is None:
                        assert np.all(np.isnan(U.real)) and np.all(np.isnan(S)) and np.all(np.isnan(Vh.real))
                    else:
                        assert np.all(np.isnan((U if right else Vh).real))


@pytest.mark.parametrize("cplx", [False, True])
def test_sweeps_at_their_limit(gpu, cplx):
    """A sector that still rotates in its last sweep answers with NaN (in LDS and
    beyond it); one sweep is enough where nothing rotates."""
    rng = np.random.default_rng(23)
    shapes = [(2, 2), (12, 30), (30, 12), (600, 7), (40, 70)]
    mats = [rng.standard_normal(s) + (1j * rng.standard_normal(s) if cplx else 0.0) for s in shapes]
    mats += [np.eye(9, 4), rng.standard_normal((1, 5)), rng.standard_normal((5, 1))]
    print("[case] sweeps", cplx, flush=True)
    for sweeps in (1, 60):
        got = factorcase.Case(gpu, mats).batched(sweeps)
        for i, (U, S, Vh) in enumerate(got):
            if sweeps == 1 and i < len(shapes):
                assert np.all(np.isnan(S)) and np.all(np.isnan(U.real)) and np.all(np.isnan(Vh.real))
            else:
                assert np.max(np.abs((U * S) @ Vh - mats[i])) <= 1e-13


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("exp", [-310, -300, -160, -156, -155, -91, 91, 154, 160, 300])
def test_extreme_entries(gpu, cplx, exp):
    """Sectors of entries near 10^exp beside one of entries near 1: factors and
    singular values of the matrix scaled to 1 within n eps (1e-13 at these
    sizes); denormals (10^-310) and what is computed from them keep 43 bits."""
    rng = np.random.default_rng(31)
    draw = lambda m, n: rng.standard_normal((m, n)) + (1j * rng.standard_normal((m, n)) if cplx else 0.0)  # noqa: E731
    for blocked, shapes in ((False, [(1, 6), (6, 1), (20, 9), (9, 31), (600, 7)]), (True, [(40, 33), (33, 200)])):
        mats = [draw(*s) for s in shapes for _ in range(2)]
        e = int(np.floor(exp / np.log10(2.0)))  # a power of two, in two factors: 2^-e may be beyond DBL_MAX
        up = lambda a, f: a * 2.0 ** (f * (e // 2)) * 2.0 ** (f * (e - e // 2))  # noqa: E731
        given = [up(a, 1) if i % 2 else a for i, a in enumerate(mats)]
        for right in (None, False, True):
            print("[case] extreme", exp, cplx, blocked, right, flush=True)
            case = factorcase.Case(gpu, given, right)
            got = case.blocked() if blocked else case.batched()
            for i, (U, S, Vh) in enumerate(got):
                down = lambda a: up(a, -1) if i % 2 else a  # noqa: E731
                tol = 1e-12 if exp == -310 and i % 2 else 1e-13
                if right is None:
                    assert np.max(np.abs(down(S) - np.linalg.svd(mats[i], compute_uv=False))) <= tol * 10
                    A = (U * down(S)) @ Vh
                    isos = (U, Vh.conj().T)
                else:
                    assert np.all(S == 1.0)
                    A = down(U) @ Vh if right else U @ down(Vh)
                    isos = (Vh.conj().T if right else U,)
                assert np.max(np.abs(A - mats[i])) <= tol * 30
                for Q in isos:
                    assert np.max(np.abs(Q.conj().T @ Q - np.eye(Q.shape[1]))) <= 1e-13


@pytest.mark.parametrize("cplx", [False, True])
def test_columns_far_below_the_rest(gpu, cplx):
    """Columns and rows down to 10^-300 of the others, in order and not: the
    large singular values as without them, the matrix within n eps of its
    largest entry, orthonormal vectors."""
    rng = np.random.default_rng(37)
    for blocked, (m, n) in ((False, (20, 9)), (False, (9, 20)), (False, (600, 6)), (True, (50, 33))):
        A = rng.standard_normal((m, n)) + (1j * rng.standard_normal((m, n)) if cplx else 0.0)
        k = min(m, n)
        mats = []
        for low in (-120, -157, -165, -300):
            d = np.ones(n)
            d[rng.permutation(n)[:k // 2]] = 10.0 ** low
            mats.append(A * d)
            mats.append(A * 10.0 ** np.linspace(0, low, n))
            mats.append(A * 10.0 ** np.linspace(low, 0, m)[:, None])
        for right in (None, False, True):
            print("[case] graded", m, n, cplx, blocked, right, flush=True)
            case = factorcase.Case(gpu, mats, right)
            got = case.blocked() if blocked else case.batched()
            for a, (U, S, Vh) in zip(mats, got):
                top = np.max(np.abs(a))
                assert np.max(np.abs((U * S) @ Vh - a)) <= 1e-13 * 30 * top
                V = Vh.conj().T
                for Q in (U[:, S > 0], V[:, S > 0]) if right is None else ((V,) if right else (U,)):
                    assert np.max(np.abs(Q.conj().T @ Q - np.eye(Q.shape[1]))) <= 1e-13
                if right is None:
                    ref = np.linalg.svd(a, compute_uv=False)
                    assert np.max(np.abs(S - ref)) <= 1e-13 * ref[0]


@pytest.mark.parametrize("m,n", [(34, 60), (80, 66), (300, 40)])
def test_blocked_sweeps_finished_by_one_workgroup(gpu, m, n):
    """Sectors that still rotate after the block rounds' sweeps (none, one, three
    here) are finished in the one-workgroup kernel's order."""
    rng = np.random.default_rng(43)
    mats = [rng.standard_normal((m, n)), rng.standard_normal((n, m))]
    for sweeps in (0, 1, 3):
        print("[case] finished", m, n, sweeps, flush=True)
        for a, (U, S, Vh) in zip(mats, factorcase.Case(gpu, mats).blocked(sweeps)):
            ref = np.linalg.svd(a, compute_uv=False)
            assert np.max(np.abs(S - ref)) <= 1e-13 * ref[0]
            assert np.max(np.abs((U * S) @ Vh - a)) <= 1e-12
            for Q in (U, Vh.T):
                assert np.max(np.abs(Q.T @ Q - np.eye(Q.shape[1]))) <= 1e-13


@pytest.mark.parametrize("low", [-60, -90, -120])
def test_split_of_columns_far_below_the_rest(gpu, low):
    """Half a sector's columns many orders below the others, where the block
    rounds alone do not converge: split as rocSOLVER's Jacobi did."""
    print("[case] split far below", low, flush=True)
    rng = np.random.default_rng(47)
    M = rng.standard_normal((50, 34)) * np.where(rng.permutation(34) < 17, 1.0, 10.0 ** low)
    M /= np.linalg.norm(M)
    out = split(gpu, one_sector(M))
    assert out["chi"] == 17
    assert np.max(np.abs(np.asarray(out["lam"][0]) - np.linalg.svd(M, compute_uv=False)[:17])) <= 1e-14


def test_split_with_a_negligible_sector(gpu):
    """A sector of entries near 10^-156 beside an ordinary one is no error: the
    ordinary one is split as without it."""
    rng = np.random.default_rng(41)
    M, T = rng.standard_normal((30, 40)), rng.standard_normal((30, 40))
    M /= np.linalg.norm(M)
    for scale in (1e-156, 1e-310):
        psi = one_sector(M)
        for k, b in one_sector(T * scale, l=7).b.items():
            psi[k] = b
        out = split(gpu, psi)
        assert out["chi"] == 30
        assert np.max(np.abs(np.asarray(out["lam"][0]) - np.linalg.svd(M, compute_uv=False))) <= 1e-14


def test_compression_refuses_what_is_not_finite(gpu):
    """The Chebyshev engine's compression of a state with a NaN is an error."""
    L = 6
    itk = [models.itokey_u1xu1()] * L
    mps, _ = synth.random_mps(L, itk, models.pack_charge(L // 2, L // 2), 8, 3)
    for bad in (False, True):
        if bad:
            k = sorted(mps[2].keys())[-1]
            mps[2].b[k] = mps[2].b[k].copy()
            mps[2].b[k][-1, -1] = NAN
        eng = native.Cheb([mps], models.hubbard_mpo(L, 1.0, 2.0), itk)
        if bad:
            with pytest.raises(native.MpsaError, match="did not converge"):
                eng.compress(0, 6)
        else:
            eng.compress(0, 6)
