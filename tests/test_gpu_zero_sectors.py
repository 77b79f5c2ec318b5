"""Zero singular values: their vectors on the shorter side are completed to an
orthonormal basis, whatever the vectors before them are."""
import numpy as np
import pytest

import factorcase
from mpstools_amd import native
from mpstools_amd.blocks import Blocks

pytestmark = pytest.mark.gpu


def check(mats, got, sweeps=0):
    """Orthonormal to n eps (1e-13), or to one eps per rotation of a column where
    sweeps made it (r rotations each; sectors with zero columns take up to 30);
    the matrix to the same times its norm."""
    for a, (U, S, Vh) in zip(mats, got):
        tol = max(1e-13, sweeps * min(a.shape) * np.finfo(float).eps)
        for Q in (U, Vh.conj().T):
            assert np.max(np.abs(Q.conj().T @ Q - np.eye(Q.shape[1]))) <= tol
        assert np.max(np.abs((U * S) @ Vh - a)) <= tol * max(1.0, np.linalg.norm(a))
        assert np.all(np.diff(S) <= 0.0)


@pytest.mark.parametrize("cplx", [False, True])
def test_zero_and_padded_sectors(gpu, cplx):
    """Sectors of zeros, and random ones with zero rows and columns, in LDS, in
    one workgroup beyond it and over several; up to 512 singular values."""
    rng = np.random.default_rng(3)
    draw = lambda m, n: rng.standard_normal((m, n)) + (1j * rng.standard_normal((m, n)) if cplx else 0.0)  # noqa: E731
    for blocked, shapes in ((False, [(1, 1), (1, 7), (9, 1), (2, 2), (13, 30), (31, 16), (600, 9), (40, 41)]),
                            (True, [(33, 33), (160, 160), (70, 200), (512, 512)])):
        mats = []
        for m, n in shapes:
            mats.append(np.zeros((m, n)) + (0j if cplx else 0.0))
            if min(m, n) >= 8 and m < 512:
                for keep in (1, min(m, n) // 2, min(m, n) - 1):
                    a = draw(m, n)
                    a[rng.permutation(m)[keep:]] = 0.0
                    mats.append(a)
                    b = draw(m, n)
                    b[:, rng.permutation(n)[keep:]] = 0.0
                    mats.append(b)
        print("[case] zeros", cplx, blocked, flush=True)
        case = factorcase.Case(gpu, mats)
        check(mats, case.blocked() if blocked else case.batched(), 30)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("r", [2, 5, 17, 64, 130])
def test_completion_of_a_spread_null_space(gpu, cplx, r):
    """Null spaces of every unit vector's residual below 1/4 (one vector of equal
    entries, up to a few random ones), from given ends of the sweeps."""
    rng = np.random.default_rng(r)
    draw = lambda *s: rng.standard_normal(s) + (1j * rng.standard_normal(s) if cplx else 0.0)  # noqa: E731
    for null in (1, 2, r // 3, r - 1):
        if not 1 <= null < r:
            continue
        for wide in (False, True):
            p = r + 3
            first = np.ones((r, 1)) if null == 1 else draw(r, null)
            Z = np.linalg.qr(np.hstack([first, draw(r, r - null)]))[0]
            s = np.concatenate([np.zeros(null), 2.0 ** -np.linspace(0, 8, r - null)])
            s[null:] = rng.permutation(s[null:])
            order = rng.permutation(r)
            A, s = (Z * s)[:, order], s[order]
            Q = np.linalg.qr(draw(p, r))[0]
            # X = Q Wm: M = X Sigma Z^H, or its adjoint when wide
            M = Q @ A.conj().T
            M = M.conj().T if wide else M
            print("[case] spread", r, cplx, null, wide, flush=True)
            case = factorcase.Case(gpu, [M])
            got = case.outputs([(A, Q)])
            assert np.count_nonzero(got[0][1] == 0.0) == null
            check([M], got)


def test_split_of_zero_sectors(gpu):
    """A zero sector of 160 x 160 and a zero-padded one beside an ordinary one:
    the nonzero values are kept, and the isometry is one."""
    rng = np.random.default_rng(11)
    psi, ref = Blocks(2), []
    for q, (m, n, keep) in ((0, (80, 80, 0)), (5, (20, 30, 7)), (9, (12, 15, 24))):
        M = rng.standard_normal((2 * m, 2 * n))
        M[keep:] = 0.0
        ref += list(np.linalg.svd(M, compute_uv=False)[:keep])
        for a in range(2):
            for b in range(2):
                psi[(q, q, a, b)] = np.asfortranarray(M[a * m:(a + 1) * m, b * n:(b + 1) * n])
    t = native.Table.from_blocks(psi)
    out = native.split(t, gpu.from_numpy(t.pack(psi)).cuda(), [0, 0], [0, 0], direction=1, chimax=10 ** 6,
                       normalize=False)
    assert out["chi"] == len(ref)
    got = np.sort(np.concatenate([np.asarray(v) for v in out["lam"].values()]))
    assert np.max(np.abs(got - np.sort(ref))) <= 1e-13 * max(ref)
