"""The sector factorisations at the limits of their routes, every output and the
workspace NaN beforehand: an element that no kernel writes fails the test.

Bars: U^H U = 1 and V^dagger V = 1 within 30 r eps of the sweeps' rotations (r
per column and sweep, at most 30 sweeps here), the matrix rebuilt and its
singular values within the same times its norm; the QR's isometry and product
within 4 r eps (r reflections)."""
import numpy as np
import pytest

import factorcase

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps
# (m, n): rows around the 64-row segments and their limit of 512, either side
# of the singular values' 31 / 32 and 64, and of the LDS's size
SVD = {False: [(1, 1), (1, 30), (30, 1), (64, 20), (20, 65), (128, 20), (20, 129), (511, 20), (20, 512), (513, 20),
               (464, 24), (24, 465), (334, 31), (31, 335), (60, 32), (64, 64), (64, 65), (66, 65), (600, 31)],
       True: [(1, 1), (1, 30), (30, 1), (64, 20), (20, 65), (128, 20), (129, 20), (267, 20), (20, 268), (46, 45),
              (45, 47), (512, 5), (513, 5), (66, 65), (600, 24)]}
QR = {False: [(1, 1), (1, 70), (70, 1), (64, 15), (65, 15), (512, 15), (513, 15), (20, 64), (100, 64), (122, 64),
              (123, 64), (100, 65), (130, 60), (131, 60)],
      True: [(1, 1), (1, 70), (70, 1), (64, 7), (65, 7), (512, 7), (513, 7), (20, 64), (61, 64), (62, 64), (100, 39),
             (101, 39), (30, 65)]}


def draw(rng, m, n, cplx):
    return rng.standard_normal((m, n)) + (1j * rng.standard_normal((m, n)) if cplx else 0.0)


def check_svd(a, U, S, Vh):
    r = min(a.shape)
    tol = 30 * r * EPS
    ref = np.linalg.svd(a, compute_uv=False)
    assert np.max(np.abs(S - ref)) <= tol * ref[0]
    assert np.max(np.abs((U * S) @ Vh - a)) <= tol * ref[0]
    for Q in (U, Vh.conj().T):
        assert np.max(np.abs(Q.conj().T @ Q - np.eye(r))) <= tol


def check_qr(a, right, U, S, Vh):
    r = min(a.shape)
    tol = 4 * max(r, 8) * EPS
    Q = Vh.conj().T if right else U
    R = U.conj().T if right else Vh
    assert np.all(S == 1.0)
    assert np.max(np.abs(Q.conj().T @ Q - np.eye(r))) <= tol
    assert np.max(np.abs(U @ Vh - a)) <= tol * np.linalg.norm(a, 2)
    assert np.all(np.tril(R, -1) == 0.0)


def test_limits_are_the_kernels():
    """The shapes above lie on both sides of each line."""
    for cplx in (False, True):
        assert {factorcase.svd_in_lds(m, n, cplx) for m, n in SVD[cplx]} == {True, False}
        assert {factorcase.qr_in_lds(m, n, False, cplx) for m, n in QR[cplx]} == {True, False}
    assert factorcase.svd_in_lds(464, 24, False) and not factorcase.svd_in_lds(24, 465, False)
    assert factorcase.svd_in_lds(267, 20, True) and not factorcase.svd_in_lds(20, 268, True)
    assert factorcase.qr_in_lds(122, 64, False, False) and not factorcase.qr_in_lds(123, 64, False, False)


@pytest.mark.parametrize("cplx", [False, True])
def test_svd_in_one_workgroup(gpu, cplx):
    """One launch of every shape, and of its transpose."""
    rng = np.random.default_rng(1)
    mats = [draw(rng, *s, cplx) for mn in SVD[cplx] for s in (mn, mn[::-1])]
    print("[case] svd", cplx, flush=True)
    for a, out in zip(mats, factorcase.Case(gpu, mats).batched()):
        check_svd(a, *out)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("right", [False, True])
def test_qr_in_one_workgroup(gpu, cplx, right):
    rng = np.random.default_rng(2)
    mats = [draw(rng, *s, cplx) for mn in QR[cplx] for s in (mn, mn[::-1])]
    print("[case] qr", cplx, right, flush=True)
    for a, out in zip(mats, factorcase.Case(gpu, mats, right).batched()):
        check_qr(a, right, *out)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("right", [None, False, True])
def test_over_several_workgroups(gpu, cplx, right):
    """Block counts odd and even, a last block of one column, panels of 128, 256
    and more rows and their ends, 1024 rows; for the QR also more columns than
    rows."""
    rng = np.random.default_rng(3)
    shapes = [(32, 32), (33, 40), (64, 65), (128, 34), (129, 47), (257, 33), (1024, 40), (48, 136), (200, 160)]
    if right is not None:
        shapes += [(8, 40), (40, 9), (130, 70)]
    mats = [draw(rng, *s, cplx) for s in shapes]
    print("[case] several", cplx, right, flush=True)
    for a, out in zip(mats, factorcase.Case(gpu, mats, right).blocked()):
        check_svd(a, *out) if right is None else check_qr(a, right, *out)
