"""Small sector factorisations against numpy: two rows or columns, 30 / 32
singular values (one workgroup's SVD below 32), wide and tall, rank-deficient
ones, and long ones beyond one workgroup's LDS.  Driven through the split of a
one-sector two-site state (the real SVD) and the orthonormalisation of a complex
MPS (QR).  The routes' exact limits are in test_gpu_sector_limits.py, zero
sectors in test_gpu_zero_sectors.py."""
import numpy as np
import pytest

import pycheb
from mpstools_amd import models, native, synth
from mpstools_amd.blocks import Blocks, twosite

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dl,dr,rank", [(1, 7, None), (7, 1, None), (13, 15, None), (15, 15, None), (15, 250, None),
                                        (250, 15, None), (15, 260, None), (200, 15, None), (15, 10, 6), (8, 8, 1)])
def test_small_real_svd(gpu, dl, dr, rank):
    """Sum of singular triplets = the state within 1e-13 relative (k <= 31 terms
    of rounding eps each), singular values within 1e-14 of the unit norm; values
    beyond the rank, where the SVD keeps any, at 16 eps."""
    torch = gpu
    print("[case] small svd", 2 * dl, 2 * dr, rank, flush=True)
    rng = np.random.default_rng(77 * dl + dr)
    k = min(2 * dl, 2 * dr) if rank is None else rank
    M = rng.standard_normal((2 * dl, k)) @ rng.standard_normal((k, 2 * dr))
    M /= np.linalg.norm(M)
    psi = Blocks(2)
    for s1 in range(2):
        for s2 in range(2):
            psi[(0, 0, s1, s2)] = M[s1 * dl:(s1 + 1) * dl, s2 * dr:(s2 + 1) * dr]
    t = native.Table.from_blocks(psi)
    out = native.split(t, torch.from_numpy(t.pack(psi)).cuda(), [0, 0], [0, 0], direction=1, chimax=10 ** 6)
    ref = np.linalg.svd(M, compute_uv=False)[:k]
    got = np.asarray(out["lam"][0])
    assert np.max(np.abs(got[:k] - ref)) <= 1e-14
    if rank is not None:
        assert np.all(got[k:] <= 1e-15 * 16)  # rounding level, where an SVD keeps any
    two = twosite(out["left"][0].unpack(out["left"][1].cpu().numpy()),
                  out["right"][0].unpack(out["right"][1].cpu().numpy()))
    assert max(np.max(np.abs(two[key] - psi[key])) for key in psi.keys()) <= 1e-13


@pytest.mark.parametrize("L,D,seed", [(6, 6, 11), (8, 40, 12)])
def test_small_complex_factorisations(gpu, L, D, seed):
    """orthonormalize(rl) of a complex Hubbard MPS keeps the (normalised) state
    and makes every site right-isometric, both within 1e-12."""
    print("[case] small complex", L, D, flush=True)
    itk = [models.itokey_u1xu1()] * L
    mps, _ = synth.random_mps(L, itk, models.pack_charge(L // 2, L // 2), D, seed)
    rng = np.random.default_rng(seed)
    for A in mps:
        for k in A.keys():
            A.b[k] = np.asfortranarray(A[k] + 1j * rng.standard_normal(A[k].shape))
        A.dtype = np.dtype(np.complex128)
    eng = native.Cheb([mps], models.hubbard_mpo(L, 1.0, 2.0), itk)
    eng.orthonormalize(0)
    got = eng.state(0, 0)
    a, b = pycheb.to_dense(pycheb.MPS(mps, itk)), pycheb.to_dense(pycheb.MPS(got, itk))
    a /= np.linalg.norm(a)
    assert abs(abs(np.vdot(a, b)) - 1.0) <= 1e-12 and abs(np.linalg.norm(b) - 1.0) <= 1e-12
    for A in got[1:]:
        by = {}
        for k in A.keys():
            by.setdefault(k[0], []).append(A[k])
        for blocks in by.values():
            X = np.hstack(blocks)
            assert np.max(np.abs(X @ X.conj().T - np.eye(X.shape[0]))) <= 1e-12


@pytest.mark.parametrize("dl,dr,scale", [(16, 17, 1.0), (17, 17, 1.0), (20, 90, 1.0), (33, 32, 1.0), (63, 64, 1.0),
                                         (65, 65, 1.0), (128, 140, 1.0), (129, 130, 1.0), (21, 30, 1e70),
                                         (7, 9, 1e70), (17, 512, 1.0), (512, 19, 1.0)])
def test_block_rounds_at_their_edges(gpu, dl, dr, scale):
    """Sectors of several column blocks: a whole last block and one of 2 to 6
    columns, odd and even block counts, either side of 128 and 256 rows (the
    shares of the vectors' update); norms near 1e140, where the rotation's
    squares leave the doubles' range.  Singular values 1 .. 2^-4 (relative
    error n eps < 1e-13 each), state rebuilt within 1e-12 relative."""
    torch = gpu
    print("[case] block rounds", 2 * dl, 2 * dr, scale, flush=True)
    rng = np.random.default_rng(31 * dl + dr)
    m, n = 2 * dl, 2 * dr
    k = min(m, n)
    U = np.linalg.qr(rng.standard_normal((m, k)))[0]
    V = np.linalg.qr(rng.standard_normal((n, k)))[0]
    sv = 2.0 ** (-4.0 * np.arange(k) / k)
    M = (U * (sv * scale)) @ V.T
    psi = Blocks(2)
    for s1 in range(2):
        for s2 in range(2):
            psi[(0, 0, s1, s2)] = M[s1 * dl:(s1 + 1) * dl, s2 * dr:(s2 + 1) * dr]
    t = native.Table.from_blocks(psi)
    out = native.split(t, torch.from_numpy(t.pack(psi)).cuda(), [0, 0], [0, 0], direction=1, chimax=10 ** 6)
    got = np.asarray(out["lam"][0])
    got = got / np.linalg.norm(got)
    assert got.shape == (k,) and np.max(np.abs(got / (sv / np.linalg.norm(sv)) - 1.0)) <= 1e-13
    two = twosite(out["left"][0].unpack(out["left"][1].cpu().numpy()),
                  out["right"][0].unpack(out["right"][1].cpu().numpy()))
    ratio = np.vdot(two[(0, 0, 0, 0)], psi[(0, 0, 0, 0)]) / np.vdot(two[(0, 0, 0, 0)], two[(0, 0, 0, 0)])
    assert max(np.max(np.abs(two[key] * (ratio / scale) - psi[key] / scale)) for key in psi.keys()) <= 1e-12
