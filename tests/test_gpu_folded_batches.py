"""Batched applies (nvec > 1) at every FP64/FP32 tile class: the vectors of a
batch are folded into one dimension of each grouped product, so tiles straddle
vector boundaries at odd block sizes.

Bars: FP64 results equal the single-vector apply bit for bit (same k order per
element) and the numpy execution of the plan's schedule within 1e-13 relative
(sums of at most a few hundred products of O(1) terms: n eps ~ 5e-14); FP32
within 2e-6 of the FP64 result (operands and products rounded once at 2^-24,
sums of the same length)."""
import numpy as np
import pytest

import complexcase as cc
import plan_interp
import problems
from mpstools_amd import native

pytestmark = pytest.mark.gpu


# block dimensions from 1 up: below, at and across one 16-row sub-tile (xxz),
# thousands of tiny blocks (hubbard), blocks over several tiles (dense, odd)
@pytest.mark.parametrize("model,L,N,D,seed,dense,nvecs", [
    ("xxz", 12, 6, 40, 901, False, (2, 17)), ("hubbard", 8, 8, 60, 902, False, (3, 16)),
    ("tv", 16, 8, 90, 903, False, (5, 64)), ("xxz", 14, 0, 67, 904, True, (2, 3))])
def test_folded_batches(gpu, oracle, model, L, N, D, seed, dense, nvecs):
    torch = gpu
    P = problems.build(oracle, model, L, N, D, seed, dense=dense)
    c, mpo, itk = P["c"], P["mpo"], P["itk"]
    Lb, Rb = P["Ls"][c - 1], P["Rs"][c + 2]
    Lt, Rt, xt = native.Table.from_blocks(Lb), native.Table.from_blocks(Rb), native.Table.from_blocks(P["psi"])
    vt = xt.union(native.heff2_outkeys(Lt, Rt, xt, mpo[c], mpo[c + 1], itk[c], itk[c + 1]))
    dL, dR = torch.from_numpy(Lt.pack(Lb)).cuda(), torch.from_numpy(Rt.pack(Rb)).cuda()
    rng = np.random.default_rng(seed)
    stride = vt.total + 5  # odd: vectors start at every alignment
    for prec in (native.F64, native.F32):
        plan = native.HeffPlan(Lt, Rt, vt, vt, (mpo[c], mpo[c + 1]), (itk[c], itk[c + 1]), prec)
        plan.bind_env(dL, dR)
        for nvec in nvecs:
            x = rng.standard_normal((nvec, stride))
            ref = np.zeros((nvec, vt.total))
            ref_plan = native.HeffPlan(Lt, Rt, vt, vt, (mpo[c], mpo[c + 1]), (itk[c], itk[c + 1]), native.F64)
            for v in range(nvec):
                plan_interp.run_heff(ref_plan.describe(), Lt.pack(Lb), Rt.pack(Rb), x[v, :vt.total], ref[v],
                                     ref_plan.info()["workspace_bytes"] // 8)
            dx = torch.from_numpy(x).cuda()
            for cls in range(5):
                print("[case]", model, prec, nvec, cls, flush=True)
                plan.set_tile_class(1, cls)
                plan.set_tile_class(2, cls)
                dy = torch.full((nvec, stride), 7.0, dtype=torch.float64, device="cuda")
                plan.apply(dx, dy, nvec, stride, stride)
                one = torch.full((nvec, stride), 7.0, dtype=torch.float64, device="cuda")
                for v in range(nvec):
                    plan.apply(dx[v], one[v])
                torch.cuda.synchronize()
                assert torch.equal(dy, one)  # also: nothing written between the vectors
                blocks = vt.unpack(dy[nvec - 1, :vt.total].cpu().numpy())
                want = vt.unpack(ref[nvec - 1])
                num = sum(float(np.sum((blocks[k] - want[k]) ** 2)) for k in want.keys())
                den = sum(float(np.sum(want[k] ** 2)) for k in want.keys())
                assert (num / den) ** 0.5 <= (1e-13 if prec == native.F64 else 2e-6), (prec, nvec, cls)


@pytest.mark.parametrize("model,L,N,D,seed,dense", [("xxz", 12, 6, 40, 911, False), ("hubbard", 8, 8, 60, 912, False),
                                                    ("xxz", 14, 0, 37, 913, True)])
@pytest.mark.parametrize("sites,cplx", [(1, False), (1, True), (2, True)])
def test_folded_one_site_and_complex_batches(gpu, oracle, model, L, N, D, seed, dense, sites, cplx):
    """One-site and complex (planar: blocks of real and imaginary parts, with
    signs) plans at every FP64/FP32 tile class: batches equal the single-vector
    applies bit for bit, and write nothing between the vectors."""
    torch = gpu
    P = problems.build(oracle, model, L, N, D, seed, dense=dense)
    c, mpo, itk = P["c"], P["mpo"], P["itk"]
    Lb = P["Ls"][c - 1]
    Rb, xb = (P["Rs"][c + 2], P["psi"]) if sites == 2 else (P["Rs"][c + 1], P["mps"][c])
    if cplx:
        Lb, Rb, xb = (cc.with_imag(b, seed + i) for i, b in enumerate((Lb, Rb, xb)))
    Lt, Rt, xt = (native.Table.from_blocks(b) for b in (Lb, Rb, xb))
    W, ik = ((mpo[c], mpo[c + 1]), (itk[c], itk[c + 1])) if sites == 2 else (mpo[c], itk[c])
    keys = native.heff2_outkeys(Lt, Rt, xt, *W, *ik) if sites == 2 else native.heff1_outkeys(Lt, Rt, xt, W, ik)
    vt = xt.union(keys)
    dL, dR = (torch.from_numpy(t.pack(b)).cuda() for t, b in ((Lt, Lb), (Rt, Rb)))
    rng = np.random.default_rng(seed)
    stride = vt.length + 5
    x = torch.from_numpy(rng.standard_normal((17, stride))).cuda()
    for prec in (native.F64,) if cplx else (native.F64, native.F32):
        plan = native.HeffPlan(Lt, Rt, vt, vt, W, ik, prec)
        plan.bind_env(dL, dR)
        for cls in range(5):
            plan.set_tile_class(1, cls)
            plan.set_tile_class(2, cls)
            for nvec in (3, 17):
                print("[case]", model, sites, cplx, prec, cls, nvec, flush=True)
                y, one = torch.full_like(x, 7.0), torch.full_like(x, 7.0)
                plan.apply(x, y, nvec, stride, stride)
                for v in range(nvec):
                    plan.apply(x[v], one[v])
                torch.cuda.synchronize()
                assert torch.equal(y, one)


@pytest.mark.parametrize("D,nvecs", [(64, (2, 64)), (100, (2, 16, 64)), (192, (3, 16)), (256, (2, 4, 16))])
def test_untuned_batches_of_a_dense_bond(gpu, oracle, D, nvecs):
    """The class that a batch takes by its number of vectors: the single-vector
    apply's result bit for bit in FP64, and within the precision's bound of it
    elsewhere (FP32 5e-6, BF16X3 2e-4, BF16 3e-2: operands rounded once, sums in
    another order); again the same after the batches, with and without a pinned
    class."""
    torch = gpu
    L = 18
    P = problems.build(oracle, "xxz", L, 0, D, 905, dense=True)
    c, mpo, itk = P["c"], P["mpo"], P["itk"]
    Lt, Rt, xt = (native.Table.from_blocks(b) for b in (P["Ls"][c - 1], P["Rs"][c + 2], P["psi"]))
    vt = xt.union(native.heff2_outkeys(Lt, Rt, xt, mpo[c], mpo[c + 1], itk[c], itk[c + 1]))
    dL, dR = (torch.from_numpy(t.pack(b)).cuda() for t, b in ((Lt, P["Ls"][c - 1]), (Rt, P["Rs"][c + 2])))
    rng = np.random.default_rng(D)
    stride = vt.total + 3
    x = torch.from_numpy(rng.standard_normal((max(nvecs), stride))).cuda()
    ref = None
    for prec, tol in ((native.F64, 0.0), (native.F32, 5e-6), (native.BF16X3, 2e-4), (native.BF16, 3e-2)):
        plan = native.HeffPlan(Lt, Rt, vt, vt, (mpo[c], mpo[c + 1]), (itk[c], itk[c + 1]), prec)
        plan.bind_env(dL, dR)
        one = torch.full_like(x, 7.0)  # the gaps between blocks stay as they were
        for v in range(max(nvecs)):
            plan.apply(x[v], one[v])
        torch.cuda.synchronize()
        ref = one if prec == native.F64 else ref
        own = (plan.stage_info()["tile_class1"], plan.stage_info()["tile_class2"])
        for pin in (False, True):
            if pin:
                plan.set_tile_class(1, 1)
                plan.set_tile_class(2, 1)
            for nvec in nvecs + (1,):
                print("[case] untuned", D, prec, nvec, pin, flush=True)
                y = torch.full_like(x, 7.0)
                plan.apply(x, y, nvec, stride, stride)
                torch.cuda.synchronize()
                for v in range(nvec):
                    got, want = y[v, :vt.total], one[v, :vt.total]
                    if prec == native.F64:
                        assert torch.equal(got, want), (nvec, v)
                    else:
                        assert float((got - ref[v, :vt.total]).norm() / ref[v, :vt.total].norm()) <= tol, (prec, nvec)
                assert bool((y[:, vt.total:] == 7.0).all()) and bool((y[nvec:] == 7.0).all())
            if not pin:
                assert (plan.stage_info()["tile_class1"], plan.stage_info()["tile_class2"]) == own
