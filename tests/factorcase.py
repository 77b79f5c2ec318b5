"""The library's sector factorisation launchers (mpsa_factor.hip) called
directly: sectors packed planar, every output and the workspace filled with
NaN beforehand, so that an element no kernel writes shows."""
import ctypes as C

import numpy as np

from mpstools_amd import native

TASK = np.dtype([("a_off", np.int64), ("u_off", np.int64), ("vt_off", np.int64), ("s_off", np.int64),
                 ("w_off", np.int64), ("m", np.int32), ("n", np.int32), ("lda", np.int32), ("pad", np.int32)])
_ARRAYS = "PKdlPdlS5_lS5_S5_l"  # M, m_plane, U, u_plane, Vt, vt_plane, S, W, w_plane
LOAD, INIT, SWEEP, BACK, OUT = 1, 4, 8, 16, 64  # the kPh* bits of mpsa_internal.h
# the one-workgroup kernels' LDS, in doubles, as mpsa_factor.hip holds it
SVD_LDS, QR_LDS = 12288, 7808


def svd_in_lds(m, n, cplx):
    p, r = max(m, n), min(m, n)
    return p <= 512 and r <= 64 and (2 if cplx else 1) * (p * r + 2 * r * r) <= SVD_LDS


def qr_in_lds(m, n, right, cplx):
    return (n if right else m) <= 512 and (m if right else n) <= 64 and (2 if cplx else 1) * m * n <= QR_LDS


def _fn(name, sig):
    f = getattr(native.lib(), "_ZN4mpsa%d%sE%s" % (len(name), name, sig))
    f.restype = C.c_int
    return f


class Case:
    def __init__(self, torch, mats, right=None):
        self.torch, self.mats = torch, mats
        self.cplx = any(np.iscomplexobj(a) for a in mats)
        self.right = right
        self.tasks = np.zeros(len(mats), TASK)
        am = au = av = ss = aw = 0
        for t, a in zip(self.tasks, mats):
            m, n = a.shape
            k, p, r = min(m, n), max(m, n), min(m, n)
            t["a_off"], t["u_off"], t["vt_off"], t["s_off"], t["w_off"] = am, au, av, ss, aw
            t["m"], t["n"], t["lda"] = m, n, m + 3  # a leading dimension of its own
            am += (m + 3) * n
            au += m * k
            av += k * n
            ss += k
            # svd_workspace / qr_workspace
            aw += 2 * p * r + 2 * r * r + r + 1 if right is None else m * n + (n if right else m) * k + k + 1
        pl = 2 if self.cplx else 1
        M = np.full(pl * am, np.nan)
        for t, a in zip(self.tasks, mats):
            m, n = a.shape
            for q in range(pl):
                v = M[q * am + t["a_off"]:q * am + t["a_off"] + (m + 3) * n].reshape(n, m + 3)
                v[:, :m] = (a.imag if q else a.real).T
        self.plane = (am, au, av, aw)
        nan = lambda n: torch.full((max(n, 1),), float("nan"), dtype=torch.float64, device="cuda")  # noqa: E731
        self.M = torch.from_numpy(M).cuda()
        self.U, self.V, self.S, self.W = nan(pl * au), nan(pl * av), nan(ss), nan(pl * aw)
        self.dt = self._put(self.tasks)

    def _put(self, a):
        return self.torch.from_numpy(np.ascontiguousarray(a).view(np.uint8).copy()).cuda()

    def _arrays(self):
        p = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
        am, au, av, aw = (C.c_int64(x) for x in self.plane)
        return [p(self.M), am, p(self.U), au, p(self.V), av, p(self.S), p(self.W), aw]

    def _call(self, f, *args):
        assert f(*args) == 0
        self.torch.cuda.synchronize()

    def _st(self):
        return native._stream()

    def batched(self, max_sweeps=60):
        """All sectors in one launch, one workgroup each."""
        c, n, t = int(self.cplx), len(self.mats), C.c_void_p(self.dt.data_ptr())
        if self.right is None:
            self._call(_fn("launch_svd_batched", "iPKNS_7SvdTaskEi" + _ARRAYS + "P12ihipStream_ti"), c, t, n,
                       *self._arrays(), self._st(), max_sweeps)
        else:
            self._call(_fn("launch_qr_batched", "iiPKNS_7SvdTaskEi" + _ARRAYS + "P12ihipStream_t"), c,
                       int(self.right), t, n, *self._arrays(), self._st())
        return self.results()

    def blocked(self, max_sweeps=60):
        """The same over several workgroups per sector, as svd_blocked_run does."""
        c, n, t = int(self.cplx), len(self.mats), C.c_void_p(self.dt.data_ptr())
        layout = 0 if self.right is None else 1 + int(self.right)
        base = np.zeros(n + 1, np.int32)
        for i, a in enumerate(self.mats):
            m, nn = a.shape
            r = (min(m, nn), nn, m)[layout]
            base[i + 1] = base[i] + (r + 7) // 8
        kmax = max(min(a.shape) for a in self.mats)
        db = self._put(base)
        pb = C.c_void_p(db.data_ptr())
        W, aw = C.c_void_p(self.W.data_ptr()), C.c_int64(self.plane[3])
        if layout == 0:
            f = _fn("launch_svd_phase", "iiPKNS_7SvdTaskEi" + _ARRAYS + "P12ihipStream_t")
            phase = lambda ph: self._call(f, c, ph, t, n, *self._arrays(), self._st())  # noqa: E731
        else:
            f = _fn("launch_qr_phase", "iiiPKNS_7SvdTaskEi" + _ARRAYS + "P12ihipStream_t")
            phase = lambda ph: self._call(f, c, int(self.right), ph, t, n, *self._arrays(), self._st())  # noqa: E731
        phase(LOAD)
        self._call(_fn("launch_house_panels", "iiPKNS_7SvdTaskEiPKiiiPdlP12ihipStream_t"), c, layout, t, n, pb,
                   int(base[-1]), kmax, W, aw, self._st())
        phase(INIT)
        self.rotating = False
        if layout == 0:
            nb = [(min(a.shape) + 7) // 8 for a in self.mats]
            pairs = np.concatenate([[0], np.cumsum([(b + b % 2) // 2 for b in nb])]).astype(np.int32)
            dp = self._put(pairs)
            flags = self.torch.zeros(n, dtype=self.torch.float64, device="cuda")
            g = _fn("launch_svd_block_round", "iPKNS_7SvdTaskEiPKiiiPdlS5_iP12ihipStream_t")
            for _ in range(max_sweeps):
                flags.zero_()
                for rnd in range(-1, max(b + b % 2 - 1 for b in nb)):
                    assert g(c, t, n, C.c_void_p(dp.data_ptr()), int(pairs[-1]), rnd, W, aw,
                             C.c_void_p(flags.data_ptr()), kmax, self._st()) == 0
                self.rotating = bool((flags != 0).any().item())
                if not self.rotating:
                    break
            if self.rotating or max_sweeps == 0:
                phase(SWEEP)
            phase(BACK)
        self._call(_fn("launch_house_apply", "iiPKNS_7SvdTaskEiPKiiPdlP12ihipStream_t"), c, layout, t, n, pb,
                   int(base[-1]), W, aw, self._st())
        phase(OUT)
        return self.results()

    def outputs(self, svds):
        """The SVD's outputs from given ends of the sweeps: per sector the
        rotated A (r x r, orthogonal columns) and Q Wm (p x r)."""
        pw = self.plane[3]
        W = self.W.cpu().numpy()
        for t, (A, Q) in zip(self.tasks, svds):
            p, r = Q.shape
            for q in range(2 if self.cplx else 1):
                part = lambda x: np.asfortranarray(x.imag if q else x.real).reshape(-1, order="F")  # noqa: E731
                o = q * pw + t["w_off"]
                W[o:o + p * r] = part(Q)
                o += 2 * p * r + r * r
                W[o:o + r * r] = part(A)
                W[o + r * r + r] = 1.0  # the scale, after the betas
        self.W.copy_(self.torch.from_numpy(W))
        f = _fn("launch_svd_phase", "iiPKNS_7SvdTaskEi" + _ARRAYS + "P12ihipStream_t")
        self._call(f, int(self.cplx), OUT, C.c_void_p(self.dt.data_ptr()), len(self.mats), *self._arrays(), self._st())
        return self.results()

    def results(self):
        """(U, S, V^dagger) per sector."""
        _, au, av, _ = self.plane
        U, V, S = self.U.cpu().numpy(), self.V.cpu().numpy(), self.S.cpu().numpy()
        out = []
        for t, a in zip(self.tasks, self.mats):
            m, n = a.shape
            k = min(m, n)
            get = lambda buf, off, pl, r, c: (  # noqa: E731
                (buf[off:off + r * c] + (1j * buf[pl + off:pl + off + r * c] if self.cplx else 0.0))
                .reshape(c, r).T)
            out.append((get(U, t["u_off"], au, m, k), S[t["s_off"]:t["s_off"] + k], get(V, t["vt_off"], av, k, n)))
        return out
