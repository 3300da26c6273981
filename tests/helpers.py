"""Shared helpers of the parity tests: structures, oracle runs, comparisons."""
import numpy as np

import oracle as O
from mtpx import capi
from mtpx import synth as S


def rel_err(a, b):
    """max |a - b| / max |b| (per quantity; exact zero reference -> absolute)."""
    a = np.asarray(a, float)
    b = np.asarray(b, float)
    scale = np.max(np.abs(b)) if b.size else 0.0
    diff = np.max(np.abs(a - b)) if b.size else 0.0
    return diff / scale if scale > 0 else diff


def oracle_case(model_text, s: S.Structure):
    """Wrap (Atoms::wrap), build the BOXED lists and evaluate E/F/S on the CPU."""
    m = O.Model(model_text)
    pos = O.wrap(s.cell, s.pbc, s.pos)
    nb = O.Neighbors.build(s.cell, s.pbc, pos, s.types, m.cutoff)
    E, F, St, se = O.efs(m, nb)
    return dict(model=m, pos=pos, nb=nb, E=E, F=F, S=St, se=se)


def upload_oracle_lists(ctx, nb):
    ctx.set_neighbors(nb.offsets, nb.idx, nb.types, nb.vec, nb.dist, nb.center_types)


def assert_efs_close(got, ref, tol):
    E, F, St, se = got
    assert rel_err(E, ref["E"]) < tol, (E, ref["E"])
    assert rel_err(se, ref["se"]) < tol
    assert rel_err(F, ref["F"]) < tol, rel_err(F, ref["F"])
    assert rel_err(St, ref["S"]) < tol, (St, ref["S"])


def loss_case(model_text, structs, seed):
    """Structures with the oracle's lists and labels, every label weighed.  The
    labels are half the model's own E/F/S plus noise: the residuals are then
    about half the values, and a rounding error of E/F/S reaches the gradient
    at most twice as large.  (With labels at the model's own values the
    residuals of the noise alone remain; in a dense cluster of 33 atoms, level
    20, with E = 1,010 and forces of 16,000 against noise of 0.05 and 0.16, a
    relative change of E/F/S by 1e-13 changes the gradient by 1e-7.)"""
    m = O.Model(model_text)
    rng = S.rng_for(seed)
    nbs, labels = [], []
    for s in structs:
        s.pos = O.wrap(s.cell, s.pbc, s.pos) if np.any(s.pbc) else s.pos
        nb = O.Neighbors.build(s.cell, s.pbc, s.pos, s.types, m.cutoff)
        E, F, St, _ = O.efs(m, nb)
        e, f, st = S.noisy_labels(rng, s.n, 0.5 * E, 0.5 * F, 0.5 * St)
        nbs.append(nb)
        labels.append(O.Labels(s.n, energy=e, forces=f, stress=st))
    return dict(text=model_text, model=m, structs=structs, nbs=nbs, labels=labels)


def assert_loss_grad_close(ctx, case, tol):
    """mtpx_loss_grad of a loss_case against the oracle; the model is loaded."""
    labels, structs = case["labels"], case["structs"]
    f_o, g_o = O.loss_grad_batch(case["model"], case["nbs"], labels, O.LossSettings.make(),
                                 penalty_weight=1e-4, reg_l2=1e-6, threads=8)
    off = ctx.set_structures(structs, case["model"].cutoff)
    tf = np.concatenate([lb.forces for lb in labels])
    active, wE, wF, wS = capi.loss_weights(capi.LossSettings.make(), off,
                                           np.ones((len(structs), 3), np.int32), tf)
    ctx.set_labels(active, np.array([lb.energy for lb in labels]), wE, tf, wF,
                   np.array([lb.stress for lb in labels]), wS)
    f, g, _ = ctx.loss_grad(penalty_weight=1e-4, reg_l2=1e-6)
    assert rel_err(f, f_o) < tol
    assert rel_err(g, g_o) < tol, rel_err(g, g_o)


class DeviceArray:
    """A float64 device buffer from the HIP runtime the library itself links
    (libamdhip64.so.7): hipMalloc / hipMemcpy / hipFree through ctypes, for
    tests of entry points that take device pointers."""
    _hip = None

    @classmethod
    def hip(cls):
        if cls._hip is None:
            import ctypes as C
            h = C.CDLL("libamdhip64.so.7")
            h.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
            h.hipFree.argtypes = [C.c_void_p]
            h.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
            h.hipDeviceSynchronize.argtypes = []
            cls._hip = h
        return cls._hip

    def __init__(self, values):
        import ctypes as C
        self.host = np.ascontiguousarray(values, dtype=np.float64)
        self.ptr = C.c_void_p()
        assert self.hip().hipMalloc(C.byref(self.ptr), max(self.host.nbytes, 8)) == 0
        self.upload(self.host)

    def upload(self, values):
        import ctypes as C
        v = np.ascontiguousarray(values, dtype=np.float64).reshape(self.host.shape)
        assert self.hip().hipMemcpy(self.ptr, v.ctypes.data_as(C.c_void_p), v.nbytes, 1) == 0

    def download(self):
        import ctypes as C
        out = np.empty_like(self.host)
        assert self.hip().hipMemcpy(out.ctypes.data_as(C.c_void_p), self.ptr, out.nbytes, 2) == 0
        return out

    @property
    def address(self):
        return self.ptr.value

    def free(self):
        if self.ptr:
            self.hip().hipFree(self.ptr)
            self.ptr = None
