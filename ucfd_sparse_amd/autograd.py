"""torch binding of the differentiation form: one FP64 coloured LU-SGS pass
dQ = upper(lower(pre(dt, fspr), rhsb)) as a torch.autograd.Function whose
backward is the library's hand-written adjoint (ucfd_lusgs_adjoint,
include/ucfd_ext.h).

The forward runs the legacy API's pass (parallel_pre_lusgs, ns_parallel_lower_sweep
per colour, ns_parallel_upper_sweep per colour in reverse, as one library
call) on device tensors of a colour-contiguous layout, on torch's current
stream.  The lower sweep's
output dQ* is either kept for the backward (two-array sweeps: rhsb -> dQ*,
dQ* -> dQ) or, with recompute=True, never kept: the forward runs the
in-place sweeps on one buffer (rhsb copy -> dQ* -> dQ) and the backward
recomputes dQ* (pre + lower sweeps again) and lets the adjoint overwrite it
with the rhsb gradient.  That saves 5 x neles doubles both between forward
and backward and at the peak, for half a forward of extra work.
"""
from __future__ import annotations

import ctypes

import numpy as np
import torch

from . import lib as L


class _Stream:
    """Route library calls to torch's current stream for the duration."""

    def __init__(self, lib):
        self.lib = lib

    def __enter__(self):
        self.prev = self.lib.ucfd_get_stream()
        self.lib.ucfd_set_stream(torch.cuda.current_stream().cuda_stream)

    def __exit__(self, *exc):
        self.lib.ucfd_set_stream(self.prev)
        return False


class ColoredSystem:
    """Device-resident mesh of a colour-contiguous layout
    (ucfd_sparse_amd.layout.ColoredLayout): nei_ele, fnorm_vol, vec_fnorm,
    upts, identity icolor / non-decreasing lcolor, declared to the library."""

    def __init__(self, lay, device="cuda:0"):
        self.lib = L.load()
        m, f = lay.mesh, lay.flow
        dev = torch.device(device)

        def up(a):
            return torch.from_numpy(np.ascontiguousarray(a)).to(dev)
        self.N, self.F, self.rows = m.neles, m.nface, m.ndims + 2
        self.nei, self.fnv, self.vfn = up(m.nei_ele), up(m.fnorm_vol), up(m.vec_fnorm)
        self.upts = up(f.upts)
        self.icolor, self.lcolor = up(lay.icolor), up(lay.lcolor)
        self.off = [int(x) for x in lay.off]
        L.check(self.lib.ucfd_declare_colored_layout(self.N, self.icolor.data_ptr(),
                                                     self.lcolor.data_ptr(), None),
                "ucfd_declare_colored_layout")
        h = ctypes.c_void_p()
        off = np.ascontiguousarray(lay.off, np.int32)
        L.check(self.lib.ucfd_adjoint_create(ctypes.byref(h), self.N, self.F, len(off) - 1,
                                             off.ctypes.data, self.nei.data_ptr(),
                                             self.fnv.data_ptr(), self.vfn.data_ptr(),
                                             self.upts.data_ptr()), "ucfd_adjoint_create")
        self.handle = h

    def check_inputs(self, rhsb, dt, fspr, **outs):
        """Every array the pass reads or writes: float64, contiguous, on the
        GPU, at least as large as the kernels index (ValueError otherwise)."""
        N, F = self.N, self.F
        if rhsb is not None:
            L.arr(rhsb, np.float64, 5 * N, "rhsb", device=True)
        L.arr(dt, np.float64, N, "dt", device=True)
        L.arr(fspr, np.float64, F * N, "fspr", device=True)
        sizes = {"dq": 5 * N, "dstar": 5 * N, "diag": N, "w": 5 * N}
        for k, v in outs.items():
            if v is not None:
                L.arr(v, np.float64, sizes[k], k, device=True)

    def _out(self, like):
        """An output of the pass: the sweeps write every cell of the NFVARS rows,
        only rows beyond them start from zero."""
        return (torch.empty_like if like.numel() == self.rows * self.N else torch.zeros_like)(like)

    def _pass(self, rhsb, dt, fspr, factor, dstar, dq, diag=None):
        """ucfd_lusgs_pass on torch's current stream; returns diag."""
        diag = torch.empty(self.N, dtype=torch.float64, device=rhsb.device) if diag is None else diag
        with _Stream(self.lib):
            L.check(self.lib.ucfd_lusgs_pass(
                self.handle, float(factor), self.icolor.data_ptr(), self.lcolor.data_ptr(),
                dt.data_ptr(), fspr.data_ptr(), rhsb.data_ptr(),
                None if dstar is None else dstar.data_ptr(),
                None if dq is None else dq.data_ptr(), diag.data_ptr()), "ucfd_lusgs_pass")
        return diag

    def forward_arrays(self, rhsb, dt, fspr, factor=1.0, dq=None, dstar=None, diag=None):
        """pre + lower + upper on torch's current stream; returns (dq, dstar, diag)."""
        self.check_inputs(rhsb, dt, fspr, dq=dq, dstar=dstar, diag=diag)
        dstar = self._out(rhsb) if dstar is None else dstar
        dq = self._out(rhsb) if dq is None else dq
        return dq, dstar, self._pass(rhsb, dt, fspr, factor, dstar, dq, diag)

    def forward_inplace(self, rhsb, dt, fspr, factor=1.0):
        """pre + lower + upper with the in-place C sweeps on one buffer;
        returns dQ (dQ* is overwritten by the upper sweep)."""
        self.check_inputs(rhsb, dt, fspr)
        dub = torch.empty_like(rhsb) if rhsb.numel() == self.rows * self.N else rhsb.clone()
        self._pass(rhsb, dt, fspr, factor, None, dub)
        return dub

    def recompute_dstar(self, rhsb, dt, fspr, factor=1.0):
        self.check_inputs(rhsb, dt, fspr)
        dstar = self._out(rhsb)
        self._pass(rhsb, dt, fspr, factor, dstar, None)
        return dstar

    def adjoint(self, dt, fspr, dstar, dq, w, factor=1.0, overwrite_dstar=False):
        """(rhsbar, dtbar, fsprbar) of J = sum(w * dq); with overwrite_dstar
        the rhsb gradient is written into dstar's buffer and returned."""
        w = w.contiguous()
        self.check_inputs(None, dt, fspr, dq=dq, dstar=dstar, w=w)
        rb = dstar if overwrite_dstar else self._out(dq)
        dtb = torch.empty_like(dt)
        fb = torch.empty_like(fspr)
        with _Stream(self.lib):
            L.check(self.lib.ucfd_lusgs_adjoint(self.handle, float(factor), dt.data_ptr(),
                                                fspr.data_ptr(), dstar.data_ptr(), dq.data_ptr(),
                                                w.data_ptr(), rb.data_ptr(), dtb.data_ptr(),
                                                fb.data_ptr()), "ucfd_lusgs_adjoint")
        return rb, dtb, fb

    def close(self):
        if self.handle:
            self.lib.ucfd_adjoint_destroy(self.handle)
            self.lib.ucfd_release_colored_layout(self.icolor.data_ptr(), self.lcolor.data_ptr())
            self.handle = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


class LUSGSPass(torch.autograd.Function):
    """dQ = coloured LU-SGS pass (pre + lower + upper) of rhsb [NFVARS, N],
    dt [N], fspr [F, N]; differentiable in all three."""

    @staticmethod
    def forward(ctx, rhsb, dt, fspr, system, recompute=False, factor=1.0):
        rhsb, dt, fspr = rhsb.contiguous(), dt.contiguous(), fspr.contiguous()
        system.check_inputs(rhsb, dt, fspr)
        ctx.system, ctx.recompute, ctx.factor = system, recompute, factor
        if recompute:
            dq = system.forward_inplace(rhsb, dt, fspr, factor)
            ctx.save_for_backward(rhsb, dt, fspr, dq)
        else:
            dq, dstar, _ = system.forward_arrays(rhsb, dt, fspr, factor)
            ctx.save_for_backward(rhsb, dt, fspr, dq, dstar)
        return dq

    @staticmethod
    def backward(ctx, w):
        S = ctx.system
        if ctx.recompute:
            rhsb, dt, fspr, dq = ctx.saved_tensors
            dstar = S.recompute_dstar(rhsb, dt, fspr, ctx.factor)
            rb, dtb, fb = S.adjoint(dt, fspr, dstar, dq, w, ctx.factor, overwrite_dstar=True)
        else:
            rhsb, dt, fspr, dq, dstar = ctx.saved_tensors
            rb, dtb, fb = S.adjoint(dt, fspr, dstar, dq, w, ctx.factor)
        return rb, dtb, fb, None, None, None


def lusgs_pass(system, rhsb, dt, fspr, recompute=False, factor=1.0):
    return LUSGSPass.apply(rhsb, dt, fspr, system, recompute, factor)
