"""The LTE Stokes synthesis as a differentiable torch operation.

`stokes(engine, atmos, mu)` returns the emergent Stokes vector of a batch of
columns held in a CUDA tensor, and its backward pass is the library's
hand-written adjoint (rhg_rf_lte_params: one reverse depth sweep per column
and wavelength, see include/pyrh_amd.h) contracted with the incoming
gradient.  PyTorch only carries the tensors and the autograd graph; every
number comes from the HIP library.

Gradients flow to the atmosphere rows of the six response-function
parameters: temperature (row 1), line-of-sight velocity (3), micro-
turbulence (4), field strength (5), inclination (6) and azimuth (7).  The
depth scale (row 0), the electron density (2) and the hydrogen density (8)
are held fixed: their rows receive zero gradient.  Wavelengths that the
reference solves without polarization (no Zeeman line) have zero response
(the library leaves them zero), so their Stokes values are treated as
constants.
"""
from __future__ import annotations

from .engine import RF_PARAMS, RF_ROWS, rf_contract

try:
    import torch
    from torch.autograd import forward_ad
except ImportError:  # pragma: no cover - the product path needs torch for this module
    torch = None


def _require_torch():
    if torch is None:
        raise RuntimeError("pyrh_amd.autograd needs PyTorch")


def _bare(t):
    """Whether a tensor's memory is all there is to it: no subclass, no
    wrapper of a function transform, no forward-mode tangent, no pending
    negation."""
    return (type(t) is torch.Tensor and not torch._C._functorch.is_functorch_wrapped_tensor(t)
            and forward_ad.unpack_dual(t).tangent is None and not t.is_neg())


def _watched():
    """Whether a mode sees the operations run now (make_fx and other
    dispatch modes, torch-function modes): it would not see a kernel."""
    return torch._C._len_torch_dispatch_stack() > 0 or torch._C._len_torch_function_stack() > 0


def _contract_here(rf, g, shape):
    """Whether backward may run rhg_rf_contract: plain CUDA tensors of one
    device (_bare: the kernel reads their memory and nothing else), the saved
    response functions as forward laid them out (a saved-tensor hook may
    return others), and nobody who has to see the operations: a graph of the
    backward itself (create_graph), a tracer or another mode (_watched)."""
    return (_bare(rf) and _bare(g) and not _watched() and g.is_cuda
            and rf.device == g.device and rf.dtype in (torch.float32, torch.float64)
            and tuple(rf.shape) == shape and rf.is_contiguous()
            and not (torch.is_grad_enabled() and (g.requires_grad or rf.requires_grad)))


class _StokesFn(torch.autograd.Function if torch is not None else object):
    """forward: Stokes [ncol, 4, nout] float64.  With gradients requested the
    forward runs the adjoint as well (same Stokes values) and keeps the
    response functions of the requested parameters for backward."""

    @staticmethod
    def forward(ctx, atmos, engine, mu, precision, params):
        if not atmos.is_cuda or atmos.dtype != torch.float64 or atmos.dim() != 3 \
                or atmos.shape[1] != 9:
            raise ValueError("atmos must be a CUDA float64 tensor [ncol, 9, ndep]")
        atmos = atmos.contiguous()
        ncol, _, nd = atmos.shape
        dev = atmos.device
        ndep = torch.full((ncol,), nd, dtype=torch.int32, device=dev)
        st = torch.empty((ncol, 4, engine.nout), dtype=torch.float64, device=dev)
        torch.cuda.synchronize(dev)
        if not ctx.needs_input_grad[0]:
            engine.synth_lte_device(atmos.data_ptr(), ndep.data_ptr(), ncol, nd, st.data_ptr(),
                                    mu=mu, precision=precision)
            return st
        ids = [RF_PARAMS.index(p) for p in params]
        rf = torch.empty((len(ids), nd, 4, engine.nout, ncol),
                         dtype=torch.float32 if precision == 1 else torch.float64, device=dev)
        engine.rf_lte_device(atmos.data_ptr(), ndep.data_ptr(), ncol, nd, st.data_ptr(),
                             rf.data_ptr(), mu=mu, precision=precision, params=params)
        ctx.save_for_backward(rf)
        ctx.ids = ids
        ctx.shape = atmos.shape
        return st

    @staticmethod
    def backward(ctx, grad):
        (rf,) = ctx.saved_tensors
        g = grad.to(torch.float64)                                  # [ncol, 4, nout]
        ncol, _, nd = ctx.shape
        out = torch.zeros(ctx.shape, dtype=torch.float64, device=grad.device)
        if _contract_here(rf, g, (len(ctx.ids), nd, 4, g.shape[-1], ncol)):
            g = g.contiguous()
            work = torch.empty(g.numel(), dtype=torch.float64, device=g.device)
            rf_contract(g.device.index, torch.cuda.current_stream(g.device).cuda_stream,
                        1 if rf.dtype == torch.float32 else 0, ctx.ids, ncol, nd, g.shape[-1],
                        rf.data_ptr(), g.data_ptr(), work.data_ptr(), out.data_ptr())
            return out, None, None, None, None
        # d L / d p(k) = sum over (Stokes, wavelength) of grad * rf
        contr = torch.einsum("csl,pkslc->cpk", g, rf.to(torch.float64))
        for i, p in enumerate(ctx.ids):
            out[:, RF_ROWS[p], :] = contr[:, i, :]
        return out, None, None, None, None


def stokes(engine, atmos, mu=1.0, precision=1, params=RF_PARAMS):
    """Emergent Stokes [ncol, 4, nout] (float64 tensor) of the atmospheres
    atmos [ncol, 9, ndep] (CUDA float64, pyrh's row order and units) with an
    Engine built on the run directory and wavelength grid; differentiable
    with respect to atmos through the hand-written adjoint.  precision 1 is
    the FP32 form, 0 the plain FP64 path; params selects the parameters
    whose rows receive gradients (names of pyrh_amd.engine.RF_PARAMS)."""
    _require_torch()
    params = tuple(params)
    for p in params:
        if p not in RF_PARAMS:
            raise ValueError(f"unknown parameter {p!r}; expected names of {RF_PARAMS}")
    return _StokesFn.apply(atmos, engine, float(mu), int(precision), params)


__all__ = ["stokes", "RF_PARAMS", "RF_ROWS"]
