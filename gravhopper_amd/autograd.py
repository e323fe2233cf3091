"""Differentiable leapfrog: gradients of a direct-sum N-body run with respect to the
initial positions, velocities and masses, through a hand-written adjoint.

    x, v = leapfrog(x0, v0, m, dt, eps, nsteps)
    loss = ((x - target) ** 2).sum(-1).mean(); loss.backward()

x0, v0: (n,3) float64 CUDA tensors (kpc, km/s); m: (n,) float64 (Msun); dt in Myr,
eps in kpc.  The forward is the drift-kick-drift of Simulation.run (gh_adjoint_forward,
the same kernels as gh_run).  With `checkpoint_every` it keeps (x, v) that often, 48 bytes per
particle, and backward re-runs each segment from its checkpoint.  Without, a run whose half-step
positions take at most KEEP_BYTES keeps those (gh_adjoint_forward_kept) and nothing is re-run;
a longer one has a checkpoint every 20 steps.  Backward applies the reverse step with the
vector-Jacobian products through the softened tidal tensor (gh_adjoint_backward).
Both are ordered with torch's current stream.
"""
import ctypes
import math

import torch

from . import _native

# A thousandth of the card's memory per run in the graph: 28 bytes per particle and step.
KEEP_BYTES = 256 << 20
CHECKPOINT_EVERY = 20  # where the caller names no interval and the run is longer


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _graph_is_kept():
    """Whether the backward pass that is running leaves its graph for another one."""
    return torch._C._autograd._get_current_graph_task_keep_graph()


class _OnTorchStream:
    """Orders library work with torch's current stream.  A real stream is handed to the
    library; torch's legacy default stream (handle 0) cannot be, since 0 selects the
    context's own stream, so then the call is fenced by synchronisation on both sides."""

    def __init__(self, lib, device):
        self.lib = lib
        self.torch_stream = torch.cuda.current_stream(device)
        self.handle = self.torch_stream.cuda_stream

    def __enter__(self):
        if self.handle == 0:
            self.torch_stream.synchronize()
        return ctypes.c_void_p(self.handle or None)

    def __exit__(self, *exc):
        if self.handle == 0:
            self.lib.sync()
        return False


class DirectLeapfrog(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x0, v0, m, dt, eps, nsteps, every, precision):
        lib = _native.default_context()
        n = x0.shape[0]
        x = x0.detach().to(torch.float64).contiguous().clone()
        v = v0.detach().to(torch.float64).contiguous().clone()
        mm = m.detach().to(torch.float64).contiguous()
        if every is None and n > 0 and nsteps >= 0 and 28 * n * nsteps <= KEEP_BYTES:
            return DirectLeapfrog._forward_kept(ctx, lib, x, v, mm, float(dt), float(eps),
                                                int(precision), int(nsteps))
        if every is None:
            every = CHECKPOINT_EVERY
        nseg = max(1, math.ceil(nsteps / every))
        ckpt = torch.empty((nseg, 2, n, 3), dtype=torch.float64, device=x.device)
        with _OnTorchStream(lib, x.device) as stream:
            lib.check(lib.lib.gh_adjoint_forward(lib.handle, _p(x), _p(v), _p(mm), n, float(dt),
                                                 float(eps), int(precision), int(nsteps),
                                                 int(every), _p(ckpt), stream))
        ctx.save_for_backward(mm, ckpt)
        ctx.kept = False
        ctx.params = (float(dt), float(eps), int(precision), int(nsteps), int(every))
        return x, v

    @staticmethod
    def _forward_kept(ctx, lib, x, v, mm, dt, eps, precision, nsteps):
        n = x.shape[0]
        half = torch.empty((nsteps, n, 3), dtype=torch.float64, device=x.device)
        order = torch.empty((nsteps, n), dtype=torch.int32, device=x.device)
        ordered = ctypes.c_int(0)
        with _OnTorchStream(lib, x.device) as stream:
            lib.check(lib.lib.gh_adjoint_forward_kept(lib.handle, _p(x), _p(v), _p(mm), n, dt,
                                                      eps, precision, nsteps, _p(half),
                                                      _p(order), ctypes.byref(ordered), stream))
        ctx.save_for_backward(mm, half)
        ctx.kept = True
        # indices, so not among the saved tensors: a hook may round what it packs
        ctx.order = order if ordered.value else None
        ctx.params = (dt, eps, precision, nsteps, 0)
        return x, v

    @staticmethod
    def backward(ctx, gx, gv):
        mm, ckpt = ctx.saved_tensors
        dt, eps, precision, nsteps, every = ctx.params
        n = mm.shape[0]
        dev = mm.device
        lx = (gx if gx is not None else torch.zeros((n, 3), device=dev)).to(
            torch.float64).contiguous().clone()
        lv = (gv if gv is not None else torch.zeros((n, 3), device=dev)).to(
            torch.float64).contiguous().clone()
        lm = torch.empty(n, dtype=torch.float64, device=dev)
        lib = _native.default_context()
        with _OnTorchStream(lib, dev) as stream:
            if ctx.kept:
                order = None if ctx.order is None else _p(ctx.order)
                lib.check(lib.lib.gh_adjoint_backward_kept(lib.handle, _p(ckpt), order, _p(mm),
                                                           n, dt, eps, nsteps, _p(lx), _p(lv),
                                                           _p(lm), stream))
                if not _graph_is_kept():
                    ctx.order = None  # with the saved tensors
            else:
                lib.check(lib.lib.gh_adjoint_backward(lib.handle, _p(ckpt), _p(mm), n, dt, eps,
                                                      precision, nsteps, every, _p(lx), _p(lv),
                                                      _p(lm), stream))
        return lx, lv, lm, None, None, None, None, None


def leapfrog(x0, v0, m, dt, eps, nsteps, checkpoint_every=None, precision="fp32"):
    """Final (x, v) after nsteps drift-kick-drift steps, differentiable in x0, v0, m.
    checkpoint_every: the steps between checkpoints (None: KEEP_BYTES decides, see above)."""
    every = None if checkpoint_every is None else int(checkpoint_every)
    return DirectLeapfrog.apply(x0, v0, m, dt, eps, int(nsteps), every,
                                _native.PRECISIONS[precision])
