"""Gate/up projections + SwiGLU as one autograd op.

Mirrors ``qwen3_triton/kernels/mlp_precision.py:16-66`` (``_GateUp`` / ``gate_up_swiglu``):
forward G = X Wg^T, U = X Wu^T, Y = silu(G)*U, saving G and U -- one matrix-core GEMM over both
weights with the SwiGLU in its epilogue (``q3_gemm``), else two GEMMs and the SwiGLU kernel; backward =
SwiGLU backward, dX = dG Wg + dU Wu (fp32 accumulation across both products, one rounding), dWg = dG^T X,
dWu = dU^T X, each pair one launch over the two pieces.
"""
import torch

from .. import _hip as H
from . import _ops
from .linear import MAX_LD, chunk_aligned, gemm, gemm_ok, linear, linear_residual, matmul, matmul_into


def _check(x, wg, wu):
    if not x.is_cuda or x.ndim < 2 or wg.ndim != 2 or wg.shape != wu.shape or x.shape[-1] != wg.shape[1]:
        raise ValueError('Expected ROCm X[...,K] and matching [N,K] gate/up weights')
    if x.dtype not in (torch.float32, torch.bfloat16, torch.float16) or \
            any(t.device != x.device or t.dtype != x.dtype or not t.is_contiguous() for t in (x, wg, wu)):
        raise ValueError('Matching contiguous floating point ROCm inputs required')
    m, k, n = x.numel() // x.shape[-1], x.shape[-1], wg.shape[0]
    if min(m, k, n) < 1:
        raise ValueError('Nonempty inputs required')
    return m, k, n


def _new(like, *shape):
    return torch.empty(shape, device=like.device, dtype=like.dtype)


def _gate_up_ok(flat, wg, wu):
    return wg.shape[0] % 8 == 0 and wg.shape[0] < MAX_LD and gemm_ok(flat, wg, wu)


def _gate_up_y(x, wg, wu):
    """Y alone (no autograd: nothing is saved, so the fused GEMM skips the G and U stores)."""
    m, k, n = _check(x, wg, wu)
    flat = x.view(m, k)
    if _gate_up_ok(flat, wg, wu):
        y = _new(x, m, n)
        gemm([flat], [wg, wu], [y], m, n, k, epilogue=H.GEMM_GATE_UP)
    else:
        y = _ops.swiglu_fwd(matmul(flat, wg.t()), matmul(flat, wu.t()))
    return y.view(*x.shape[:-1], n)


def _gate_up_forward(flat, wg, wu, m, n, k):
    if _gate_up_ok(flat, wg, wu):
        g, u, y = (_new(flat, m, n) for _ in range(3))
        gemm([flat], [wg, wu], [y], m, n, k, epilogue=H.GEMM_GATE_UP, g=g, u=u)
        return g, u, y
    g = matmul(flat, wg.t())
    u = matmul(flat, wu.t())
    return g, u, _ops.swiglu_fwd(g, u)


def _gate_up_grads(flat, wg, wu, dg, du, m, n, k, need):
    """(dX, dWg, dWu) of G = X Wg^T, U = X Wu^T from dg, du; ``need`` says which (weights together)."""
    dx = dwg = dwu = None
    if need[0]:
        dx = _new(flat, m, k)
        gemm([dg, du], [wg, wu], [dx], m, k, 2 * n, kmajor=(False, True), axis=1)
    if need[1] or need[2]:
        dwg, dwu = _new(flat, n, k), _new(flat, n, k)
        gemm([dg, du], [flat], [dwg, dwu], 2 * n, k, m, kmajor=(True, True), axis=3)
    return dx, dwg, dwu


class _GateUp(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, wg, wu, optimized):
        m, k, n = _check(x, wg, wu)
        g, u, y = _gate_up_forward(x.view(m, k), wg, wu, m, n, k)
        ctx.save_for_backward(x, wg, wu, g, u)
        return y.view(*x.shape[:-1], n)

    @staticmethod
    def backward(ctx, dy):
        x, wg, wu, g, u = ctx.saved_tensors
        m, k, n = x.numel() // x.shape[-1], x.shape[-1], wg.shape[0]
        flat = x.view(m, k)
        dyf = dy.contiguous().view(m, n)
        dg, du = _ops.swiglu_bwd(g, u, dyf)
        if _gate_up_ok(flat, wg, wu):
            dx, dwg, dwu = _gate_up_grads(flat, wg, wu, dg, du, m, n, k, ctx.needs_input_grad)
            return None if dx is None else dx.view(x.shape), dwg, dwu, None
        acc = torch.empty((m, k), device=x.device, dtype=torch.float32)
        matmul_into(dg, wg, acc)
        matmul_into(du, wu, acc, accumulate=True)
        dx = _ops.cast(acc, x.dtype).view(x.shape)
        dwg = matmul(dg.t(), flat)
        dwu = matmul(du.t(), flat)
        return dx, dwg, dwu, None


def gate_up_swiglu(x, gate_weight, up_weight, *, optimized=False):
    """``kernels/mlp_precision.py:65``.  Without autograd (inference, or no input needing a gradient)
    only Y is formed: the same values, without the G and U the backward would need."""
    if not (torch.is_grad_enabled() and any(t.requires_grad for t in (x, gate_weight, up_weight))):
        return _gate_up_y(x, gate_weight, up_weight)
    return _GateUp.apply(x, gate_weight, up_weight, optimized)


class _MLPBlock(torch.autograd.Function):
    """out = (silu(X Wg^T) * (X Wu^T)) Wd^T as one op, so the backward can run the SwiGLU backward in the
    epilogue of the down projection's input-gradient GEMM: dY never reaches memory.  Every GEMM and
    rounding point is the one of ``gate_up_swiglu`` followed by ``linear``."""

    @staticmethod
    def forward(ctx, x, wg, wu, wd, res):
        m, k, n = x.numel() // x.shape[-1], x.shape[-1], wg.shape[0]
        h = wd.shape[0]
        g, u, y = _gate_up_forward(x.view(m, k), wg, wu, m, n, k)
        out = _new(x, m, h)
        if res is None:
            gemm([y], [wd], [out], m, h, n)
        else:  # the residual sum rides in the down GEMM's epilogue
            gemm([y], [wd], [out], m, h, n, epilogue=H.GEMM_RESIDUAL, res=res.view(m, h))
        ctx.save_for_backward(x, wg, wu, wd, g, u, y)
        ctx.has_res = res is not None
        return out.view(*x.shape[:-1], h)

    @staticmethod
    def backward(ctx, dout):
        x, wg, wu, wd, g, u, y = ctx.saved_tensors
        m, k, n = x.numel() // x.shape[-1], x.shape[-1], wg.shape[0]
        h = wd.shape[0]
        need = ctx.needs_input_grad
        dof = chunk_aligned(dout).view(m, h)
        dwd = dx = dwg = dwu = None
        if need[3]:
            dwd = _new(x, h, n)
            gemm([dof], [y], [dwd], h, n, m, kmajor=(True, True))
        if any(need[:3]):
            dg, du = _new(x, m, n), _new(x, m, n)
            gemm([dof], [wd], [dg, du], m, n, h, kmajor=(False, True), epilogue=H.GEMM_SWIGLU_BWD, g=g, u=u)
            dx, dwg, dwu = _gate_up_grads(x.view(m, k), wg, wu, dg, du, m, n, k, need)
        return None if dx is None else dx.view(x.shape), dwg, dwu, dwd, (dout if ctx.has_res else None)


def mlp_block(x, gate_weight, up_weight, down_weight, *, optimized=False, residual=None):
    """down(silu(gate(x)) * up(x)) (+ ``residual``) -- ``components.py`` MLP: ``gate_up_swiglu`` then the
    down ``linear`` (then the residual sum) -- with the fused backward above when every operand suits
    the matrix-core epilogue (16-bit contiguous operands, feature counts multiples of 8); otherwise
    exactly that composition."""
    m, k, n = x.numel() // x.shape[-1], x.shape[-1], gate_weight.shape[0]
    ok = x.is_cuda and x.ndim >= 2 and x.is_contiguous() and gate_weight.ndim == down_weight.ndim == 2 and \
        down_weight.shape[1] == n and gate_weight.shape == up_weight.shape and gate_weight.shape[1] == k and \
        all(t.dtype == x.dtype and t.device == x.device and t.is_contiguous()
            for t in (gate_weight, up_weight, down_weight)) and \
        x.dtype in (torch.bfloat16, torch.float16) and m > 0 and n % 8 == 0 and down_weight.shape[0] % 8 == 0 and \
        down_weight.shape[0] < MAX_LD and \
        gemm_ok(x.view(m, k), gate_weight, up_weight, down_weight)
    if residual is not None:
        ok = ok and residual.is_contiguous() and residual.dtype == x.dtype and residual.device == x.device and \
            residual.shape == (*x.shape[:-1], down_weight.shape[0])
    if not ok:
        y = gate_up_swiglu(x, gate_weight, up_weight, optimized=optimized)
        if residual is None:
            return linear(y, down_weight, optimized=optimized)
        return linear_residual(y, down_weight, residual, optimized=optimized)
    return _MLPBlock.apply(x, gate_weight, up_weight, down_weight, residual)
