"""Fused LM head + causal cross-entropy without materialising full fp32 logits.

New here (the reference materialises [B,S,V] logits: ``qwen3_triton/_model.py:131-132``
``lm_head`` then ``kernels/loss.py:46-71``).  On the matrix cores one GEMM over the vocabulary forms the
logits and folds them into per-row (max, sum-exp) partials plus the target logit; a final merge gives lse and
the token-mean loss.  Whole 8-token groups at a ``chunk`` of whole 8-column groups also keep the logits in the
activation dtype (bf16: the reference's own lm_head output, whose [T, V] copy it materialises too) and take the
statistics from those stored values; the backward turns them in place into dz = (softmax - onehot) * up / count
and forms dW = dz^T . h and dX = dz . W from them as they lie, one GEMM each (a second backward forms the consumed
logits again).  Elsewhere the statistics and dz come from fp32 logits, which the backward recomputes: in the epilogue
of a second logits GEMM (for token counts off that grid by chunks of ``chunk`` vocabulary columns, dX summed over
them in fp32: no [T, V] buffer), or, for other types and widths, in one reusable fp32 [T, chunk] buffer.  The same
math as ``linear`` followed by ``causal_cross_entropy``.
"""
import torch

from . import _ops
from .linear import MAX_LD, gemm, gemm_nt_into, gemm_ok, matmul_into

DEFAULT_CHUNK = 16384


def _mfma_ok(x, w):
    return x.dtype in (torch.bfloat16, torch.float16) and x.shape[-1] % 8 == 0 and w.shape[0] % 8 == 0


def _chunk_logits(x, w, c0, n, zbuf):
    """zbuf[:, :n] = x . w[c0:c0+n]^T in fp32."""
    t, h = x.shape
    if _mfma_ok(x, w):
        gemm_nt_into(x, h, w[c0:c0 + n], h, zbuf, t, n, h)
    else:
        matmul_into(x, w[c0:c0 + n].t(), zbuf[:, :n])


def _fused_ok(x, w):
    """The logits GEMM's statistics and gradient epilogues, and q3_gemm over the [T, V] dz (row stride V)."""
    return _mfma_ok(x, w) and x.shape[-1] % 64 == 0 and gemm_ok(x, w) and w.shape[0] < MAX_LD


def _stored_logits(x, w, tgt):
    """(statistics, logits [T, V] in the activation dtype): the statistics are of the stored, rounded logits."""
    t, v = x.shape[0], w.shape[0]
    st = _ops.CEState(t, -(-v // 128), x.device)   # a partial per 128 columns
    z = torch.empty((t, v), device=x.device, dtype=x.dtype)
    st.gemm_stats_store(0, x, w, 0, v, tgt, z)
    return st, z


class _LMHeadCE(torch.autograd.Function):
    @staticmethod
    def forward(ctx, hidden, weight, labels, ignore_index, chunk):
        if not hidden.is_cuda or hidden.ndim != 3 or weight.ndim != 2 or weight.shape[1] != hidden.shape[-1]:
            raise ValueError('ROCm hidden [B,S,H] and weight [V,H] required')
        if labels.shape != hidden.shape[:2] or labels.dtype != torch.int64 or labels.device != hidden.device:
            raise ValueError('int64 [B,S] labels on the hidden device required')
        if hidden.dtype != weight.dtype or not hidden.is_contiguous() or not weight.is_contiguous():
            raise ValueError('Contiguous hidden/weight of one dtype required')
        b, s, h = hidden.shape
        v = weight.shape[0]
        if s < 2:
            raise ValueError('At least 2 tokens required')
        x = hidden.view(b * s, h)
        tgt = _ops.ce_shift_labels(labels, ignore_index)
        chunk = min(chunk, v)
        nch = -(-v // chunk)
        z = None
        if _fused_ok(x, weight):
            if (b * s) % 8 == 0 and chunk % 8 == 0:
                st, z = _stored_logits(x, weight, tgt)
            else:
                st = _ops.CEState(b * s, -(-v // 128), hidden.device)
                st.gemm_stats(0, x, weight, 0, v, tgt)
        else:
            st = _ops.CEState(b * s, nch, hidden.device)
            zbuf = torch.empty((b * s, chunk), device=hidden.device, dtype=torch.float32)
            for c in range(nch):
                c0 = c * chunk
                n = min(chunk, v - c0)
                _chunk_logits(x, weight, c0, n, zbuf)
                st.stats(c, zbuf, chunk, n, c0, tgt)
        loss = st.finish(tgt, v, ignore_index)
        ctx.save_for_backward(hidden, weight, tgt, st.lse, st.count)
        ctx.ignore, ctx.chunk = ignore_index, chunk
        ctx.z = z
        return loss.clone()

    @staticmethod
    def backward(ctx, dy):
        hidden, weight, tgt, lse, count = ctx.saved_tensors
        b, s, h = hidden.shape
        v, t, chunk = weight.shape[0], b * s, ctx.chunk
        x = hidden.view(t, h)
        up = dy.float().contiguous()
        mfma = _mfma_ok(x, weight) and t % 8 == 0
        z, ctx.z = ctx.z, None   # consumed: dz overwrites the stored logits in place
        fused = _fused_ok(x, weight)
        if mfma and fused:   # [T, V] dz
            if chunk % 8:
                z = torch.empty((t, v), device=x.device, dtype=x.dtype)
                _ops.gemm_ce_grad(x, weight, 0, v, tgt, lse, count, up, z, v, ctx.ignore)
            else:
                if z is None:   # a second backward: the logits that lse was formed from, again
                    z = _stored_logits(x, weight, tgt)[1]
                _ops.ce_grad(z, v, v, 0, tgt, lse, count, up, z, v, v, ctx.ignore)
            dx = dw = None
            if ctx.needs_input_grad[1]:
                dw = torch.empty_like(weight)
                gemm([z], [x], [dw], v, h, t, kmajor=(True, True))
            if ctx.needs_input_grad[0]:
                dx = torch.empty((t, h), device=x.device, dtype=x.dtype)
                gemm([z], [weight], [dx], t, h, v, kmajor=(False, True))
                dx = dx.view(b, s, h)
            return dx, dw, None, None, None
        dw = torch.empty_like(weight)
        zbuf = None if fused else torch.empty((t, chunk), device=x.device, dtype=torch.float32)
        dz = torch.empty((t, chunk), device=x.device, dtype=x.dtype)
        dx = torch.empty((t, h), device=x.device, dtype=torch.float32)
        if mfma:
            wt = _ops.transpose_last2(weight, pad_to=8)   # [H, Vp]
            xt = _ops.transpose_last2(x)                  # [H, T]
        for c in range(-(-v // chunk)):
            c0 = c * chunk
            n = min(chunk, v - c0)
            if fused:
                _ops.gemm_ce_grad(x, weight, c0, n, tgt, lse, count, up, dz, v, ctx.ignore)
            else:
                _chunk_logits(x, weight, c0, n, zbuf)
                _ops.ce_grad(zbuf, chunk, n, c0, tgt, lse, count, up, dz, chunk, v, ctx.ignore)
            if mfma:
                gemm_nt_into(dz, chunk, wt[:, c0:], wt.shape[1], dx, t, h, n, accumulate=c > 0)
                dzt = _ops.transpose_last2(dz)            # [chunk, T]
                gemm_nt_into(dzt, t, xt, t, dw[c0:c0 + n], n, h, t)
            else:
                matmul_into(dz[:, :n], weight[c0:c0 + n], dx, accumulate=c > 0)
                matmul_into(dz[:, :n].t(), x, dw[c0:c0 + n])
        return _ops.cast(dx, x.dtype).view(b, s, h), dw, None, None, None


def lm_head_cross_entropy(hidden, weight, labels, *, ignore_index=-100, chunk=DEFAULT_CHUNK):
    """Causal token-mean CE of ``hidden @ weight.T`` against ``labels`` (shift inside), fused."""
    return _LMHeadCE.apply(hidden, weight, labels, ignore_index, chunk)
