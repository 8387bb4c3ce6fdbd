"""q3_gemm's rules on the host: what it takes, and the launches and tiles that it plans (nothing runs)."""
import ctypes

import pytest
import torch

from qwen3_triton import _hip as H
from qwen3_triton.kernels import linear


def desc(layout, m, n, k, *, epilogue=H.GEMM_PLAIN, axis=0, parts=(), lda=None, ldb=None):
    """A call on made-up aligned addresses; ``parts`` are the pieces along ``axis``."""
    d = H.GemmDesc()
    d.dtype, d.a_kmajor, d.b_kmajor = H.BF16, layout == "TN", layout != "NT"
    d.m, d.n, d.k, d.axis, d.pieces, d.epilogue, d.eps = m, n, k, axis, max(1, len(parts)), epilogue, 1e-6
    for i in range(3):
        size = {1: k, 2: n, 3: m}
        if i < len(parts):
            size[axis] = parts[i]
            d.end[i] = sum(parts[:i + 1])
        d.a[i] = d.b[i] = d.c[i] = 1 << 20
        d.lda[i] = lda or (size[3] if layout == "TN" else size[1])
        d.ldb[i] = ldb or (size[1] if layout == "NT" else size[2])
        d.ldc[i] = size[2]
    d.res = d.norm_w = d.y = 1 << 20
    d.ldres = d.ldy = d.ldgu = n
    if epilogue in (H.GEMM_GATE_UP, H.GEMM_SWIGLU_BWD):
        d.g = d.u = 1 << 20
    return d


def plan(*args, **kw):
    """[(first row, rows, tile rows, tile columns, splits)] of a call, [] when it is refused."""
    d, out = desc(*args, **kw), (ctypes.c_int64 * 10)()
    n = H.query("q3_gemm_plan", ctypes.addressof(d), ctypes.addressof(out))
    return [tuple(out[5 * i:5 * i + 5]) for i in range(n)]


@pytest.mark.parametrize("rows,cols,ld", [(8, 8, 8), (8, 12, 16), (8, 8, 12), (40, 64, (1 << 22) - 8), (40, 64, 1 << 22),
                                          (8200, 64, 1 << 21), (113080, 151936, 151936), (1 << 20, 64, 1 << 20),
                                          ((1 << 28) - 1, 8, 8), (1 << 31, 8, 8)])
def test_python_and_c_take_the_same_operands(rows, cols, ld):
    """What gemm_ok lets through, the library takes in every role (past 2^34 elements too); what it refuses in a
    role, gemm_ok keeps from it."""
    t = torch.empty(0, dtype=torch.bfloat16, device="meta").as_strided((rows, cols), (ld, 1))
    roles = [plan("NT", rows, 8, cols, lda=ld), plan("NT", 8, rows, cols, ldb=ld),
             plan("TN", 8, cols, rows, ldb=ld), plan("TN", cols, 8, rows, lda=ld)]
    if linear._operand_ok(t):
        assert all(roles)
    else:
        assert not all(roles)


@pytest.mark.parametrize("layout,axis,epilogue", [("NT", 0, H.GEMM_RESIDUAL), ("NT", 2, 0), ("NT", 0, H.GEMM_GATE_UP),
                                                  ("NN", 1, 0), ("NN", 0, H.GEMM_SWIGLU_BWD), ("TN", 3, 0), ("TN", 0, 0)])
def test_launches_cover_every_row_once(layout, axis, epilogue):
    """The second launch, where there is one, starts at the first row that the first has not formed."""
    two = 0
    for m in range(256, 20000, 328):
        for n in (1024, 2048, 4096, 8192):
            parts = {1: (256, 256), 2: (n // 2, n // 2), 3: (m // 2 // 256 * 256, m - m // 2 // 256 * 256)}.get(axis, ())
            if 0 in parts:
                continue
            launches = plan(layout, m, n, 512, epilogue=epilogue, axis=axis, parts=parts)
            end = 0
            for first, rows, bm, bn, splits in launches:
                assert first == end and rows > 0 and (end + rows == m or rows % bm == 0)
                end += rows
            assert end == m
            two += len(launches) == 2
    assert two
