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


# kind -> (operand layout, axis of its pieces, epilogue)
KINDS = {"plain NT": ("NT", 0, H.GEMM_PLAIN), "plain NN": ("NN", 0, H.GEMM_PLAIN), "plain TN": ("TN", 0, H.GEMM_PLAIN),
         "residual NT": ("NT", 0, H.GEMM_RESIDUAL), "residual NN": ("NN", 0, H.GEMM_RESIDUAL),
         "norm": ("NT", 0, H.GEMM_RESIDUAL_NORM), "gate/up": ("NT", 0, H.GEMM_GATE_UP),
         "swiglu bwd": ("NN", 0, H.GEMM_SWIGLU_BWD), "pieces of n": ("NT", 2, H.GEMM_PLAIN),
         "pieces of k": ("NN", 1, H.GEMM_PLAIN), "pieces of m": ("TN", 3, H.GEMM_PLAIN)}
# Ragged m, n, k per kind that between them take every tile the plan chooses from, without and with a K split, and a
# second launch on tiles of 192 rows (256 where both operands are K-major) and of fewer: found by running the plan.
SHAPES = {
    "plain NT": [(17, 8, 72), (21, 8, 1624), (2087, 8, 4264), (6674, 8, 72), (420, 208, 2200), (8485, 136, 80),
        (3141, 8, 4104), (577, 8680, 72), (4061, 136, 5816), (8085, 408, 72), (4161, 8, 4360), (8839, 776, 72),
        (1357, 696, 6568), (801, 13328, 72), (8203, 144, 4104), (6343, 8080, 248), (6462, 7968, 520),
        (6559, 3976, 88)],
    "plain NN": [(2748, 8, 3168), (17, 8, 72), (17, 8, 1696), (8213, 152, 72), (5657, 8, 2136), (597, 8240, 72),
        (205, 4880, 4824), (8354, 408, 72), (1356, 408, 3920), (5697, 1288, 72), (4557, 136, 5464), (8106, 1304, 72),
        (8853, 144, 4104), (8399, 8024, 200), (7161, 8088, 136), (6571, 4008, 72)],
    "plain TN": [(2736, 8, 3194), (24, 8, 17), (24, 8, 1631), (8752, 136, 31), (6456, 8, 2054), (8568, 392, 18),
        (3664, 136, 4384), (5560, 1440, 18), (8224, 144, 3263), (8208, 4056, 25), (3072, 8080, 77), (3136, 8008, 24)],
    "residual NT": [(17, 8, 72), (17, 8, 1648), (2836, 8, 3080), (6697, 8, 72), (409, 200, 2272), (8607, 136, 72),
        (1348, 160, 4584), (787, 6544, 72), (193, 4504, 4968), (4525, 776, 72), (3041, 136, 3376), (8795, 808, 72),
        (8785, 136, 2728), (8223, 1296, 72), (4118, 392, 4104), (6291, 8168, 72), (4901, 8072, 72), (6180, 4008, 72)],
    "residual NN": [(4226, 8, 2152), (17, 8, 72), (17, 8, 1672), (8685, 136, 72), (3094, 8, 4104), (390, 11344, 72),
        (4071, 144, 5984), (5325, 656, 72), (1795, 264, 4104), (8205, 800, 72), (8293, 144, 2464), (8543, 1304, 72),
        (8625, 152, 4104), (6318, 8168, 200), (6411, 8184, 72), (6566, 4088, 72)],
    "norm": [(17, 8, 72), (17, 8, 1032), (8369, 8, 1032), (6597, 8, 72), (391, 456, 1032), (8737, 136, 72),
        (1471, 152, 4576), (1163, 4624, 72), (212, 5072, 4104), (7950, 408, 72), (8487, 136, 1032), (6583, 1048, 72),
        (6228, 136, 4104), (8639, 1296, 72), (197, 6536, 4872), (6357, 8096, 136), (4996, 8120, 112),
        (6219, 4016, 136)],
    "gate/up": [(17, 8, 72), (391, 496, 72), (66, 8360, 72), (194, 8488, 72), (257, 6328, 72), (267, 11664, 72),
        (431, 10920, 72), (8401, 4088, 72), (4889, 3984, 112), (3090, 4040, 72)],
    "swiglu bwd": [(17, 8, 72), (8229, 144, 72), (405, 11000, 72), (4505, 800, 72), (6754, 1072, 72),
        (8487, 1288, 72), (6219, 8080, 136), (5087, 8072, 520), (6519, 3888, 72)],
    "pieces of n": [(17, 8, 72), (17, 8, 1672), (5451, 24, 72), (1395, 32, 2168), (2183, 24, 72), (257, 24, 4104),
        (7553, 24, 72), (1945, 24, 2272), (8351, 432, 72), (3143, 440, 2872), (5430, 416, 72), (1298, 24, 4376),
        (5399, 1312, 72), (1401, 432, 5416), (1163, 9592, 72), (2798, 432, 4104), (6197, 7984, 520),
        (6442, 7952, 200), (6290, 4088, 104)],
    "pieces of k": [(4161, 8, 2128), (17, 8, 72), (17, 8, 1680), (8244, 144, 72), (3083, 8, 4104), (438, 11128, 72),
        (2044, 408, 7592), (8250, 400, 72), (2955, 144, 3160), (8818, 784, 72), (4718, 136, 4920), (6931, 1608, 72),
        (4278, 392, 4104), (6207, 7984, 136), (5065, 8184, 104), (3291, 8168, 72)],
    "pieces of m": [(4232, 8, 2178), (24, 8, 18), (24, 8, 1634), (224, 6096, 20), (1440, 136, 4457), (224, 10992, 23),
        (232, 2192, 6045), (408, 15864, 18), (424, 1912, 6853), (8360, 3928, 77), (6096, 3960, 23),
        (3296, 8008, 139)],
}


def pieces(kind, m, n, k):
    """Three pieces along the kind's axis (one where it is too short), those along m whole 256-row tiles where that
    leaves any (the condition of a second launch)."""
    axis = KINDS[kind][1]
    size = (0, k, n, m)[axis]
    a = size // 3 // 256 * 256 or size // 3 // 8 * 8
    return () if axis == 0 else (a, a, size - 2 * a) if a else (size,)


def planned(kind, m, n, k):
    layout, axis, epilogue = KINDS[kind]
    return plan(layout, m, n, k, axis=axis, epilogue=epilogue, parts=pieces(kind, m, n, k))


@pytest.mark.parametrize("kind", KINDS)
def test_shapes_take_every_tile(kind):
    """The shapes that the GPU tests compare still reach every tile (a changed plan needs other shapes)."""
    layout, axis, epilogue = KINDS[kind]
    calls = [planned(kind, *s) for s in SHAPES[kind]]
    assert all(calls)
    tiles = {(64, 64), (64, 128), (128, 128), (128, 256), (256, 256)}
    tiles |= {(192, 128), (192, 256)} if layout != "TN" else set()
    tiles |= {(32, 64)} if layout == "NT" else set()
    one = {c[0][2:4] for c in calls if len(c) == 1 and c[0][4] == 1}
    assert one >= tiles - {(64, 64)}   # 64 x 64: two workgroups per CU, chosen with a split
    if epilogue not in (H.GEMM_GATE_UP, H.GEMM_SWIGLU_BWD):
        assert {c[0][2:4] for c in calls if c[0][4] > 1} >= tiles
    rest = {c[1][2] for c in calls if len(c) == 2}
    assert max(rest) == (256 if layout == "TN" else 192) and min(rest) < 192
