"""Which kernel a call runs on (yr_hip_fused_plan, host only)."""
import ctypes

import pytest

from product_tiles import KN, NK, STAGED, TILES
from yirage_amd import _lib

KINDS = {"linear": _lib.OP_LINEAR, "rmsnorm_linear": _lib.OP_RMSNORM_LINEAR, "gated_mlp": _lib.OP_GATED_MLP}
ONE_ROW, PRODUCT, ATTENTION = 0, 1, 2


def product_plan(kind, M, K, N, layout, aligned=True):
    """kernel, rows, columns, splits, row pass, through registers"""
    p = (ctypes.c_int64 * 6)(M, K, N, _lib.DTYPE_BF16, layout, 0)
    plan = (ctypes.c_int * 6)()
    n = 6 if kind == _lib.OP_RMSNORM_LINEAR else 5
    assert _lib.lib().yr_hip_fused_plan(kind, n, p, int(aligned), plan) == 0, _lib.last_error()
    return tuple(plan)


@pytest.mark.parametrize("kind", [_lib.OP_LINEAR, _lib.OP_RMSNORM_LINEAR, _lib.OP_GATED_MLP])
@pytest.mark.parametrize("layout", [_lib.W_NK, _lib.W_KN])
@pytest.mark.parametrize("M,K,N", [(1, 4096, 4096), (16, 3000, 72), (40, 1096, 200), (130, 584, 392),
                                   (300, 2056, 264), (2048, 4096, 14336)])
def test_unaligned_operands_pass_through_registers(kind, layout, M, K, N):
    """Direct loads into LDS need 16-byte aligned operands; others take a tile
    that loads through registers, within the same workspace."""
    assert product_plan(kind, M, K, N, layout)[5] == 0
    kernel, rows, cols, splits, row_pass, staged = product_plan(kind, M, K, N, layout, aligned=False)
    if kernel == ONE_ROW:  # loads x and W through registers always
        return
    assert kernel == PRODUCT and staged == 1 and row_pass == 0 and (rows, cols) in ((32, 128), (64, 128))
    name = {_lib.OP_LINEAR: "linear", _lib.OP_RMSNORM_LINEAR: "rmsnorm_linear", _lib.OP_GATED_MLP: "gated_mlp"}[kind]
    have = getattr(_lib.lib(), f"yr_hip_{name}_workspace")(M, K, N, _lib.DTYPE_BF16, layout)
    if splits > 1:
        ncol = cols // 2 if kind == _lib.OP_GATED_MLP else cols
        records = -(-M // rows) * -(-N // ncol) * splits * rows * cols * 4
        assert 64 * 1024 + records <= have


@pytest.mark.parametrize("kind", [_lib.OP_LINEAR, _lib.OP_RMSNORM_LINEAR, _lib.OP_GATED_MLP])
def test_longest_k(kind):
    """K of 2^26 and more while the rows of x and the weights stay below 4 GiB;
    one row on N x K weights as far as the one-row kernel's grid reaches."""
    K = 1 << 26
    for M, N, layout, kernel in ((1, 8, _lib.W_NK, ONE_ROW), (1, 8, _lib.W_KN, PRODUCT), (3, 16, _lib.W_KN, PRODUCT),
                                 (31, 8, _lib.W_KN, PRODUCT), (20, 8, _lib.W_NK, PRODUCT)):
        assert product_plan(kind, M, K, N, layout)[0] == kernel
    assert product_plan(kind, 1, 65535 * 2048, 8, _lib.W_NK)[0] == ONE_ROW
    for M, k, layout in ((2, K, _lib.W_NK), (32, K, _lib.W_KN), (1, 65536 * 2048, _lib.W_NK)):
        p = (ctypes.c_int64 * 6)(M, k, 8, _lib.DTYPE_BF16, layout, 0)
        n = 6 if kind == _lib.OP_RMSNORM_LINEAR else 5
        assert _lib.lib().yr_hip_fused_plan(kind, n, p, 1, (ctypes.c_int * 6)()) != 0


def test_product_scratch_is_bounded():
    """The workspace of a stream lives as long as the process: 64 MiB of K-split
    records and 128 MiB for the row pass's copy of x, whatever the shape."""
    lib = _lib.lib()
    most = 64 * 1024 + (64 << 20) + (128 << 20) + 4 * 8192 + 512
    for M in (256, 257, 700, 1110, 1654, 2048, 4096, 8192, 8193, 20000):
        for K in (1024, 4096, 6648, 13984, 14336, 28672, 1 << 18):
            for N in (256, 3376, 4096, 7744, 11848, 14336):
                for layout in (_lib.W_NK, _lib.W_KN):
                    for kind in ("linear", "rmsnorm_linear", "gated_mlp"):
                        b = getattr(lib, f"yr_hip_{kind}_workspace")(M, K, N, _lib.DTYPE_F16, layout)
                        assert b <= most, (kind, M, K, N, layout, b)


def test_few_rows_of_rmsnorm_fill_the_chip():
    """Up to 16 rows are bound by the weights: the CU with the most workgroups
    has at most half as many again as the average one."""
    worst, total, n = 0.0, 0.0, 0
    for K in (2048, 3072, 4096, 5120, 8192, 11264):
        for N in (2048, 3072, 4096, 5120, 6144, 7168, 8192, 9216, 10240, 11264, 14336):
            if K * N * 2 < 16 << 20:
                continue
            for M in (1, 8, 16):
                _, _, cols, splits, _, _ = product_plan(_lib.OP_RMSNORM_LINEAR, M, K, N, _lib.W_KN)
                groups = -(-N // cols) * splits
                uneven = -(-groups // 256) * 256 / groups
                worst, total, n = max(worst, uneven), total + uneven, n + 1
    assert worst <= 1.5 and total / n <= 1.2


@pytest.mark.parametrize("kind,K,N,kernel", [
    (_lib.OP_RMSNORM_LINEAR, 2048, 14336, ONE_ROW), (_lib.OP_RMSNORM_LINEAR, 10240, 1024, ONE_ROW),
    (_lib.OP_RMSNORM_LINEAR, 4096, 4096, ONE_ROW), (_lib.OP_RMSNORM_LINEAR, 4096, 4104, PRODUCT),
    (_lib.OP_LINEAR, 2048, 8192, ONE_ROW), (_lib.OP_LINEAR, 2048, 8200, PRODUCT),
    (_lib.OP_LINEAR, 9224, 952, ONE_ROW), (_lib.OP_LINEAR, 14336, 4096, PRODUCT),
    (_lib.OP_GATED_MLP, 2048, 7168, ONE_ROW), (_lib.OP_GATED_MLP, 2048, 8200, PRODUCT),
    (_lib.OP_GATED_MLP, 2056, 1024, PRODUCT),
])
def test_one_row_of_n_by_k_weights(kind, K, N, kernel):
    """Both sides of the rule; it never holds for K x N weights or two rows."""
    assert product_plan(kind, 1, K, N, _lib.W_NK)[0] == kernel
    assert product_plan(kind, 1, K, N, _lib.W_KN)[0] == product_plan(kind, 2, K, N, _lib.W_NK)[0] == PRODUCT


def test_every_tile_has_its_shapes():
    """The shapes of product_tiles.py get the tile they stand for, all tiles are
    there, and every one of them leaves partial tiles and a partial chunk."""
    for (op, layout, rows, cols, row_pass), shapes in TILES.items():
        for split, (M, K, N) in enumerate(shapes):
            kernel, r, c, s, p, staged = product_plan(KINDS[op], M, K, N, layout)
            assert (kernel, r, c, s > 1, p, staged) == (PRODUCT, rows, cols, split == 1, row_pass, 0), (op, M, K, N)
            ncols = cols // 2 if op == "gated_mlp" else cols
            assert M % rows and N % ncols and K % 64 and (s > 1 or K >= 840)
    for (op, layout, rows, cols), shapes in STAGED.items():
        for split, (M, K, N) in enumerate(shapes):
            kernel, r, c, s, p, staged = product_plan(KINDS[op], M, K, N, layout, aligned=False)
            assert (kernel, r, c, s > 1, p, staged) == (PRODUCT, rows, cols, split == 1, 0, 1), (op, M, K, N)
            assert M % rows and N % (cols // 2 if op == "gated_mlp" else cols) and K % 64
    assert len(STAGED) == 3 * 2 * 2
    small, large = [(32, 64), (32, 128), (64, 128)], [(128, 128), (128, 192), (128, 256), (256, 256)]
    for layout in (NK, KN):
        for r, c in small + large:
            assert ("linear", layout, r, c, False) in TILES
            assert ("rmsnorm_linear", layout, r, c, (r, c) in large) in TILES
            assert (("gated_mlp", layout, r, c, False) in TILES) == ((r, c) not in ((32, 64), (128, 192)))


@pytest.mark.parametrize("G,M,L,d,rows,split", [
    (3, 16, 264, 64, 16, True), (515, 3, 136, 64, 16, False), (2, 5, 328, 128, 16, True),
    (1, 33, 520, 128, 32, True), (4, 64, 4096, 64, 32, True), (260, 65, 8, 128, 64, False),
    (9, 3601, 72, 128, 64, False), (5, 13001, 72, 64, 64, False), (5, 13057, 72, 64, 128, False),
    (6, 11009, 1544, 64, 128, False),
])
def test_graph_attention_tiles(G, M, L, d, rows, split):
    """Rows of a workgroup and whether tokens are split; tests/test_gpu_graph_attn.py
    runs these shapes."""
    strides = [M * d, d, 1, d * L, L, 1, L * d, d, 1, M * d, d, 1]
    p = (ctypes.c_int64 * 18)(G, M, L, d, _lib.DTYPE_F16, 0, *strides)
    plan = (ctypes.c_int * 6)()
    assert _lib.lib().yr_hip_fused_plan(_lib.OP_ATTENTION, 18, p, 1, plan) == 0, _lib.last_error()
    assert plan[0] == ATTENTION and plan[1] == rows and (plan[3] > 1) == split, list(plan)
