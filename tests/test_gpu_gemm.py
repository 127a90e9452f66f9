"""GPU parity of the matrix-product kernel (csrc/gemm_kernel.h): rows, columns
and K around the tile sizes and the 64-k chunk, every epilogue, both weight
layouts, and every tile, whole and with K splits (product_tiles.py).

Reference: float64 products of the same 16-bit inputs, x * gamma rounded to
the storage type first (the operand the kernels form).  Tolerance: the fp32
sums differ from it by less than K 2^-24 sum|x w| <= 2e-3 here, and the
result is rounded once to 16 bits (2^-9 relative for bf16): 1e-2 covers both.
"""
import pytest
import torch

from product_tiles import STAGED, TILES

pytestmark = pytest.mark.gpu

NK, KN = 0, 1


def _case(M, K, N, layout, dtype, gen):
    x = torch.randn((M, K), generator=gen).to(dtype).cuda()
    shape = (K, N) if layout == KN else (N, K)
    ws = [(torch.randn(shape, generator=gen) * K ** -0.5).to(dtype).cuda() for _ in range(2)]
    gamma = (1 + 0.1 * torch.randn(K, generator=gen)).to(dtype).cuda()
    res = torch.randn((M, N), generator=gen).to(dtype).cuda()
    return x, ws, gamma, res


def _check(got, ref, what):
    err = (got.double() - ref).abs()
    bad = err > 1e-2 + 1e-2 * ref.abs()
    print(f"[{what}] max err {err.max().item():.2e}", flush=True)
    assert not bad.any(), f"{what}: {int(bad.sum())} of {bad.numel()} outside 1e-2"


@pytest.mark.parametrize("layout", [NK, KN])
@pytest.mark.parametrize("M,K,N", [
    (1, 8, 8),             # the one-row kernel (N x K)
    (1, 2056, 40),         # its second K slice; the product kernel's for the gated MLP
    (1, 2048, 6152),
    (1, 2048, 8200),       # the other side of its rule for linear and gated
    (2, 1096, 136),        # the smallest row tile, mostly empty
    (16, 3000, 72),        # many K splits of one column tile
    (17, 8, 8),            # one chunk of 8 k, one column group
    (31, 72, 72),          # a chunk and a piece; a tile and a piece of columns
    (32, 1000, 520),       # whole rows of the 32-row tiles, a partial last chunk
    (33, 1024, 200),       # one row more, whole chunks
    (64, 2056, 136),       # K splits of unequal length
    (65, 640, 1096),       # one row more than two 32-row tiles
    (127, 4096, 72),       # many K splits of two column tiles
    (129, 584, 392),
    (250, 1216, 2056),     # the 128-column tiles of 32 and 64 rows
    (257, 64, 264),        # RMSNorm by its row pass from here on; a single chunk
    (600, 1088, 1544),     # 32, 64 and, for RMSNorm, 128 rows
])
def test_tile_edges(M, K, N, layout):
    import yirage_amd.fused as F

    print(f"case gemm M={M} K={K} N={N} layout={layout}", flush=True)
    gen = torch.Generator().manual_seed(M * 7 + K)
    dtype = torch.bfloat16 if (M + K // 8) % 2 else torch.float16
    x, (w, w3), gamma, res = _case(M, K, N, layout, dtype, gen)
    wd, w3d = ((t if layout == KN else t.t()).double() for t in (w, w3))
    xd = x.double()
    for residual in (None, res):
        out = F.linear(x, w, residual=residual, w_layout=layout)
        _check(out, xd @ wd + (0 if residual is None else res.double()), "linear")
        again = F.linear(x, w, residual=residual, w_layout=layout)  # tickets re-armed, same order of sums
        assert torch.equal(out, again)
    a = xd @ wd
    _check(F.gated_mlp(x, w, w3, w_layout=layout), a * torch.sigmoid(a) * (xd @ w3d), "gated_mlp")
    rs = torch.rsqrt((xd * xd).mean(-1, keepdim=True) + 1e-6)
    _check(F.rmsnorm_linear(x, gamma, w, w_layout=layout), ((x * gamma).double() @ wd) * rs, "rmsnorm_linear")
    _check(F.rmsnorm_linear(x, None, w, w_layout=layout), a * rs, "rmsnorm_linear, no gamma")


def _run_tile(op, layout, M, K, N, place):
    """One call of `op` with operands as `place` puts them, twice (the second
    finds the tickets as the first left them), against float64."""
    import yirage_amd.fused as F

    print(f"case tile {op} M={M} K={K} N={N} layout={layout}", flush=True)
    gen = torch.Generator().manual_seed(M + K + N)
    x, (w, w3), gamma, res = _case(M, K, N, layout, torch.bfloat16 if N % 16 else torch.float16, gen)
    wd = (w if layout == KN else w.t()).double()
    if op == "linear":
        ref = x.double() @ wd + res.double()
        call = lambda a, b, c: F.linear(a, b, residual=c, w_layout=layout)
        ops = (x, w, res)
    elif op == "gated_mlp":
        a = x.double() @ wd
        ref = a * torch.sigmoid(a) * (x.double() @ (w3 if layout == KN else w3.t()).double())
        call = lambda a, b, c: F.gated_mlp(a, b, c, w_layout=layout)
        ops = (x, w, w3)
    else:
        rs = torch.rsqrt((x.double() ** 2).mean(-1, keepdim=True) + 1e-6)
        ref = ((x * gamma).double() @ wd) * rs
        call = lambda a, b, c: F.rmsnorm_linear(a, c, b, w_layout=layout)
        ops = (x, w, gamma)
    ops = [place(t) for t in ops]
    out = call(*ops)
    _check(out, ref, op)
    assert torch.equal(call(*ops), out)


@pytest.mark.parametrize("split", [0, 1], ids=["whole", "split"])
@pytest.mark.parametrize("tile", list(TILES), ids=lambda t: "-".join(map(str, t)))
def test_every_tile(tile, split):
    _run_tile(tile[0], tile[1], *TILES[tile][split], lambda t: t)


@pytest.mark.parametrize("split", [0, 1], ids=["whole", "split"])
@pytest.mark.parametrize("tile", list(STAGED), ids=lambda t: "-".join(map(str, t)))
def test_every_tile_through_registers(tile, split):
    _run_tile(tile[0], tile[1], *STAGED[tile][split], _odd)


def _odd(t):
    """The same values one element off a 16-byte boundary."""
    return torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape).copy_(t)


@pytest.mark.parametrize("layout", [NK, KN])
@pytest.mark.parametrize("M,K,N", [
    (1, 4096, 4096),       # N x K: the one-row kernel (not gated); K x N: K splits
    (3, 8, 8),             # a piece of one chunk
    (16, 3000, 72),        # many K splits of one column tile
    (40, 1096, 200),       # a partial last chunk
    (130, 584, 392),
    (300, 2056, 264),      # past the rows that scale x in LDS when aligned
])
def test_operands_off_16_byte_boundaries(M, K, N, layout):
    """Contiguous tensors at any element address, as views of a larger one are."""
    import yirage_amd.fused as F

    print(f"case unaligned M={M} K={K} N={N} layout={layout}", flush=True)
    gen = torch.Generator().manual_seed(M + K)
    dtype = torch.bfloat16 if M % 2 else torch.float16
    x, (w, w3), gamma, res = _case(M, K, N, layout, dtype, gen)
    wd, w3d = ((t if layout == KN else t.t()).double() for t in (w, w3))
    xd = x.double()
    a = xd @ wd
    rs = torch.rsqrt((xd * xd).mean(-1, keepdim=True) + 1e-6)
    out = _odd(torch.zeros_like(res))
    xo, wo, w3o, go, ro = (_odd(t) for t in (x, w, w3, gamma, res))
    for ops in ((xo, wo, ro), (x, wo, res), (xo, w, res)):
        F.linear(ops[0], ops[1], residual=ops[2], w_layout=layout, out=out)
        _check(out, a + res.double(), "linear")
        first = out.clone()
        F.linear(ops[0], ops[1], residual=ops[2], w_layout=layout, out=out)  # tickets re-armed
        assert torch.equal(out, first)
    _check(F.gated_mlp(xo, wo, w3o, w_layout=layout), a * torch.sigmoid(a) * (xd @ w3d), "gated_mlp")
    _check(F.gated_mlp(x, w, w3o, w_layout=layout), a * torch.sigmoid(a) * (xd @ w3d), "gated_mlp, W3 off")
    ref = ((x * gamma).double() @ wd) * rs
    _check(F.rmsnorm_linear(xo, go, wo, w_layout=layout), ref, "rmsnorm_linear")
    _check(F.rmsnorm_linear(x, go, w, w_layout=layout), ref, "rmsnorm_linear, gamma off")
    _check(F.rmsnorm_linear(xo, None, w, w_layout=layout), a * rs, "rmsnorm_linear, no gamma")


@pytest.mark.parametrize("M", [40, 300])
def test_special_values_stay_in_their_rows(M):
    """Inf and NaN in one row of x (and none elsewhere) reach that row only:
    rows past M, columns past N and k past K are read as copies or zeros."""
    import yirage_amd.fused as F

    gen = torch.Generator().manual_seed(5)
    x, (w, _), gamma, _ = _case(M, 200, 136, NK, torch.bfloat16, gen)
    x[M - 1, 3] = float("inf")
    x[M - 2, 199] = float("nan")
    for out in (F.linear(x, w), F.rmsnorm_linear(x, gamma, w, w_layout=NK)):
        assert torch.isfinite(out[: M - 2]).all()
        assert torch.isnan(out[M - 2]).all() and not torch.isfinite(out[M - 1]).any()


def test_more_rows_than_a_panel():
    """More rows than one launch takes (8192), the last panel a single row."""
    import yirage_amd.fused as F

    gen = torch.Generator().manual_seed(6)
    x, (w, _), gamma, res = _case(8193, 128, 136, NK, torch.float16, gen)
    xd, wd = x.double(), w.t().double()
    _check(F.linear(x, w, residual=res), xd @ wd + res.double(), "linear")
    rs = torch.rsqrt((xd * xd).mean(-1, keepdim=True) + 1e-6)
    _check(F.rmsnorm_linear(x, gamma, w, w_layout=NK), ((x * gamma).double() @ wd) * rs, "rmsnorm_linear")


def test_n_by_k_weights_past_4_gib():
    """Up to 16 rows take N x K weights of any size: every tile has its own
    32-bit offsets.  First and last columns against the reference."""
    import yirage_amd.fused as F

    K, N = 8192, 262152
    x = torch.randn((3, K), generator=torch.Generator().manual_seed(7)).to(torch.bfloat16).cuda()
    w = torch.empty((N, K), dtype=torch.bfloat16, device="cuda").normal_(0.0, K ** -0.5)
    out = F.linear(x, w)
    for cols in (slice(0, 72), slice(N - 72, N)):
        _check(out[:, cols], x.double() @ w[cols].double().t(), "linear")


@pytest.mark.parametrize("M,layout", [(1, NK), (3, KN), (17, NK)])
def test_long_k(M, layout):
    """K = 2^26: few rows and columns, operands below 4 GiB."""
    import yirage_amd.fused as F

    K, N = 1 << 26, 8
    print(f"case long K M={M} layout={layout}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(8)
    x = torch.empty((M, K), dtype=torch.bfloat16, device="cuda").normal_(generator=gen)
    w = torch.empty((K, N) if layout == KN else (N, K), dtype=torch.bfloat16, device="cuda")
    w.normal_(0.0, K ** -0.5, generator=gen)
    ref = torch.zeros((M, N), dtype=torch.float64, device="cuda")
    ss = torch.zeros((M, 1), dtype=torch.float64, device="cuda")
    for k in range(0, K, 1 << 22):
        xd = x[:, k:k + (1 << 22)].double()
        ref += xd @ (w[k:k + (1 << 22)] if layout == KN else w[:, k:k + (1 << 22)].t()).double()
        ss += (xd * xd).sum(-1, keepdim=True)
    # fp32 sums in chunks: each of the K / 64 chunk sums adds at most half an
    # ulp of the running sum (about 1): 2^20 2^-24 at worst, 2^10 2^-24 at random
    _check(F.linear(x, w, w_layout=layout), ref, "linear")
    _check(F.rmsnorm_linear(x, None, w, w_layout=layout), ref * torch.rsqrt(ss / K + 1e-6), "rmsnorm_linear")
