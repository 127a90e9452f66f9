"""Graph attention on the operands as they lie (K as [g][d][l]): row and token
remainders of each tile, one and several token splits, strided operands, and
operands that are not 16-byte aligned (packed first), against float64."""
import ctypes
import math
import struct

import pytest
import torch

from yirage_amd import _lib

pytestmark = pytest.mark.gpu

# outputs are averages of unit normals; a 16-bit P and a 16-bit result round by
# half an ulp each, 2^-11 (f16) or 2^-8 (bf16) of at most 4.5 (the largest |v|)
TOL = {torch.float16: 2 * 4.5 * 2.0 ** -11, torch.bfloat16: 2 * 4.5 * 2.0 ** -8}


def _call(q, k, v, out, scale, ws=None, misses=0):
    G, M, d = q.shape
    dt = _lib.DTYPE_F16 if q.dtype == torch.float16 else _lib.DTYPE_BF16
    bits = struct.unpack("<i", struct.pack("<f", scale))[0]
    params = [G, M, v.shape[1], d, dt, bits, *q.stride(), *k.stride(), *v.stride(), *out.stride()]
    P = (ctypes.c_int64 * len(params))(*params)
    lib = _lib.lib()
    nb = lib.yr_hip_fused_workspace(_lib.OP_ATTENTION, len(params), P)
    if ws is None:
        ws = torch.zeros(max(nb, 1), dtype=torch.uint8, device="cuda")
    ins = (ctypes.c_void_p * 3)(q.data_ptr(), k.data_ptr(), v.data_ptr())
    outs = (ctypes.c_void_p * 1)(out.data_ptr())
    rc = lib.yr_hip_run_fused(_lib.OP_ATTENTION, 3, ins, 1, outs, len(params), P, ctypes.c_void_p(ws.data_ptr()),
                              nb - misses, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    return rc, ws


def _operands(G, M, L, d, dt, seed=0):
    gen = torch.Generator().manual_seed(seed)
    return [torch.randn(s, generator=gen).to(dt).cuda() for s in ((G, M, d), (G, d, L), (G, L, d))]


def _check(out, q, k, v, scale):
    p = torch.softmax(scale * (q.double() @ k.double()), -1)
    err = (out.double() - p @ v.double()).abs().max().item()
    assert err <= TOL[q.dtype], err


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("G,M,L,d", [
    (1, 1, 8, 64), (3, 16, 264, 64), (2, 5, 4096, 64),            # 16 rows
    (2, 17, 64, 64), (1, 33, 520, 128), (3, 100, 2040, 128), (4, 64, 4096, 64),  # 32 rows
    (9, 3601, 72, 128), (260, 65, 8, 128), (5, 13001, 72, 64),    # 64 rows, no split
    (5, 13057, 72, 64), (6, 11009, 1544, 64),                     # 128 rows, the last tile 1 row
    (515, 3, 136, 64),                                            # 16 rows, no split
    (2, 5, 328, 128), (1, 16, 328, 128), (1, 65, 12, 64),         # 12 tokens: packed
])
def test_rows_and_tokens(G, M, L, d, dt):
    print("case", G, M, L, d, dt, flush=True)
    q, k, v = _operands(G, M, L, d, dt)
    scale = 1.0 / math.sqrt(d)
    out = torch.full_like(q, math.nan)
    rc, ws = _call(q, k, v, out, scale)
    assert rc == 0, _lib.last_error()
    _check(out, q, k, v, scale)
    again = torch.empty_like(out)  # the tickets are zero again, and the merge order is fixed
    rc, _ = _call(q, k, v, again, scale, ws)
    assert rc == 0 and torch.equal(again, out)


@pytest.mark.parametrize("d", [64, 128])
def test_strides_alignment_and_workspace(d):
    G, M, L, dt = 2, 40, 712, torch.float16
    print("case strides", d, flush=True)
    q, k, v = _operands(G, M, L, d, dt, 1)
    scale = 1.0 / math.sqrt(d)
    ref = torch.empty_like(q)
    assert _call(q, k, v, ref, scale)[0] == 0
    _check(ref, q, k, v, scale)
    # other strides of the same values: the same bits
    qs = q.transpose(0, 1).contiguous().transpose(0, 1)
    ks = torch.nn.functional.pad(k, (0, 8))[..., :L]
    vs = v.transpose(0, 1).contiguous().transpose(0, 1)
    out = torch.empty((M, G, d), dtype=dt, device="cuda").transpose(0, 1)
    assert _call(qs, ks, vs, out, scale)[0] == 0
    assert torch.equal(out, ref)
    # K with its head dims contiguous, and an operand at an odd address: packed
    kt = k.transpose(1, 2).contiguous().transpose(1, 2)
    qo = torch.empty(q.numel() + 1, dtype=dt, device="cuda")[1:].view(q.shape).copy_(q)
    for ops in ((q, kt, v), (qo, k, v)):
        out = torch.empty_like(q)
        assert _call(*ops, out, scale)[0] == 0
        _check(out, q, k, v, scale)
    # refused: a workspace a byte short, a scale that is not positive
    assert _call(q, k, v, ref, scale, misses=1)[0] != 0
    assert _call(q, k, v, ref, 0.0)[0] != 0


def test_infinite_scores_and_weights():
    """A row whose scores are all -inf gives 0 (as the packed kernels do), and
    a token of weight 0 does not leak; +-65504 scores stay finite."""
    G, M, L, d, dt = 1, 33, 600, 64, torch.float16
    print("case extremes", flush=True)
    q, k, v = _operands(G, M, L, d, dt, 2)
    q[:, :2] = 0
    q[:, 0, 0] = -math.inf
    k[:, 0] = k[:, 0].abs() + 1
    q[:, 1, 0] = 65504
    out = torch.empty_like(q)
    assert _call(q, k, v, out, 0.125)[0] == 0
    assert (out[:, 0] == 0).all()
    _check(out[:, 1:], q[:, 1:], k, v, 0.125)


@pytest.mark.parametrize("M", [1, 3, 33])
def test_long_tail_of_small_weights(M):
    """Weights that round to 0 in f16 beside the row's maximum (2^-26 each)
    still count in the row sum, which is fp32: a token of weight 1 and V = 1,
    then 65535 whose V is +1 and -1 in turn, give 1 / (1 + 65535 2^-26).  The
    numerator loses at most one such weight (2^-26), the sum is fp32, and the
    result is rounded once to f16."""
    G, L, d, dt = 512, 65536, 64, torch.float16
    print("case tail", M, flush=True)
    q = torch.zeros((G, M, d), dtype=dt, device="cuda")
    q[..., 0] = 1
    k = torch.zeros((1, d, L), dtype=dt, device="cuda")
    k[:, 0] = -26
    k[:, 0, 0] = 0
    v = torch.ones((1, L, d), dtype=dt, device="cuda")
    v[:, 2::2] = -1
    out = torch.empty_like(q)
    assert _call(q, k.expand(G, d, L), v.expand(G, L, d), out, math.log(2))[0] == 0
    ref = 1 / (1 + 65535 * 2.0 ** -26)
    assert (out.double() - ref).abs().max().item() <= 2.0 ** -12 + 2.0 ** -20
