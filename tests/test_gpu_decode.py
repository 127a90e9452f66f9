"""Paged decode: every group size, lengths around the 32-token blocks, one to
many splits, page sizes on both page-table paths, and caches that are not
16-byte aligned, against float64."""
import math

import numpy as np
import pytest
import torch

import yirage_amd.fused as F

pytestmark = pytest.mark.gpu

# outputs are averages of unit normals (at most 4.5): half an ulp each for the
# 16-bit P and the 16-bit result
TOL = {torch.float16: 2 * 4.5 * 2.0 ** -11, torch.bfloat16: 2 * 4.5 * 2.0 ** -8}


def _odd(t):
    return torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape).copy_(t)


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("G,hkv,page,lens", [
    (1, 1, 64, [1]), (16, 1, 32, [8193]),                # one pair: up to 256 splits
    (2, 2, 16, [31, 4096]), (4, 2, 64, [33, 1000, 257]), (8, 4, 48, [95, 2049]),
    (16, 16, 128, [700] * 17), (1, 16, 64, [32] * 16),   # one split
])
def test_lengths_and_splits(G, hkv, page, lens, dt):
    print("case", G, hkv, page, len(lens), max(lens), dt, flush=True)
    gen = torch.Generator().manual_seed(G + page)
    npg = [-(-n // page) for n in lens]
    pool = sum(npg)
    q = torch.randn((len(lens), G * hkv, 128), generator=gen).to(dt).cuda()
    k, v = (torch.randn((pool, page, hkv, 128), generator=gen).to(dt).cuda() for _ in range(2))
    indptr = torch.from_numpy(np.concatenate([[0], np.cumsum(npg)]).astype(np.int32)).cuda()
    indices = torch.randperm(pool, generator=gen).int().cuda()
    ls = torch.tensor(lens, dtype=torch.int32).cuda()
    out = F.gqa_decode_paged(q, k, v, indptr, indices, ls, max_kv_len=max(lens))
    pages = indices.long().split(npg)
    for b, n in enumerate(lens):
        kb, vb = (c[pages[b]].reshape(-1, hkv, 128)[:n].double() for c in (k, v))
        for h in range(hkv):
            p = torch.softmax(q[b, h * G:(h + 1) * G].double() @ kb[:, h].t() / math.sqrt(128), -1)
            err = (out[b, h * G:(h + 1) * G].double() - p @ vb[:, h]).abs().max().item()
            assert err <= TOL[dt], (b, h, err)
    # the same bits again, and from caches at an odd address
    assert torch.equal(F.gqa_decode_paged(q, k, v, indptr, indices, ls, max_kv_len=max(lens)), out)
    assert torch.equal(F.gqa_decode_paged(q, _odd(k), _odd(v), indptr, indices, ls, max_kv_len=max(lens)), out)
