"""argmax at the edges of its pieces: rows that start off 16-byte boundaries
(odd n), fewer valid columns than n, ties across and within pieces, -inf and
NaN rows; indices are exact."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(x, n_valid):
    """Lowest index of the largest value that is not NaN, -1 if there is none."""
    out = []
    for row in x[:, :n_valid].float().cpu():
        ok = ~torch.isnan(row)
        out.append(int(torch.nonzero(ok & (row == row[ok].max()))[0]) if ok.any() else -1)
    return out


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,n,n_valid", [(1, 1, 1), (3, 7, 7), (5, 9, 8), (4, 63, 61), (9, 2051, 2050),
                                            (3, 8193, 8193), (2, 32771, 32768), (3, 128256, 128251)])
def test_argmax_edges(rows, n, n_valid, dtype):
    import yirage_amd.fused as F

    print(f"case argmax rows={rows} n={n} n_valid={n_valid} {dtype}", flush=True)
    gen = torch.Generator().manual_seed(rows * n)
    x = (torch.randn((rows, n), generator=gen) * 4).round().to(dtype)  # many ties
    if n > n_valid:
        x[:, n_valid:] = 1000  # never looked at
    cases = [x, torch.full_like(x, float("-inf")), torch.full_like(x, float("nan"))]
    mixed = torch.full_like(x, float("-inf"))
    mixed[:, ::3] = float("nan")
    mixed[:, n_valid // 2] = float("-inf")
    cases.append(mixed)
    last = x.clone()
    last[:, n_valid - 1] = 900
    cases.append(last)
    for c in cases:
        got = F.argmax(c.cuda(), n_valid=n_valid).cpu().tolist()
        assert got == _reference(c, n_valid)
