"""The forward's bias loads at every row alignment, against the float64 oracle.

The forward reads its bias [H, Sq, Sk] in one of three ways, chosen by Sk and the address: rows on
4-byte boundaries (Sk even) and rows of odd Sk, both through LDS, and 2-byte loads for the rest (Sk
even at an odd element offset; odd Sk up to 16, ungated at D <= 32 up to 55). The cases sit at the edges of a 64-key tile, where an odd row's
last key lies past the tile, with no dead key, a few (among them key 63), and more than the
tile-wide limit of 8 for single stores. With odd Sk the same values at an odd element offset, which
swaps the roles of even and odd queries within the same kernel, must give the same bits.
"""
import numpy as np
import pytest
import torch

from conftest import abs_excess
from oracle import attention as ora

pytestmark = pytest.mark.gpu

OUT_ATOL = 2e-3  # beyond each fp16 result's half-ulp rounding, as for every forward


def mask(kind, n, sk, rng):
    m = np.ones((n, sk), np.uint8)
    if kind == "few":
        m[:, sk // 3] = 0
        m[0, min(63, sk - 1)] = 0
    elif kind == "many":
        m[:, -(sk // 4 + 1):] = 0
        m[1] = (rng.random(sk) > 0.5)
        m[1, 0] = 1
    return m


@pytest.mark.parametrize("kind", ["none", "few", "many"])
@pytest.mark.parametrize("sq,sk,d", [(33, 1, 32), (5, 7, 8), (20, 15, 64), (20, 17, 64), (40, 55, 16), (40, 57, 16), (63, 63, 32), (64, 65, 16), (130, 127, 32), (129, 129, 32),
                                     (131, 191, 64), (37, 193, 96), (66, 130, 32), (65, 132, 32), (64, 134, 64),
                                     (257, 261, 32)])
def test_bias_rows(hip, sq, sk, d, kind):
    n, h = 2, 3
    rng = np.random.default_rng(sq * 1000 + sk)
    q = (rng.standard_normal((n, h, sq, d)) * 0.7).astype(np.float16)
    k, v = (rng.standard_normal((n, h, sk, d)).astype(np.float16) for _ in range(2))
    bias = (rng.standard_normal((h, sq, sk)) * 2).astype(np.float16)
    km = mask(kind, n, sk, rng)
    tq, tk, tv, tm = (torch.from_numpy(a).cuda() for a in (q, k, v, km))
    flat = torch.from_numpy(bias.reshape(-1)).cuda()
    got = []
    for offset in (0, 1):  # an element offset moves every row's alignment
        buf = torch.full((flat.numel() + 8,), float("nan"), dtype=torch.float16, device="cuda")
        buf[offset:offset + flat.numel()] = flat
        tb = buf[offset:offset + flat.numel()].view(h, sq, sk)
        got.append(hip.attention_fwd(tq, tk, tv, tb, tm, d ** -0.5, *((64, 64) if d == 64 else (64, 32))))
    torch.cuda.synchronize()
    want_out, want_lse = ora.attention_fwd(q, k, v, bias, km, d ** -0.5)
    for out, lse in got:
        assert abs_excess(out.float().cpu().numpy(), want_out) <= OUT_ATOL
        assert abs_excess(lse.cpu().numpy(), want_lse, fp16_out=False) <= OUT_ATOL
    if sk % 2:
        assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
