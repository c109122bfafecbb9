"""The dK/dV kernels at head dims up to 32 where the route is chosen by estimated time, against the
float64 oracle: the register kernels at head dims below 32 and in query windows (Sq > 384), with window
edges and ragged last tiles, several rows per workgroup, and the running sum of dK and dV that a window
hands to the next; and the LDS-partial kernel, over several passes of its row groups. dk and dv must
not depend on want_dbias, repeat bit for bit, and be the same from clk_attention_bwd_noalloc.
"""
import numpy as np
import pytest
import torch

from conftest import abs_excess
from oracle import attention as ora

pytestmark = pytest.mark.gpu

GRAD_ATOL = 5e-3  # beyond each fp16 result's half-ulp rounding, as for every backward


@pytest.mark.parametrize("n,h,sq,sk,d,windows", [
    (3, 2, 100, 90, 8, 1), (2, 2, 128, 65, 16, 1), (2, 3, 140, 60, 16, 1), (2, 2, 257, 64, 24, 1), (700, 1, 384, 33, 8, 1),
    (2, 2, 385, 100, 32, 2), (600, 1, 520, 40, 32, 2), (2, 2, 513, 130, 16, 2), (2, 1, 640, 129, 8, 2), (2, 2, 768, 70, 24, 2),
    (2, 1, 769, 64, 32, 3), (300, 2, 900, 20, 32, 3),
    (700, 1, 200, 33, 8, 1), (1500, 1, 256, 20, 16, 1), (901, 1, 560, 40, 16, 2)])
def test_register_windows(hip, n, h, sq, sk, d, windows):
    plan = hip.attention_bwd_plan(n, h, sq, sk, d)
    assert plan["registers"] == 1 and plan["windows"] == windows, plan
    compare(hip, n, h, sq, sk, d)


@pytest.mark.parametrize("n,h,sq,sk,d,registers,passes", [
    # 13 to 15 query tiles at D >= 24: the LDS-partial kernel (one row of a pass absent, ragged Sq)
    (64, 4, 400, 400, 32, 0, 2), (600, 1, 416, 40, 32, 0, 1), (61, 4, 390, 400, 24, 0, 2), (99, 2, 480, 470, 32, 0, 2),
    # but where its plan has the many more partials, few rows, or 16 tiles or 12
    (256, 4, 386, 400, 32, 1, 29), (2, 2, 385, 100, 32, 1, 1), (64, 4, 481, 470, 32, 1, 8), (64, 4, 384, 400, 32, 1, 8),
    # one or two tiles at D < 32: the LDS-partial kernel with one or two row groups; three not
    (3000, 1, 31, 33, 8, 0, 11), (1111, 2, 64, 64, 16, 0, 3), (751, 1, 33, 130, 24, 0, 3), (300, 1, 65, 64, 24, 1, 2),
    # 5 and 6 tiles at D = 24
    (561, 8, 164, 136, 24, 0, 7), (850, 4, 142, 142, 24, 0, 6), (144, 8, 158, 99, 24, 1, 9), (150, 4, 190, 200, 16, 1, 10)])
def test_route(hip, n, h, sq, sk, d, registers, passes):
    plan = hip.attention_bwd_plan(n, h, sq, sk, d)
    assert plan["registers"] == registers and plan["passes"] == passes, plan
    if n * h * sq * sk <= 6e7:  # the oracle's time
        compare(hip, n, h, sq, sk, d)


def compare(hip, n, h, sq, sk, d):
    rng = np.random.default_rng(sq + sk + d)
    f16 = lambda *shape: (rng.standard_normal(shape) * 0.5).astype(np.float16)
    q, k, v, bias, dout = f16(n, h, sq, d), f16(n, h, sk, d), f16(n, h, sk, d), f16(h, sq, sk), f16(n, h, sq, d)
    km = (rng.random((n, sk)) > 0.15).astype(np.uint8)
    km[0] = 0
    scale = d ** -0.5
    tq, tk, tv, tb, tm, tdo = (torch.from_numpy(a).cuda() for a in (q, k, v, bias, km, dout))
    out, lse = hip.attention_fwd(tq, tk, tv, tb, tm, scale)
    args = (tq, tk, tv, tb, tm, out, tdo, lse, scale)
    got, again = hip.attention_bwd(*args), hip.attention_bwd_noalloc(*args)
    off = hip.attention_bwd(*args, want_dbias=False)
    torch.cuda.synchronize()
    want = ora.attention_bwd(q, k, v, bias, km, dout, scale)
    for i, name in enumerate(("dq", "dk", "dv", "dbias")):
        assert abs_excess(got[i].float().cpu().numpy(), want[i], fp16_out=name != "dbias") <= GRAD_ATOL, name
        assert torch.equal(got[i], again[i]), name + " differs on repeat"
        assert torch.equal(got[i], off[i]) or name == "dbias", name + " changed without want_dbias"
    assert not off[3].any()
