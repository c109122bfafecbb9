"""The transition's streamed kernel (128 and 256 channels) at the edges of its row tiles, against the
float64 oracle: 128-row tiles up to 32768 rows, 256-row tiles past that; a tile of one row, waves
with no row at all, keep units computed, padded and not written, and the residual in place. The bytes
after the result stay as they were.
"""
import numpy as np
import pytest
import torch

from conftest import abs_excess
from oracle import fused as orf

pytestmark = pytest.mark.gpu

EPS, ATOL, FILL = 1e-5, 2e-3, 7.0  # ATOL: beyond each fp16 result's half-ulp rounding


def run(hip, c, mult, m, add, keep, alias, check_rows=None):
    rng = np.random.default_rng(c + mult + m)
    hd = mult * c
    x = (rng.standard_normal((m, c)) * 2).astype(np.float16)
    sc, of = (1 + 0.1 * rng.standard_normal(c)).astype(np.float32), (0.1 * rng.standard_normal(c)).astype(np.float32)
    w1, w2 = (rng.standard_normal((c, hd)) * c ** -.5).astype(np.float16), (rng.standard_normal((hd, c)) * hd ** -.5).astype(np.float16)
    b1, b2 = (0.1 * rng.standard_normal(hd)).astype(np.float16), (0.1 * rng.standard_normal(c)).astype(np.float16)
    w1T, w2T = np.ascontiguousarray(w1.T), orf.w2_blocked(w2)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (x, sc, of, w1T, b1, w2T, b2)]
    store = torch.full((m + 3, c), FILL, dtype=torch.float16, device="cuda")
    out = store[:m]
    if alias:
        out.copy_(dev[0])
        dev[0] = out
    k = None if keep is None else torch.from_numpy(keep).cuda()
    hip.transition(*dev, keep=k, eps=EPS, add_input=add, out=out)
    torch.cuda.synchronize()
    got = out.float().cpu().numpy()
    rows = np.arange(m) if check_rows is None else check_rows
    want = orf.transition(x[rows], sc, of, w1T, b1, w2T, b2, None, EPS, add)
    if keep is not None:
        unit = 32 if c > 128 else 64
        for u in range(0, m, unit):
            part = keep[u:u + unit]
            if not (part > 0).any():
                fill = x[u:u + unit].astype(np.float64) if add else (0.0 if (part == 0).any() else FILL)
                want[u:u + unit] = fill
    assert abs_excess(got[rows], want) <= ATOL
    assert (store[m:] == FILL).all()


@pytest.mark.parametrize("c,mult", [(128, 2), (128, 4), (256, 2), (256, 4)])
@pytest.mark.parametrize("m", [1, 16, 127, 129, 300])
@pytest.mark.parametrize("add", [False, True])
def test_tile_edges(hip, c, mult, m, add):
    run(hip, c, mult, m, add, None, add)


@pytest.mark.parametrize("c", [128, 256])
@pytest.mark.parametrize("add", [False, True])
@pytest.mark.parametrize("m", [700, 33001])
def test_keep_units(hip, c, add, m):
    keep = (np.random.default_rng(m).random(m) > 0.3).astype(np.float16)
    keep[64:160] = 0
    keep[256:384] = -1
    keep[m - 30:] = 0
    rows = None
    run(hip, c, 2, m, add, keep, add, rows)


@pytest.mark.parametrize("c,m", [(128, 32768), (128, 32769), (256, 32768), (256, 32769), (128, 131313), (256, 70001)])
def test_dispatch_line(hip, c, m):
    rows = np.unique(np.concatenate([np.arange(300), np.arange(m - 300, m), np.random.default_rng(0).choice(m, 300)]))
    run(hip, c, 4, m, True, None, True, rows)


@pytest.mark.parametrize("c", [128, 256])
def test_padding_costs_no_products(hip, c):
    """Whole tiles of padding are only stored: the same call with every row kept takes several times as
    long (256 rows a tile, each of whose products read all weights)."""
    m = 131072
    rng = np.random.default_rng(0)
    dev = [torch.from_numpy(a).cuda() for a in (
        rng.standard_normal((m, c)).astype(np.float16), np.ones(c, np.float32), np.zeros(c, np.float32),
        (rng.standard_normal((4 * c, c)) * c ** -.5).astype(np.float16), np.zeros(4 * c, np.float16),
        orf.w2_blocked((rng.standard_normal((4 * c, c)) * c ** -.5).astype(np.float16)), np.zeros(c, np.float16))]
    out, ms = torch.empty_like(dev[0]), {}
    for value in (1, 0) * 4:
        keep = torch.full((m,), value, dtype=torch.float16, device="cuda")
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        hip.transition(*dev, keep=keep, eps=EPS, out=out)
        a.record()
        for _ in range(20):
            hip.transition(*dev, keep=keep, eps=EPS, out=out)
        b.record()
        b.synchronize()
        ms[value] = min(ms.get(value, 1e9), a.elapsed_time(b))
        assert value or not out.any()
    assert ms[0] < 0.7 * ms[1], ms
