"""ln_gdp where M is not a multiple of 8, so that a channel's row of results starts off the 16-byte
boundaries (odd M: every second channel off the 4-byte ones): against the float64 oracle at the
edges of its 64-row tiles, with skipped tiles and the bytes around both results left as they were; and
results so large that their offsets need more than 32 bits.
"""
import numpy as np
import pytest
import torch

from conftest import abs_excess
from oracle import fused as orf

pytestmark = pytest.mark.gpu

EPS, ATOL, FILL = 1e-5, 2e-3, 7.0  # ATOL: beyond each fp16 result's half-ulp rounding


@pytest.mark.parametrize("a,ci", [(64, 64), (128, 128), (64, 128)])
@pytest.mark.parametrize("m", [2, 15, 63, 65, 66, 127, 129, 190, 257, 33001, 66006])
def test_ragged_rows(hip, a, ci, m):
    rng = np.random.default_rng(m * 7 + a + ci)
    x = (rng.standard_normal((m, a)) * 2).astype(np.float16)
    sc, of = (1 + 0.1 * rng.standard_normal(a)).astype(np.float32), (0.1 * rng.standard_normal(a)).astype(np.float32)
    wpT, wgT = ((0.1 * rng.standard_normal((2 * ci, a))).astype(np.float16) for _ in range(2))
    bp, bg = ((0.1 * rng.standard_normal(2 * ci)).astype(np.float16) for _ in range(2))
    mask = (rng.uniform(size=m) > .2).astype(np.float16)
    if m > 128:
        mask[64:128] = -1  # a tile that is not written
    n = ci * m
    store = torch.full((2, n + 16 + 8 - n % 8), FILL, dtype=torch.float16, device="cuda")
    left, right = (s[8:8 + n].view(ci, m) for s in store)
    dev = [torch.from_numpy(t).cuda() for t in (x, sc, of, wpT, bp, wgT, bg, mask)]
    bufs = [hip.buffer(t) for t in dev + [left, right]]
    hip._check(hip.lib().clk_ln_gdp(hip._stream(dev[0]), *map(hip._ref, bufs), EPS))
    torch.cuda.synchronize()
    for got, want in zip((left, right), orf.ln_gdp(x, sc, of, wpT, bp, wgT, bg, mask, EPS)):
        got, unwritten = got.float().cpu().numpy(), np.isnan(want)
        assert unwritten.any() == (m > 128)
        assert (got[unwritten] == FILL).all()
        assert abs_excess(got[~unwritten], want[~unwritten]) <= ATOL
    assert (store[:, :8] == FILL).all() and (store[:, 8 + n:] == FILL).all()


@pytest.mark.parametrize("m", [2 ** 24 - 1, 2 ** 24, 2 ** 24 + 3])
def test_results_past_32_bit_offsets(hip, m):
    """Results of 2^31 bytes each (4096 residues squared, 64 channels) are the general kernel's, just
    below them the other's with its largest offsets: every value against calls of a sixteenth of the
    rows, which may round one sum differently (an fp16 ulp), and rows at both ends against the oracle."""
    rng = np.random.default_rng(m)
    c = 64
    sc, of = (1 + 0.1 * rng.standard_normal(c)).astype(np.float32), (0.1 * rng.standard_normal(c)).astype(np.float32)
    wpT, wgT = ((0.1 * rng.standard_normal((2 * c, c))).astype(np.float16) for _ in range(2))
    bp, bg = ((0.1 * rng.standard_normal(2 * c)).astype(np.float16) for _ in range(2))
    x = torch.empty((m, c), dtype=torch.float16, device="cuda").normal_(std=2, generator=torch.Generator("cuda").manual_seed(0))
    mask = torch.ones(m, dtype=torch.float16, device="cuda")
    mask[5::7] = 0
    mask[-200:-40] = 0
    par = [torch.from_numpy(a).cuda() for a in (sc, of, wpT, bp, wgT, bg)]
    got = hip.ln_gdp(x, *par, mask, eps=EPS)
    step = 2 ** 20
    for a in range(0, m, step):
        b = min(a + step, m)
        for g, want in zip(got, hip.ln_gdp(x[a:b], *par, mask[a:b], eps=EPS)):
            want = want.float()
            assert ((g[:, a:b].float() - want).abs() <= 2.0 ** -10 * want.abs() + 1e-5).all(), a
    for rows in (slice(0, 300), slice(m - 300, m)):
        want = orf.ln_gdp(x[rows].cpu().numpy(), sc, of, wpT, bp, wgT, bg, mask[rows].cpu().numpy(), EPS)
        for g, w in zip(got, want):
            assert abs_excess(g[:, rows].float().cpu().numpy(), w) <= ATOL
