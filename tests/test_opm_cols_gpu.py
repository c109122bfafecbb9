"""opm_update where K is 128, 256 or 512 against the float64 oracle: but for small products t^T is in
registers and the lhs rows are streamed. Row blocks and column tiles cut short, rows split over
workgroups or not, the residual absent, apart and in place.
"""
import numpy as np
import pytest
import torch

from conftest import abs_excess
from oracle import opm as oro

pytestmark = pytest.mark.gpu

ATOL = 2e-3  # beyond each fp16 result's half-ulp rounding


@pytest.mark.parametrize("k", [128, 256, 512])
@pytest.mark.parametrize("b,d,f", [(17, 9, 16), (113, 449, 128), (121, 3590, 16), (520, 260, 64),
                                   # too few row blocks, one round of half the places, splits with a last workgroup cut short
                                   (65, 1500, 32), (161, 161, 128), (1000, 33, 64), (1290, 70, 64), (899, 170, 64)])
@pytest.mark.parametrize("residual", ["none", "apart", "in place"])
def test_columns(hip, k, b, d, f, residual):
    rng = np.random.default_rng(k + b + d + f)
    lhs = rng.standard_normal((b, k)).astype(np.float16)
    t = (rng.standard_normal((k, d, f)) * k ** -0.5).astype(np.float16)
    bias = (rng.standard_normal(f) * 0.1).astype(np.float32)
    norm = rng.integers(1, k // 32 + 1, size=(b, d)).astype(np.float32)
    res = None if residual == "none" else (rng.standard_normal((b, d, f)) * 2).astype(np.float16)
    dev = [torch.from_numpy(a).cuda() for a in (lhs, t, bias, norm)]
    n = b * d * f
    store = torch.full((n + 64,), 7.0, dtype=torch.float16, device="cuda")
    out = store[:n].view(b, d, f)
    tr = None
    if res is not None:
        tr = torch.from_numpy(res).cuda()
        if residual == "in place":
            out.copy_(tr)
            tr = out
    hip.opm_update(*dev, tr, eps=1e-3, out=out)
    torch.cuda.synchronize()
    assert abs_excess(out.float().cpu().numpy(), oro.opm_update(lhs, t, bias, norm, 1e-3, res)) <= ATOL
    assert (store[n:] == 7.0).all()


@pytest.mark.parametrize("k", [128, 512])
@pytest.mark.parametrize("b,d,f", [(17, 9, 128), (256, 256, 128)])
def test_division(hip, k, b, d, f):
    """Sums that are 7 times a value halfway between two fp16 numbers: divided by 7 they round to the
    even one, from both kernels. A multiplication by the rounded 1 / 7 misses it at every third value."""
    m = 1 + (2 * np.arange(1024) + 1) * 2.0 ** -11
    s = np.resize(7 * m, (d, f))
    t = np.zeros((k, d, f), np.float16)
    t[0] = s
    t[1] = s - t[0].astype(np.float64)
    assert (t[0].astype(np.float64) + t[1] == s).all()
    lhs = np.zeros((b, k), np.float16)
    lhs[:, :2] = 1
    dev = [torch.from_numpy(a).cuda() for a in (lhs, t, np.zeros(f, np.float32), np.full((b, d), 7, np.float32))]
    got = hip.opm_update(*dev, None, eps=0.0).cpu().numpy()
    assert (got == np.resize(m, (d, f)).astype(np.float16)).all()
