"""The activation quantisers' rounded quotients: bit for bit the division's,
over scales and values across bf16's range, and on the rows of a padded order
(the GEMM1 output inside a quantised layer)."""

import pytest
import torch

from flaggems_sglang.ops import fused_moe as fm

pytestmark = pytest.mark.gpu


def _rows(n, cols, seed):
    """bf16 rows whose largest value runs over bf16's exponents (down to
    values the 1e-10 floor of the scale takes over), the others uniform in
    exponent below it or near it, both signs."""
    g = torch.Generator().manual_seed(seed)
    top = 2.0 ** (torch.rand(n, 1, generator=g) * 200 - 100)
    near = torch.rand(n, cols, generator=g) * 2 - 1
    far = torch.sign(near) * 2.0 ** (-40 * torch.rand(n, cols, generator=g))
    x = torch.where(torch.rand(n, cols, generator=g) < 0.7, near, far) * top
    x[:, 5] = top[:, 0]
    x[0] = 0.0
    x[1, :] = 3.3e38 * near[1]
    x[2, :] = 1e-40 * near[2]
    return x.bfloat16()


def _fp8(x, group):
    g = x.float().reshape(x.shape[0], -1, group)
    scale = g.abs().amax(-1, keepdim=True).clamp(min=1e-10) / 448.0
    q = (g / scale).clamp(-448, 448).to(torch.float8_e4m3fn)
    return q.reshape(x.shape).view(torch.uint8), scale.squeeze(-1)


def _int8(x):
    f = x.float()
    scale = f.abs().amax(-1, keepdim=True).clamp(min=1e-10) / 127.0
    return (f / scale).round().clamp(-127, 127).to(torch.int8), scale.squeeze(-1)


@pytest.mark.parametrize("n,cols,group", [(4000, 1024, 128), (777, 136, 8), (900, 512, 512)])
def test_fp8_codes(gpu, n, cols, group):
    x = _rows(n, cols, n + cols)
    q, s = fm.per_token_group_quant_fp8(x.to(gpu), group)
    rq, rs = _fp8(x, group)
    assert torch.equal(s.cpu(), rs)
    assert torch.equal(q.view(torch.uint8).cpu(), rq)


@pytest.mark.parametrize("n,cols", [(1023, 1024), (1024, 1032), (5, 8), (4000, 520), (1200, 8192),
                                    (1100, 8200)])
def test_int8_codes(gpu, n, cols):
    x = _rows(n, cols, n + cols)
    q, s = fm.per_token_quant_int8(x.to(gpu))
    rq, rs = _int8(x)
    assert torch.equal(s.cpu(), rs)
    assert torch.equal(q.cpu(), rq)


def test_infinite_values(gpu):
    """An infinity makes its scale infinite: every finite value's code is 0
    (x / inf), in its own group or row only."""
    x = _rows(8, 256, 3)
    x[4, 7] = float("inf")
    q, s = fm.per_token_group_quant_fp8(x.to(gpu), 128)
    rq, rs = _fp8(x, 128)
    assert torch.equal(s.cpu(), rs)
    keep = torch.ones_like(rq, dtype=torch.bool)
    keep[4, 7] = False
    assert torch.equal(q.view(torch.uint8).cpu()[keep] & 0x7f, rq[keep] & 0x7f)
    q, s = fm.per_token_quant_int8(x.to(gpu))
    rq, rs = _int8(x)
    assert torch.equal(q.cpu()[keep], rq[keep])
