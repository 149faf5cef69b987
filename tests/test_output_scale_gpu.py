"""The routed scaling factor applied by the kernel that writes the output: bit
for bit the unscaled call followed by the in-place multiplication, on every
schedule that ends a layer, with infinities and zeros of the factor."""

import pytest
import torch

from flaggems_sglang import _capi, testing
from flaggems_sglang.ops import fused_moe as fm
from test_fused_moe_gpu import _bias_inputs

pytestmark = pytest.mark.gpu

# m, hidden, inter, experts, topk, mode, flags, the schedule (in full)
SHAPES = [(1, 4096, 256, 8, 2, "bf16", 0, "direct_sum"),
          (1, 2048, 768, 16, 8, "bf16", 0, "direct_sum pair"),
          (1, 2048, 128, 8, 3, "fp8", 0, "direct_sum pair qfold"),
          (1, 4096, 256, 8, 2, "int8", 0, "direct_sum qfold_a2"),
          (1, 512, 256, 8, 2, "bf16", 0, "direct"),
          (7, 512, 256, 8, 8, "bf16", 0, "stream mt=1"),
          (7, 640, 128, 8, 3, "bf16", 0, "stream mt=1"),
          (9, 512, 256, 8, 2, "int8", 0, "stream mt=1"),
          (300, 512, 256, 8, 1, "fp8", _capi.flag_tile(0), "tiled cfg=0 cfg2=0"),
          (300, 512, 256, 8, 4, "int8", _capi.flag_tile(1), "tiled cfg=1 cfg2=1"),
          (128, 4096, 2560, 8, 2, "bf16", 0, "tiled cfg=1 cfg2=1 ksplit2=2")]


@pytest.mark.parametrize("M,K,N,E,topk,mode,flags,sched", SHAPES)
@pytest.mark.parametrize("bias", [False, True])
def test_scaled_is_mul(gpu, M, K, N, E, topk, mode, flags, sched, bias):
    x, _, _, b1, b2, w, ids = _bias_inputs(M, K, N, E, topk, gpu)
    ids = ids.clone()
    ids.view(-1)[::5] = -1
    wts = testing.make_weights(K, N, E, mode, 0.05, device=gpu, seed=M + K)
    kw = wts.kwargs(mode)
    qm = {"bf16": _capi.QMODE_BF16, "fp8": _capi.QMODE_FP8_BLOCK,
          "int8": _capi.QMODE_INT8_CHANNEL}[mode]
    assert _capi.schedule(M, K, N, E, topk, qm, flags) == sched

    def run(scale):
        if bias:
            return fm.fused_moe_with_bias(x, wts.w1, b1, wts.w2, b2, w, ids, interleaved=False,
                                          routed_scaling_factor=scale, _flags=flags, **kw)
        return fm.fused_moe(x, wts.w1, wts.w2, w, ids, routed_scaling_factor=scale,
                            _flags=flags, **kw)

    plain = run(None)
    assert torch.equal(run(1.0), plain)
    for scale in (2.5, 0.1, -3, 0, 1e300, 1e-300, float("inf")):
        torch.testing.assert_close(run(scale), plain.clone().mul_(scale), rtol=0, atol=0,
                                   equal_nan=True)


def test_other_factors(gpu):
    x, w1, w2, _, _, w, ids = _bias_inputs(5, 256, 128, 4, 2, gpu)
    plain = fm.fused_moe(x, w1, w2, w, ids)
    for scale in (torch.tensor(1.7, device=gpu), torch.tensor(0.3), 2 ** 53 + 1):
        assert torch.equal(fm.fused_moe(x, w1, w2, w, ids, routed_scaling_factor=scale),
                           plain.clone().mul_(scale))
    for scale in ("2", 1j, torch.ones(2, device=gpu)):
        with pytest.raises((TypeError, RuntimeError)):
            fm.fused_moe(x, w1, w2, w, ids, routed_scaling_factor=scale)
