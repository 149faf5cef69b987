"""Shapes and epilogues the tiled schedules took over from slower ones.

Hidden sizes that are an odd multiple of 128: GEMM2's 256-column tiles end in
a half tile there. Every tiled configuration against the oracle (the
tolerances of test_fused_moe_gpu.py) and bit for bit against each other, the
split tail and the k split on half tiles, and the allocation-free entry point
where only the streaming workspace fits. gelu and swiglu on the 4-wave kernel."""

import pytest
import torch

from flaggems_sglang import _capi, testing
from flaggems_sglang.ops import fused_moe as fm
from oracle import moe_ref
from test_fused_moe_gpu import _bias_inputs, _check, _routing_with_counts, _sample
from test_zz_no_alloc import _no_alloc, _with_workspace

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,K,N", [("bf16", 128, 256), ("bf16", 384, 128), ("bf16", 1152, 384),
                                      ("fp8", 128, 256), ("fp8", 640, 384)])
def test_odd_hidden_tiled_configs(gpu, mode, K, N):
    rem = [1, 33, 128, 160, 161, 255, 64, 0]
    counts = [256 * (e % 2) + r for e, r in enumerate(rem)]
    w, ids = _routing_with_counts(counts, gpu, seed=N)
    wts = testing.make_weights(K, N, len(counts), mode, 0.05, device=gpu, seed=K + N)
    g = torch.Generator(device=gpu).manual_seed(K)
    x = torch.randn(ids.shape[0], K, generator=g, device=gpu).to(torch.bfloat16)
    ref = moe_ref.fused_moe(x, wts.w1, wts.w2, w, ids, mode=mode, w1_scale=wts.w1_scale,
                            w2_scale=wts.w2_scale, return_mag=True)
    outs = [fm.fused_moe(x, wts.w1, wts.w2, w, ids, _flags=_capi.flag_tile(cfg),
                         **wts.kwargs(mode)) for cfg in range(_capi.TILED_CONFIGS)]
    # (fp8: every token, as in test_block_remainders, so its bound of 8 ulps)
    _check(outs[0].cpu(), ref, mode, f"odd hidden {K} {N} {mode}",
           ulp_mag=8.0 if mode == "fp8" else None)
    for cfg in range(1, _capi.TILED_CONFIGS):
        assert torch.equal(outs[0], outs[cfg]), f"{mode} K={K} N={N}: tile 0 vs tile {cfg}"


def _within_ulps(res, ref):
    """Against the oracle, in bf16 ulps of the summed terms' magnitude: sums in
    another order may round each slot's row (together at most one ulp of the
    magnitude) and the result (one more) to the neighbouring value, and an
    intermediate element with them (well under another). Over the ~200k
    outputs compared here both do at once now and then, and two ulps are up to
    1.6 % of the magnitude, past the elementwise tolerance of 1 %."""
    st = testing.regression_stats(res, *ref)
    assert st["max_ulp_mag"] <= 4 and st["mean_rel"] <= 1e-3, st


# the split tail on half tiles (1 to 8 rounds of tiles, 40 stages of k) and a
# k split of them
@pytest.mark.parametrize("shape,split", [((2100, 4224, 3200, 8, 2), "tail2"),
                                         ((128, 3968, 2560, 8, 2), "ksplit2=2")])
def test_odd_hidden_splits(gpu, shape, split):
    M, K, N, E, topk = shape
    sched = _capi.schedule(M, K, N, E, topk, _capi.QMODE_BF16)
    assert split in sched.split(), sched
    x, w1, w2, b1, b2, w, ids = _bias_inputs(M, K, N, E, topk, gpu)
    toks = _sample(M, 48)
    res = fm.fused_moe(x, w1, w2, w, ids)
    ref = moe_ref.fused_moe(x, w1, w2, w, ids, tokens=toks, return_mag=True)
    _within_ulps(res.cpu()[toks], ref)
    res = fm.fused_moe_with_bias(x, w1, b1, w2, b2, w, ids, interleaved=False)
    ref = moe_ref.fused_moe(x, w1, w2, w, ids, tokens=toks, return_mag=True,
                            activation="swiglu", b1=b1, b2=b2)
    _within_ulps(res.cpu()[toks], ref)


def test_odd_hidden_no_alloc_streams(gpu):
    """The tiled schedule's split-tail workspace alone is the whole device
    scratch; the streaming one fits, and the call is still served."""
    M, K, N, E, topk = 2100, 4224, 3200, 8, 2
    wts = testing.make_weights(K, N, E, "bf16", 0.05, device=gpu, seed=K)
    x, w, ids = testing.make_tokens(M, K, E, topk, device=gpu)
    out = _no_alloc(x, wts.w1, wts.w2, w, ids)
    ref = _with_workspace(x, wts.w1, wts.w2, w, ids, flags=_capi.FLAG_FORCE_DECODE)
    assert torch.equal(out, ref)


@pytest.mark.parametrize("on_input", [False, True], ids=["gammas_out", "gammas_in"])
@pytest.mark.parametrize("mode", ["bf16", "int8"])
@pytest.mark.parametrize("act", ["gelu", "swiglu"])
def test_wide_activations(gpu, act, mode, on_input):
    """gelu and the bias variant's swiglu in the 4-wave kernel's epilogue
    (256-row blocks, every partial block) against the oracle and the 8-wave
    kernels' epilogues, which round at the same points."""
    K, N = 512, 256
    rem = [1, 33, 128, 160, 161, 255, 64, 0]
    counts = [256 * (e % 2) + r for e, r in enumerate(rem)]
    w, ids = _routing_with_counts(counts, gpu, seed=N)
    M, E = ids.shape[0], len(counts)
    wts = testing.make_weights(K, N, E, mode, 0.05, device=gpu, seed=K + N)
    g = torch.Generator(device=gpu).manual_seed(K)
    x = torch.randn(M, K, generator=g, device=gpu).to(torch.bfloat16)
    b1 = torch.randn(E, 2 * N, generator=g, device=gpu) * 0.5
    b2 = torch.randn(E, K, generator=g, device=gpu) * 0.5

    def run(cfg):
        kw = dict(apply_router_weight_on_input=on_input, _flags=_capi.flag_tile(cfg),
                  **wts.kwargs(mode))
        if act == "gelu":
            return fm.fused_moe(x, wts.w1, wts.w2, w, ids, activation="gelu", **kw)
        return fm.fused_moe_with_bias(x, wts.w1, b1, wts.w2, b2, w, ids, gemm1_alpha=1.702,
                                      gemm1_clamp_limit=7.0, interleaved=False, **kw)

    kw = dict(mode=mode, w1_scale=wts.w1_scale, w2_scale=wts.w2_scale, activation=act,
              apply_router_weight_on_input=on_input, return_mag=True)
    if act == "swiglu":
        kw.update(b1=b1, b2=b2, alpha=1.702, limit=7.0)
    ref = moe_ref.fused_moe(x, wts.w1, wts.w2, w, ids, **kw)
    out = run(0)
    _check(out.cpu(), ref, mode, f"wide {act} {mode} {on_input}")
    for cfg in (1, 3):
        assert torch.equal(out, run(cfg)), f"{act} {mode}: tile 0 vs tile {cfg}"


_QM = {"bf16": _capi.QMODE_BF16, "fp8": _capi.QMODE_FP8_BLOCK, "int8": _capi.QMODE_INT8_CHANNEL}
_SCHEDULED = [
    # 128x128 tiles, one per CU: k rows of one or two stages, of less and of
    # more than the ring, the last block of an expert partly filled
    ("bf16", (60, 128, 128, 4, 2), "cfg=1 cfg2=1 deep1 deep2"),
    ("bf16", (61, 384, 256, 4, 2), "cfg=1 cfg2=1 deep1 deep2"),
    ("bf16", (700, 1152, 640, 4, 2), "cfg=1 cfg2=1 deep1 deep2"),
    ("int8", (60, 256, 256, 4, 2), "cfg=1 cfg2=1 deep1 deep2"),
    ("int8", (500, 1280, 768, 4, 2), "cfg=1 cfg2=1 deep1 deep2"),
    ("fp8", (60, 128, 128, 4, 2), "cfg=1 cfg2=1 deep1 deep2"),
    ("fp8", (333, 896, 640, 4, 2), "cfg=1 cfg2=1 deep1 deep2"),
    # fp8 GEMM1 two workgroups per CU on halves of 256-row blocks
    ("fp8", (1700, 128, 1024, 32, 4), "cfg=0 cfg2=1 dual1"),
    ("fp8", (1801, 384, 1152, 32, 4), "cfg=0 cfg2=1 dual1"),
    # fp8 GEMM2 on the 160-row ring
    ("fp8", (1050, 384, 2560, 16, 2), "cfg=0 cfg2=0 ksplit2=2"),
    # the split tail, a k split
    ("bf16", (2600, 1152, 2560, 32, 2), "cfg=0 cfg2=0 tail2"),
    ("int8", (2600, 1280, 5120, 32, 2), "cfg=0 cfg2=0 tail2"),
    ("bf16", (128, 4096, 4096, 8, 2), "cfg=1 cfg2=1 ksplit2=2"),
    ("bf16", (128, 1280, 4096, 8, 2), "cfg=1 cfg2=1 deep2 ksplit2=3"),
]


@pytest.mark.parametrize("mode,shape,expect", _SCHEDULED,
                         ids=[f"{m}-{s}-{e}".replace(" ", "") for m, s, e in _SCHEDULED])
def test_scheduled_shapes(gpu, mode, shape, expect):
    """What the schedule's rules pick off the benchmarked sizes, against the
    oracle and (tiled) bit for bit against the 128-row configuration."""
    M, K, N, E, topk = shape
    sched = _capi.schedule(M, K, N, E, topk, _QM[mode])
    assert sched == "tiled " + expect
    wts = testing.make_weights(K, N, E, mode, 0.05, device=gpu, seed=M + K + N)
    x, w, ids = testing.make_tokens(M, K, E, topk, device=gpu, seed=M + K + N)
    res = fm.fused_moe(x, wts.w1, wts.w2, w, ids, **wts.kwargs(mode))
    toks = _sample(M, 48)
    ref = moe_ref.fused_moe(x, wts.w1, wts.w2, w, ids, mode=mode, w1_scale=wts.w1_scale,
                            w2_scale=wts.w2_scale, tokens=toks, return_mag=True)
    _check(res.cpu()[toks], ref, mode, f"{sched} {shape} {mode}",
           ulp_mag=8.0 if mode == "fp8" else None)
    if ("deep" in sched or "dual" in sched) and "ksplit" not in sched:
        other = fm.fused_moe(x, wts.w1, wts.w2, w, ids, _flags=_capi.flag_tile(1),
                             **wts.kwargs(mode))
        assert torch.equal(res, other)


# the gathered activation scales (256-row fp8 tiles): k blocks below, at and
# across a thread's 16, in fours and not
@pytest.mark.parametrize("kblocks", [1, 4, 15, 16, 17, 20, 33, 36])
def test_gathered_scales(gpu, kblocks):
    K, N = 128 * kblocks, 256
    g = torch.Generator(device=gpu).manual_seed(kblocks)
    counts = [300, 1, 257, 0, 65, 255]
    w, ids = _routing_with_counts(counts, gpu, seed=kblocks)
    wts = testing.make_weights(K, N, len(counts), "fp8", 0.05, device=gpu, seed=K)
    # a factor per token and k block, so that a wrong block's scale shows
    x = torch.randn(ids.shape[0], kblocks, 128, generator=g, device=gpu)
    x *= 4.0 ** torch.randint(-3, 4, (ids.shape[0], kblocks, 1), generator=g, device=gpu)
    x = x.reshape(-1, K).to(torch.bfloat16)
    outs = [fm.fused_moe(x, wts.w1, wts.w2, w, ids, _flags=_capi.flag_tile(cfg),
                         **wts.kwargs("fp8")) for cfg in (0, 1)]
    assert torch.equal(outs[0], outs[1])
