"""The activation quantisers' rounded quotients: bit for bit the division's,
over scales and values across bf16's range, and on the rows of a padded order
(the GEMM1 output inside a quantised layer)."""

import pytest
import torch

from flaggems_sglang import _capi, testing
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


@pytest.mark.parametrize("flags", [_capi.FLAG_FORCE_DECODE, _capi.flag_tile(0), _capi.flag_tile(1)],
                         ids=["stream", "tile0", "tile1"])
@pytest.mark.parametrize("mode", ["fp8", "int8"])
def test_repeated_slots_of_a_routing_tuple(gpu, mode, flags):
    """A routing tuple whose gathered order names some slots twice inside their
    expert's range, some never and some outside: every row that holds a slot is
    quantised (both of a repeated one's, which GEMM2 both reads), whatever the
    workspace held. The same bits as the layer with the unnamed slots dropped."""
    M, K, N, E, topk = 384, 512, 256, 4, 2
    n, qm = M * topk, {"fp8": _capi.QMODE_FP8_BLOCK, "int8": _capi.QMODE_INT8_CHANNEL}[mode]
    wts = testing.make_weights(K, N, E, mode, 0.05, device=gpu, seed=K)
    x, w, ids = testing.make_tokens(M, K, E, topk, device=gpu, seed=M)
    w, ids = fm._routing_to_topk(*fm.standard_topk_to_routing(w, ids, E)[:2], M)
    rd, gi, _ = fm.standard_topk_to_routing(w, ids, E)
    src, gate, hist = gi.src_indx.cpu().clone(), rd.gate_scal.cpu().clone(), rd.expt_hist.cpu()
    g = torch.Generator().manual_seed(1)
    dropped = torch.zeros(n, dtype=torch.bool)
    start = 0
    for c in hist.tolist():
        p = start + torch.randperm(c, generator=g)
        for a, b in zip(p[: c // 4].tolist(), p[c // 4: c // 4 * 2].tolist()):
            dropped[int(src[a])] = True           # a names b's slot instead of its own
            src[a], gate[a] = src[b], gate[b]
        dropped[int(src[p[-1]])] = True
        src[p[-1]] = n + 7 if start % 2 else -3
        start += c
    src, gate = src.to(gpu), gate.to(gpu)
    lib = _capi.load()
    need = lib.fgs_moe_workspace_bytes(M, K, N, E, topk, qm, flags)
    ws = torch.full((need,), 0xff, dtype=torch.uint8, device=gpu)  # fp8 codes and scales: NaN
    out = torch.empty((M, K), dtype=torch.bfloat16, device=gpu)
    _capi.check(lib.fgs_moe_fused_routed(
        qm, x.data_ptr(), wts.w1.data_ptr(), wts.w2.data_ptr(), wts.w1_scale.data_ptr(),
        wts.w2_scale.data_ptr(), None, None, 1.0, 0.0, gate.data_ptr(), src.data_ptr(),
        rd.expt_hist.data_ptr(), M, K, N, E, topk, flags, ws.data_ptr(), need, out.data_ptr(),
        torch.cuda.current_stream().cuda_stream), "fused_moe (routing tuple)")
    ids = torch.where(dropped.view(M, topk).to(gpu), torch.full_like(ids, -1), ids)
    ref = fm.fused_moe(x, wts.w1, wts.w2, w, ids, _flags=flags, **wts.kwargs(mode))
    # (a token with an unnamed slot reads what the workspace held for it: here -1, dropped)
    assert torch.equal(out, ref)


@pytest.mark.parametrize("M", [110, 450])
@pytest.mark.parametrize("mode", ["fp8", "int8"])
def test_rows_of_many_experts(gpu, mode, M):
    """880 and 3600 slots of 1024 experts: the alignment for more experts than
    the single-workgroup one's LDS takes records the padded rows. The bits of
    the routing-tuple path (its own order kernel), slots dropped and outside."""
    K, N, E, topk = 256, 256, 1024, 8
    wts = testing.make_weights(K, N, E, mode, 0.05, device=gpu, seed=M)
    x, w, ids = testing.make_tokens(M, K, E, topk, device=gpu, seed=M)
    w, ids = (t.gather(1, ids.argsort(1)) for t in (w, ids))
    ids[::3, -1] = -1
    known = ids >= 0
    key = torch.where(known, ids, torch.full_like(ids, E)).reshape(-1)
    src = key.sort(stable=True).indices.int()
    hist = torch.bincount(key, minlength=E + 1)[:E].int()
    rd = fm.RoutingData(w.reshape(-1)[src.long()].float(), hist, E, topk)
    qm = {"fp8": _capi.QMODE_FP8_BLOCK, "int8": _capi.QMODE_INT8_CHANNEL}[mode]
    ref = fm._fused_routed(x, wts.w1, wts.w2, rd, fm.GatherIndx(src, src), qmode=qm,
                           w1_scale=wts.w1_scale, w2_scale=wts.w2_scale)
    ids[::3, -1] = torch.where(torch.arange(len(ids[::3]), device=gpu) % 2 == 0, -1, E).int()
    assert torch.equal(fm.fused_moe(x, wts.w1, wts.w2, w, ids, **wts.kwargs(mode)), ref)
