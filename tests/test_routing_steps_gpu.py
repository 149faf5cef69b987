"""The small routing kernels at the sizes and values where they can go wrong:
whole and partial waves of experts, ties, signed zeros, masked (-inf) and
infinite logits, against the oracle."""

import pytest
import torch

from flaggems_sglang.ops import fused_moe as fm
from oracle import moe_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scoring", ["softmax", "sigmoid"])
@pytest.mark.parametrize("E", [1, 2, 63, 64, 65, 128, 250, 512, 1023, 1024])
def test_gating_ranks(gpu, E, scoring):
    k = min(E, 64)
    g = torch.Generator().manual_seed(E)
    logits = torch.randn(9, E, generator=g)
    logits[1] = torch.randint(-2, 3, (E,), generator=g).float()      # ties
    logits[2] = torch.where(torch.arange(E) % 2 == 0, 0.0, -0.0)     # equal zeros
    logits[3, : E // 2] = float("-inf")                              # masked experts
    logits[4] = -torch.rand(E, generator=g) * 1e-40                  # denormal, negative
    logits[5] = 80.0 * torch.randn(E, generator=g)                   # scores at 0 and 1
    logits[6, E - 1] = logits[6].max()                               # a tie across the row
    logits[7] = logits[7].bfloat16().float()
    w, ids = fm.fused_topk(torch.empty(9, 8, device=gpu), logits.to(gpu), k, renormalize=False,
                           scoring_func=scoring)
    rw, rids = moe_ref.topk_gating(logits, k, scoring=scoring, renormalize=False)
    assert torch.equal(ids.cpu(), rids)
    # a score: the exponential's and the sum's fp32 rounding (2 ulps each)
    assert torch.allclose(w.cpu(), rw, rtol=2e-6, atol=1e-7)


@pytest.mark.parametrize("M,k,E", [(0, 4, 65), (8, 8, 64), (9, 8, 65), (64, 4, 128),
                                   (512, 8, 129), (513, 8, 256), (700, 6, 1022), (3, 1, 1),
                                   (110, 8, 1022), (450, 8, 1022)])
def test_conversion_tables(gpu, M, k, E):
    """One, 64, 65, 4095.. slots and whole and partial waves of experts: the
    single-wave, single- and many-workgroup alignments (and, at 880 and 3600
    slots of 1022 experts, the one for more experts than the single-workgroup
    one's LDS takes) write the histogram, the last workgroup of the finishing
    launch the tables. Ids on either side
    of [0, E) sort behind the experts and count for none."""
    g = torch.Generator().manual_seed(M + E)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(M)]).int() if M else \
        torch.empty(0, k, dtype=torch.int32)
    ids[::3, -1] = -1
    ids[1::5, 0] = E
    ids[2::5, 0] = 2 ** 30
    w = torch.rand(M, k, generator=g)
    rd, gi, si = fm.standard_topk_to_routing(w.to(gpu), ids.to(gpu), E)
    # the oracle's dropped id is -1
    known = torch.where((ids >= 0) & (ids < E), ids, torch.full_like(ids, -1))
    hist = torch.bincount(known[known >= 0].long().reshape(-1), minlength=E).int()
    assert torch.equal(rd.expt_hist.cpu(), hist)
    raw, pad, pid = moe_ref.expt_data(hist.numpy(), E, M * k)
    assert torch.equal(rd.expt_data.token_offs_raw.cpu(), torch.from_numpy(raw))
    for bm in moe_ref.ROUTING_BLOCK_MS:
        assert torch.equal(rd.expt_data.token_offs_pad[bm].cpu(), torch.from_numpy(pad[bm]))
        assert torch.equal(rd.expt_data.block_pid_map[bm].cpu(), torch.from_numpy(pid[bm]))
    # every expert's range of the gathered order holds its slots, in slot order
    rank = torch.argsort(ids, dim=1, stable=True)            # slot of each row-sorted place
    slot = (rank + torch.arange(M)[:, None] * k).reshape(-1)
    src = gi.src_indx.cpu().long()
    got = known.reshape(-1)[slot[src]] if M else src
    n = int(hist.sum())
    assert torch.equal(got[:n], torch.repeat_interleave(torch.arange(E), hist.long()).int())
    assert bool((got[n:] == -1).all())
    for e in range(E):
        assert bool((slot[src[raw[e]:raw[e + 1]]].diff() > 0).all())
    assert torch.equal(si.src_indx.cpu().long()[src], torch.arange(M * k))
    assert torch.equal(rd.gate_scal.cpu(), w.reshape(-1)[slot[src]] if M else w.reshape(-1))


@pytest.mark.parametrize("E", [1, 64, 65, 130, 1024])
def test_order_from_extreme_histograms(gpu, E):
    """Counts of a caller's histogram up to the type's limits: the running
    sums are cut at the gate count without wrapping in 32 bits."""
    n = 3 * E
    hist = torch.full((E,), 2 ** 31 - 1, dtype=torch.int32)
    hist[::2] = -(2 ** 31)
    hist[0] = 2
    g = torch.Generator().manual_seed(E)
    src = torch.randperm(n, generator=g).int()
    gs = torch.rand(n, generator=g)
    _, _, _, rid, rwt = moe_ref.routing_order(gs.numpy(), src.numpy(), hist.numpy(), n, 1)
    tw, ti = fm._routing_to_topk(fm.RoutingData(gs.to(gpu), hist.to(gpu), E, 3),
                                 fm.GatherIndx(src.to(gpu), src.to(gpu)), E)
    assert torch.equal(ti.cpu().reshape(-1), torch.from_numpy(rid))
    assert torch.equal(tw.cpu().reshape(-1), torch.from_numpy(rwt))


@pytest.mark.parametrize("numel", [65, 128, 129, 1000, 1024, 1025, 2048, 2049, 4095, 4096,
                                   4097, 8191, 8192, 8193])
@pytest.mark.parametrize("E,B", [(1, 16), (7, 100), (64, 1), (256, 16), (257, 256), (1023, 8),
                                 (1024, 256)])
def test_align_a_wave_per_chunk(gpu, numel, E, B):
    """65 to 4096 slots, one to four runs of 64 of them per wave, and the
    sizes on either side; dropped and outside ids, experts without slots and
    one with most."""
    g = torch.Generator().manual_seed(numel + E)
    ids = torch.randint(-1, E + 2, (numel,), generator=g).int()
    ids[::4] = E // 2
    s, eids, npp = fm.moe_align_block_size(ids.reshape(-1, 1).to(gpu), E, B)
    rs, reids, rnpp = moe_ref.align(ids.numpy().reshape(-1, 1), E, B)
    assert int(npp.item()) == rnpp
    assert torch.equal(s.cpu(), torch.from_numpy(rs))
    assert torch.equal(eids.cpu(), torch.from_numpy(reids))


def test_align_skewed_ids_in_parallel(gpu):
    """4096 slots in blocks of one row: all on one expert cost about what
    spread ones do (the block -> expert map is written by the slots, not by a
    thread per expert: 12 times as long). Whole launches, replayed in turn."""
    from flaggems_sglang import _capi

    lib, n, E = _capi.load(), 4096, 64
    out = [torch.empty(s, dtype=torch.int32, device=gpu) for s in (n, n, 1)]
    ids = {"spread": torch.arange(n, device=gpu).remainder(E).int(),
           "one": torch.full((n,), E - 1, device=gpu).int()}

    def launch(x):
        stream = torch.cuda.current_stream().cuda_stream
        for _ in range(20):
            _capi.check(lib.fgs_moe_align_block_size(
                x.data_ptr(), n, E, 1, *(t.data_ptr() for t in out), n, None, 0, stream), "align")

    graphs = {}
    for name, x in ids.items():
        launch(x)
        torch.cuda.synchronize()
        graphs[name] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graphs[name]):
            launch(x)
    times = {name: [] for name in ids}
    for _ in range(5):
        for name, g in graphs.items():
            t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            t0.record()
            g.replay()
            t1.record()
            torch.cuda.synchronize()
            times[name].append(t0.elapsed_time(t1))
            assert torch.equal(out[1].cpu(), ids[name].sort().values.cpu())
    assert min(times["one"]) < 3 * min(times["spread"]), times
