"""Host-side shortcuts of the Python layer, on the CPU."""

import os
import subprocess
import sys
import time
import types

import pytest
import torch

from flaggems_sglang import _capi
from flaggems_sglang.ops import fused_moe as fm


def test_combine_class_follows_a_later_import(monkeypatch):
    """Without SGLang the stand-in, remembered; once something has imported
    SGLang, its class."""
    monkeypatch.setattr(fm, "_combine_cls", None)
    monkeypatch.setattr(fm, "_sglang_absent", False)
    name = "sglang.srt.layers.moe.token_dispatcher.standard"
    parts = [".".join(name.split(".")[: i + 1]) for i in range(len(name.split(".")))]
    for p in parts:
        monkeypatch.delitem(sys.modules, p, raising=False)
    assert fm._combine_input_cls() is fm.StandardCombineInput
    assert fm._sglang_absent
    for p in parts:
        mod = types.ModuleType(p)
        mod.__path__ = []
        monkeypatch.setitem(sys.modules, p, mod)
    sys.modules[name].StandardCombineInput = type("StandardCombineInput", (), {})
    cls = fm._combine_input_cls()
    assert cls is sys.modules[name].StandardCombineInput
    assert fm._combine_input_cls() is cls


def test_conversion_view_shortcut():
    """A transposed view of a native-layout weight converts to the native
    tensor itself and is not cached; a reference-layout one is converted once
    per version."""
    cache = fm._ConversionCache(lambda t: t.transpose(-1, -2).contiguous(),
                                view=lambda t: t.transpose(-1, -2))
    native = torch.randn(2, 6, 4)
    assert cache(native.transpose(-1, -2)).data_ptr() == native.data_ptr()
    assert len(cache) == 0
    ref = torch.randn(2, 4, 6)
    first = cache(ref)
    assert first.is_contiguous() and torch.equal(first, ref.transpose(-1, -2))
    assert cache(ref) is first and len(cache) == 1
    ref.add_(1.0)
    assert torch.equal(cache(ref), ref.transpose(-1, -2))
    # one row or column: both orders are contiguous, so the view serves
    row = torch.randn(2, 1, 6)
    assert cache(row).data_ptr() == row.data_ptr() and cache(row).is_contiguous()


def test_scaled_entry_refusals():
    """The scaled entry's checks are the entry points' it covers."""
    lib, nul, shape = _capi.load(), None, (4, 256, 128, 4, 2)
    need = lib.fgs_moe_workspace_bytes(*shape, _capi.QMODE_BF16, 0)

    def call(b13=nul, b2=nul, w=16, flags=0, alpha=1.0, ws_bytes=need):
        return lib.fgs_moe_fused_scaled(0, 16, 16, 16, nul, nul, b13, b2, alpha, 0.0, w, 16,
                                        *shape, flags, 2.5, 256, ws_bytes, 16, nul)

    for kw, code, text in [({"b13": 16}, -1, "b13 and b2"), ({"b2": 16}, -1, "b13 and b2"),
                           ({"b13": 16, "b2": 16, "flags": _capi.FLAG_ACT_GELU}, -2, "swiglu"),
                           ({"b13": 16, "b2": 16, "alpha": float("nan")}, -1, "NaN"),
                           ({"w": nul}, -1, "null pointer"), ({"ws_bytes": need - 1}, -1,
                                                              "workspace")]:
        assert call(**kw) == code and text in _capi.last_error()


def test_split_scale():
    t = torch.tensor([1.0, 2.0])
    for factor, want in [(None, (None, None)), (1, (None, None)), (True, (None, None)),
                         (2, (2.0, None)), (0.5, (0.5, None)), (False, (0.0, None)),
                         (2 ** 53 + 1, (None, 2 ** 53 + 1)), (1j, (None, 1j))]:
        assert fm._split_scale(factor) == want
    with pytest.raises(RuntimeError):  # ambiguous, as the comparison was before
        fm._split_scale(t)


# (problem, flags), whether the allocation-free entry point takes it, and under
# which tuning switches that turns over
_T4 = _capi.flag_tile(4)
_NOALLOC = [((582, 6912, 1920, 16, 2), _T4, True, ("KSPLIT=3",)),
            ((94, 7680, 1792, 8, 8), _T4, True, ("KSPLIT=3",)),
            ((3220, 1536, 1280, 60, 2), _T4, False, ()),
            ((138, 4352, 5632, 16, 4), _T4, False, ("KSPLIT=3",)),
            ((1503, 3328, 128, 32, 4), 0, False, ("KSPLIT=3", "TILE=4", "TAIL=0")),
            ((582, 6912, 1920, 16, 2), 0, True, ("KSPLIT=3",)),
            ((2100, 4224, 3200, 8, 2), 0, True, ())]


def _noalloc_taken(lib):
    """Null pointers: a problem past the scratch is refused as unsupported, any
    other for its pointers (or, without a GPU, its scratch), before a launch."""
    out = []
    for shape, flags, _, _ in _NOALLOC:
        rc = lib.fgs_moe_fused_bf16_noalloc(*[None] * 5, *shape, flags, None, None)
        assert rc < 0
        out.append(rc != _capi.FGS_EUNSUPPORTED)
    return out


@pytest.mark.parametrize("switch", ["", "TILE=4", "TAIL=0", "KSPLIT=3"])
def test_no_alloc_accepted_set(switch):
    """The problems the allocation-free entry point takes do not move with the
    schedule rules: the 160-row configuration's split counts one block per
    expert below 160 rows, and the tuning switches count as in a call."""
    want = [taken != (switch in turns) for _, _, taken, turns in _NOALLOC]
    if not switch:
        assert _noalloc_taken(_capi.load()) == want
        return
    here = os.path.dirname(os.path.abspath(__file__))
    code = (f"import sys; sys.path[:0] = {[here] + sys.path!r}\n"
            "import test_host_paths as t\nprint(t._noalloc_taken(t._capi.load()))")
    name, value = switch.split("=")
    env = dict(os.environ, FGS_MOE_TUNING="1", **{"FGS_MOE_" + name: value})
    r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    assert r.stdout.strip().splitlines()[-1] == str(want)


def test_plan_time_of_long_calls():
    """A plan's block estimate does not walk a long call's blocks one by one
    (2^27 tokens on one expert: 0.25 s for these plans)."""
    _capi.schedule(2, 128, 128, 1, 1)
    t0 = time.perf_counter()
    for _ in range(30):
        assert "tiled" in _capi.schedule(2 ** 27, 128, 128, 1, 1)
    assert time.perf_counter() - t0 < 0.05


@pytest.mark.parametrize("qmode,shape,split", [
    (_capi.QMODE_BF16, (92, 2688, 3584, 8, 2), "ksplit2=2"),       # 88 tiles
    (_capi.QMODE_FP8_BLOCK, (381, 1408, 13312, 8, 2), "ksplit2=2"),  # 88 of 128 columns
    (_capi.QMODE_BF16, (83, 4224, 11648, 8, 2), ""),               # 136
    (_capi.QMODE_BF16, (128, 1280, 4096, 8, 2), "ksplit2=3")])     # 80 of 128 columns
def test_k_split_fits_one_round(qmode, shape, split):
    """GEMM2's k split stays within one round of the 256 CUs: a few tiles past
    it make a second round (88 tiles in three 16 % slower than in two)."""
    sched = _capi.schedule(*shape, qmode)
    assert [w for w in sched.split() if "split" in w] == split.split(), sched
