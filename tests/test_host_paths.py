"""Host-side shortcuts of the Python layer, on the CPU."""

import sys
import types

import torch

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
