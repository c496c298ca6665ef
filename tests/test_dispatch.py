"""Which entry points the operators reach, on the CPU with the launches
recorded instead of made: no launch on tensors the GPU does not own."""

import pytest
import torch

import keep_amd
from keep_amd import _lib, ops


@pytest.fixture
def launches(monkeypatch):
    """The entry points called, none of them run; a GPU's stream and capture state stubbed."""
    calls, real = [], _lib.call
    host = ("keep_e8p_packed_abs_grid", "keep_e8_1bit_packed")  # tables built on the host
    monkeypatch.setattr(_lib, "call", lambda name, *a: real(name, *a) if name in host else calls.append(name))
    monkeypatch.setattr(ops, "_raw_stream", lambda index: 0)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    monkeypatch.setattr(ops, "_PREPARED", {})
    return calls


def _moe(T, H=512, I=256, E=4, k=2):
    codes = lambda n, K: (torch.zeros((E, n, K // 8), dtype=torch.int16), torch.ones((E, n, 1), dtype=torch.float16))  # noqa: E731
    return (torch.zeros((T, H), dtype=torch.float16), torch.zeros((T, E)), (codes(I, H), codes(I, H), codes(H, I)),
            torch.zeros((T, k), dtype=torch.int32), torch.ones((T, k)))


@pytest.mark.parametrize("call", ["decode", "decode_packed", "tiles_layer", "layer", "wide"])
def test_cpu_activations_are_refused_before_any_launch(launches, call):
    x, z, pool, idx, w = _moe(1 if call == "layer" else 3, **({"H": 4096, "I": 512} if call == "layer" else
                                                              {"H": 4608} if call == "wide" else {}))
    with pytest.raises(ValueError, match="cuda device"):
        if call in ("decode", "wide"):
            keep_amd.moe_decode(x, idx, w, *pool)
        elif call == "decode_packed":
            keep_amd.moe_decode(x, idx, w, *pool, prepared=False)
        elif call == "tiles_layer":
            keep_amd.moe_tiles_layer(x, z, *pool, k=2)
        else:
            keep_amd.moe_layer(x, z, *pool, k=2)
    assert launches == []


def test_a_table_prepared_under_capture_is_not_kept(launches, monkeypatch):
    """It holds nothing before that graph's first replay: the next eager call builds its own, once."""
    cb = torch.from_numpy(ops.e8p_packed_abs_grid().view("int32"))
    monkeypatch.setattr(ops, "_stream", lambda device: 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: type("S", (), {"synchronize": lambda self: None})())
    captured = ops.prepared_table(cb)
    assert launches == ["keep_e8p_prepare"] and not ops._may_prepare(cb)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    assert ops._may_prepare(cb)
    eager = ops.prepared_table(cb)
    assert eager is not captured and launches == ["keep_e8p_prepare"] * 2
    assert ops.prepared_table(cb) is eager
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert ops._may_prepare(cb) and ops.prepared_table(cb) is eager
    assert len(launches) == 2
