"""Which expert weights the grouped GEMM wrappers take, by dtype: host logic
only, so the library's entry points are stood in for by a recorder."""
import pytest
import torch

from ubridge_amd import moe

T, K, N, E = 4, 64, 16, 2


class Recorder:
    """Takes the place of the library: the names of the entry points called."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append(name)
            return 0
        return call


@pytest.fixture
def rec(monkeypatch):
    r = Recorder()
    monkeypatch.setattr(moe, "lib", r)
    monkeypatch.setattr(moe, "check", lambda rc=None: None)
    monkeypatch.setattr(moe, "_need_cuda", lambda *ts: None)
    monkeypatch.setattr(moe, "stream_ptr", lambda stream=None: None)
    return r


def _routing():
    i = torch.zeros(T, dtype=torch.int32)
    return i, i, i


@pytest.mark.parametrize("a,b,scales,entry", [
    (torch.bfloat16, torch.int8, True, "ubridge_fused_moe_w8a16_silu"),
    (torch.float16, torch.uint8, True, "ubridge_fused_moe_w8a16_silu"),  # int8 codes as bytes
    (torch.bfloat16, torch.int8, False, "ubridge_fused_moe_w8a16_silu"),  # which refuses it
    (torch.bfloat16, torch.bfloat16, False, "ubridge_fused_moe_silu"),
    (torch.float16, torch.float16, False, "ubridge_fused_moe_silu"),
    (torch.bfloat16, torch.float16, False, None),
    (torch.float16, torch.bfloat16, True, None),
    (torch.bfloat16, torch.float32, False, None),
    (torch.bfloat16, torch.float8_e4m3fn, True, None)])
def test_gate_up_silu_weight_dtypes(rec, a, b, scales, entry):
    A, B = torch.zeros(T, K, dtype=a), torch.zeros(E, N, K).to(b)
    S = torch.ones(E, N, dtype=a) if scales else None
    if entry is None:
        with pytest.raises(ValueError):
            moe.fused_moe_gate_up_silu(A, B, S, *_routing(), 1, 4)
        assert rec.calls == []
    else:
        moe.fused_moe_gate_up_silu(A, B, S, *_routing(), 1, 4)
        assert rec.calls == [entry]


@pytest.mark.parametrize("a,b,entry", [
    (torch.bfloat16, torch.int8, "ubridge_fused_moe_w8a16"),
    (torch.bfloat16, torch.bfloat16, "invoke_fused_moe_bf16"),
    (torch.float16, torch.float16, "invoke_fused_moe_f16"),
    (torch.bfloat16, torch.float16, None), (torch.float16, torch.uint8, None),
    (torch.bfloat16, torch.float32, None)])
def test_expert_gemm_weight_dtypes(rec, a, b, entry):
    A, B, C = torch.zeros(T, K, dtype=a), torch.zeros(E, N, K).to(b), torch.zeros(T, N, dtype=a)
    S = torch.ones(E, N, dtype=a)
    call = lambda: moe.invoke_fused_moe(A, B, C, None, *_routing(), 1, 4, False, B_scale=S)
    if entry is None:
        with pytest.raises(ValueError):
            call()
        assert rec.calls == []
    else:
        call()
        assert rec.calls == [entry]
    ids = torch.zeros(T, 1, dtype=torch.int32)
    call = lambda: moe.topsaten_fused_moe_gemm(A, B, None, ids, *_routing(), False, 4)
    if a == b:
        call()
        assert rec.calls[-1] == "topsaten_fused_moe_gemm"
    else:
        with pytest.raises(ValueError):
            call()
