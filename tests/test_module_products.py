"""The drop-in modules' torch route for a masked prompt (CPU): no batched
product over a transposed right operand, which has faulted the GPU in bfloat16
(at batch 1 torch passes a transposed U_k through as it is)."""
import importlib

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode


class _Products(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.transposed = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        if func.overloadpacket in (torch.ops.aten.bmm, torch.ops.aten.baddbmm):
            right = args[-1]
            if right.stride(-1) != 1:
                self.transposed.append((tuple(right.shape), right.stride()))
        return func(*args, **(kwargs or {}))


class _Pair(torch.nn.Module):
    def __init__(self, vs, u):
        super().__init__()
        self.VS, self.U = vs, u


@pytest.mark.parametrize("module", ["LlamaLoRaAttention_headwise", "LlamaLoRaAttention_headwise_quant"])
def test_no_batched_product_over_a_transposed_operand(module, monkeypatch):
    from transformers import LlamaConfig
    mod = importlib.import_module("starkv." + module)
    Hq, Hkv, r, Rv, T = 4, 2, 40, 300, 6
    cfg = LlamaConfig(hidden_size=Hq * 128, num_attention_heads=Hq, num_key_value_heads=Hkv, intermediate_size=64,
                      num_hidden_layers=1)
    torch.manual_seed(0)
    m = mod.LlamaCustomAttention(cfg, layer_idx=0, decomp_goup_num=Hq)
    m.k_proj = _Pair(torch.nn.Linear(cfg.hidden_size, Hkv * r, bias=False), torch.randn(Hkv, 128, r) / r ** 0.5)
    m.v_proj = _Pair(torch.nn.Linear(cfg.hidden_size, Rv, bias=False), torch.nn.Linear(Rv, Hkv * 128, bias=False))
    m.k_proj.VS, m.v_proj.VS, m.v_proj.U = (x.bfloat16() for x in (m.k_proj.VS, m.v_proj.VS, m.v_proj.U))
    m.k_proj.U = m.k_proj.U.bfloat16()
    m = m.bfloat16().eval()
    if module.endswith("quant"):                       # its quantiser is a device kernel

        def quantised(x, split):
            rest = x.shape[-1] - split
            z = lambda n, dt: torch.zeros(*x.shape[:-1], n, dtype=dt)
            return z(split, torch.int8), z(1, torch.float16), z((rest + 1) // 2, torch.uint8), z(1, torch.float16), rest

        monkeypatch.setattr(mod, "quantize_r_split_int8_int4_packed", quantised)
    # the attention itself is torch's, with products of its own
    monkeypatch.setattr(mod.F, "scaled_dot_product_attention", lambda q, K, V, **kw: q + 0 * (K + V))
    hidden = (torch.randn(1, T, cfg.hidden_size) * 0.5).bfloat16()
    mask = torch.zeros(1, 1, T, T, dtype=torch.bfloat16)
    cos, sin = torch.ones(1, T, 128).bfloat16(), torch.zeros(1, T, 128).bfloat16()
    with torch.no_grad(), _Products() as seen:
        m(hidden, (cos, sin), mask)
    assert not seen.transposed, seen.transposed
