"""P.V over the per-token block formats at the edges of its raw kernel: one,
four, five and seven column tiles a wave, upper blocks of one and of many
tiles, int8 and int4, alone and over a lower block, rows of any alignment,
steps of 32 positions, and latents it leaves to the other kernels."""
import pytest
import torch

from _util import check_output, make_case
from test_gpu_quant import _dequant_one_hot, make_quant_v

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16
# kind, rank, split, pad
SHAPES = [("ref_int8", 64, 32, 0), ("ref_int8", 93, 32, 0), ("ref_int4", 288, 256, 0), ("ref_int4", 1024, 64, 1),
          ("ref_int8", 1025, 256, 0), ("ref_int4", 1279, 256, 0), ("ref_int8", 1281, 128, 2), ("ref_int8", 1640, 256, 0),
          ("ref_int4", 1792, 512, 0), ("ref_int8", 1791, 288, 3), ("int4_whole", 33, 33, 0), ("int4_whole", 1640, 1640, 1),
          ("int8", 16, 16, 0), ("int8", 1001, 1001, 0),
          # an upper block of part of a tile, rows below one piece, too many pieces, too many tiles
          ("ref_int8", 300, 40, 0), ("int8", 9, 9, 0), ("int8", 1100, 1100, 0), ("ref_int4", 1920, 256, 0)]


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("kind,R,split,pad", SHAPES)
def test_dequant_bit_exact(kind, R, split, pad, dtype):
    print(f"[pv block one-hot] {kind} R={R} split={split} pad={pad} {dtype}", flush=True)
    _dequant_one_hot(kind, R, split, dtype, pad)


# rows of whole dwords past 1280 ranks: the context length at which the drop-in product changes kernels; unaligned ones
@pytest.mark.parametrize("S", [2047, 2048])
@pytest.mark.parametrize("kind,R,split,pad", [("int4_whole", 1640, 1640, 0), ("ref_int4", 1792, 512, 0), ("ref_int8", 1288, 256, 0),
                                              ("ref_int4", 1288, 256, 1)])
def test_many_ranks(kind, R, split, pad, S):
    test_products(kind, R, split, pad, F16, 1, S, 8)


@pytest.mark.parametrize("B,S,H", [(1, 1, 32), (2, 31, 8), (1, 33, 40), (3, 500, 32)])
@pytest.mark.parametrize("kind,R,split,pad,dtype", [SHAPES[0] + (F16,), SHAPES[5] + (F16,), SHAPES[7] + (F16,), SHAPES[9] + (BF16,),
                                                    SHAPES[13] + (BF16,), SHAPES[14] + (F16,)])
def test_products(kind, R, split, pad, dtype, B, S, H):
    """The drop-in product and the fused decode against fp64 over the dequantised values."""
    from oracle import starkv_oracle as o
    from starkv import RopeConfig, decode_attention, pv_latent
    print(f"[pv block] {kind} R={R} B={B} S={S} H={H} {dtype}", flush=True)
    spec, deq, _ = make_quant_v(kind, B, S, R, split=split, seed=5, pad=pad)
    deq = torch.from_numpy(deq).to(dtype).double()
    g = torch.Generator(device="cuda").manual_seed(2)
    p = torch.softmax(torch.randn(B, H, S, generator=g, device="cuda") * 3, dim=-1).to(dtype)
    check_output(pv_latent(p, spec), p.double().cpu() @ deq, "P.V ")
    case = make_case(B, H, 8, S, [32] * 8, R, dtype=dtype, seed=3)
    out = decode_attention(case.q, case.kspec, spec, case.uv, out_dtype=torch.float32)
    rope = RopeConfig()
    cos, sin = o.rope_cos_sin(rope.inv_freq(), torch.arange(S), rope.attention_scaling)
    ref = o.decode_attention(case.q.cpu(), [b.cpu() for b in case.bk_heads], [x.cpu() for x in case.xk_heads], deq,
                             case.uv.cpu(), cos, sin)[0]
    check_output(out, ref, "decode ")
