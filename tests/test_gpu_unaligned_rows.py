"""Dense K latents whose rows are contiguous but not 16-byte aligned whole
chunks (odd ranks, odd offsets, odd context lengths), staged as runs of bytes,
against the oracle; rows that are not contiguous keep the other routes."""
import pytest
import torch

from _util import check_logits, check_output, make_case, oracle_decode, oracle_logits

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16
# MHA (one odd rank misaligns every later head, whole-chunk ranks included) and grouped queries (ranks at both ends of the
# linear range, K-steps of 16 ranks at every remainder); one to many tiles per workgroup, contexts ending inside a tile
CASES = [
    ("mha_odd", 3, 8, 8, 1003, [9, 16, 101, 32, 128, 33, 96, 127], 200, F16),
    ("mha_even", 2, 4, 4, 33, [102, 10, 66, 8], 64, F16),
    ("mha_bf16", 1, 6, 6, 4099, [15, 17, 31, 64, 65, 88], 40, BF16),
    ("mha_one_position", 2, 3, 3, 1, [11, 24, 55], 64, F16),
    ("gqa_odd", 2, 16, 4, 1003, [9, 8, 127, 49], 200, F16),
    ("gqa_102", 1, 32, 8, 2100, [102] * 8, 64, F16),
    ("gqa_bf16", 3, 8, 4, 777, [113, 97, 33, 15], 64, BF16),
    ("gqa_odd_heads", 1, 6, 3, 65, [81, 23, 119], 64, F16),
    ("gqa_too_wide", 1, 4, 2, 500, [128, 31], 64, F16),       # 128 misaligned: copied (K logits) / register streaming
    ("below_a_chunk", 2, 4, 4, 130, [7, 12, 40, 1], 64, F16),
    ("mha_few_ranks", 2, 6, 6, 300, [8, 9, 13, 15, 11, 14], 64, F16),    # (decode streams them in registers)
    ("mha_few_ranks_bf16", 1, 5, 5, 129, [10, 11, 12, 14, 15], 40, BF16),
]


@pytest.mark.parametrize("name,B,Hq,Hkv,S,ranks,Rv,dtype", CASES, ids=[c[0] for c in CASES])
def test_odd_ranks(name, B, Hq, Hkv, S, ranks, Rv, dtype):
    from starkv import decode_attention, k_logits
    print(f"[unaligned rows] {name}", flush=True)
    case = make_case(B, Hq, Hkv, S, ranks, Rv, dtype=dtype, seed=11)
    scale = 128 ** -0.5
    check_logits(k_logits(case.q, case.kspec, S, scale=scale), oracle_logits(case, scale=scale), scale, name)
    out = decode_attention(case.q, case.kspec, case.xv, case.uv, out_dtype=torch.float32)
    check_output(out, oracle_decode(case)[0], name)


@pytest.mark.parametrize("Hq,Hkv,ranks", [(4, 4, [40, 24, 128, 64]), (8, 2, [104, 56]), (4, 4, [41, 15, 99, 12]),
                                          (8, 2, [101, 57])])
@pytest.mark.parametrize("shift", [1, 3, 7])
def test_shifted_base(Hq, Hkv, ranks, shift):
    """Rows from a base 2, 6 or 14 bytes off, with infinities planted just
    outside every head's rows: nothing of them may reach a logit."""
    from starkv import KLatentSpec, k_logits
    S, B = 100, 2
    case = make_case(B, Hq, Hkv, S, ranks, 64, dtype=F16, seed=12)
    gap = 5
    sizes = [S * r for r in ranks]
    buf = torch.full((B, shift + sum(sizes) + gap * Hkv + 8), float("inf"), dtype=F16, device="cuda")
    offs, o = [], shift
    for h, n in enumerate(sizes):
        offs.append(o)
        buf[:, o:o + n] = case.xk_heads[h].reshape(B, n)
        o += n + gap
    k = KLatentSpec(buf, ranks, offs, ranks, buf.stride(0), case.kspec.bk, case.kspec.bk_head_offset,
                    case.kspec.bk_row_stride)
    print(f"[shifted base] {shift} {ranks}", flush=True)
    a, b = k_logits(case.q, k, S), k_logits(case.q, case.kspec, S)
    # the same products in the same order, whatever the alignment
    assert torch.equal(a, b)


@pytest.mark.parametrize("layout_ranks", [[33, 48, 7, 101], [30, 42, 50, 66]])
def test_rows_not_contiguous(layout_ranks):
    """All heads of a position side by side (odd ranks): not a linear run."""
    from starkv import decode_attention, k_logits
    case = make_case(2, 8, 4, 333, layout_ranks, 64, dtype=F16, layout="posmajor", seed=13)
    print(f"[posmajor] {layout_ranks}", flush=True)
    scale = 128 ** -0.5
    check_logits(k_logits(case.q, case.kspec, 333, scale=scale), oracle_logits(case, scale=scale), scale, "posmajor")
    check_output(decode_attention(case.q, case.kspec, case.xv, case.uv, out_dtype=torch.float32), oracle_decode(case)[0],
                 "posmajor")


# V ranks around a chunk, a wave's slab (4, 8 and 13 tiles) and a column block; rows 2-byte aligned
@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("Rv,B,S,pad", [(5, 2, 70, 0), (9, 1, 33, 0), (127, 2, 300, 0), (129, 3, 17, 2), (257, 1, 1000, 1),
                                        (1023, 2, 250, 0), (417, 1, 129, 0), (1249, 2, 200, 0), (1637, 3, 500, 0),
                                        (1664, 1, 100, 3), (3001, 1, 260, 0),
                                        # one, two and four chunks a lane: their last and first ranks
                                        (128, 2, 130, 1), (255, 1, 65, 0), (256, 2, 47, 3)])
def test_dense_v_rows(Rv, B, S, pad, dtype):
    """Dense V latents of odd ranks and pitches, in the drop-in P.V and the
    fused decode; what lies between the rows and past the last is infinite."""
    from starkv import decode_attention, pv_latent
    print(f"[dense v rows] Rv={Rv} B={B} S={S} pad={pad} {dtype}", flush=True)
    case = make_case(B, 8, 8, S, [16] * 8, Rv, dtype=dtype, seed=14)
    buf = torch.full((B * S * (Rv + pad) + 64,), float("inf"), dtype=dtype, device="cuda")
    xv = torch.as_strided(buf, (B, S, Rv), (S * (Rv + pad), Rv + pad, 1), 1)
    xv.copy_(case.xv)
    p = torch.softmax(torch.randn(B, 8, S, device="cuda", generator=torch.Generator("cuda").manual_seed(1)), -1).to(dtype)
    ref = torch.matmul(p.double().cpu(), case.xv.double().cpu())
    check_output(pv_latent(p, xv), ref, "P.V ")
    out = decode_attention(case.q, case.kspec, xv, case.uv, out_dtype=torch.float32)
    check_output(out, oracle_decode(case)[0], "decode ")


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("ranks,S", [([102, 49, 127, 9], 333), ([8, 33, 64, 119], 32), ([31, 95], 2049)])
def test_gqa_linear_rows_masked(ranks, S, dtype):
    """Grouped queries over contiguous odd ranks under an additive mask and
    under a device-held last position, contexts ending inside a tile: both
    against the oracle, and the two forms of the same mask against each other."""
    from starkv import decode_attention, k_logits
    B, Hkv = 2, len(ranks)
    print(f"[gqa linear masked] {ranks} S={S} {dtype}", flush=True)
    case = make_case(B, 4 * Hkv, Hkv, S, ranks, 64, dtype=dtype, seed=16)
    last, scale = S - 1 - S // 5, 128 ** -0.5
    mask = torch.zeros(B, 1, S, device="cuda")
    mask[..., last + 1:] = -1e30
    mask[0, 0, :last + 1:7] = -3.0
    out = decode_attention(case.q, case.kspec, case.xv, case.uv, mask=mask, out_dtype=torch.float32)
    check_output(out, oracle_decode(case, mask=mask.double().cpu())[0], "additive mask ")
    got = k_logits(case.q, case.kspec, S, scale=scale, mask=mask)
    plain = k_logits(case.q, case.kspec, S, scale=scale)
    # scale * sum + mask rounds once in the kernel (a fused multiply-add), scale * sum first here: at most half a unit in
    # the last place of the product, and one of the result
    assert bool(((got - (plain + mask)).abs() <= 2.0 ** -23 * (plain.abs() + (plain + mask).abs())).all())
    mask[0, 0, :last + 1] = 0.0
    lp = torch.tensor([last], dtype=torch.int32, device="cuda")
    a = decode_attention(case.q, case.kspec, case.xv, case.uv, last_pos=lp, out_dtype=torch.float32)
    m = decode_attention(case.q, case.kspec, case.xv, case.uv, mask=mask, out_dtype=torch.float32)
    check_output(a, oracle_decode(case, mask=mask.double().cpu())[0], "last position ")
    # (past the last position -1e30 against a logit plus -1e30: the same fp32 number)
    assert torch.equal(a, m)


@pytest.mark.parametrize("latent_scale,q_scale", [(30000.0, 1.0), (1.0, 1e5), (3000.0, 3e4)], ids=["keys", "queries", "both"])
def test_gqa_linear_bf16_beyond_fp16_range(latent_scale, q_scale):
    """bf16 keys or queries past fp16's range over contiguous odd ranks: the
    rerun with scaled keys (test_gpu_decode.py has it for aligned rows)."""
    from starkv import k_logits
    ranks = [101, 102, 33, 127, 49, 64, 97, 15]
    case = make_case(1, 32, 8, 300, ranks, 64, dtype=BF16, seed=17, latent_scale=latent_scale)
    case.q.mul_(q_scale)
    print(f"[gqa linear bf16 range] {latent_scale} {q_scale}", flush=True)
    out = k_logits(case.q, case.kspec, 300)
    ref = oracle_logits(case)
    assert torch.isfinite(out).all()
    rms = float(ref.pow(2).mean().sqrt())
    d = (out.double().cpu() - ref).abs() / rms
    assert float(d.max()) <= 2e-2 and float(d.mean() / (ref.abs().mean() / rms)) <= 1e-3
