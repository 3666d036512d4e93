"""The cache writer's kernel for runs of positions against its row-per-wave
kernel: one append of a whole run must store the bytes, scales and zero points
that appends of a few positions at a time store (those are pinned to the
oracle's quantisers in test_gpu_cache.py)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# ranks and V ranks at the edges of 8-rank chunks, 64-rank groups, the split
# blocks (16 of K, 256 of V) and one, two and four chunks per thread
SHAPES = [
    ("harness", [96, 56, 48, 32, 16] * 6 + [88, 16], 1640, 2, 600),
    ("odd", [1, 7, 9, 33, 101, 127, 128, 15], 1637, 3, 1379),
    ("narrow", [8], 5, 1025, 35),
    ("gqa", [32, 128, 32, 80, 32, 64, 80, 64], 512, 7, 613),
    ("two_per_thread", [128] * 20, 2056, 5, 331),
    ("four_per_thread", [128] * 40, 4203, 3, 277),
    ("split_edges", [16, 17, 24, 128], 256, 8, 1030),
    ("split_edges_v", [3, 31], 263, 900, 21),
    # V rows of one chunk per thread in the block kernel: past a rank's row count, past 28 groups
    ("block_v", [16], 300, 30, 820),
    ("block_v_split_edge", [8], 257, 25, 1000),
    ("block_v_wide", [16, 9], 1793, 4, 4100),
]


def _inputs(B, T, ranks, Rv, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    k = torch.randn(B, T, sum(ranks), generator=g, device="cuda")
    v = torch.randn(B, T, Rv, generator=g, device="cuda")
    for x in (k, v):
        x[..., ::97] *= 10
        # quotients that are exact ties: scale 1 (int8) on halves of integers, and multiples of a group's step
        x[:, 1::7] = torch.randint(-254, 255, x[:, 1::7].shape, generator=g, device="cuda").float() / 2
        x[:, 1::7, ::5] = 127.0
        x[:, 2::11] = torch.randint(0, 31, x[:, 2::11].shape, generator=g, device="cuda").float() / 2
        x[:, 3::13] = 0.0
        x[:, 4::17] *= 1e-6
        x[:, 5::19] *= 2000.0
        x[:, 6, ::41] = float("nan")
        x[:, 8, ::43] = float("inf")
        x[:, 9, ::43] = float("-inf")
    if dtype == torch.bfloat16:
        k[:, 10] *= 1e30
        v[:, 10] *= 1e30
    return k.to(dtype), v.to(dtype)


@pytest.mark.parametrize("fmt", ["dense", "int8_g64", "reference"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("name,ranks,Rv,B,T", SHAPES, ids=[s[0] for s in SHAPES])
def test_run_equals_rows(name, ranks, Rv, B, T, dtype, fmt):
    from starkv.cache import LatentCache
    print(f"[append run] {name} {fmt} {dtype}", flush=True)
    k, v = _inputs(B, T, ranks, Rv, dtype, 3)
    bk = torch.zeros(len(ranks), max(ranks), 128, device="cuda", dtype=dtype)
    cap = T + 5
    run = LatentCache(B, ranks, Rv, cap, dtype, "cuda", fmt=fmt)
    rows = LatentCache(B, ranks, Rv, cap, dtype, "cuda", fmt=fmt)
    for t in (slice(0, 2), slice(2, T)):              # the run starts at position 2
        run.append(k[:, t], v[:, t], bk)
    for t in range(0, T, 15):                         # runs of fewer than 16 positions: the row-per-wave kernel
        rows.append(k[:, t:t + 15], v[:, t:t + 15], bk)
    for n in ("k_data", "k_scale", "k_data2", "k_scale2", "v_data", "v_scale", "v_zero", "v_data2", "v_scale2"):
        if hasattr(run, n):
            a, b = getattr(run, n).contiguous(), getattr(rows, n).contiguous()
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), n


def test_run_past_the_capacity_skips_and_flags():
    """A device-held position: rows of the run that land outside the capacity
    are skipped and set the error flag, the others are written."""
    from starkv.cache import LatentCache
    B, T, cap, ranks, Rv = 16, 1100, 1000, [32, 24], 300
    for fmt in ("dense", "int8_g64", "reference"):
        k, v = _inputs(B, T, ranks, Rv, torch.float16, 4)
        bk = torch.zeros(2, 32, 128, device="cuda", dtype=torch.float16)
        a, b = (LatentCache(B, ranks, Rv, cap, torch.float16, "cuda", fmt=fmt) for _ in range(2))
        err = torch.zeros(1, dtype=torch.int32, device="cuda")
        pos = torch.tensor([50], dtype=torch.int32, device="cuda")
        a.append_at(k, v, bk, pos, error_flag=err)
        assert int(err) == 1
        b.length = 50
        for t in range(0, 950, 10):
            b.append(k[:, t:min(t + 10, 950)], v[:, t:min(t + 10, 950)], bk)
        for n in ("k_data", "k_scale", "k_data2", "v_data", "v_scale", "v_zero", "v_data2"):
            if hasattr(a, n):
                assert torch.equal(getattr(a, n).contiguous().view(torch.uint8),
                                   getattr(b, n).contiguous().view(torch.uint8)), (fmt, n)
