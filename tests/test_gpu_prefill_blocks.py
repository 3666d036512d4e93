"""The causal attention's block loop at the context lengths where its pipelining
can go wrong: one key block, an odd and an even number of them, waves with
blocks wholly in their future, a chunk whose first block is already past the
mask; gates as in test_gpu_prefill.py."""
import pytest
import torch

from test_gpu_prefill import _run


@pytest.mark.gpu
@pytest.mark.parametrize("T,pos0", [(1, 0), (1, 63), (1, 64), (33, 31), (64, 0), (65, 0), (129, 0), (192, 0), (257, 0),
                                    (256, 1), (300, 130), (31, 500)])
def test_prefill_block_edges(T, pos0):
    _run(1, 4, [32, 64], 136, T, pos0, torch.float16, seed=T + pos0)
