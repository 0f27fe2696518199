"""Kernels and dispatch rules at the sizes where they can go wrong: edges of tiles, remainders, the smallest and the
largest of a variant's range."""
import pytest
import torch

from _util import randn_bf16

pytestmark = pytest.mark.gpu


def test_grouped_wgrad_of_many_one_block_experts_is_the_same_every_time(gpu):
    """Tiles of a single k-block store almost without pause, the state in which a store's data registers were once
    overwritten before the store had read them: an expert without rows must have a weight gradient of exact zeros and
    every launch the same bits."""
    from hpfp8 import ops
    counts = [2155, 0, 983, 7145, 0, 100, 1528, 3, 3362, 1211, 0, 128]
    rows, n, k = sum(counts), 2048, 3584
    offs = torch.tensor(counts).cumsum(0).to(torch.int32).to(gpu)
    x, go = randn_bf16((rows, k), 1).to(gpu), randn_bf16((rows, n), 2).to(gpu)
    layout = ops.grouped_layout(offs, rows)
    xt, sxt = ops.quantize_128x1_t_grouped(x, layout, len(counts))
    got, sgot = ops.quantize_128x1_t_grouped(go, layout, len(counts))
    first = ops.gemm_grouped_wgrad(got, sgot, xt, sxt, layout, len(counts), rows)
    for e, c in enumerate(counts):
        if c == 0:
            assert int(first[e].count_nonzero()) == 0
    for _ in range(20):
        assert torch.equal(ops.gemm_grouped_wgrad(got, sgot, xt, sxt, layout, len(counts), rows), first)
