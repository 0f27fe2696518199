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


def _ints(shape, seed, gpu, lo=-4, hi=5):
    """Small integers as E4M3 codes: products and their sums over any of the contractions here are exact in fp32."""
    g = torch.Generator(device="cpu").manual_seed(seed)
    return torch.randint(lo, hi, shape, generator=g).float().to(torch.float8_e4m3fn).to(gpu)


def _pow2(shape, seed, gpu):
    g = torch.Generator(device="cpu").manual_seed(seed)
    return torch.exp2(torch.randint(-2, 3, shape, generator=g).float()).to(gpu)


def _dequantized(q, s, rows, cols=128):
    """float64 values of codes q[R, C] with one scale per rows x cols block (exact for the inputs here)."""
    v = q.double()
    r, c = v.shape
    return (v.view(r // rows, rows, c // cols, cols) * s.double().view(r // rows, 1, c // cols, 1)).view(r, c)


@pytest.mark.parametrize("m", [1, 16, 17, 32, 33, 48, 49, 64, 65])
@pytest.mark.parametrize("n,k", [(128, 128), (256, 640), (1152, 1152), (33024, 384), (384, 2048), (256, 2432), (33024, 2048)])
def test_gemm_with_few_rows_is_exact_on_integer_inputs(gpu, m, n, k):
    """Every row-fragment count of the few-rows GEMM and the first row count beyond it; contractions on both sides of the
    shortest it takes, k-blocks that divide among its waves and that do not; fewer units of columns than compute units,
    uneven runs of them, and wide ones.  All
    partial sums are integers below 2^24 (k / 128 blocks of 128 products of at most 16, times scales of at most 16 in
    steps of 2^-4), so every order of summation gives the exact result."""
    from hpfp8 import ops
    a, b = _ints((m, k), 1, gpu), _ints((n, k), 2, gpu)
    kb = k // 128
    sa, sb = _pow2((kb, m), 3, gpu).t(), _pow2((n // 128, kb), 4, gpu)
    bias = _pow2((n,), 5, gpu).to(torch.bfloat16)
    want = _dequantized(a, sa.contiguous(), 1) @ _dequantized(b, sb, 128).t()
    assert torch.equal(ops.gemm_blockwise(a, sa, b, sb, out_dtype=torch.float32).double(), want)
    assert torch.equal(ops.gemm_blockwise(a, sa.contiguous(), b, sb, bias=bias), (want + bias.double()).to(torch.bfloat16))
    assert torch.equal(ops.gemm_blockwise(a, sa, b, sb, pow2_scales=True, out_dtype=torch.float32).double(), want)
    one = a.double() @ b.double().t() * 0.125
    ta, tb = torch.tensor(0.5, device=gpu), torch.tensor(0.25, device=gpu)
    assert torch.equal(ops.gemm_per_tensor(a, ta, b, tb, out_dtype=torch.float32).double(), one)
    assert torch.equal(ops.gemm_per_tensor(a, ta, b, tb, bias=bias), (one + bias.double()).to(torch.bfloat16))


@pytest.mark.parametrize("counts", [[1], [0, 1, 0], [16, 17, 32, 0, 33], [48, 49, 0, 64, 65, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0],
                                    [200] + [0] * 69 + [3, 0, 7], [5] * 130])
@pytest.mark.parametrize("n,k", [(128, 128), (384, 640), (256, 2176)])
def test_grouped_gemm_with_few_rows_is_exact_on_integer_inputs(gpu, counts, n, k):
    """Row counts around every fragment count and around the 64-row chunks, empty experts, more experts than a wave has
    lanes, fewer units than workgroups; rows past the last offset stay as they are.  Exact for the reason above."""
    from hpfp8 import _lib, ops
    e, rows = len(counts), sum(counts) + 2
    a, b = _ints((rows, k), 1, gpu), _ints((e * n, k), 2, gpu)
    kb = k // 128
    sa, sb = _pow2((kb, rows), 3, gpu).t(), _pow2((e * n // 128, kb), 4, gpu)
    offs = torch.tensor(counts).cumsum(0).to(torch.int32).to(gpu)
    av, bv = _dequantized(a, sa.contiguous(), 1), _dequantized(b, sb, 128).view(e, n, k)
    out = torch.full((rows, n), 7.0, dtype=torch.float32, device=gpu)
    _lib.call("hpfp8_gemm_grouped_blockwise", a.data_ptr(), k, sa.data_ptr(), sa.stride(0), sa.stride(1), b.data_ptr(), sb.data_ptr(),
              offs.data_ptr(), e, rows, n, k, out.data_ptr(), n, _lib.OUT_F32, ops._stream())
    r = 0
    for i, c in enumerate(counts):
        assert torch.equal(out[r:r + c].double(), av[r:r + c] @ bv[i].t())
        r += c
    assert bool((out[r:] == 7.0).all())
    y = ops.gemm_grouped_blockwise(a, sa, b.view(e, n, k), sb.view(e, n // 128, kb), offs)
    assert torch.equal(y[:r], out[:r].to(torch.bfloat16))
