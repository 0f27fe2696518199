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
@pytest.mark.parametrize("n,k", [(128, 128), (256, 640), (1152, 1152), (33024, 384), (384, 512), (1152, 896), (384, 2048), (256, 2432), (33024, 2048)])
def test_gemm_with_few_rows_is_exact_on_integer_inputs(gpu, m, n, k):
    """Every row-fragment count of the few-rows GEMM and the first row count beyond it; contractions on both sides of the
    shortest it takes, k-blocks that divide into its stages and that do not; fewer runs of columns than compute units and
    more.  All partial sums are integers below 2^24 (k / 128 blocks of 128 products of at most 16, times scales of at most 16 in
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


# (n, k) of the few-rows form: with the row counts below every number of fragments per workgroup (1, 2, 3, 4, 6 and 9 on 256
# compute units) in one run and in several, last runs that are partly missing, stages of two, four and eight k-blocks that
# divide the contraction and that do not, or that are longer than it
FEW_ROWS_SHAPES = [(128, 2048), (1152, 2432), (8320, 2176), (12160, 2304), (16384, 2432), (24704, 2176), (36736, 2432), (38400, 2176),
                   (1152, 512), (8320, 640), (24704, 1024), (33024, 1920)]


def _normal(shape, seed, gpu, std=1.0, outliers=False):
    """Normal values drawn on the GPU (the wide weights here would take seconds on the CPU)."""
    g = torch.Generator(device=gpu).manual_seed(seed)
    x = torch.empty(shape, dtype=torch.bfloat16, device=gpu).normal_(0.0, std, generator=g)
    if outliers:
        x.view(-1)[torch.randint(0, x.numel(), (1 + x.numel() // 1000,), device=gpu, generator=g)] *= 50.0
    return x


def _both_tiles(run):
    """What `run` gives under the default rule and with the 256 x 256 tiles of the general form."""
    from hpfp8 import _lib
    got = run()
    _lib.load().hpfp8_debug_set_small_gemm(1)
    try:
        return got, run()
    finally:
        _lib.load().hpfp8_debug_set_small_gemm(0)


@pytest.mark.parametrize("m", [1, 8, 9, 23, 37, 48, 57, 64])
@pytest.mark.parametrize("n,k", FEW_ROWS_SHAPES)
def test_gemm_with_few_rows_has_the_bits_of_the_general_form(gpu, m, n, k):
    """Random values, so that the order and the rounding of the sums show: an element of c does not depend on how many
    rows there are or which kernel computes it.  Against 64 bits: what the matrix instruction leaves of products some 2^12
    times smaller than the largest of its 128 (test_gpu_gemm.py measures that and derives the 1e-4 used here)."""
    from hpfp8 import ops
    x, w = _normal((m, k), 1, gpu, outliers=True), _normal((n, k), 2, gpu, 0.02)
    bias = _normal((n,), 3, gpu)
    for pow2 in (False, True):
        a, sa = ops.quantize_1x128(x, kmajor=True, pow2=pow2)
        b, sb = ops.quantize_128x128(w, pow2=pow2)
        got, want = _both_tiles(lambda: ops.gemm_blockwise(a, sa, b, sb, pow2_scales=pow2, out_dtype=torch.float32))
        assert torch.equal(got, want)
        exact = _dequantized(a, sa.contiguous(), 1) @ _dequantized(b, sb, 128).t()
        assert float((got.double() - exact).norm() / exact.norm()) < 1e-4
        got, want = _both_tiles(lambda: ops.gemm_blockwise(a, sa.contiguous(), b, sb, bias=bias, pow2_scales=pow2))
        assert torch.equal(got, want)
    a, _, sa = ops.quantize_per_tensor(x)
    b, _, sb = ops.quantize_per_tensor(w)
    got, want = _both_tiles(lambda: ops.gemm_per_tensor(a, sa, b, sb, out_dtype=torch.float32))
    assert torch.equal(got, want)
    got, want = _both_tiles(lambda: ops.gemm_per_tensor(a, sa, b, sb, bias=bias))
    assert torch.equal(got, want)


@pytest.mark.parametrize("m", [1, 17, 40, 64])
@pytest.mark.parametrize("n,k", [(1152, 2432), (8320, 2176), (16384, 2432)])
def test_gemm_with_few_rows_on_rows_with_strides(gpu, m, n, k):
    """Row strides of a, b and c beyond the width: the same bits, and c untouched outside its columns and rows."""
    from hpfp8 import _lib, ops
    x, w = _normal((m, k), 1, gpu), _normal((n, k), 2, gpu, 0.02)
    a, sa = ops.quantize_1x128(x, kmajor=True)
    b, sb = ops.quantize_128x128(w)
    want = ops.gemm_blockwise(a, sa, b, sb)
    a8, b8 = _strided_rows(a.view(torch.uint8), 48, gpu), _strided_rows(b.view(torch.uint8), 16, gpu)
    c = torch.full((m + 3, n + 24), 7.0, dtype=torch.bfloat16, device=gpu)
    _lib.call("hpfp8_gemm_blockwise", a8.data_ptr(), a8.stride(0), sa.data_ptr(), sa.stride(0), sa.stride(1), b8.data_ptr(),
              b8.stride(0), sb.data_ptr(), sb.stride(0), sb.stride(1), 128, m, n, k, None, c.data_ptr(), c.stride(0), _lib.OUT_BF16, 0,
              ops._stream())
    assert torch.equal(c[:m, :n], want)
    assert bool((c[:m, n:] == 7.0).all()) and bool((c[m:] == 7.0).all())


@pytest.mark.parametrize("m", [2, 9, 33, 64])
@pytest.mark.parametrize("pow2", [False, True])
def test_gemm_with_few_rows_keeps_nan_and_infinity_to_their_rows(gpu, m, pow2):
    """A NaN code, a NaN scale and an infinite scale in a row of a, a NaN code in a row of b: that row or column of c as the
    general form has it, every other element unchanged."""
    from hpfp8 import ops
    n, k = 8320, 2432
    x, w = _normal((m, k), 1, gpu), _normal((n, k), 2, gpu, 0.02)
    a, sa = ops.quantize_1x128(x, kmajor=True, pow2=pow2)
    b, sb = ops.quantize_128x128(w, pow2=pow2)
    clean = ops.gemm_blockwise(a, sa, b, sb, pow2_scales=pow2)
    bad = m // 2
    for what in ("code", "nan", "inf", "weight"):
        a2, s2, b2 = a.clone(), sa.t().clone().t(), b.clone()
        if what == "code":
            a2.view(torch.uint8)[bad, 200] = 0x7F
        elif what == "weight":
            b2.view(torch.uint8)[4000, k - 1] = 0xFF
        else:
            s2[bad, 3] = float(what)
        got, want = _both_tiles(lambda: ops.gemm_blockwise(a2, s2, b2, sb, pow2_scales=pow2))
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)) or torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))
        keep = torch.ones((m, n), dtype=torch.bool, device=gpu)
        if what == "weight":
            assert bool(got[:, 4000].isnan().all())
            keep[:, 4000] = False
        else:
            assert not bool(got[bad].isfinite().all())
            keep[bad] = False
        assert torch.equal(got[keep], clean[keep])


@pytest.mark.parametrize("m", [1, 2, 7, 8])
@pytest.mark.parametrize("n,k", [(128, 128), (256, 512), (1152, 640), (4096, 2432), (7168, 4096), (8320, 1152), (36864, 512)])
def test_rows_quantized_inside_the_few_rows_product_have_the_bits_of_the_two_launches(gpu, m, n, k):
    """1, 2 and 3 fragments of columns per workgroup, one run of them and several, k-blocks that fill the last stage and that do not;
    a row of zeros, one below the smallest scale, and a NaN and an infinity that stay in their row."""
    from hpfp8 import _lib, ops
    x, w = _normal((m, k), 1, gpu, outliers=True), _normal((n, k), 2, gpu, 0.02)
    bias = _normal((n,), 3, gpu)
    if m > 2:
        x[1] = 0.0
        x[2] *= 2.0 ** -60
    x_bad = x.clone()
    x_bad[-1, 5], x_bad[-1, k - 1] = float("nan"), float("inf")
    for pow2 in (False, True):
        b, sb = ops.quantize_128x128(w, pow2=pow2)
        for src in (x, x_bad):
            q, s = ops.quantize_1x128(src, kmajor=True, pow2=pow2)
            for dtype, with_bias in ((torch.bfloat16, bias), (torch.float32, None)):
                want = ops.gemm_blockwise(q, s, b, sb, bias=with_bias, pow2_scales=pow2, out_dtype=dtype)
                c = torch.full((m + 1, n + 8), 7.0, dtype=dtype, device=gpu)
                _lib.call("hpfp8_linear_few_rows_bf16", src.data_ptr(), b.data_ptr(), b.stride(0), sb.data_ptr(), sb.stride(0), sb.stride(1),
                          m, n, k, pow2, None if with_bias is None else with_bias.data_ptr(), c.data_ptr(), c.stride(0),
                          _lib.OUT_F32 if dtype == torch.float32 else _lib.OUT_BF16, ops._stream())
                assert torch.equal(c[:m, :n].nan_to_num(3.0), want.nan_to_num(3.0))
                assert torch.equal(c[:m, :n].isnan(), want.isnan())
                assert bool((c[:m, n:] == 7.0).all()) and bool((c[m] == 7.0).all())


def test_rows_quantized_inside_the_few_rows_product_may_be_as_long_as_those_of_codes(gpu):
    """The limit on a row is the product's, 8 MiB of codes; the same row of bf16 is twice as many bytes."""
    from hpfp8 import _lib, ops
    m, n, k = 8, 128, (1 << 22) + 128
    x, w = _normal((m, k), 1, gpu), _normal((n, k), 2, gpu, 0.02)
    b, sb = ops.quantize_128x128(w)
    q, s = ops.quantize_1x128(x, kmajor=True)
    want = ops.gemm_blockwise(q, s, b, sb)
    c = torch.zeros((m, n), dtype=torch.bfloat16, device=gpu)
    _lib.call("hpfp8_linear_few_rows_bf16", x.data_ptr(), b.data_ptr(), b.stride(0), sb.data_ptr(), sb.stride(0), sb.stride(1), m, n, k, False,
              None, c.data_ptr(), c.stride(0), _lib.OUT_BF16, ops._stream())
    assert torch.equal(c, want)


def test_gemm_with_few_rows_and_power_of_two_scales_whose_product_is_out_of_range(gpu):
    """Two scales of 2^80: their product is no fp32 number, but a product of codes that is zero stays zero."""
    from hpfp8 import ops
    m, n, k = 5, 256, 2048
    a, b = _ints((m, k), 1, gpu), _ints((n, k), 2, gpu)
    a.view(torch.uint8)[:, 128:256] = 0
    sa = torch.ones((m, k // 128), dtype=torch.float32, device=gpu)
    sb = torch.ones((n // 128, k // 128), dtype=torch.float32, device=gpu)
    want = ops.gemm_blockwise(a, sa, b, sb, pow2_scales=True, out_dtype=torch.float32)
    sa[:, 1], sb[:, 1] = 2.0 ** 80, 2.0 ** 80
    assert torch.equal(ops.gemm_blockwise(a, sa, b, sb, pow2_scales=True, out_dtype=torch.float32), want)


def test_gemm_with_few_rows_does_not_depend_on_the_column_or_the_batch(gpu):
    """The same rows of b in other places (a column shard, a rolled weight) and more rows of a: the same bits."""
    from hpfp8 import ops
    n, k = 7168, 16384
    x, w = _normal((65, k), 1, gpu), _normal((n, k), 2, gpu, 0.02)
    a, sa = ops.quantize_1x128(x, kmajor=True)
    b, sb = ops.quantize_128x128(w)
    c = ops.gemm_blockwise(a, sa, b, sb)
    for m in (1, 8, 37, 64):
        am, sm = ops.quantize_1x128(x[:m], kmajor=True)
        assert torch.equal(ops.gemm_blockwise(am, sm, b, sb), c[:m])
        half = ops.gemm_blockwise(am, sm, b[n // 2:], sb[n // 256:])
        assert torch.equal(half, c[:m, n // 2:])
        rolled = ops.gemm_blockwise(am, sm, b.view(torch.uint8).roll(1280, 0).view(b.dtype), sb.roll(10, 0))
        assert torch.equal(rolled, c[:m].roll(1280, 1))


@pytest.mark.parametrize("m", [1, 37, 64, 65])
@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("pow2_in,pow2_out", [(False, False), (True, False), (False, True), (True, True)])
def test_swiglu_epilogue_is_its_two_calls_at_decode_row_counts(gpu, m, fast, pow2_in, pow2_out):
    """What `hpfp8_gemm_blockwise_swiglu_quantize` promises, on both sides of the few-rows GEMM's last row count: bit for bit
    the GEMM followed by the SwiGLU quantizer, by the C entry point and by the operator, which takes two launches there."""
    from hpfp8 import _lib, ops
    k, inter = 7168, 4608
    x, w = _normal((m, k), 1, gpu), _normal((2 * inter, k), 2, gpu, 0.05)
    a, sa = ops.quantize_1x128(x, kmajor=True, pow2=pow2_in)
    b, sb = ops.quantize_128x128(w, pow2=pow2_in)
    h = ops.gemm_blockwise(a, sa, b, sb, pow2_scales=pow2_in)
    q, si = ops.swiglu_quantize_1x128(h, fast=fast, pow2=pow2_out)
    cq = torch.zeros((m, inter), dtype=torch.uint8, device=gpu)
    cs, csi = (torch.zeros((inter // 128, m), dtype=torch.float32, device=gpu) for _ in range(2))
    _lib.call("hpfp8_gemm_blockwise_swiglu_quantize", a.data_ptr(), k, sa.data_ptr(), sa.stride(0), sa.stride(1), b.data_ptr(), k,
              sb.data_ptr(), sb.stride(0), sb.stride(1), m, inter, k, int(fast), int(pow2_in), int(pow2_out), cq.data_ptr(), inter,
              cs.data_ptr(), csi.data_ptr(), ops._stream())
    assert torch.equal(cq, q.view(torch.uint8)) and torch.equal(csi.t(), si)
    got = ops.gemm_blockwise_swiglu_quantize(a, sa, b, sb, fast=fast, pow2_scales=pow2_in, pow2_out=pow2_out, want_scale=True)
    assert torch.equal(got[0].view(torch.uint8), cq) and torch.equal(got[1], si) and torch.equal(got[2], cs.t())


@pytest.mark.parametrize("m", [64, 65])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_swiglu_operator_takes_two_launches_where_the_gemm_takes_few_rows(gpu, m, mode, monkeypatch):
    """One rule for both, the library's: the operator splits exactly where the GEMM would take its few-rows form, so a tile
    that the test hook asks for reaches the epilogue it belongs to."""
    from hpfp8 import _lib, ops
    k, inter = 2048, 128
    a, sa = ops.quantize_1x128(_normal((m, k), 1, gpu), kmajor=True)
    b, sb = ops.quantize_128x128(_normal((2 * inter, k), 2, gpu, 0.05))
    names, call, gemm = [], _lib.call, ops.gemm_blockwise
    monkeypatch.setattr(_lib, "call", lambda name, *args: (names.append(name), call(name, *args))[1])
    monkeypatch.setattr(ops, "gemm_blockwise", lambda *args, **kw: (names.append("gemm_blockwise"), gemm(*args, **kw))[1])
    _lib.load().hpfp8_debug_set_small_gemm(mode)
    try:
        few = m <= _lib.load().hpfp8_gemm_few_rows(k)
        ops.gemm_blockwise_swiglu_quantize(a, sa, b, sb)
    finally:
        _lib.load().hpfp8_debug_set_small_gemm(0)
    assert few == (m == 64 and mode == 0)
    assert names == (["gemm_blockwise", "hpfp8_swiglu_quantize_1x128_bf16"] if few else ["hpfp8_gemm_blockwise_swiglu_quantize"])


@pytest.mark.parametrize("m", [1, 64, 65])
def test_swiglu_operator_refuses_a_weight_of_two_gib_at_every_row_count(gpu, m):
    """512 rows of codes 4 MiB apart: what the fused call refuses is not taken on where the operator would split it."""
    from hpfp8 import _lib, ops
    k = 2048
    b = torch.empty(512 << 22, dtype=torch.uint8, device=gpu).view(512, 1 << 22)[:, :k]
    a = torch.zeros((m, k), dtype=torch.uint8, device=gpu)
    sa, sb = torch.ones((m, k // 128), device=gpu), torch.ones((4, k // 128), device=gpu)
    with pytest.raises(_lib.Hpfp8Error, match="2 GiB"):
        ops.gemm_blockwise_swiglu_quantize(a, sa, b, sb)


@pytest.mark.parametrize("counts", [[1], [0, 1, 0], [16, 17, 32, 0, 33], [48, 49, 0, 64, 65, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0],
                                    [200] + [0] * 69 + [3, 0, 7], [5] * 130])
@pytest.mark.parametrize("n,k", [(128, 128), (384, 640), (256, 2176)])
def test_grouped_gemm_with_few_rows_is_exact_on_integer_inputs(gpu, counts, n, k):
    """Experts of a few rows each, so that every tile is a partial one; empty experts, many of them in a row, more experts
    than a wave has lanes, fewer tiles than workgroups; rows past the last offset stay as they are.  Exact for the reason
    above."""
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


def _strided_rows(t, pad, gpu):
    """The same rows with a row stride of pad elements more."""
    wide = torch.zeros((t.shape[0], t.shape[1] + pad), dtype=t.dtype, device=gpu)
    wide[:, :t.shape[1]] = t
    return wide[:, :t.shape[1]]


@pytest.mark.parametrize("m,n", [(300, 6784), (385, 5504), (256, 16384), (300, 14208), (129, 32512), (257, 10880)])
@pytest.mark.parametrize("k", [128, 256, 640])
def test_gemm_tiles_are_exact_on_integer_inputs(gpu, m, n, k):
    """Problems that take 128 x 128 tiles (the first three) and 128 x 256 tiles (the last three) under the default rule,
    with ragged rows, an odd number of 128-column blocks, contractions of one, two and five k-blocks; every scale form,
    output type, bias and accumulation.  Exact for the reason above (with scales on both operands' rows sums are multiples
    of 2^-4 too)."""
    from hpfp8 import ops
    a, b = _ints((m, k), 1, gpu), _ints((n, k), 2, gpu)
    kb = k // 128
    sa, sb = _pow2((kb, m), 3, gpu).t(), _pow2((n // 128, kb), 4, gpu)
    sr = _pow2((kb, n), 6, gpu).t()
    bias = _pow2((n,), 5, gpu).to(torch.bfloat16)
    av = _dequantized(a, sa.contiguous(), 1)
    want = av @ _dequantized(b, sb, 128).t()
    rows = av @ _dequantized(b, sr.contiguous(), 1).t()
    for pow2 in (False, True):
        assert torch.equal(ops.gemm_blockwise(a, sa, b, sb, pow2_scales=pow2, out_dtype=torch.float32).double(), want)
        assert torch.equal(ops.gemm_blockwise(_strided_rows(a, 16, gpu), sa.contiguous(), b, sb, bias=bias, pow2_scales=pow2),
                           (want + bias.double()).to(torch.bfloat16))
        assert torch.equal(ops.gemm_blockwise(a, sa, b, sr, sb_gran=1, pow2_scales=pow2), rows.to(torch.bfloat16))
        c = torch.full((m, n), 3.0, dtype=torch.float32, device=gpu)
        ops.gemm_blockwise(a, sa, b, sr, sb_gran=1, out=c, accumulate=True, pow2_scales=pow2)
        assert torch.equal(c.double(), rows + 3.0)
        ops.gemm_blockwise(a, sa, b, sb, out=c, accumulate=True, pow2_scales=pow2)
        assert torch.equal(c.double(), rows + 3.0 + want)
    one = a.double() @ b.double().t() * 0.125
    ta, tb = torch.tensor(0.5, device=gpu), torch.tensor(0.25, device=gpu)
    assert torch.equal(ops.gemm_per_tensor(a, ta, b, tb, out_dtype=torch.float32).double(), one)
    assert torch.equal(ops.gemm_per_tensor(a, ta, b, tb, bias=bias), (one + bias.double()).to(torch.bfloat16))


@pytest.mark.parametrize("m,n,k", [(1, 128, 128), (127, 384, 256), (129, 640, 640), (300, 2432, 384), (1000, 1152, 1152)])
def test_every_tile_shape_gives_the_same_bits(gpu, m, n, k):
    """256 x 256, 64 x 64 (64 x 256 for the SwiGLU epilogue), 128 x 256, 128 x 128 and 64 x 128 tiles, asked for one after the other (so
    whatever the number of compute units; a form that lacks one takes the next larger) on random values: all scale forms, output types,
    bias, accumulation, the SwiGLU epilogue and experts."""
    from hpfp8 import _lib, ops
    x, w = _normal((m, k), 1, gpu, outliers=True), _normal((2 * n, k), 2, gpu, 0.05)
    bias, c0 = _normal((n,), 3, gpu), _normal((m, n), 4, gpu).float()
    rows = torch.tensor([m // 3, 0, m - m // 3]).cumsum(0).to(torch.int32).to(gpu)
    out = {}
    for mode in (1, 2, 3, 4, 5):
        _lib.load().hpfp8_debug_set_small_gemm(mode)
        try:
            r = out[mode] = []
            for pow2 in (False, True):
                a, sa = ops.quantize_1x128(x, kmajor=True, pow2=pow2)
                b, sb = ops.quantize_128x128(w, pow2=pow2)
                br, sr = ops.quantize_1x128(w[:n], kmajor=True, pow2=pow2)
                b1, sb1 = b[:n], sb[:n // 128]
                r.append(ops.gemm_blockwise(a, sa, b1, sb1, pow2_scales=pow2, out_dtype=torch.float32))
                r.append(ops.gemm_blockwise(a, sa.contiguous(), b1, sb1, bias=bias, pow2_scales=pow2))
                r.append(ops.gemm_blockwise(a, sa, br, sr, sb_gran=1, pow2_scales=pow2))
                r.append(ops.gemm_blockwise(a, sa.contiguous(), br, sr, sb_gran=1, pow2_scales=pow2, out_dtype=torch.float32))
                for gran, bb, ss in ((128, b1, sb1), (1, br, sr)):
                    r.append(ops.gemm_blockwise(a, sa, bb, ss, sb_gran=gran, out=c0.clone(), accumulate=True, pow2_scales=pow2))
                r += ops.gemm_blockwise_swiglu_quantize(a, sa, b, sb, fast=pow2, pow2_scales=pow2, pow2_out=pow2, want_scale=True)
                stack = b.view(2, n, k), sb.view(2, n // 128, k // 128)
                experts = [torch.cat((t, t[:1])) if t.dtype == torch.float32 else torch.cat((t.view(torch.uint8), t[:1].view(torch.uint8)))
                           for t in stack]
                for dtype in (torch.bfloat16, torch.float32):
                    r.append(ops.gemm_grouped_blockwise(a, sa, *experts, rows, pow2_scales=pow2, out_dtype=dtype))
            a, _, sa = ops.quantize_per_tensor(x)
            b, _, sb = ops.quantize_per_tensor(w[:n])
            r.append(ops.gemm_per_tensor(a, sa, b, sb, out_dtype=torch.float32))
            r.append(ops.gemm_per_tensor(a, sa, b, sb, bias=bias))
        finally:
            _lib.load().hpfp8_debug_set_small_gemm(0)
    for mode in (2, 3, 4, 5):
        for got, want in zip(out[mode], out[1]):
            assert torch.equal(got.view(torch.uint8) if got.dtype == torch.float8_e4m3fn else got,
                               want.view(torch.uint8) if want.dtype == torch.float8_e4m3fn else want)


@pytest.mark.parametrize("m,inter,k", [(65, 128, 128), (127, 384, 384), (129, 1280, 256), (300, 10752, 128)])
@pytest.mark.parametrize("fast,pow2", [(True, False), (False, True)])
def test_swiglu_epilogue_is_the_same_with_both_tile_heights(gpu, m, inter, k, fast, pow2):
    from hpfp8 import _lib, ops
    x, w = randn_bf16((m, k), 1).to(gpu), randn_bf16((2 * inter, k), 2, 0.05).to(gpu)
    xq, sx = ops.quantize_1x128(x, kmajor=True, pow2=pow2)
    wq, sw = ops.quantize_128x128(w, pow2=pow2)
    got = ops.gemm_blockwise_swiglu_quantize(xq, sx, wq, sw, fast=fast, pow2_scales=pow2, want_scale=True)
    _lib.load().hpfp8_debug_set_small_gemm(1)
    try:
        want = ops.gemm_blockwise_swiglu_quantize(xq, sx, wq, sw, fast=fast, pow2_scales=pow2, want_scale=True)
    finally:
        _lib.load().hpfp8_debug_set_small_gemm(0)
    assert torch.equal(got[0].view(torch.uint8), want[0].view(torch.uint8))
    assert torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])


@pytest.mark.parametrize("counts", [[127, 128, 129, 0, 1, 255, 257], [0, 0, 1000, 3], [2048, 0, 1, 700]])
@pytest.mark.parametrize("n,k", [(128, 128), (640, 384)])
def test_grouped_tiles_are_exact_on_integer_inputs(gpu, counts, n, k):
    """Row counts around the 128-row tile of the grouped form, the tile it takes for few rows per expert."""
    test_grouped_gemm_with_few_rows_is_exact_on_integer_inputs(gpu, counts, n, k)


@pytest.mark.parametrize("rows,experts,n", [(513, 8, 4096), (2048, 8, 4096), (2049, 8, 4096), (4096, 32, 2048), (8192, 32, 4096),
                                            (1024, 4, 16384)])
@pytest.mark.parametrize("spread", ["even", "zipf", "half", "two", "one", "none"])
def test_grouped_gemm_leaves_the_tile_height_to_the_device(gpu, rows, experts, n, spread):
    """Row counts at which the host cannot know which tile is better and the kernel chooses (and some at which it knows): every row is
    computed, with the bits of 256 x 256 tiles."""
    from hpfp8 import _lib, ops
    k = 256
    counts = {"even": [rows // experts] * experts, "zipf": [int(rows / 4 / (i + 1)) for i in range(experts)],
              "half": [rows // 2] + [rows // 2 // experts] * (experts - 1), "two": [0, rows // 2] + [0] * (experts - 3) + [rows // 2],
              "one": [0] * (experts - 1) + [rows], "none": [0] * experts}[spread]
    a, sa = ops.quantize_1x128(_normal((rows, k), 1, gpu), kmajor=True)
    b, sb = ops.quantize_128x128(_normal((experts * n, k), 2, gpu, 0.05))
    offs = torch.tensor(counts).cumsum(0).clamp(max=rows).to(torch.int32).to(gpu)

    def run():
        out = torch.full((rows, n), 7.0, dtype=torch.bfloat16, device=gpu)
        _lib.call("hpfp8_gemm_grouped_blockwise", a.data_ptr(), k, sa.data_ptr(), sa.stride(0), sa.stride(1), b.data_ptr(), sb.data_ptr(),
                  offs.data_ptr(), experts, rows, n, k, out.data_ptr(), n, _lib.OUT_BF16, ops._stream())
        return out
    got, want = _both_tiles(run)
    assert torch.equal(got, want)
    assert bool((got[int(offs[-1]):] == 7.0).all())


@pytest.mark.parametrize("m", [1, 63, 64, 65, 127, 128, 129, 383])
@pytest.mark.parametrize("k", [128, 640, 2048])
@pytest.mark.parametrize("pow2", [False, True])
def test_dual_quantizers_of_ragged_rows_equal_those_of_zero_padded_rows(gpu, m, k, pow2):
    """Both row quads of a tile partly or wholly missing, one tile and several, both walking orders (row stride a multiple
    of 4 KB or not): every result bit for bit that of the source with zero rows appended, whose own rows are unchanged."""
    from hpfp8 import ops
    u8 = torch.uint8
    mp = (m + 127) // 128 * 128
    x = torch.full((mp + 8, k), 77.0, dtype=torch.bfloat16, device=gpu)      # what lies behind the rows must not be read
    x[:m] = randn_bf16((m, k), m, 1.0, 0.01, 50.0).to(gpu)
    pad = torch.zeros((mp, k), dtype=torch.bfloat16, device=gpu)
    pad[:m] = x[:m]
    q, s, qt, st, cs = ops.quantize_1x128_and_128x1_t_rows(x[:m], pow2=pow2, column_sum=True)
    w = ops.quantize_1x128_and_128x1_t(pad, pow2=pow2, column_sum=True)
    assert torch.equal(q.view(u8), w[0][:m].view(u8)) and torch.equal(s, w[1][:m])
    assert torch.equal(qt.view(u8), w[2].view(u8)) and torch.equal(st, w[3]) and torch.equal(cs, ops.column_sum(x[:m]))
    for a, b in zip(ops.quantize_1x128_and_128x1_t_rows(x[:m], pow2=pow2), (q, s, qt, st)):
        assert torch.equal(a.float(), b.float())
    qt2, st2 = ops.quantize_128x1_t_rows(x[:m], pow2=pow2)
    assert torch.equal(qt2.view(u8), qt.view(u8)) and torch.equal(st2, st)
    if pow2:
        return
    inter = k
    h = torch.full((mp + 8, 2 * inter), 77.0, dtype=torch.bfloat16, device=gpu)
    h[:m] = randn_bf16((m, 2 * inter), m + 1).to(gpu)
    dact = randn_bf16((m, inter), m + 2).to(gpu)
    hp, dp = torch.zeros((mp, 2 * inter), dtype=torch.bfloat16, device=gpu), torch.zeros((mp, inter), dtype=torch.bfloat16, device=gpu)
    hp[:m], dp[:m] = h[:m], dact
    for got, want in [(ops.swiglu_quantize_1x128_and_128x1_t_rows(h[:m], fast=f), ops.swiglu_quantize_1x128_and_128x1_t(hp, fast=f))
                      for f in (False, True)] + [(ops.swiglu_backward_quantize_1x128_and_128x1_t_rows(h[:m], dact),
                                                  ops.swiglu_backward_quantize_1x128_and_128x1_t(hp, dp))]:
        assert torch.equal(got[0].view(u8), want[0][:m].view(u8)) and torch.equal(got[1], want[1][:m])
        assert torch.equal(got[2].view(u8), want[2].view(u8)) and torch.equal(got[3], want[3])


@pytest.mark.parametrize("rows", [1, 100, 129])
def test_mlp_block_of_ragged_tokens_is_that_of_its_two_linears(gpu, rows):
    """The one-node training path of the MLP block at a ragged token count gives the bits of the linear and SwiGLU nodes
    it replaces (which a frozen weight still selects)."""
    import hpfp8
    x0, gu0, dn0, go = (randn_bf16(s, i, sd).to(gpu) for i, (s, sd) in enumerate((((rows, 256), 1.0), ((512, 256), 0.05),
                                                                               ((384, 256), 0.05), ((rows, 384), 0.1))))
    x, gu, dn = (t.clone().requires_grad_(True) for t in (x0, gu0, dn0))
    y = hpfp8.fp8_swiglu_mlp(x, gu, dn)
    dx, dgu, ddn = torch.autograd.grad(y, (x, gu, dn), go)
    x2, gu2 = (t.clone().requires_grad_(True) for t in (x0, gu0))
    y2 = hpfp8.fp8_swiglu_mlp(x2, gu2, dn0)                      # frozen down projection
    dx2, dgu2 = torch.autograd.grad(y2, (x2, gu2), go)
    x3, dn3 = (t.clone().requires_grad_(True) for t in (x0, dn0))
    y3 = hpfp8.fp8_swiglu_mlp(x3, gu0, dn3)                      # frozen gate/up projection
    dx3, ddn3 = torch.autograd.grad(y3, (x3, dn3), go)
    for a, b in ((y, y2), (y, y3), (dx, dx2), (dx, dx3), (dgu, dgu2), (ddn, ddn3)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("m", [0, 1, 5, 128, 200])
@pytest.mark.parametrize("x_grad,w_grad", [(True, True), (True, False), (False, True), (False, False)])
def test_per_tensor_linear_without_output_features_has_an_empty_result(gpu, m, x_grad, w_grad):
    """A weight of no rows: nothing to quantize in any form, whatever gradients are to come."""
    import hpfp8
    x, w = randn_bf16((m, 256), 1).to(gpu).requires_grad_(x_grad), torch.empty((0, 256), dtype=torch.bfloat16, device=gpu, requires_grad=w_grad)
    for bias in (None, torch.empty((0,), dtype=torch.bfloat16, device=gpu)):
        assert tuple(hpfp8.fp8_linear(x, w, bias, recipe="per_tensor").shape) == (m, 0)


def _between_vectors(t):
    """The same values in memory that starts two bytes past a 16-byte boundary."""
    buf = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)
    v = buf[1:1 + t.numel()].view(t.shape)
    return v.copy_(t)


@pytest.mark.parametrize("recipe", ["blockwise", "blockwise_pow2", "per_tensor"])
@pytest.mark.parametrize("m", [5, 128, 200])
def test_what_starts_between_two_vectors_is_refused_at_every_number_of_rows(gpu, recipe, m):
    """Input, weight and grad_out of a training step: refused or taken alike for whole and for ragged token counts, but for a
    ragged grad_out of which only the weight gradient is made."""
    import hpfp8
    from hpfp8 import _lib
    x, w, go = (randn_bf16(s, i, sd).to(gpu) for i, (s, sd) in enumerate((((m, 256), 1.0), ((384, 256), 0.05), ((m, 384), 0.1))))
    for x_grad, w_grad in ((True, True), (False, True)):
        with pytest.raises(_lib.Hpfp8Error, match="16-byte aligned"):
            hpfp8.fp8_linear(_between_vectors(x).requires_grad_(x_grad), w.clone().requires_grad_(w_grad), recipe=recipe)
        with pytest.raises(_lib.Hpfp8Error, match="16-byte aligned"):
            hpfp8.fp8_linear(x.clone().requires_grad_(x_grad), _between_vectors(w).requires_grad_(w_grad), recipe=recipe)
        ins = [t for t, g in ((x.clone(), x_grad), (w.clone(), w_grad)) if t.requires_grad_(g).requires_grad]
        y = hpfp8.fp8_linear(ins[0] if x_grad else x, ins[-1], recipe=recipe)
        if x_grad or m == 128:
            with pytest.raises(_lib.Hpfp8Error, match="16-byte aligned"):
                torch.autograd.grad(y, ins, _between_vectors(go))
        else:
            want = torch.autograd.grad(y, ins, go, retain_graph=True)
            assert torch.equal(torch.autograd.grad(y, ins, _between_vectors(go))[0], want[0])
    if recipe == "blockwise":
        dn = randn_bf16((256, 128), 4, 0.05).to(gpu)
        w2, d2 = w[:256].clone().requires_grad_(True), dn.clone().requires_grad_(True)
        with pytest.raises(_lib.Hpfp8Error, match="16-byte aligned"):
            hpfp8.fp8_swiglu_mlp(_between_vectors(x), w2, d2)


@pytest.mark.parametrize("m,k", [(1, 128), (127, 128), (129, 384), (1024, 1024), (1000, 2048), (2048, 1024), (2049, 2048), (4096, 1024),
                                 (4097, 1024), (300, 16384)])
@pytest.mark.parametrize("one_launch,polls", [(True, None), (True, 0), (False, None)])
def test_per_tensor_codes_with_their_transpose(gpu, m, k, one_launch, polls, monkeypatch):
    """One, two and four tiles per workgroup with whole and partly empty last workgroups, the first sizes past 256 tiles,
    ragged rows, workgroups that stop waiting for the others and find the maximum alone (no polls), and the form without a
    block to agree through: the codes and scale of the plain quantizer, their transpose, the column sums; twice in a row,
    since the block must have been left as it was found."""
    from hpfp8 import _lib, ops
    x = torch.full((m + 8, k), 1e30, dtype=torch.bfloat16, device=gpu)       # what lies behind the rows must not be read
    x[:m] = randn_bf16((m, k), m, 1.0, 0.001, 50.0).to(gpu)
    x = x[:m]
    want, _, si = ops.quantize_per_tensor(x)
    mp = (m + 127) // 128 * 128
    if not one_launch:
        monkeypatch.setattr(ops, "_sync_words", lambda device: None)
    if polls is not None:
        _lib.load().hpfp8_debug_set_spin_limit(polls)
    try:
        for column_sum in (False, True):
            out = ops.quantize_per_tensor_t(x, column_sum=column_sum)
            assert torch.equal(out[0].view(torch.uint8), want.view(torch.uint8)) and torch.equal(out[1], si)
            t = out[2].view(torch.uint8)
            assert tuple(t.shape) == (k, mp) and torch.equal(t[:, :m].t(), want.view(torch.uint8)) and not t[:, m:].any()
            if column_sum:
                assert torch.equal(out[3], ops.column_sum(x))
    finally:
        _lib.load().hpfp8_debug_set_spin_limit(256)


@pytest.mark.parametrize("mode", [2, 3, 4, 5])
@pytest.mark.parametrize("m,n,blocks", [(70, 256, 1), (200, 384, 2), (130, 128, 3), (129, 640, 4), (64, 128, 6), (65, 256, 7), (65, 256, 9), (1300, 2560, 3),
                                        (2300, 4224, 1)])
def test_tiles_with_fetching_waves_give_the_bits_of_256_x_256_ones(gpu, mode, m, n, blocks):
    """Contractions of fewer k-blocks than the rings hold, as many and more; ragged rows and columns; several tiles per workgroup (the last
    two shapes: 840 and 2376 tiles of 64 x 64, 420 and 1188 of 64 x 128, 220 and 594 of 128 x 128, 110 and 306 of 128 x 256); scales of a in both layouts."""
    from hpfp8 import _lib, ops
    k = 128 * blocks
    x, w = _normal((m, k), 1, gpu, outliers=True), _normal((n, k), 2, gpu, 0.05)
    bias, c0 = _normal((n,), 3, gpu), _normal((m, n), 4, gpu).float()
    got = {}
    for hook in (1, mode):
        _lib.load().hpfp8_debug_set_small_gemm(hook)
        try:
            r = got[hook] = []
            for pow2 in (False, True):
                a, sa = ops.quantize_1x128(x, kmajor=True, pow2=pow2)
                for gran, (b, sb) in ((128, ops.quantize_128x128(w, pow2=pow2)), (1, ops.quantize_1x128(w, kmajor=True, pow2=pow2))):
                    for s in (sa, sa.contiguous()):
                        r.append(ops.gemm_blockwise(a, s, b, sb, bias=bias, sb_gran=gran, pow2_scales=pow2))
                        r.append(ops.gemm_blockwise(a, s, b, sb, sb_gran=gran, out=c0.clone(), accumulate=True, pow2_scales=pow2))
            a, _, sa = ops.quantize_per_tensor(x)
            b, _, sb = ops.quantize_per_tensor(w)
            r.append(ops.gemm_per_tensor(a, sa, b, sb, bias=bias))
            r.append(ops.gemm_per_tensor(a, sa, b, sb, out_dtype=torch.float32))
        finally:
            _lib.load().hpfp8_debug_set_small_gemm(0)
    for one, other in zip(got[1], got[mode]):
        assert torch.equal(one, other)


@pytest.mark.parametrize("counts", [[5], [0, 64, 0, 65, 1], [300] * 3, [0] * 63 + [200], [3] * 64, [0] * 64 + [129], [1, 0, 2] * 43, [40] * 70,
                                    [2500, 7, 0, 1]])
@pytest.mark.parametrize("n", [128, 640])
def test_grouped_rows_give_the_same_bits_with_every_tile(gpu, counts, n):
    """The tile that the kernel chooses and each one asked for, rows of an expert around the tiles' heights, experts around a
    wave's 64; rows past the last offset are left as they are."""
    from hpfp8 import _lib, ops
    k, e, m = 384, len(counts), sum(counts)
    a, sa = ops.quantize_1x128(_normal((m + 3, k), 1, gpu, outliers=True), kmajor=True)
    b, sb = ops.quantize_128x128(_normal((8 * n, k), 2, gpu, 0.05))
    pick = torch.arange(e, device=gpu) % 8
    b, sb = b.view(torch.uint8).view(8, n, k)[pick].view(b.dtype), sb.view(8, n // 128, k // 128)[pick].contiguous()
    offs = torch.tensor(counts).cumsum(0).to(torch.int32).to(gpu)
    got = {}
    for mode in (1, 0, 2, 3, 5):
        _lib.load().hpfp8_debug_set_small_gemm(mode)
        try:
            got[mode] = [ops.gemm_grouped_blockwise(a, s, b, sb, offs)[:m] for s in (sa, sa.contiguous())]
        finally:
            _lib.load().hpfp8_debug_set_small_gemm(0)
        assert torch.equal(got[mode][0], got[1][0]) and torch.equal(got[mode][1], got[1][0])
    for i, c in enumerate(counts[:6]):
        rows = slice(int(sum(counts[:i])), int(sum(counts[:i + 1])))
        assert torch.equal(got[0][0][rows], ops.gemm_blockwise(a[rows], sa[rows], b[i], sb[i]))


def _chosen_rows(counts, n, cus=256):
    """The height that grouped_tile_rows (csrc/gemm.hip) chooses for these rows of the experts."""
    tiles = {tm: sum(-(-c // tm) for c in counts) * -(-n // tn) for tm, tn in ((64, 128), (128, 256), (256, 256))}
    cost = {tm: w * -(-tiles[tm] // cus) for tm, w in ((64, 26), (128, 50), (256, 83))}
    return min(cost, key=lambda tm: (cost[tm], tm))


@pytest.mark.parametrize("rows,counts", [(64, [70] + [0] * 31), (128, [64] * 31 + [61]), (256, [7900] + [0] * 30 + [100])])
@pytest.mark.parametrize("pow2", [False, True])
def test_grouped_kernel_that_chooses_its_tile_has_the_bits_of_one_that_does_not(gpu, rows, counts, pow2):
    """Each of the three forms inside the kernel that chooses, reached through the default rule: both output types, scales of a in both
    layouts."""
    from hpfp8 import _lib, ops
    n, k, e, m = 4096, 256, len(counts), sum(counts)
    assert torch.cuda.get_device_properties(0).multi_processor_count != 256 or _chosen_rows(counts, n) == rows
    a, sa = ops.quantize_1x128(_normal((m, k), 1, gpu, outliers=True), kmajor=True, pow2=pow2)
    b, sb = ops.quantize_128x128(_normal((e * n, k), 2, gpu, 0.05), pow2=pow2)
    b, sb = b.view(e, n, k), sb.view(e, n // 128, k // 128)
    offs = torch.tensor(counts).cumsum(0).to(torch.int32).to(gpu)
    got = {}
    for mode in (1, 0):
        _lib.load().hpfp8_debug_set_small_gemm(mode)
        try:
            got[mode] = [ops.gemm_grouped_blockwise(a, s, b, sb, offs, out_dtype=dtype, pow2_scales=pow2)
                         for s in (sa, sa.contiguous()) for dtype in (torch.bfloat16, torch.float32)]
        finally:
            _lib.load().hpfp8_debug_set_small_gemm(0)
    for one, other in zip(got[0], got[1]):
        assert torch.equal(one, other)


@pytest.mark.parametrize("mode,m,n", [(1, 2304, 8704), (2, 640, 2048), (3, 1152, 8704), (4, 1152, 4352), (5, 640, 4352)])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_scales_that_are_not_finite_stay_with_their_tile(gpu, mode, m, n, value):
    """Several tiles per compute unit with every tile shape: a NaN or an infinity among the scales of a tile's last k-block makes its own
    rows (columns) NaN or infinite, and none of the tile that the same waves compute next."""
    from hpfp8 import _lib, ops
    k = 256
    x, w = _normal((m, k), 1, gpu), _normal((n, k), 2, gpu)
    a, sa = ops.quantize_1x128(x, kmajor=True)
    bad = torch.tensor([3, 21, 40, 63], device=gpu)
    sa[bad, -1] = value
    _lib.load().hpfp8_debug_set_small_gemm(mode)
    try:
        for b, sb, gran in ((*ops.quantize_128x128(w), 128), (*ops.quantize_1x128(w, kmajor=True), 1)):
            c = ops.gemm_blockwise(a, sa, b, sb, sb_gran=gran)
            assert torch.equal((~c.isfinite()).any(1).nonzero().flatten(), bad)
            assert not bool(c[bad].isfinite().any())
    finally:
        _lib.load().hpfp8_debug_set_small_gemm(0)


@pytest.mark.parametrize("mode,m,n", [(1, 300, 640), (2, 65, 256), (3, 129, 384), (4, 130, 384), (5, 65, 640), (1, 2305, 8704), (2, 1100, 1152)])
@pytest.mark.parametrize("k", [128, 384])
def test_per_row_scales_on_both_operands_are_those_of_their_rows_and_blocks(gpu, mode, m, n, k):
    """Scales with full mantissas, another in every row and k-block, on integer codes: the sum of a k-block is an exact integer below 2^12, so
    with one k-block c is that integer times the fp32 product of the two scales, rounded once; with more of them each adds at most
    its own rounding, 2^-24 of the sum so far."""
    from hpfp8 import _lib, ops
    a, b, kb = _ints((m, k), 1, gpu), _ints((n, k), 2, gpu), k // 128
    g = torch.Generator(device="cpu").manual_seed(3)
    sa, sb = ((torch.rand((kb, r), generator=g) + 0.5).to(gpu).t() for r in (m, n))
    part = torch.stack([a.double()[:, i * 128:(i + 1) * 128] @ b.double()[:, i * 128:(i + 1) * 128].t() for i in range(kb)])
    scale = torch.stack([sa[:, i:i + 1] * sb[:, i] for i in range(kb)])
    _lib.load().hpfp8_debug_set_small_gemm(mode)
    try:
        for s in (sa, sa.contiguous()):
            c = ops.gemm_blockwise(a, s, b, sb, sb_gran=1, out_dtype=torch.float32)
            if kb == 1:
                assert torch.equal(c, part[0].float() * scale[0])
            terms = part * scale.double()
            assert bool(((c.double() - terms.sum(0)).abs() <= kb * 2.0 ** -23 * terms.abs().sum(0)).all())
    finally:
        _lib.load().hpfp8_debug_set_small_gemm(0)


@pytest.mark.parametrize("m,n,k", [(1, 128, 128), (100, 128, 384), (256, 128, 256), (129, 256, 256), (65, 1024, 128), (300, 1024, 640), (1531, 2048, 1152), (2048, 1152, 2176)])
@pytest.mark.parametrize("recipe", [0, 1, 2])
def test_both_products_of_a_backward_in_one_launch_have_the_bits_of_two(gpu, m, n, k, recipe):
    """Every tile shape for both products (the sizes end inside tiles of each), the rule's own choice, and the launches one by one; fewer
    tiles than XCDs, and more than one per compute unit."""
    import ctypes
    from hpfp8 import _lib, ops

    class Operand(ctypes.Structure):
        _fields_ = [("codes", ctypes.c_void_p), ("ld", ctypes.c_int64), ("scale_inv", ctypes.c_void_p), ("stride_r", ctypes.c_int64),
                    ("stride_k", ctypes.c_int64)]

        def __init__(self, codes, s):
            strides = s.stride() if s.dim() == 2 else (0, 0)
            super().__init__(codes.data_ptr(), codes.stride(0), s.data_ptr(), *strides)

    go, x, w = _normal((m, n), 1, gpu, outliers=True), _normal((m, k), 2, gpu, outliers=True), _normal((n, k), 3, gpu, 0.02)
    blocks = (m + 127) // 128
    part = torch.randn((blocks, n), generator=torch.Generator("cpu").manual_seed(4)).to(gpu)
    db = torch.empty(n, dtype=torch.bfloat16, device=gpu)
    _lib.call("hpfp8_column_sum_finish", part.data_ptr(), blocks, n, db.data_ptr(), None, ops._stream())
    if recipe == 2:
        (g, sg, gt), (_, sx, xt), (_, sw, wt) = (ops.quantize_per_tensor_t(t)[:3] for t in (go, x, w))
        sgt = sg
        want = [ops.gemm_per_tensor(g, sg, wt, sw), ops.gemm_per_tensor(gt, sg, xt, sx), db]
    else:
        g, sg, gt, sgt = ops.quantize_1x128_and_128x1_t_rows(go, pow2=recipe == 1)
        _, _, xt, sx = ops.quantize_1x128_and_128x1_t_rows(x, pow2=recipe == 1)
        _, sw, wt = ops.quantize_128x128(w, with_transpose=True, pow2=recipe == 1)
        sw = sw.t()
        want = [ops.gemm_blockwise(g, sg, wt, sw, pow2_scales=recipe == 1), ops.gemm_blockwise(gt, sgt, xt, sx, sb_gran=1, pow2_scales=recipe == 1), db]
    operands = [Operand(g, sg), Operand(wt, sw), Operand(gt, sgt), Operand(xt, sx)]
    if recipe != 2:
        old = torch.randn((n, k), generator=torch.Generator("cpu").manual_seed(5)).to(gpu)
        summed = ops.gemm_blockwise(gt, sgt, xt, sx, sb_gran=1, pow2_scales=recipe == 1, out=old.clone(), accumulate=True)
    for mode in (0, 1, 2, 3, 4, 5):
        got = [torch.full(s, 7.0, dtype=torch.bfloat16, device=gpu) for s in ((m + 1, k), (n + 1, k), (n + 8,))]
        _lib.load().hpfp8_debug_set_small_gemm(mode)
        try:
            _lib.call("hpfp8_linear_backward", *(ctypes.addressof(o) for o in operands), m, n, k, got[0].data_ptr(), got[1].data_ptr(), 0,
                      part.data_ptr(), got[2].data_ptr(), recipe, ops._stream())
            if recipe != 2 and mode < 2:        # (scales that are not k-block-major: the launches one by one)
                sg_rows, sgt_rows = sg.contiguous(), sgt.contiguous()
                rows = [Operand(g, sg_rows), operands[1], Operand(gt, sgt_rows), operands[3]]
                apart = [torch.full_like(t, 7.0) for t in got]
                _lib.call("hpfp8_linear_backward", *(ctypes.addressof(o) for o in rows), m, n, k, apart[0].data_ptr(), apart[1].data_ptr(), 0,
                          part.data_ptr(), apart[2].data_ptr(), recipe, ops._stream())
                assert all(torch.equal(a[:len(b)], b) for a, b in zip(apart, want))
            if recipe != 2:
                onto = [torch.full_like(got[0], 7.0), old.clone()]
                _lib.call("hpfp8_linear_backward", *(ctypes.addressof(o) for o in operands), m, n, k, onto[0].data_ptr(), onto[1].data_ptr(), 1,
                          None, None, recipe, ops._stream())
                assert torch.equal(onto[0][:m], want[0]) and torch.equal(onto[1], summed)
        finally:
            _lib.load().hpfp8_debug_set_small_gemm(0)
        for a, b, rows in zip(got, want, (m, n, n)):
            assert torch.equal(a[:rows], b)
            assert bool((a[rows:] == 7.0).all())


@pytest.mark.parametrize("m,n,k", [(1, 128, 128), (300, 128, 384), (2048, 1024, 1024), (128, 4096, 1024), (1025, 256, 2048), (8192, 512, 512)])
@pytest.mark.parametrize("spins", [256, 0])
def test_two_tensors_quantized_in_one_launch_have_the_bits_of_two(gpu, m, n, k, spins):
    """One, two and four tiles per workgroup, the fewest and the most workgroups per tensor, and workgroups that never see the others'
    maximum and find it by themselves; three times over the same words, which have to be zero again in between."""
    from hpfp8 import _lib, ops
    x, w = _normal((m, k), 1, gpu, outliers=True), _normal((n, k), 2, gpu, 0.02)
    (q, s, qt), (wq, sw, wqt) = ops.quantize_per_tensor_t(x), ops.quantize_per_tensor_t(w)
    sync = torch.zeros(256, dtype=torch.int32, device=gpu)
    _lib.load().hpfp8_debug_set_spin_limit(spins)
    try:
        for _ in range(3):
            got = [torch.zeros_like(q), torch.empty(k, qt.stride(0), dtype=torch.float8_e4m3fn, device=gpu).zero_(), torch.zeros_like(s),
                   torch.zeros_like(wq), torch.empty(k, wqt.stride(0), dtype=torch.float8_e4m3fn, device=gpu).zero_(), torch.zeros_like(sw)]
            _lib.call("hpfp8_quantize_two_per_tensor_t_bf16", x.data_ptr(), m, k, got[0].data_ptr(), got[1].data_ptr(), qt.stride(0), got[2].data_ptr(),
                      w.data_ptr(), n, got[3].data_ptr(), got[4].data_ptr(), wqt.stride(0), got[5].data_ptr(), sync.data_ptr(), ops._stream())
            for a, b in zip(got, (q, qt, s, wq, wqt, sw)):
                a = a[:, :b.shape[1]] if b.dim() == 2 else a
                assert torch.equal(a.contiguous().view(torch.uint8) if b.dim() == 2 else a, b.contiguous().view(torch.uint8) if b.dim() == 2 else b)
            assert int(sync.count_nonzero()) == 0
    finally:
        _lib.load().hpfp8_debug_set_spin_limit(256)


def _fastest(run):
    """The shortest of seven times of twenty launches, ms."""
    times = []
    for _ in range(7):
        start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        for i in range(4):
            run(i)
        start.record()
        for i in range(20):
            run(i)
        end.record()
        end.synchronize()
        times.append(start.elapsed_time(end))
    return min(times)


@pytest.mark.parametrize("grouped", [False, True])
def test_a_weight_that_stays_in_the_caches_is_read_from_them(gpu, grouped):
    """Streamed past them, one weight used again and again would take as long as several in turn that do not fit together (measured: 97 %
    of it dense, 100 % grouped; kept 68 % and 70 %)."""
    from hpfp8 import ops
    m, k = (512, 7168) if grouped else (128, 7168)
    n = 8 * 4096 if grouped else 18432
    a, sa = ops.quantize_1x128(_normal((m, k), 1, gpu), kmajor=True)
    weights = [ops.quantize_128x128(_normal((n, k), seed, gpu, 0.02)) for seed in range(4)]
    sizes = [188, 94, 63, 47, 37, 31, 27, 25]
    offs = torch.tensor(sizes, device=gpu).cumsum(0).int()

    def product(b, sb):
        if grouped:
            return ops.gemm_grouped_blockwise(a, sa, b.view(8, 4096, k), sb.view(8, 32, k // 128), offs)
        return ops.gemm_blockwise(a, sa, b, sb)

    one, several = (_fastest(lambda i: product(*of[i % len(of)])) for of in (weights[:1], weights))
    assert one < 0.85 * several


def test_grouped_products_whose_weight_is_streamed_past_the_caches_have_the_bits_of_those_that_keep_it(gpu):
    """Experts with rows on both sides of the size from which on rows of b that one low tile reads alone are streamed, among 12 and among
    70 (two chunks of 64 lanes), with none, one tile's and several tiles' rows; 256 x 256 tiles stream nothing."""
    from hpfp8 import ops
    for experts, n, k, counts in ((12, 4096, 7168, [1, 0, 64, 65, 128, 129, 7, 300, 16, 2, 1, 1]), (12, 4096, 7168, [10] * 12), (12, 4096, 7168, [10] * 10 + [0] * 2),
                                  (70, 2048, 2560, [3] * 30 + [0] * 10 + [70] + [1] * 29)):
        b, sb = ops.quantize_128x128(_normal((experts * n, k), 2, gpu, 0.02))
        a, sa = ops.quantize_1x128(_normal((sum(counts), k), 1, gpu), kmajor=True)
        offs = torch.tensor(counts, device=gpu).cumsum(0).int()
        got, want = _both_tiles(lambda: ops.gemm_grouped_blockwise(a, sa, b.view(experts, n, k), sb.view(experts, n // 128, k // 128), offs))
        assert torch.equal(got, want)


@pytest.mark.parametrize("tiles", [0, 1, 3, 4, 5])
@pytest.mark.parametrize("gran", [1, 128])
def test_the_product_of_two_scales_is_formed_first_and_rounded_to_fp32(gpu, gran, tiles):
    """part * (sa * sb), the oracle's order, at both ends of the range: a product below the smallest normal number keeps the bits that a
    subnormal one has, and one that overflows is infinite for every element it scales (times a zero sum: NaN), and for no other."""
    from hpfp8 import _lib, ops
    m, n, k = 256, 256, 384
    a, b = _ints((m, k), 1, gpu), _ints((n, k), 2, gpu)
    a.view(torch.uint8)[5, 128:256] = 0
    sa, sb = torch.ones((k // 128, m), device=gpu), torch.ones((k // 128, n // gran), device=gpu)
    sa[0], sb[0] = 1.25 * 2.0 ** -70, 1.625 * 2.0 ** -76        # 16.25 * 2^-149: rounded to the subnormal number 16 * 2^-149
    sa[2], sb[2] = 2.0 ** -100, 2.0 ** -40                      # (with it every sum is a whole number of 2^-149 below 2^24 of them)
    sa[1] = 0.0
    sa[1, 3:8], sb[1, 1] = 2.0 ** 100, 2.0 ** 100
    part = [a.float()[:, i * 128:(i + 1) * 128].cpu() @ b.float()[:, i * 128:(i + 1) * 128].cpu().t() for i in range(k // 128)]
    want = torch.zeros((m, n))
    for i, p in enumerate(part):
        want = torch.addcmul(want.double(), p.double(), torch.outer(sa[i].cpu(), sb[i].cpu().repeat_interleave(gran)).double()).float()
    _lib.load().hpfp8_debug_set_small_gemm(tiles)
    try:
        got = ops.gemm_blockwise(a, sa.t(), b, sb.t() if gran == 1 else sb.t().contiguous(), sb_gran=gran, out_dtype=torch.float32).cpu()
    finally:
        _lib.load().hpfp8_debug_set_small_gemm(0)
    assert bool(want[5].isnan().any()) and bool(want[3].isinf().any()) and bool(want[8].isfinite().all())
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(0.0, 1.0, -1.0), want.nan_to_num(0.0, 1.0, -1.0))


def test_few_rows_of_a_wide_weight_with_a_short_contraction_take_no_longer_than_tiles(gpu):
    """64 rows of [131072, 1024], one weight for every call: 25.6 us with tiles, 38.2 in the few-rows form."""
    from hpfp8 import _lib, ops
    a, sa = ops.quantize_1x128(_normal((64, 1024), 1, gpu), kmajor=True)
    b, sb = ops.quantize_128x128(_normal((131072, 1024), 2, gpu, 0.02))
    fastest = {}
    for tiles in (1, 3, 0):
        _lib.load().hpfp8_debug_set_small_gemm(tiles)
        try:
            fastest[tiles] = _fastest(lambda i: ops.gemm_blockwise(a, sa, b, sb))
        finally:
            _lib.load().hpfp8_debug_set_small_gemm(0)
    assert fastest[0] < 1.2 * min(fastest[1], fastest[3])
