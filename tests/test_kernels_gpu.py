"""Kernel-level parity on the GPU, through the C ABI (via the ctypes wrappers).

Comparators are the eager ATen ops of the oracle on the same device and
dtype (the rounding chain each kernel mirrors) and an fp32 evaluation of the
same inputs.  Bars, per test:

* GEMM (bias, GELU, residual, masks, packed QKV): bitwise equal to the eager
  chain (F.linear / F.gelu / x + y on hipBLASLt and ATen) at every shape
  whose library kernel accumulates K in order or in the local split-K order
  that gemm_lsu_kernel reproduces (M <= 256, K >= 2048); only M = 100000,
  where the library runs a Stream-K kernel, is compared to 1 ulp;
* attention, eager softmax: bitwise equal to the eager chain at every tested
  length, S = 8192 included;
* attention, online softmax: no worse than twice eager's own deviation from
  fp32 attention;
* LayerNorm: mean, rstd and output bitwise equal to torch.native_layer_norm.
"""

import math

import pytest
import torch
import torch.nn.functional as F

from transformer_optimization_amd import _C
from _util import log, ulp, ulp_diff_stats

pytestmark = pytest.mark.gpu

DTYPES = [torch.bfloat16, torch.float16]


def _gen(seed):
    return torch.Generator("cpu").manual_seed(seed)


def _randn(shape, dtype, dev, seed, scale=1.0):
    return (torch.randn(shape, generator=_gen(seed)) * scale).to(dev, dtype)


# ------------------------------------------------------------------ LayerNorm
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,d", [(256, 256), (64, 512), (8192, 1024), (8192, 2048), (100000, 1024), (7, 1032),
                                    (9, 2056), (64, 4096), (16, 8192)])
def test_layernorm_matches_eager(cuda, dtype, rows, d):
    log(f"layernorm {rows}x{d} {dtype}")
    x = _randn((rows, d), dtype, cuda, 1, 2.0) + 0.5
    g = _randn((d,), dtype, cuda, 2, 0.2) + 1.0
    b = _randn((d,), dtype, cuda, 3, 0.2)
    mean = torch.empty(rows, device=cuda)
    rstd = torch.empty(rows, device=cuda)
    y = _C.layernorm_residual(x, g, b, mean_out=mean, rstd_out=rstd)
    ref, ref_mean, ref_rstd = torch.native_layer_norm(x, [d], g, b, 1e-5)
    mx, frac = ulp_diff_stats(y, ref, dtype)
    bad_mean = int((mean != ref_mean.view(-1)).sum())
    bad_rstd = int((rstd != ref_rstd.view(-1)).sum())
    log(f"  max_ulp={mx:.2f} frac_diff={frac:.2e} mean_rows_diff={bad_mean} rstd_rows_diff={bad_rstd}")
    # ATen's reduction order and rounding points: bit-identical moments and output.
    assert bad_mean == 0 and bad_rstd == 0
    assert torch.equal(y, ref)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows", [1000, 5003])  # one row / four rows per workgroup (ragged tail)
def test_layernorm_residual_flags(cuda, dtype, rows):
    d = 1024
    x = _randn((rows, d), dtype, cuda, 4)
    delta = _randn((rows, d), dtype, cuda, 5, 0.3)
    g = _randn((d,), dtype, cuda, 6, 0.2) + 1.0
    b = _randn((d,), dtype, cuda, 7, 0.2)
    valid = torch.rand(rows, generator=_gen(8)) > 0.3
    valid = valid.to(cuda)
    x_out = torch.empty_like(x)
    flags = _C.LN_MASK_DELTA | _C.LN_MASK_X | _C.LN_MASK_OUT
    y = _C.layernorm_residual(x, g, b, delta=delta, x_out=x_out, row_valid=valid, flags=flags)
    # eager chain: x' = mask_x(x + mask_d(delta)); y = mask_o(LN(x'))
    dm = delta.masked_fill(~valid[:, None], 0)
    xr = (x + dm).masked_fill(~valid[:, None], 0)
    assert torch.equal(x_out, xr)
    ref = F.layer_norm(xr, (d,), g, b, 1e-5).masked_fill(~valid[:, None], 0)
    assert torch.equal(y, ref)
    assert torch.count_nonzero(y[~valid]) == 0


# ----------------------------------------------------------------------- GEMM
GEMM_SHAPES = [
    (64, 64, 64),
    (100, 192, 136),       # ragged M, N; K not a multiple of 64
    (64, 512, 48),         # K % 32 == 16: the 32x32 skinny kernel
    (200, 192, 80),        # same, ragged M
    (64, 1536, 512),       # c2 QKV
    (64, 512, 2048),       # c2 FFN out (library: local split-K over 4 waves)
    (200, 512, 2048),      # ragged M on the local split-K path
    (256, 768, 256),       # c1 QKV
    (8192, 3072, 1024),    # c3 QKV
    (8192, 1024, 1024),    # c3 out_proj
    (8192, 4096, 1024),    # c3 FFN in
    (8192, 1024, 4096),    # c3 FFN out
    (8192, 6144, 2048),    # c4 QKV
    (8192, 2048, 2048),    # c4 q/k/v/out_proj
    (8192, 8192, 2048),    # c4 FFN in
    (8192, 2048, 8192),    # c4 FFN out
    (100000, 1024, 1024),  # c5 out_proj
]


# hipBLASLt picks Stream-K kernels at M = 100000; their partial sums are
# added in a different order.  (Its local split-K kernel at small M and
# K = 2048 is reproduced bit for bit by gemm_lsu_kernel.)
NON_INORDER_LIBRARY_SHAPES = {(100000, 1024)}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", GEMM_SHAPES)
def test_gemm_bias_matches_eager_linear(cuda, dtype, m, n, k):
    log(f"gemm {m}x{n}x{k} {dtype}")
    a = _randn((m, k), dtype, cuda, 11)
    w = _randn((n, k), dtype, cuda, 12, 0.02)
    bias = _randn((n,), dtype, cuda, 13, 0.1)
    c = _C.gemm(a, w, bias)
    ref = F.linear(a, w, bias)
    mx, frac = ulp_diff_stats(c, ref, dtype)
    # Against an fp32 evaluation: one rounding of the output plus fp32
    # accumulation error, which matters only where |c| << the summands.
    ref32 = a.float() @ w.float().t() + bias.float()
    scale = (a.float().abs() @ w.float().abs().t()).amax(1, keepdim=True)
    err32 = (c.float() - ref32).abs() - 0.5 * ulp(ref32, dtype)
    log(f"  vs eager max_ulp={mx:.2f} frac={frac:.2e}; vs fp32 excess {float((err32 / scale).max()):.2e}")
    assert float((err32 / scale).max()) <= k * 2.0 ** -24
    if (m, k) in NON_INORDER_LIBRARY_SHAPES:
        assert frac < 1e-2
    else:
        assert torch.equal(c, ref)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", [(300, 1024, 512), (8192, 4096, 1024)])
def test_gemm_gelu_epilogue(cuda, dtype, m, n, k):
    a = _randn((m, k), dtype, cuda, 21)
    w = _randn((n, k), dtype, cuda, 22, 0.05)
    bias = _randn((n,), dtype, cuda, 23, 0.1)
    c = _C.gemm(a, w, bias, gelu=True)
    ref = F.gelu(F.linear(a, w, bias), approximate="none")
    mx, frac = ulp_diff_stats(c, ref, dtype)
    log(f"gelu {m}x{n}x{k} max_ulp={mx:.2f} frac={frac:.2e}")
    # GELU reads the rounded GEMM value (TTB:1795-1798) through the device
    # erff, as ATen's gelu kernel does: bitwise equal.
    assert torch.equal(c, ref)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("variant", [-1, 256, 192, 128, 1283, 20, 0])
def test_gemm_gelu_every_16bit_input(cuda, dtype, variant, gemm_variant):
    """The GELU epilogue on every one of the 2^16 values of the dtype (NaN,
    infinities, subnormals and signed zeros included), through each GEMM
    kernel: A = [1, 0, ...] rows and W[n, 0] = the n-th bit pattern make the
    pre-activation exactly that value, and C must equal F.gelu(F.linear(...))
    bit for bit."""
    log(f"gelu every input {dtype} variant {variant}")
    m, n, k = 256, 1 << 16, 64
    a = torch.zeros((m, k), dtype=dtype, device=cuda)
    a[:, 0] = 1
    w = torch.zeros((n, k), dtype=dtype, device=cuda)
    w[:, 0] = torch.arange(n, dtype=torch.int32, device=cuda).to(torch.int16).view(dtype)
    bias = torch.zeros((n,), dtype=dtype, device=cuda)
    gemm_variant(variant)
    out = _C.gemm(a, w, bias, gelu=True)
    ref = F.gelu(F.linear(a, w, bias))
    same = (out.view(torch.int16) == ref.view(torch.int16)) | (torch.isnan(out) & torch.isnan(ref))
    n_diff = int((~same).sum())
    log(f"  differing outputs {n_diff} of {out.numel()}")
    assert n_diff == 0


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("m,n,k", [(1000, 1024, 4096), (64, 512, 2048), (200, 192, 80)])
def test_gemm_residual_epilogue_inplace(cuda, dtype, masked, m, n, k):
    log(f"residual {m}x{n}x{k} masked={masked} {dtype}")
    a = _randn((m, k), dtype, cuda, 31)
    w = _randn((n, k), dtype, cuda, 32, 0.02)
    bias = _randn((n,), dtype, cuda, 33, 0.1)
    x = _randn((m, n), dtype, cuda, 34)
    valid = (torch.rand(m, generator=_gen(35)) > 0.25).to(cuda) if masked else None
    delta = F.linear(a, w, bias)
    # mask_delta: invalid rows keep x; eager x + masked_fill(delta, 0)
    want_d = x + (delta.masked_fill(~valid[:, None], 0) if masked else delta)
    xs = x.clone()
    _C.gemm(a, w, bias, residual=xs, out=xs, row_valid=valid, mask_delta=masked)
    mx, frac = ulp_diff_stats(xs, want_d, dtype)
    log(f"  max_ulp={mx:.2f} frac={frac:.2e}")
    # round(x + round(acc + b)), the eager residual chain: bitwise equal.
    assert torch.equal(xs, want_d)
    if masked:
        assert torch.equal(xs[~valid], x[~valid])
        # mask_out: invalid rows become 0 (end of block, TTB:219-220)
        xo = x.clone()
        _C.gemm(a, w, bias, residual=xo, out=xo, row_valid=valid, mask_out=True)
        assert torch.count_nonzero(xo[~valid]) == 0
        assert torch.equal(xo[valid], (x + delta)[valid])


# ------------------------------------------------------------ packed QKV
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("b,s,d,h", [(1, 64, 512, 8), (2, 100, 256, 4), (8, 1024, 1024, 16), (1, 8192, 2048, 16)])
def test_qkv_proj_layouts(cuda, dtype, b, s, d, h):
    log(f"qkv b{b} s{s} d{d} h{h} {dtype}")
    hd = d // h
    x = _randn((b * s, d), dtype, cuda, 41)
    w = _randn((3 * d, d), dtype, cuda, 42, 0.02)
    bias = _randn((3 * d,), dtype, cuda, 43, 0.1)
    qk, vt = _C.qkv_proj(x, w, bias, b, s, h)
    ref = F.linear(x, w, bias)
    # The packed projection is F.linear of the packed weights, bit for bit,
    # stored as qk [M, 2D] and head-transposed V.
    assert torch.equal(qk, ref[:, : 2 * d])
    v_ref = ref[:, 2 * d:].reshape(b, s, h, hd).permute(0, 2, 3, 1)  # [B,H,hd,S]
    assert torch.equal(vt[..., :s], v_ref)
    # Closed form of the packing (TTB:440-504): the three projections.
    for j in range(3):
        assert torch.equal(ref[:, j * d:(j + 1) * d], F.linear(x, w[j * d:(j + 1) * d], bias[j * d:(j + 1) * d]))


# The 256-row kernel's three tile widths against the in-order register-staged
# kernel (tx_select_kernel; 0 = gemm_kernel): ragged
# M and N, N % 8 == 4 (the direct epilogue), K = 64 (one k step per tile), the
# in-place residual with row masks, GELU, and packed QKV whose sequence length
# is not a multiple of 16 (V^T written without staging).
# The last shape gives every CU four 128-wide tiles (tile transitions of the
# persistent kernel with two and three K stages).
HP_EDGE_SHAPES = [(520, 196, 192), (777, 584, 128), (300, 256, 64), (1000, 1032, 256), (4096, 8192, 192)]


@pytest.fixture
def gemm_variant():
    yield lambda v: _C.select_kernel(_C.SELECT_GEMM, v)
    _C.select_kernel(_C.SELECT_GEMM, -1)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", HP_EDGE_SHAPES)
def test_gemm_hp_widths_match_inorder_kernel(cuda, dtype, m, n, k, gemm_variant):
    log(f"gemm hp widths {m}x{n}x{k} {dtype}")
    a = _randn((m, k), dtype, cuda, 71)
    w = _randn((n, k), dtype, cuda, 72, 0.02)
    bias = _randn((n,), dtype, cuda, 73, 0.1)
    x = _randn((m, n), dtype, cuda, 74)
    rows = (torch.arange(m, device=cuda) % 7 != 3).to(torch.uint8)

    def run_all():
        outs = [_C.gemm(a, w, bias), _C.gemm(a, w, bias, gelu=True)]
        c = x.clone()
        _C.gemm(a, w, bias, residual=c, out=c)
        outs.append(c)
        c = x.clone()
        _C.gemm(a, w, bias, residual=c, out=c, row_valid=rows, mask_delta=True)
        outs.append(c)
        return outs

    gemm_variant(0)
    ref = run_all()
    for v in (256, 192, 128, 1283, -1):
        gemm_variant(v)
        got = run_all()
        for r, g in zip(ref, got):
            assert torch.equal(g, r), f"variant {v}"


@pytest.mark.parametrize("dtype", DTYPES)
def test_qkv_proj_unstaged_v_matches_inorder_kernel(cuda, dtype, gemm_variant):
    b, s, d, h = 3, 100, 256, 4
    hd = d // h
    log(f"qkv hp b{b} s{s} {dtype}")
    x = _randn((b * s, d), dtype, cuda, 81)
    w = _randn((3 * d, d), dtype, cuda, 82, 0.02)
    bias = _randn((3 * d,), dtype, cuda, 83, 0.1)
    gemm_variant(0)
    qk0, vt0 = _C.qkv_proj(x, w, bias, b, s, h)
    for v in (256, 192, 128, 1283, -1):
        gemm_variant(v)
        qk, vt = _C.qkv_proj(x, w, bias, b, s, h)
        assert torch.equal(qk, qk0), f"variant {v}"
        assert torch.equal(vt[..., :s], vt0[..., :s]), f"variant {v}"
    ref = F.linear(x.float(), w.float(), bias.float())
    assert float((qk.float() - ref[:, : 2 * d]).abs().max()) < 0.05


# gemm_ring_kernel's tile configurations (variants 1000 ..) against the
# in-order kernel, bit for bit: one to five K steps (fewer than the ring's
# stages, equal, more), one tile and a ragged last tile in M and N, N % 8 == 4
# (the direct epilogue), fp32 results and hi/lo pairs.
RING_SHAPES = [(1, 8, 64), (64, 64, 256), (65, 196, 128), (129, 200, 192), (300, 584, 320), (1000, 1032, 512)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", RING_SHAPES)
def test_gemm_ring_configurations_match_inorder_kernel(cuda, dtype, m, n, k, gemm_variant):
    log(f"gemm ring {m}x{n}x{k} {dtype}")
    a = _randn((m, k), dtype, cuda, 71)
    w = _randn((n, k), dtype, cuda, 72, 0.02)
    bias = _randn((n,), dtype, cuda, 73, 0.1)
    x = _randn((m, n), dtype, cuda, 74)
    x32 = _randn((m, n), torch.float32, cuda, 75)
    rows = (torch.arange(m, device=cuda) % 7 != 3).to(torch.uint8)

    def run_all():
        outs = [_C.gemm(a, w), _C.gemm(a, w, bias, gelu=True), _C.gemm(a, w, bias, gelu=True, split_out=True),
                _C.gemm(a, w, bias, residual=x32, out_dtype=torch.float32, row_valid=rows, mask_out=True)]
        for kw in ({"mask_delta": True}, {"mask_out": True}):
            c = x.clone()
            outs.append(_C.gemm(a, w, bias, residual=c, out=c, row_valid=rows, **kw))
        return outs

    gemm_variant(0)
    ref = run_all()
    for v in [*range(1000, 1006), -1]:
        gemm_variant(v)
        for i, (r, g) in enumerate(zip(ref, run_all())):
            assert torch.equal(g, r), f"variant {v} output {i}"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", [(17, 72, 2048), (64, 512, 2176), (200, 1024, 2048), (256, 4096, 2048)])
def test_gemm_ring_four_sum_order(cuda, dtype, m, n, k, gemm_variant):
    """M <= 256, K >= 2048: the ring tiles add K in the order of the 16x16
    kernel's four waves (variant 10), bit for bit."""
    log(f"gemm ring four sums {m}x{n}x{k} {dtype}")
    a = _randn((m, k), dtype, cuda, 76)
    w = _randn((n, k), dtype, cuda, 77, 0.02)
    bias = _randn((n,), dtype, cuda, 78, 0.1)
    x = _randn((m, n), torch.float32, cuda, 79)
    got = {}
    for v in (10, 1000, 1001, -1):
        gemm_variant(v)
        got[v] = (_C.gemm(a, w, bias, gelu=True), _C.gemm(a, w, bias, residual=x, out_dtype=torch.float32))
    for v in (1000, 1001, -1):
        assert all(torch.equal(p, q) for p, q in zip(got[10], got[v])), f"variant {v}"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("b,s,d,h", [(1, 64, 64, 1), (3, 100, 256, 4), (5, 129, 320, 5), (2, 421, 192, 3),
                                     (9, 40, 256, 2), (1, 1023, 128, 1)])
def test_qkv_proj_ring_configurations(cuda, dtype, b, s, d, h, gemm_variant):
    """Packed Q/K/V through every ring tile: tiles that hold k and V columns,
    V^T runs that start and end inside an eight-position chunk, two sequences
    in a tile, and sequences shorter than a tile (written unstaged).  The
    columns of V^T past the sequence stay as they were."""
    log(f"qkv ring b{b} s{s} d{d} {dtype}")
    x = _randn((b * s, d), dtype, cuda, 81)
    w = _randn((3 * d, d), dtype, cuda, 82, 0.02)
    bias = _randn((3 * d,), dtype, cuda, 83, 0.1)

    def run():
        vt = torch.full((b, h, d // h, _C.vt_ld(s)), 7.0, dtype=dtype, device=cuda)
        return _C.qkv_proj(x, w, bias, b, s, h, vt=vt)

    gemm_variant(0)
    qk0, vt0 = run()
    for v in [*range(1000, 1006), -1]:
        gemm_variant(v)
        qk, vt = run()
        assert torch.equal(qk, qk0) and torch.equal(vt, vt0), f"variant {v}"


def test_gemm_kernel_choice_is_per_thread_and_not_the_environment(cuda, gemm_variant, monkeypatch):
    """Variant 9 adds K in eight parts, which shows in the bits.  Set in the
    environment after the first launch it changes nothing (no launch reads the
    environment, which another thread may be writing), and selected in another
    thread it changes that thread's calls only."""
    import threading

    log("gemm kernel choice")
    a = _randn((64, 1024), torch.bfloat16, cuda, 91)
    w = _randn((64, 1024), torch.bfloat16, cuda, 92)
    own = _C.gemm(a, w, out_dtype=torch.float32)
    gemm_variant(9)
    split = _C.gemm(a, w, out_dtype=torch.float32)
    gemm_variant(-1)
    assert not torch.equal(own, split)
    monkeypatch.setenv("TX_GEMM_VARIANT", "9")
    assert torch.equal(_C.gemm(a, w, out_dtype=torch.float32), own)
    monkeypatch.delenv("TX_GEMM_VARIANT")
    stream, got = torch.cuda.current_stream(), []

    def other():
        with torch.cuda.stream(stream):
            _C.select_kernel(_C.SELECT_GEMM, 9)
            got.append(_C.gemm(a, w, out_dtype=torch.float32))

    t = threading.Thread(target=other)
    t.start()
    t.join()
    assert torch.equal(got[0], split)
    assert torch.equal(_C.gemm(a, w, out_dtype=torch.float32), own)


def test_gemm_wide_row_stride_takes_64bit_kernel(cuda):
    """lda past the 256-row kernel's 32-bit DMA offsets ((255 lda + 56) * 2 >
    2^31 - 1) routes to the 64-bit-addressed 128x128 kernel: the product of
    the strided view is bitwise equal to the same product on a contiguous
    copy (which takes the 256-row kernel) and to F.linear."""
    m, n, k = 512, 256, 64
    lda = 4210760
    assert (255 * lda + 56) * 2 > 2**31 - 1
    log(f"gemm wide lda {lda}: {m * lda * 2 / 2**30:.1f} GiB operand")
    big = torch.empty((m, lda), dtype=torch.bfloat16, device=cuda)
    big[:, :k] = _randn((m, k), torch.bfloat16, cuda, 141)
    a = big[:, :k]
    assert a.stride(0) == lda
    w = _randn((n, k), torch.bfloat16, cuda, 142, 0.05)
    bias = _randn((n,), torch.bfloat16, cuda, 143, 0.1)
    got = _C.gemm(a, w, bias)
    same = _C.gemm(a.contiguous(), w, bias)
    torch.cuda.synchronize()
    del big
    assert torch.equal(got, same)
    assert torch.equal(got, F.linear(a.contiguous(), w, bias))


# ------------------------------------------------------------------ attention
def _split(qk, vt, b, s, h, hd):
    d = h * hd
    q = qk[:, :d].reshape(b, s, h, hd).permute(0, 2, 1, 3).contiguous()
    k = qk[:, d:].reshape(b, s, h, hd).permute(0, 2, 1, 3).contiguous()
    v = vt[..., :s].permute(0, 1, 3, 2).contiguous()
    return q, k, v


def _eager_attention(q, k, v, scale, causal, valid):
    """The oracle's chain (TTB:173-188) in the model dtype: QK^T on the
    transposed view as TTB:173 writes it, except in bf16, where a batched
    product with a transposed right operand has faulted GPUs of the test
    pool and the transpose is materialised (test_qkt_layouts_same_bits
    measures, in fp16, that the two layouts give the same bits)."""
    s = q.shape[2]
    kt = k.transpose(-2, -1)
    if q.dtype == torch.bfloat16:
        kt = kt.contiguous()
    scores = torch.matmul(q, kt) * scale
    if causal:
        scores = scores.masked_fill(torch.ones(s, s, dtype=torch.bool, device=q.device).triu(1), float("-inf"))
    if valid is not None:
        scores = scores.masked_fill(~valid[:, None, None, :], float("-inf"))
    p = torch.softmax(scores.float(), dim=-1).to(q.dtype)
    return _pv_in_key_order(p, v)


# Batched products below which the library's P.V GEMM may split the key
# dimension (measured: 2-4 products at 1024-2048 keys differ from the same
# products in a larger batch in 0.03-0.1% of outputs; 32 products at 2048
# keys and 16 at 8192 do not).
PV_INORDER_BATCH = 64


def _pv_in_key_order(p, v):
    """P.V with the keys accumulated in order, as the library computes it
    when it runs many batched products: with few products and long rows it
    picks a split-K kernel instead (a different summation order).  The
    kernels keep key order at every shape, so the comparator replicates the
    batch until the library does too."""
    n = p.shape[0] * p.shape[1]
    if n >= PV_INORDER_BATCH:
        return torch.matmul(p, v)
    rep = -(-PV_INORDER_BATCH // n)
    pb = p.reshape(n, *p.shape[2:]).repeat(rep, 1, 1).contiguous()
    vb = v.contiguous().reshape(n, *v.shape[2:]).repeat(rep, 1, 1).contiguous()
    return torch.matmul(pb, vb)[:n].reshape(*p.shape[:-1], v.shape[-1])


@pytest.mark.parametrize("b,h,s,hd", [(1, 8, 64, 64), (4, 16, 384, 64), (8, 16, 1024, 64),
                                      (1, 16, 8192, 128)])
def test_qkt_layouts_same_bits(cuda, b, h, s, hd):
    """TTB:173 multiplies q by the transposed view k.transpose(-2, -1) (the
    library's NT layout); the bf16 comparators materialise the transpose (NN
    layout), because bf16 batched products with a transposed right operand
    have faulted GPUs of the test pool.  In fp16, where both are safe, the
    two layouts give identical bits at the workload and mask-test head
    shapes (c2, masked tests, c3, c4)."""
    log(f"QK^T layouts b{b} h{h} s{s} hd{hd} fp16")
    q = _randn((b, h, s, hd), torch.float16, cuda, 101, 0.8)
    k = _randn((b, h, s, hd), torch.float16, cuda, 102, 0.8)
    nt = torch.matmul(q, k.transpose(-2, -1))
    nn_ = torch.matmul(q, k.transpose(-2, -1).contiguous())
    n_diff = int((nt != nn_).sum())
    log(f"  elements differing between NT and NN: {n_diff} of {nt.numel()}")
    assert n_diff == 0


def _fp32_attention(q, k, v, scale, causal, valid, q_rows=None):
    qf = q.float() if q_rows is None else q[:, :, q_rows].float()
    scores = torch.matmul(qf, k.float().transpose(-2, -1).contiguous()) * scale
    s = k.shape[2]
    if causal:
        rows = torch.arange(q.shape[2], device=q.device) if q_rows is None else q_rows
        scores = scores.masked_fill(torch.arange(s, device=q.device)[None, :] > rows[:, None], float("-inf"))
    if valid is not None:
        scores = scores.masked_fill(~valid[:, None, None, :], float("-inf"))
    return torch.matmul(torch.softmax(scores, -1), v.float())


ATTN_CASES = [
    # b, h, s, hd, causal, masked
    (1, 8, 64, 64, False, False),      # c2
    (2, 4, 128, 64, True, False),      # c1 shape, causal
    (2, 4, 200, 64, False, True),      # ragged S, key padding
    (8, 16, 1024, 64, False, False),   # c3
    (2, 16, 1024, 64, True, True),
    (1, 16, 8192, 128, False, False),  # c4
    (1, 4, 1000, 128, True, True),
    (3, 2, 77, 128, False, True),
    # rows of one key tile (S <= 64): stats formed inside the kernel (head
    # dim 64: two waves per 32 queries, one key half each)
    (3, 4, 37, 64, True, True),
    (2, 3, 1, 64, False, False),
    (1, 2, 8, 64, True, False),
    (2, 2, 63, 64, False, True),
    (1, 4, 33, 64, True, True),
    (2, 4, 1, 128, False, False),
    (1, 8, 50, 128, False, True),
    # S > 1024: ATen's warp softmax up to 2048 keys (two-kernel path), its
    # 512-thread block softmax above (__expf, reciprocal multiply); causal
    # and key padding (TTB:175-184) at both head dims, ragged lengths, and
    # the reference's long_fp16 attention shape (B4 H8 S2048 hd64,
    # run_bench.py:211-212)
    (1, 4, 2048, 64, True, True),
    (4, 8, 2048, 64, False, False),
    (2, 4, 2048, 64, False, True),
    (2, 8, 3000, 128, True, True),
    (1, 4, 1500, 128, True, False),
    (2, 4, 2048, 128, False, True),
    (1, 2, 4100, 64, True, True),
]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("b,h,s,causal,masked", [(2, 4, 50, True, True), (1, 8, 64, False, False),
                                                 (2, 4, 200, False, True), (1, 4, 300, True, False)])
def test_flash_attention_scale_not_power_of_two(cuda, dtype, b, h, s, causal, masked):
    """Head dim 64 with a caller's scale that is not a power of two: the
    scores are rounded, scaled and rounded again, as the eager chain does
    (the default 1/8 is exact and skips the second rounding)."""
    hd, scale = 64, 0.1
    log(f"attn scale {scale} b{b} h{h} s{s} causal={causal} masked={masked} {dtype}")
    d = h * hd
    qk = _randn((b * s, 2 * d), dtype, cuda, 54, 0.8)
    vt = torch.zeros((b, h, hd, _C.vt_ld(s)), dtype=dtype, device=cuda)
    vt[..., :s] = _randn((b, h, hd, s), dtype, cuda, 55)
    valid = None
    if masked:
        from transformer_optimization_amd.workloads import padding_mask
        valid = padding_mask(b, s, 0.5, seed=56).to(cuda)
    q, k, v = _split(qk, vt, b, s, h, hd)
    eager16 = _eager_attention(q, k, v, scale, causal, valid)
    o = _C.flash_attn(qk, vt, b, s, h, hd, scale, causal, key_valid=valid, softmax="eager")
    ex = o.reshape(b, s, h, hd).permute(0, 2, 1, 3)
    rows_ok = torch.isfinite(eager16).all(-1)
    assert int((ex != eager16)[rows_ok].sum()) == 0


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("b,h,s,hd,causal,masked", ATTN_CASES)
def test_flash_attention(cuda, dtype, b, h, s, hd, causal, masked):
    log(f"attn b{b} h{h} s{s} hd{hd} causal={causal} masked={masked} {dtype}")
    d = h * hd
    qk = _randn((b * s, 2 * d), dtype, cuda, 51, 0.8)
    vt = torch.zeros((b, h, hd, _C.vt_ld(s)), dtype=dtype, device=cuda)
    vt[..., :s] = _randn((b, h, hd, s), dtype, cuda, 52)
    valid = None
    if masked:
        from transformer_optimization_amd.workloads import padding_mask
        valid = padding_mask(b, s, 0.5, seed=53).to(cuda)
    scale = hd ** -0.5
    q, k, v = _split(qk, vt, b, s, h, hd)
    eager16 = _eager_attention(q, k, v, scale, causal, valid)
    # eager-exact mode: bitwise equal to the eager chain on every row that
    # has at least one admissible key.
    o_exact = _C.flash_attn(qk, vt, b, s, h, hd, scale, causal, key_valid=valid, softmax="eager")
    ex = o_exact.reshape(b, s, h, hd).permute(0, 2, 1, 3)
    rows_ok = torch.isfinite(eager16).all(-1)
    n_diff = int((ex != eager16)[rows_ok].sum())
    log(f"  eager-exact: differing elements {n_diff} of {int(rows_ok.sum()) * hd}")
    assert n_diff == 0
    o = _C.flash_attn(qk, vt, b, s, h, hd, scale, causal, key_valid=valid, softmax="online")
    ours = o.reshape(b, s, h, hd).permute(0, 2, 1, 3).float()
    eager = eager16.float()
    exact = _fp32_attention(q, k, v, scale, causal, valid)
    assert torch.isfinite(ours[rows_ok]).all()
    err_ours = (ours - exact)[rows_ok].abs().max().item()
    err_eager = (eager - exact)[rows_ok].abs().max().item()
    diff = (ours - eager)[rows_ok].abs().max().item()
    log(f"  online: |ours-fp32|={err_ours:.3e} |eager-fp32|={err_eager:.3e} |ours-eager|={diff:.3e}")
    # No worse than twice eager's own deviation from fp32, plus one output ulp.
    tol = 2 * err_eager + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) * exact.abs().max().item()
    assert err_ours <= tol
    assert diff <= 2 * tol


@pytest.mark.parametrize("s,causal,masked", [(1028, False, True), (2048, True, False), (2052, False, False),
                                             (2056, True, True), (16384, False, False)])
def test_flash_attention_softmax_kernel_boundaries(cuda, s, causal, masked):
    """Both sides of the change from ATen's warp softmax (rows of up to 2048
    fp32 values) to its 512-thread block softmax, and a row of 16384 keys
    (past the block's shared-memory copy with 64 KiB per block), bitwise
    against the eager chain (fp16, head dim 64)."""
    b, h, hd, dtype = 1, 2, 64, torch.float16
    d = h * hd
    log(f"softmax boundaries s{s} causal={causal} masked={masked}")
    assert _C.eager_softmax_supported(s, cuda)
    qk = _randn((b * s, 2 * d), dtype, cuda, 151, 0.8)
    vt = torch.zeros((b, h, hd, _C.vt_ld(s)), dtype=dtype, device=cuda)
    vt[..., :s] = _randn((b, h, hd, s), dtype, cuda, 152)
    valid = None
    if masked:
        from transformer_optimization_amd.workloads import padding_mask
        valid = padding_mask(b, s, 0.5, seed=153).to(cuda)
    q, k, v = _split(qk, vt, b, s, h, hd)
    eager = _eager_attention(q, k, v, hd ** -0.5, causal, valid)
    o = _C.flash_attn(qk, vt, b, s, h, hd, hd ** -0.5, causal, key_valid=valid, softmax="eager")
    got = o.reshape(b, s, h, hd).permute(0, 2, 1, 3)
    rows_ok = torch.isfinite(eager).all(-1)
    n_diff = int((got != eager)[rows_ok].sum())
    log(f"  eager-exact: differing elements {n_diff} of {int(rows_ok.sum()) * hd}")
    assert n_diff == 0


@pytest.mark.parametrize("s,causal", [(50, False), (200, True), (512, True), (1024, False), (2048, True)])
def test_flash_attention_fp16_tiny_scores(cuda, s, causal):
    """fp16 scores near zero: eager rounds round(q.k) * scale to fp16, and
    below 2^-14 that product is a subnormal that drops bits, so even a
    power-of-two scale must be applied with its own rounding.  q is scaled so
    that most |q.k| fall below 2^-11; bitwise against the eager chain."""
    b, h, hd, dtype = 2, 2, 64, torch.float16
    d = h * hd
    log(f"fp16 tiny scores s{s} causal={causal}")
    qk = _randn((b * s, 2 * d), dtype, cuda, 161, 0.8)
    qk[:, :d] *= 2.0 ** -12
    vt = torch.zeros((b, h, hd, _C.vt_ld(s)), dtype=dtype, device=cuda)
    vt[..., :s] = _randn((b, h, hd, s), dtype, cuda, 162)
    q, k, v = _split(qk, vt, b, s, h, hd)
    sc = torch.matmul(q, k.transpose(-2, -1))
    frac_tiny = float((sc.abs() < 2.0 ** -11).float().mean())
    log(f"  scores below 2^-11: {frac_tiny:.2f}")
    assert frac_tiny > 0.2
    eager = _eager_attention(q, k, v, hd ** -0.5, causal, None)
    o = _C.flash_attn(qk, vt, b, s, h, hd, hd ** -0.5, causal, softmax="eager")
    got = o.reshape(b, s, h, hd).permute(0, 2, 1, 3)
    n_diff = int((got != eager).sum())
    log(f"  eager-exact: differing elements {n_diff} of {got.numel()}")
    assert n_diff == 0


@pytest.mark.parametrize("b,h,s,causal", [(1, 2, 1028, False), (2, 2, 1500, True), (1, 1, 2048, False)])
def test_flash_attention_few_products_vs_library_split(cuda, b, h, s, causal):
    """Few batched products with long rows: the eager chain's P.V runs a
    split-K library kernel there.  The kernel's output equals the eager chain
    with P.V in key order bit for bit, and the eager chain itself within the
    repository gate (atol 0.002, rtol 0.02) -- the split order moves a few
    outputs by one ulp."""
    from oracle.gate import compare_outputs
    hd, dtype = 64, torch.bfloat16
    d = h * hd
    qk = _randn((b * s, 2 * d), dtype, cuda, 181, 0.8)
    vt = torch.zeros((b, h, hd, _C.vt_ld(s)), dtype=dtype, device=cuda)
    vt[..., :s] = _randn((b, h, hd, s), dtype, cuda, 182)
    q, k, v = _split(qk, vt, b, s, h, hd)
    inorder = _eager_attention(q, k, v, hd ** -0.5, causal, None)
    kt = k.transpose(-2, -1).contiguous()
    sc = torch.matmul(q, kt) * hd ** -0.5
    if causal:
        sc = sc.masked_fill(torch.ones(s, s, dtype=torch.bool, device=cuda).triu(1), float("-inf"))
    library = torch.matmul(torch.softmax(sc.float(), -1).to(dtype), v)
    o = _C.flash_attn(qk, vt, b, s, h, hd, hd ** -0.5, causal, softmax="eager")
    got = o.reshape(b, s, h, hd).permute(0, 2, 1, 3)
    n_split = int((library != inorder).sum())
    log(f"few products b{b} h{h} s{s}: library split-K vs in-order differ in {n_split}; "
        f"ours vs in-order {int((got != inorder).sum())}")
    assert torch.equal(got, inorder)
    r = compare_outputs(library, got)
    log(f"  vs the eager chain: {r.summary()}")
    assert r.passed


def test_eager_softmax_refuses_unmirrorable_lengths(cuda):
    """Lengths whose ATen block-softmax order is not reproduced (past 2048,
    not whole 4-value vectors) are refused rather than computed in another order; the
    library's device query and torch's device properties agree on the rule."""
    lib = _C.load_library()
    smem = torch.cuda.get_device_properties(cuda).shared_memory_per_block
    log(f"shared memory per block: {smem}")
    for s in (64, 1024, 2048, 2049, 2052, 8192, 16376, 16384, 18432, 40000, 65536, 65540):
        assert lib.tx_eager_softmax_supported(s, 0) == lib.tx_eager_softmax_supported(s, smem), s
    b, h, hd, s = 1, 2, 64, 2050
    qk = _randn((b * s, 2 * h * hd), torch.bfloat16, cuda, 171)
    vt = torch.zeros((b, h, hd, _C.vt_ld(s)), dtype=torch.bfloat16, device=cuda)
    with pytest.raises(_C.TxError) as err:
        _C.flash_attn(qk, vt, b, s, h, hd, hd ** -0.5, False, softmax="eager")
    assert err.value.code == _C.TX_EUNSUPPORTED
    o = _C.flash_attn(qk, vt, b, s, h, hd, hd ** -0.5, False, softmax="online")
    assert torch.isfinite(o).all()


STRIDED_CASES = [
    # b, s, h, hd, causal, masked, dtype
    (1, 64, 8, 64, False, False, torch.float16),      # c2
    (8, 1024, 16, 64, False, False, torch.bfloat16),  # c3
    (1, 8192, 16, 128, False, False, torch.bfloat16), # c4
    (2, 200, 4, 64, True, True, torch.float16),       # ragged, causal, key padding
    (3, 77, 2, 128, False, True, torch.bfloat16),
    (2, 37, 4, 64, True, False, torch.bfloat16),      # one key tile
    (1, 1000, 4, 128, True, True, torch.float16),
    # S > 1024 (warp softmax to 2048, block softmax above) on natural-layout V
    (1, 2048, 4, 64, True, True, torch.float16),
    (4, 2048, 8, 64, False, False, torch.float16),    # long_fp16 attention shape
    (2, 1500, 4, 128, True, True, torch.bfloat16),
    (1, 3000, 2, 64, False, True, torch.bfloat16),
]


@pytest.mark.parametrize("b,s,h,hd,causal,masked,dtype", STRIDED_CASES)
def test_flash_attention_strided_views(cuda, b, s, h, hd, causal, masked, dtype):
    """tx_flash_attn_fwd_strided on the reference's call shape: q / k / v are
    [B, H, S, hd] column views of one packed F.linear [B, S, 3D] projection
    (TTB:1596-1668, 4220-4222), V in its natural layout, output heads merged.
    Eager softmax: bitwise equal to the eager chain on the head-split
    tensors; online softmax: no worse than twice eager's deviation from fp32."""
    log(f"strided attn b{b} s{s} h{h} hd{hd} causal={causal} masked={masked} {dtype}")
    d = h * hd
    x = _randn((b, s, d), dtype, cuda, 111)
    w = _randn((3 * d, d), dtype, cuda, 112, 0.06)
    bias = _randn((3 * d,), dtype, cuda, 113, 0.1)
    qkv = F.linear(x, w, bias)                                   # [B, S, 3D]
    q, k, v = (qkv[..., j * d:(j + 1) * d].view(b, s, h, hd).transpose(1, 2) for j in range(3))
    assert not q.is_contiguous()
    valid = None
    if masked:
        from transformer_optimization_amd.workloads import padding_mask
        valid = padding_mask(b, s, 0.5, seed=114).to(cuda)
    scale = hd ** -0.5
    eager = _eager_attention(q.contiguous(), k.contiguous(), v.contiguous(), scale, causal, valid)
    got = _C.flash_attn_strided(q, k, v, scale, causal, key_valid=valid, softmax="eager")
    assert got.shape == (b, h, s, hd)
    merged = got.transpose(1, 2)                                 # [B, S, H, hd]
    assert merged.is_contiguous()                                # heads merged in memory
    rows_ok = torch.isfinite(eager).all(-1)
    n_diff = int((got != eager)[rows_ok].sum())
    log(f"  eager-exact: differing elements {n_diff} of {int(rows_ok.sum()) * hd}")
    assert n_diff == 0
    # The packed-layout entry point gives the same bits.
    qk = torch.cat([qkv[..., :2 * d]], -1).reshape(b * s, 2 * d).contiguous()
    vt = torch.zeros((b, h, hd, _C.vt_ld(s)), dtype=dtype, device=cuda)
    vt[..., :s] = v.transpose(2, 3)
    packed = _C.flash_attn(qk, vt, b, s, h, hd, scale, causal, key_valid=valid, softmax="eager")
    assert torch.equal(packed.view(b, s, h, hd), merged)
    # Online softmax on the same views.
    on = _C.flash_attn_strided(q, k, v, scale, causal, key_valid=valid, softmax="online").float()
    exact = _fp32_attention(q, k, v, scale, causal, valid)
    err_on = (on - exact)[rows_ok].abs().max().item()
    err_eager = (eager.float() - exact)[rows_ok].abs().max().item()
    tol = 2 * err_eager + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) * exact.abs().max().item()
    log(f"  online: |ours-fp32|={err_on:.3e} |eager-fp32|={err_eager:.3e}")
    assert err_on <= tol


def test_flash_attention_strided_explicit_output_view(cuda):
    """An explicit output view with its own strides ([B, H, S, hd] contiguous)
    and a key mask with a padded row stride."""
    b, s, h, hd, dtype = 2, 300, 4, 64, torch.bfloat16
    d = h * hd
    qkv = _randn((b, s, 3 * d), dtype, cuda, 121)
    q, k, v = (qkv[..., j * d:(j + 1) * d].view(b, s, h, hd).transpose(1, 2) for j in range(3))
    from transformer_optimization_amd.workloads import padding_mask
    valid_wide = torch.ones(b, s + 13, dtype=torch.bool, device=cuda)
    valid_wide[:, :s] = padding_mask(b, s, 0.4, seed=122).to(cuda)
    valid = valid_wide[:, :s]
    out = torch.empty((b, h, s, hd), dtype=dtype, device=cuda)
    got = _C.flash_attn_strided(q, k, v, hd ** -0.5, False, key_valid=valid, out=out)
    assert got.data_ptr() == out.data_ptr()
    eager = _eager_attention(q.contiguous(), k.contiguous(), v.contiguous(), hd ** -0.5, False, valid)
    assert torch.equal(out, eager)


@pytest.mark.parametrize("dtype", [torch.bfloat16])
def test_flash_attention_c5_rows(cuda, dtype):
    # S = 100000, hd 64: dense scores are impossible; check 512 seeded query
    # rows against fp32 attention over all keys.
    from transformer_optimization_amd.workloads import sample_rows
    b, h, s, hd = 1, 16, 100000, 64
    d = h * hd
    log("attn c5 S=100000")
    qk = _randn((b * s, 2 * d), dtype, cuda, 61, 0.8)
    vt = torch.zeros((b, h, hd, _C.vt_ld(s)), dtype=dtype, device=cuda)
    vt[..., :s] = _randn((b, h, hd, s), dtype, cuda, 62)
    scale = hd ** -0.5
    o = _C.flash_attn(qk, vt, b, s, h, hd, scale, False, softmax="online")
    torch.cuda.synchronize()
    rows = sample_rows(s).to(cuda)
    q, k, v = _split(qk, vt, b, s, h, hd)
    exact = torch.cat([_fp32_attention(q, k, v, scale, False, None, rows[i:i + 64])
                       for i in range(0, rows.numel(), 64)], dim=2)
    ours = o.reshape(b, s, h, hd)[:, rows].permute(0, 2, 1, 3).float()
    err = (ours - exact).abs().max().item()
    log(f"  c5 rows |ours-fp32| = {err:.3e}")
    assert err <= 4 * 2.0 ** -8 * max(exact.abs().max().item(), 1e-3)


@pytest.mark.parametrize("dtype,hd", [(torch.bfloat16, 64), (torch.float16, 128)])
@pytest.mark.parametrize("pattern", ["outlier", "staircase", "negative", "masked_prefix"])
def test_online_softmax_running_max_rebase(cuda, pattern, dtype, hd):
    """Online softmax where the running row max must move mid-row.

    Every query of a head is close to one direction u, so a key's score is
    set by how much of u it carries (a key g u scores ~11.5 g in log2 units
    at hd 64):
      * outlier: one key 10 units above the rest at position 700, worth about
        as much as the 700 keys before it, which were summed against the old
        max;
      * staircase: the level rises 3.5 units every 100 keys (a re-base about
        every third step, each carrying the earlier sums along);
      * negative: every score near -200 units (the first max is far below 0);
      * masked_prefix: batch 1 has its first 150 keys masked (no admissible
        key in the first two tiles), plus the outlier.
    At hd 128 the same levels are 1.41x larger.  A wrong rescale factor or
    shift changes the outputs by O(|v|); the bound is the c5 rows test's."""
    b, h, s = 2, 2, 1000
    d = h * hd
    g = torch.Generator().manual_seed(131)
    u = torch.randn(h, hd, generator=g)
    q = u[None, :, None, :] + 0.1 * torch.randn(b, h, s, hd, generator=g)
    k = 0.3 * torch.randn(b, h, s, hd, generator=g)
    level = torch.zeros(s)
    if pattern in ("outlier", "masked_prefix"):
        level[700] = 10.0 / 11.54
    elif pattern == "staircase":
        level = 0.3 * (torch.arange(s) // 100).float()
    elif pattern == "negative":
        level[:] = -200.0 / 11.54
    k = k + level[None, None, :, None] * u[None, :, None, :]
    v = torch.randn(b, h, s, hd, generator=g)
    valid = None
    if pattern == "masked_prefix":
        valid = torch.ones(b, s, dtype=torch.bool)
        valid[1, :150] = False
        valid = valid.to(cuda)
    qk = torch.cat([q.permute(0, 2, 1, 3).reshape(b * s, d), k.permute(0, 2, 1, 3).reshape(b * s, d)],
                   dim=1).to(cuda, dtype)
    vt = torch.zeros((b, h, hd, _C.vt_ld(s)), dtype=dtype, device=cuda)
    vt[..., :s] = v.permute(0, 1, 3, 2).to(cuda, dtype)
    scale = hd ** -0.5
    log(f"online re-base {pattern} {dtype} hd {hd}")
    o = _C.flash_attn(qk, vt, b, s, h, hd, scale, False, key_valid=valid, softmax="online")
    qs, ks, vs = _split(qk, vt, b, s, h, hd)
    exact = _fp32_attention(qs, ks, vs, scale, False, valid)
    natural = _C.flash_attn_strided(qs, ks, vs, scale, False, key_valid=valid, softmax="online")
    for ours in (o.reshape(b, s, h, hd).permute(0, 2, 1, 3).float(), natural.float()):
        err = (ours - exact).abs().max().item()
        log(f"  |ours-fp32| = {err:.3e}, max |o| = {exact.abs().max().item():.3e}")
        assert torch.isfinite(ours).all()
        assert err <= 4 * 2.0 ** -8 * max(exact.abs().max().item(), 1e-3)


@pytest.mark.parametrize("dtype,hd", [(torch.bfloat16, 64), (torch.float16, 64), (torch.bfloat16, 128)])
@pytest.mark.parametrize("b,h,s,causal,masked", [(1, 2, 1, False, False), (2, 4, 63, True, False),
                                                 (1, 3, 65, True, True), (2, 2, 128, False, True),
                                                 (2, 8, 333, True, False), (1, 4, 449, False, True)])
def test_online_softmax_short_rows_and_masks(cuda, dtype, hd, b, h, s, causal, masked):
    """Both V layouts: one to eight key tiles, full and ragged, and a fully
    masked sequence (its rows are 0).  Against fp32 attention: q is rounded
    once more (scaled into log2 units) and p once, 2^-p relative each, so 2^-p
    times a few row magnitudes bounds the difference."""
    log(f"online b{b} h{h} s{s} hd{hd} causal={causal} masked={masked} {dtype}")
    qkv = _randn((b, s, 3 * h * hd), dtype, cuda, 171, 0.8)
    q, k, v = (qkv[..., j * h * hd:(j + 1) * h * hd].view(b, s, h, hd).transpose(1, 2) for j in range(3))
    valid = None
    if masked:
        valid = torch.rand((b, s), generator=_gen(172)).to(cuda) < 0.6
        valid[-1] = False
    sc = (q.float() @ k.float().transpose(2, 3).contiguous()) * hd ** -0.5
    if causal:
        sc = sc.masked_fill(torch.ones((s, s), dtype=torch.bool, device=cuda).triu(1), float("-inf"))
    if masked:
        sc = sc.masked_fill(~valid[:, None, None, :], float("-inf"))
    ref = torch.softmax(sc, -1).nan_to_num(0.0) @ v.float()
    qk = qkv[..., :2 * h * hd].reshape(b * s, 2 * h * hd).contiguous()
    vt = torch.zeros((b, h, hd, _C.vt_ld(s)), dtype=dtype, device=cuda)
    vt[..., :s] = v.transpose(2, 3)
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    o1 = _C.flash_attn(qk, vt, b, s, h, hd, hd ** -0.5, causal, key_valid=valid, softmax="online")
    o2 = _C.flash_attn_strided(q, k, v, hd ** -0.5, causal, key_valid=valid, softmax="online")
    for o in (o1.view(b, s, h, hd).transpose(1, 2), o2):
        err = (o.float() - ref).abs().amax()
        assert float(err) <= 8 * eps * float(v.float().abs().amax()), float(err)
        if masked:
            assert not o[-1].any()


@pytest.mark.parametrize("softmax", ["eager", "online"])
@pytest.mark.parametrize("dtype,hd,h,s,causal", [(torch.bfloat16, 64, 8, 333, False), (torch.float16, 64, 8, 1000, True),
                                                 (torch.bfloat16, 128, 4, 449, True), (torch.float16, 128, 8, 200, False),
                                                 (torch.bfloat16, 64, 8, 64, False)])
def test_attention_of_a_sequence_does_not_depend_on_the_batch(cuda, softmax, dtype, hd, h, s, causal):
    """One sequence alone (a grid far below the CUs) and as the last of 40 (a
    grid that fills them): the same bits, in both V layouts."""
    b = 40
    log(f"batch independence {softmax} h{h} s{s} hd{hd} causal={causal} {dtype}")
    qkv = _randn((b, s, 3 * h * hd), dtype, cuda, 175, 0.8)

    def run(t):
        n = t.shape[0]
        q, k, v = (t[..., j * h * hd:(j + 1) * h * hd].view(n, s, h, hd).transpose(1, 2) for j in range(3))
        vt = torch.zeros((n, h, hd, _C.vt_ld(s)), dtype=dtype, device=cuda)
        vt[..., :s] = v.transpose(2, 3)
        qk = t[..., :2 * h * hd].reshape(n * s, 2 * h * hd).contiguous()
        o = _C.flash_attn(qk, vt, n, s, h, hd, hd ** -0.5, causal, softmax=softmax)
        return o.view(n, s, h, hd).transpose(1, 2), _C.flash_attn_strided(q, k, v, hd ** -0.5, causal, softmax=softmax)

    for alone, batch in zip(run(qkv[-1:]), run(qkv)):
        assert torch.equal(alone[0], batch[-1])


@pytest.fixture
def rowres():
    yield lambda n: _C.select_kernel(_C.SELECT_ATTN_ROWRES, n)
    _C.select_kernel(_C.SELECT_ATTN_ROWRES, -1)


# At head dim 64 rows of one key tile have their own kernels: neither path runs.
ROWRES_ROWS = [(1, False, False), (64, True, False), (65, False, True), (129, True, True), (256, False, False),
               (257, True, False), (500, False, True), (513, True, True), (1000, False, True), (1024, True, False)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hd,s,causal,masked", [(hd, *row) for hd in (64, 128) for row in ROWRES_ROWS
                                                if hd == 128 or row[0] > 64])
def test_exact_attention_row_resident_equals_two_kernels(cuda, dtype, hd, s, causal, masked, rowres):
    """The row-resident kernel at the edges of its tile runs (one, two and four
    tiles a wave, waves without a tile) and the two-kernel path: same bits, in
    both V layouts."""
    b, h = 2, 3
    log(f"row-resident s{s} hd{hd} causal={causal} masked={masked} {dtype}")
    qkv = _randn((b, s, 3 * h * hd), dtype, cuda, 173, 0.8)
    q, k, v = (qkv[..., j * h * hd:(j + 1) * h * hd].view(b, s, h, hd).transpose(1, 2) for j in range(3))
    qk = qkv[..., :2 * h * hd].reshape(b * s, 2 * h * hd).contiguous()
    # The padding columns of V^T hold NaN: nothing may read them into a sum.
    vt = torch.full((b, h, hd, _C.vt_ld(s)), float("nan"), dtype=dtype, device=cuda)
    vt[..., :s] = v.transpose(2, 3)
    valid = (torch.rand((b, s), generator=_gen(174)) < 0.6).to(cuda) if masked else None
    got = []
    for n in (0, 1):
        rowres(n)
        got.append(_C.flash_attn(qk, vt, b, s, h, hd, hd ** -0.5, causal, key_valid=valid).view(b, s, h, hd).transpose(1, 2))
        got.append(_C.flash_attn_strided(q, k, v, hd ** -0.5, causal, key_valid=valid))
    for g in got:
        assert torch.isfinite(g).all() and torch.equal(g, got[0])


@pytest.mark.parametrize("hd,s,causal,masked", [(64, 40, False, False), (64, 64, True, True), (64, 200, False, True),
                                                (64, 1000, True, False), (64, 1500, False, True),
                                                (64, 2304, False, True), (128, 40, False, True), (128, 300, True, False),
                                                (128, 1500, True, True), (128, 2304, True, False)])
def test_rows_that_overflow_to_minus_inf_are_nan_as_in_eager(cuda, hd, s, causal, masked):
    """fp16 rows whose admissible scores all lie below -65520 (every third
    query): they round to -inf, and eager's softmax of such a row is NaN.
    Through every exact kernel (one tile, row-resident, two kernels with the
    wave and the block softmax), both V layouts: the same rows are NaN, and
    the others have eager's bits."""
    b, h = 2, 2
    log(f"overflow to -inf s{s} hd{hd} causal={causal} masked={masked}")
    q = _randn((b, h, s, hd), torch.float16, cuda, 181, 0.02)
    q[:, :, ::3] = 45.0
    k = _randn((b, h, s, hd), torch.float16, cuda, 182) - 45.0
    v = _randn((b, h, s, hd), torch.float16, cuda, 183)
    valid = None
    if masked:
        valid = torch.rand((b, s), generator=_gen(184)).to(cuda) < 0.6
        valid[:, 0] = True  # no query without an admissible key
    ref = _eager_attention(q, k, v, hd ** -0.5, causal, valid).float()
    bad = torch.zeros(s, dtype=torch.bool, device=cuda)
    bad[::3] = True
    assert torch.equal(ref.isnan().all(-1), bad.expand(b, h, s))
    qk = torch.cat([t.transpose(1, 2).reshape(b * s, h * hd) for t in (q, k)], 1)
    vt = torch.zeros((b, h, hd, _C.vt_ld(s)), dtype=torch.float16, device=cuda)
    vt[..., :s] = v.transpose(2, 3)
    o1 = _C.flash_attn(qk, vt, b, s, h, hd, hd ** -0.5, causal, key_valid=valid)
    o2 = _C.flash_attn_strided(q, k, v, hd ** -0.5, causal, key_valid=valid)
    for o in (o1.view(b, s, h, hd).transpose(1, 2).float(), o2.float()):
        assert torch.equal(o.isnan(), ref.isnan())
        assert torch.equal(o.nan_to_num(0.0), ref.nan_to_num(0.0))


@pytest.mark.parametrize("s,hd,causal", [(96, 64, False), (40, 64, False), (17, 64, True), (1500, 64, True),
                                          (2048, 128, False), (1100, 128, True)])
def test_fully_masked_rows_are_zero_not_nan(cuda, s, hd, causal):
    """Batch 1 has no valid key: its rows come out 0 (the eager chain gives
    NaN there, and the model masks those rows anyway); batch 0's rows stay
    bitwise equal to the eager chain."""
    b, h = 2, 2
    d = h * hd
    log(f"fully masked batch s{s} hd{hd} causal={causal}")
    qk = _randn((b * s, 2 * d), torch.bfloat16, cuda, 71)
    vt = _randn((b, h, hd, _C.vt_ld(s)), torch.bfloat16, cuda, 72)
    valid = torch.ones(b, s, dtype=torch.bool, device=cuda)
    valid[0, s // 3:s // 2] = False
    valid[1] = False  # batch 1 has no valid key at all
    q, k, v = _split(qk, vt, b, s, h, hd)
    eager = _eager_attention(q, k, v, hd ** -0.5, causal, valid)
    for mode in ("eager", "online"):
        o = _C.flash_attn(qk, vt, b, s, h, hd, hd ** -0.5, causal, key_valid=valid, softmax=mode)
        assert torch.isfinite(o).all()
        assert torch.count_nonzero(o[s:]) == 0
        if mode == "eager":
            got0 = o[:s].reshape(s, h, hd).permute(1, 0, 2)
            assert torch.equal(got0, eager[0])


# ------------------------------------------------ fp32-residual policy pieces
@pytest.mark.parametrize("dtype", DTYPES)
def test_layernorm_split_and_fp32_input(cuda, dtype):
    rows, d = 2048, 1024
    x = (torch.randn(rows, d, generator=_gen(81)) * 1.7 + 0.2).to(cuda)  # fp32 residual
    g = _randn((d,), dtype, cuda, 82, 0.2) + 1.0
    b = _randn((d,), dtype, cuda, 83, 0.2)
    y = _C.layernorm_residual(x, g, b, y_dtype=dtype, split=True)
    hi, lo = y[:, :d].float(), y[:, d:].float()
    ref = F.layer_norm(x.double(), (d,), g.double(), b.double(), 1e-5)
    assert torch.equal(hi, hi.to(dtype).float())
    # hi + lo carries the fp32 value to ~2^-16 relative (plus fp32 moments).
    err = ((hi + lo).double() - ref).abs().max().item()
    assert err <= 2e-5 * ref.abs().max().item()
    y1 = _C.layernorm_residual(x, g, b, y_dtype=dtype)
    assert torch.equal(y1, y[:, :d])


@pytest.mark.parametrize("dtype", DTYPES)
def test_gemm_split_gelu_and_fp32_residual(cuda, dtype):
    m, n, k = 1000, 2048, 1024
    a_hi = _randn((m, k), dtype, cuda, 91)
    a_lo = (a_hi.float() * 2.0 ** -9 * torch.randn(m, k, generator=_gen(92)).to(cuda)).to(dtype)
    a2 = torch.cat([a_hi, a_lo], 1).contiguous()
    w = _randn((n, k), dtype, cuda, 93, 0.02)
    w2 = torch.cat([w, w], 1).contiguous()
    bias = _randn((n,), dtype, cuda, 94, 0.1)
    out = _C.gemm(a2, w2, bias, gelu=True, split_out=True)
    got = out[:, :n].double() + out[:, n:].double()
    a64 = a_hi.double() + a_lo.double()
    ref = F.gelu(a64 @ w.double().t() + bias.double())
    err = (got - ref).abs().max().item()
    log(f"split gelu max err {err:.3e}")
    assert err <= 1e-5 * max(1.0, ref.abs().max().item())
    # fp32 residual: x <- x + (acc + b) without rounding the GEMM term
    res = torch.randn(m, n, generator=_gen(95)).to(cuda)
    x32 = res.clone()
    _C.gemm(a2, w2, bias, residual=x32, out=x32)
    ref2 = res.double() + a64 @ w.double().t() + bias.double()
    err2 = (x32.double() - ref2).abs().max().item()
    assert err2 <= 1e-5 * max(1.0, ref2.abs().max().item())
    # bf16/fp16 residual into an fp32 output (first layer of the policy)
    r16 = _randn((m, n), dtype, cuda, 96)
    o32 = torch.empty(m, n, device=cuda)
    _C.gemm(a_hi, w, bias, residual=r16, out=o32)
    ref3 = r16.double() + a_hi.double() @ w.double().t() + bias.double()
    assert (o32.double() - ref3).abs().max().item() <= 1e-5 * max(1.0, ref3.abs().max().item())


@pytest.mark.parametrize("dtype", [torch.bfloat16])
def test_gemm_tall_shapes_match_across_kernels(cuda, dtype, gemm_variant):
    """Tall short-K shapes (M >= 32768, K <= 2048: the c5 projections) run on
    128-wide three-stage tiles; every kernel accumulates K in the same order,
    so the outputs equal those of the 128x128 kernel (variant 20) bit for
    bit: the bf16 GELU epilogue, the split-output (hi/lo) FFN-in epilogue and
    the fp32-output residual epilogues of the fp32-residual policy."""
    m, n, k = 40000, 1024, 1024
    log(f"gemm tall {m}x{n}x{k} {dtype}")
    a = _randn((m, k), dtype, cuda, 101)
    w = _randn((n, k), dtype, cuda, 102, 0.02)
    bias = _randn((n,), dtype, cuda, 103, 0.1)
    r16 = _randn((m, n), dtype, cuda, 104)
    res32 = torch.randn(m, n, generator=_gen(105)).to(cuda)

    def run_all():
        outs = [_C.gemm(a, w, bias, gelu=True), _C.gemm(a, w, bias, gelu=True, split_out=True)]
        o32 = torch.empty(m, n, device=cuda)
        _C.gemm(a, w, bias, residual=r16, out=o32)
        outs.append(o32)
        x32 = res32.clone()
        _C.gemm(a, w, bias, residual=x32, out=x32)
        outs.append(x32)
        return outs

    gemm_variant(20)
    ref = run_all()
    for v in (-1, 1283):
        gemm_variant(v)
        for r, g in zip(ref, run_all()):
            assert torch.equal(g, r), f"variant {v}"
