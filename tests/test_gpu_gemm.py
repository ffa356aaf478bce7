"""dc_w8a8_gemm / dc_rescale on the GPU against the oracle: the int32 GEMM is
exact and the fused epilogue rounds bit for bit like ``rescale(int_mm())``
(reference ``_int8.py:200-207, 313-323``; ``tests/test_int8.py:174-183``)."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch
import torch.nn as nn

from diffucore_amd import _int8, _lib
from oracle import gemm as OG
from oracle import quant as OQ
from tests._util import DT, np32, rel_l2

pytestmark = pytest.mark.gpu

REF_SHAPES = [(33, 2048, 1024), (300, 512, 768), (4096, 2048, 2048), (1000, 8192, 2048)]
EDGE_SHAPES = [(1, 64, 16), (17, 37, 48), (129, 200, 336), (512, 3072, 3072)]


def _qw(m, n, k, seed):
    g = torch.Generator().manual_seed(seed)
    q = torch.randint(-127, 128, (m, k), generator=g, dtype=torch.int8)
    w = torch.randint(-127, 128, (n, k), generator=g, dtype=torch.int8)
    sx = torch.rand(m, generator=g) * 1e-2
    sw = torch.rand(n, generator=g) * 1e-3
    return q, w, sx, sw


@pytest.mark.parametrize("m,n,k", REF_SHAPES + EDGE_SHAPES)
def test_int_mm_exact(gpu, m, n, k):
    q, w, _, _ = _qw(m, n, k, 6)
    acc = _int8.int_mm(q.to(gpu), w.to(gpu))
    assert acc.dtype == torch.int32
    assert np.array_equal(acc.cpu().numpy(), OG.int_mm(q.numpy(), w.numpy()))


@pytest.mark.parametrize("m,n,k", REF_SHAPES + EDGE_SHAPES)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_fused_epilogue_bit_exact(gpu, m, n, k, dtype):
    q, w, sx, sw = _qw(m, n, k, 7)
    out = _int8.scaled_mm(q.to(gpu), w.to(gpu), sx.to(gpu), sw.to(gpu), dtype)
    ref = OG.rescale(OG.int_mm(q.numpy(), w.numpy()), sx.numpy(), sw.numpy(), None, DT[dtype])
    assert out.dtype == dtype
    assert np.array_equal(np32(out).view(np.uint32), ref.view(np.uint32))
    # the reference's own contract: fused == rescale(int_mm())
    two = _int8.rescale(_int8.int_mm(q.to(gpu), w.to(gpu)), sx.to(gpu), sw.to(gpu), None, dtype)
    assert torch.equal(out, two)


@pytest.mark.parametrize("dtype,bias_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32),
                                              (torch.float32, torch.float32), (torch.bfloat16, torch.float32)])
def test_bias_double_rounding(gpu, dtype, bias_dtype):
    q, w, sx, sw = _qw(300, 520, 768, 8)
    bias = (torch.randn(520) * 0.5).to(bias_dtype)
    lin = _int8.Int8Linear(768, 520, bias=True, group=0, device=gpu)
    lin.weight.copy_(w.to(gpu))
    lin.scale_bits.copy_(sw.to(gpu).view(torch.int32))
    lin.bias = nn.Parameter(bias.to(gpu), requires_grad=False)
    out = lin.matmul_quantized(q.to(gpu), sx.to(gpu), dtype)
    ref = OG.rescale(OG.int_mm(q.numpy(), w.numpy()), sx.numpy(), sw.numpy(), np32(bias), DT[dtype])
    assert np.array_equal(np32(out).view(np.uint32), ref.view(np.uint32))
    two = _int8.rescale(_int8.int_mm(q.to(gpu), w.to(gpu)), sx.to(gpu), sw.to(gpu), bias.to(gpu), dtype)
    assert torch.equal(out, two)


@pytest.mark.parametrize("pad", [1, 4])
def test_rescale_strided_accumulator(gpu, pad):
    """dc_rescale on a row-strided int32 view (row stride N + pad: the one-
    output-per-thread pass for pad 1, the four-output pass for pad 4) equals
    the same values laid out contiguously, and the oracle."""
    q, w, sx, sw = _qw(257, 516, 512, 12)
    acc = _int8.int_mm(q.to(gpu), w.to(gpu))
    big = torch.zeros(257, 516 + pad, device=gpu, dtype=torch.int32)
    big[:, :516] = acc
    bias = (torch.randn(516) * 0.5).to(torch.bfloat16).to(gpu)
    got = _int8.rescale(big[:, :516], sx.to(gpu), sw.to(gpu), bias, torch.bfloat16)
    want = _int8.rescale(acc, sx.to(gpu), sw.to(gpu), bias, torch.bfloat16)
    assert torch.equal(got, want)
    ref = OG.rescale(acc.cpu().numpy(), sx.numpy(), sw.numpy(), np32(bias), DT[torch.bfloat16])
    assert np.array_equal(np32(got).view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("k,n,group", [(2048, 2048, 256), (768, 512, 256), (1024, 8192, 256), (320, 1280, 0)])
def test_int8_linear_matches_oracle_and_float(gpu, k, n, group):
    torch.manual_seed(4)
    lin = nn.Linear(k, n, bias=n == 512).to(gpu).half()
    m = _int8.Int8Linear.from_linear(lin, group)
    x = torch.randn(3, 333, k, device=gpu, dtype=torch.float16)
    y = m(x)
    assert y.dtype == torch.float16 and y.shape == (3, 333, n)
    qa, sa = OQ.quantize_activation(np32(x).reshape(-1, k), group)
    bias = np32(m.bias) if m.bias is not None else None
    ref = OG.w8a8_linear(qa, sa, m.weight.cpu().numpy(), m.scale.cpu().numpy(), bias, "f16")
    assert np.array_equal(np32(y).reshape(-1, n).view(np.uint32), ref.view(np.uint32))
    assert rel_l2(np32(y), np32(lin(x))) < 0.02


def test_cfg1_sd15_linear_exact(gpu):
    """Benchmark config 1 itself, seeded as specified: x fp32 [8192, 320] ~N(0, 1)
    with 0.5% of its channels (2 of 320) scaled x20, W [1280, 320] ~N(0, 0.02),
    group 0, fp32 out, through ``Int8Linear.forward``. The weight codes and
    scales (quantized on the CPU) equal the oracle's weight quantizer; the
    activation codes and scales and the fp32 output equal the oracle's
    quantize -> int_mm -> rescale bit for bit. K = 320 = 2 x 128 + 64 runs the
    DMA-fed kernel's 64-byte stages."""
    g = torch.Generator().manual_seed(0)
    x = torch.randn(8192, 320, generator=g)
    idx = torch.randperm(320, generator=g)[:2]
    x[:, idx] *= 20
    w = torch.randn(1280, 320, generator=g) * 0.02
    lin = nn.Linear(320, 1280, bias=False)
    with torch.no_grad():
        lin.weight.copy_(w)
    m = _int8.Int8Linear.from_linear(lin, 0).to(gpu)
    wq, ws = OQ.quantize_weight(w.numpy(), 0)
    assert np.array_equal(m.weight.cpu().numpy(), wq)
    assert np.array_equal(m.scale.cpu().numpy().view(np.uint32), np.asarray(ws, np.float32).view(np.uint32))
    assert _int8.gemm_plan(8192, 1280, 320) != "dma_256x256"
    assert _int8.gemm_kernel(8192, 1280, 320) == ("dma_128x128_k64", 1)
    xg = x.to(gpu)
    qa, sa = _int8.quantize_activation(xg, 0)
    oq, osc = OQ.quantize_activation(x.numpy(), 0)
    assert np.array_equal(qa.cpu().numpy(), oq)
    assert np.array_equal(sa.cpu().numpy().view(np.uint32), np.asarray(osc, np.float32).view(np.uint32))
    y = m(xg)
    assert y.dtype == torch.float32 and y.shape == (8192, 1280)
    ref = OG.w8a8_linear(oq, osc, wq, ws, None, "f32")
    assert np.array_equal(y.cpu().numpy().view(np.uint32), np.asarray(ref, np.float32).view(np.uint32))
    # group 0 on rows with x20 outlier channels: the outliers set each row's
    # int8 step, so the other channels lose precision (measured rel 0.032)
    assert rel_l2(np32(y), x.numpy() @ w.numpy().T) < 0.05


def test_short_input(gpu):
    lin = nn.Linear(256, 64, bias=False).to(gpu)
    x = torch.randn(3, 256, device=gpu)
    assert rel_l2(np32(_int8.Int8Linear.from_linear(lin)(x)), np32(lin(x))) < 0.02


# shapes of each tile class (by how full the last round of tiles is on a
# 256-CU device, and K % 256 for DMA_256x256) and the kernel that runs them,
# with M, N and K tails among them; the register-staged kernel at each of its
# four tiles
TILE_SHAPES = [((4096, 12288, 512), "dma_256x256", "dma_256x256"), ((4608, 3072, 256), "dma_256x256", "dma_128x128"),
               ((4096, 12288, 272), "256x256", "256x256"), ((4096, 3072, 512), "192x256", "dma_192x256"),
               ((4000, 3000, 272), "192x256", "192x256"), ((512, 3072, 512), "128x128", "dma_64x128"),
               ((4001, 12200, 768), "dma_256x256", "dma_256x256"), ((512, 12288, 3072), "192x128", "dma_128x128"),
               ((500, 12200, 336), "192x128", "192x128"), ((500, 3070, 528), "128x128", "128x128"),
               ((2500, 6140, 1024), "dma_256x256", "dma_256x256")]


@pytest.mark.parametrize("mnk,plan,kernel", TILE_SHAPES)
def test_every_tile_configuration(gpu, mnk, plan, kernel):
    m, n, k = mnk
    if torch.cuda.get_device_properties(gpu).multi_processor_count == 256:
        assert _int8.gemm_plan(m, n, k) == plan and _int8.gemm_kernel(m, n, k) == (kernel, 1)
    q, w, sx, sw = _qw(m, n, k, 9)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(9)) * 0.5).to(torch.bfloat16)
    lin = _int8.Int8Linear(k, n, bias=True, group=0, device=gpu)
    lin.weight.copy_(w.to(gpu))
    lin.scale_bits.copy_(sw.to(gpu).view(torch.int32))
    lin.bias = nn.Parameter(bias.to(gpu), requires_grad=False)
    acc_ref = OG.int_mm(q.numpy(), w.numpy())
    for dtype in (torch.bfloat16, torch.float16, torch.float32):
        out = lin.matmul_quantized(q.to(gpu), sx.to(gpu), dtype)
        ref = OG.rescale(acc_ref, sx.numpy(), sw.numpy(), np32(bias), DT[dtype])
        assert np.array_equal(np32(out).view(np.uint32), ref.view(np.uint32)), dtype
    acc = _int8.int_mm(q.to(gpu), w.to(gpu))
    assert np.array_equal(acc.cpu().numpy(), acc_ref)


def _int8_layers(gpu, k, ns, bias, seed):
    torch.manual_seed(seed)
    group = 256 if k % 256 == 0 else 0
    return [_int8.Int8Linear.from_linear(nn.Linear(k, n, bias=bias).to(gpu).half(), group) for n in ns]


@pytest.mark.parametrize("bias", [False, True])
def test_shared_qkv_equals_separate_layers(gpu, bias):
    """Self-attention q/k/v on one rotated + quantized copy of x (the Anima
    pattern, anima_dit.py:307-315) equals each layer on its own (the
    quantization is deterministic); cross-attention keeps k/v on the context."""
    projs = _int8_layers(gpu, 640, (640, 640, 640), bias, 21)
    x = torch.randn(2, 1000, 640, device=gpu, dtype=torch.float16)
    got = _int8.shared_qkv(x, projs)
    for p, y in zip(projs, got):
        assert torch.equal(y, p(x))
    ctx = torch.randn(2, 77, 640, device=gpu, dtype=torch.float16)
    q, k, v = _int8.shared_qkv(x, projs, ctx, is_selfattn=False)
    assert torch.equal(q, projs[0](x)) and torch.equal(k, projs[1](ctx)) and torch.equal(v, projs[2](ctx))


@pytest.mark.parametrize("bias", [False, True])
def test_fused_linears_equal_concatenated_outputs(gpu, bias):
    """One GEMM over stacked weights / scales / biases gives each layer's
    output bit for bit (per-channel scales, per-channel bias rounding)."""
    layers = _int8_layers(gpu, 1280, (1280, 640, 2560), bias, 22)
    fused = _int8.fuse_linears(layers)
    x = torch.randn(3, 333, 1280, device=gpu, dtype=torch.float16)
    y = fused(x)
    assert torch.equal(y, torch.cat([l(x) for l in layers], -1))


@pytest.mark.parametrize("mnk", [(4608, 12288, 3072), (4096, 3072, 3072), (512, 3072, 3072)])
def test_repeat_calls_identical(gpu, mnk):
    """The same launch gives the same bits every time (the DMA kernel stages
    its output through LDS with a cross-lane hand-off; a missing fence there
    would show as run-to-run differences)."""
    m, n, k = mnk
    q, w, sx, sw = _qw(m, n, k, 13)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(13)) * 0.5).to(torch.bfloat16).to(gpu)
    q, w, sx, sw = q.to(gpu), w.to(gpu), sx.to(gpu), sw.to(gpu)
    first = _int8._gemm(q, w, sx, sw, bias, torch.bfloat16).clone()
    for _ in range(8):
        assert torch.equal(_int8._gemm(q, w, sx, sw, bias, torch.bfloat16), first)


def _gemm_unsplit(q, w, sx, sw, bias, dtype):
    """dc_w8a8_gemm with no workspace (always one pass over k)."""
    from diffucore_amd import _lib
    so = _lib.require()
    M, K = q.shape
    N = w.shape[0]
    out = torch.empty(M, N, device=q.device, dtype=dtype)
    b_p, b_code = (bias.data_ptr(), _lib.dtype_code(bias.dtype)) if bias is not None else (None, _lib.NONE)
    rc = so.dc_w8a8_gemm(q.data_ptr(), K, w.data_ptr(), K, sx.data_ptr(), sw.data_ptr(), b_p, b_code, out.data_ptr(),
                         _lib.dtype_code(dtype), N, M, N, K, None, 0, _lib.stream_ptr(q.device))
    _lib.check(rc, "dc_w8a8_gemm")
    return out


# (M, N, K), and what runs it on 256 CUs: the DMA-fed kernel (K % 128 == 0)
# unsplit, then on each tile it splits (ragged rows and columns, slices that do
# not divide K); then the register-staged one, whose last slice is a short one
SPLIT_K = [((512, 3072, 3072), "dma_64x128", 1), ((154, 1280, 2048), "dma_64x64", 1), ((77, 640, 2048), "dma_64x64", 1),
           ((154, 640, 4096), "dma_64x64", 3), ((77, 1280, 4096), "dma_64x64", 3), ((300, 520, 8192), "dma_64x64", 4),
           ((1, 5120, 7680), "dma_64x64", 6), ((33, 9000, 7808), "dma_64x64", 3), ((231, 2040, 8320), "dma_64x64", 4),
           ((400, 640, 12416), "dma_64x128", 6), ((100, 3069, 15360), "dma_64x128", 5),
           ((500, 1276, 6272), "dma_64x128", 3), ((512, 3072, 12288), "dma_128x128_8w", 2),
           ((154, 3069, 7680), "dma_128x128_8w", 4), ((300, 3072, 8192), "dma_128x128_8w", 3),
           ((512, 3072, 8192), "dma_64x128", 1),
           ((154, 640, 4112), "128x128", 7), ((77, 1280, 3088), "128x128", 4), ((300, 520, 2112), "128x128", 4),
           ((77, 640, 2064), "128x128", 4), ((512, 3072, 3088), "128x128", 4)]


@pytest.mark.parametrize("mnk,kernel,slices", SPLIT_K)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_split_k_is_bit_identical(gpu, mnk, kernel, slices, dtype):
    """Small-M, long-K problems split k over workgroups into int32 partials;
    the epilogue over their exact sum equals the unsplit GEMM and the oracle
    bit for bit. The workspace is what those slices need, no more."""
    from diffucore_amd import _lib
    m, n, k = mnk
    ws = _lib.require().dc_w8a8_gemm_workspace_bytes(m, n, k, k, k)
    if torch.cuda.get_device_properties(gpu).multi_processor_count == 256:
        assert _int8.gemm_kernel(m, n, k) == (kernel, slices)
        assert ws == (slices * m * n * 4 if slices > 1 else 0)
    q, w, sx, sw = _qw(m, n, k, 14)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(14)) * 0.5).to(torch.bfloat16)
    ref = OG.rescale(OG.int_mm(q.numpy(), w.numpy()), sx.numpy(), sw.numpy(), np32(bias), DT[dtype])
    q, w, sx, sw, bias = q.to(gpu), w.to(gpu), sx.to(gpu), sw.to(gpu), bias.to(gpu)
    split = _int8._gemm(q, w, sx, sw, bias, dtype)
    assert np.array_equal(np32(split).view(np.uint32), ref.view(np.uint32))
    assert torch.equal(split, _gemm_unsplit(q, w, sx, sw, bias, dtype))
    for _ in range(4):
        assert torch.equal(_int8._gemm(q, w, sx, sw, bias, dtype), split)


# grouped launches (dc_w8a8_gemm_grouped): (row counts, N, K); M = 0 problems
# are skipped, ragged M and N exercise the partial tiles
GROUPS = [([4096, 512], 3072, 3072), ([1000, 77, 300], 1000, 512), ([257, 0, 513, 64], 640, 256),
          ([512, 4096], 3072, 1024)]


@pytest.mark.parametrize("ms,n,k", GROUPS)
@pytest.mark.parametrize("dtype,bias_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, None),
                                              (torch.float32, torch.float32), (torch.int32, None)])
def test_grouped_gemm_equals_separate_calls(gpu, ms, n, k, dtype, bias_dtype):
    """One grouped launch over problems with their own activations, weights,
    scales and biases: every output bit-identical to dc_w8a8_gemm on that
    problem alone (and the first one to the oracle)."""
    items, seps = [], []
    for i, m in enumerate(ms):
        q, w, sx, sw = _qw(m, n, k, 40 + i)
        b = (torch.randn(n, generator=torch.Generator().manual_seed(50 + i)) * 0.5).to(bias_dtype) \
            if bias_dtype is not None else None
        q, w, sx, sw = q.to(gpu), w.to(gpu), sx.to(gpu), sw.to(gpu)
        b = b.to(gpu) if b is not None else None
        items.append((q, w, sx, sw, b))
        seps.append(_gemm_unsplit(q, w, sx, sw, b, dtype) if dtype != torch.int32 else _int8.int_mm(q, w))
    outs = _int8._gemm_grouped(items, dtype)
    for m, out, sep in zip(ms, outs, seps):
        assert out.shape == (m, n) and out.dtype == dtype
        assert torch.equal(out, sep)
    q, w, sx, sw, b = (t.cpu() if t is not None else None for t in items[0])
    acc = OG.int_mm(q.numpy(), w.numpy())
    if dtype == torch.int32:
        assert np.array_equal(outs[0].cpu().numpy(), acc)
    else:
        ref = OG.rescale(acc, sx.numpy(), sw.numpy(), np32(b) if b is not None else None, DT[dtype])
        assert np.array_equal(np32(outs[0]).view(np.uint32), ref.view(np.uint32))


def test_grouped_gemm_strided_rows(gpu):
    """Row strides above K (a column slice of wider activations and weights)."""
    k, n = 512, 384
    a_wide = torch.randint(-127, 128, (700, 1024), dtype=torch.int8, device=gpu)
    w_wide = torch.randint(-127, 128, (n, 768), dtype=torch.int8, device=gpu)
    sx, sw = torch.rand(700, device=gpu) * 1e-2, torch.rand(n, device=gpu) * 1e-3
    items = [(a_wide[:300, :k], w_wide[:, :k], sx[:300], sw, None), (a_wide[300:, 256:256 + k], w_wide[:, 128:128 + k],
                                                                    sx[300:], sw, None)]
    outs = _int8._gemm_grouped(items, torch.bfloat16)
    for (q, w, x_s, w_s, _), out in zip(items, outs):
        assert torch.equal(out, _gemm_unsplit(q.contiguous(), w.contiguous(), x_s.contiguous(), w_s, None,
                                              torch.bfloat16))


def test_group_plan_and_layers(gpu):
    """The plan groups FLUX's double-block pairs whose 256 x 256 tiles add no
    round (qkv, proj, MLP down on 256 CUs) and not MLP up; grouped W8A8 layers
    equal the layers run one by one."""
    if torch.cuda.get_device_properties(gpu).multi_processor_count == 256:
        assert _int8.gemm_group_plan([4096, 512], 9216, 3072)
        assert _int8.gemm_group_plan([4096, 512], 3072, 3072)
        assert _int8.gemm_group_plan([4096, 512], 3072, 12288)
        assert not _int8.gemm_group_plan([4096, 512], 12288, 3072)
    assert not _int8.gemm_group_plan([4096], 3072, 3072)
    assert not _int8.gemm_group_plan([4096, 512], 3072, 3000)
    torch.manual_seed(3)
    la = _int8.Int8Linear.from_linear(nn.Linear(3072, 3072).to(gpu).to(torch.bfloat16), 256)
    lb = _int8.Int8Linear.from_linear(nn.Linear(3072, 3072).to(gpu).to(torch.bfloat16), 256)
    xa = torch.randn(2, 2048, 3072, device=gpu).to(torch.bfloat16)
    xb = torch.randn(1, 512, 3072, device=gpu).to(torch.bfloat16)
    ya, yb = _int8.linear_group([la, lb], [xa, xb])
    assert torch.equal(ya, la(xa)) and torch.equal(yb, lb(xb))


GATED = [([4096, 512], 3072, 3072), ([300], 1000, 768), ([257, 0, 513, 64], 640, 256), ([4608], 3072, 1024)]


def _res_gate(m, n, dtype, gpu, seed):
    g = torch.Generator().manual_seed(seed)
    return ((torch.randn(m, n, generator=g) * 2).to(dtype).to(gpu), (torch.randn(n, generator=g)).to(dtype).to(gpu))


@pytest.mark.parametrize("ms,n,k", GATED)
@pytest.mark.parametrize("dtype,bias_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, None),
                                              (torch.float32, torch.float32), (torch.bfloat16, torch.float32)])
def test_gated_grouped_gemm_equals_torch_ops(gpu, ms, n, k, dtype, bias_dtype):
    """dc_w8a8_gemm_grouped_gated: each output bit-identical to torch's
    res + gate * y on the plain grouped GEMM's y (FLUX's x + gate * out,
    reference flux_dit.py:298-301, 336), full and partial tiles."""
    items, gates = [], []
    for i, m in enumerate(ms):
        q, w, sx, sw = _qw(m, n, k, 60 + i)
        b = (torch.randn(n, generator=torch.Generator().manual_seed(70 + i)) * 0.5).to(bias_dtype) \
            if bias_dtype is not None else None
        items.append((q.to(gpu), w.to(gpu), sx.to(gpu), sw.to(gpu), b.to(gpu) if b is not None else None))
        gates.append(_res_gate(m, n, dtype, gpu, 80 + i))
    ys = _int8._gemm_grouped(items, dtype)
    outs = _int8._gemm_grouped(items, dtype, gates)
    for m, y, out, (res, gate) in zip(ms, ys, outs, gates):
        assert out.shape == (m, n) and out.dtype == dtype
        assert torch.equal(out, res + gate * y)


def test_gated_gemm_in_place_and_strided_residual(gpu):
    """The residual may be the output itself (in place), or a strided view."""
    n, k, dtype = 1024, 512, torch.bfloat16
    q, w, sx, sw = (t.to(gpu) for t in _qw(1000, n, k, 90))
    bias = torch.randn(n, device=gpu).to(dtype)
    y = _int8._gemm_grouped([(q, w, sx, sw, bias)], dtype)[0]
    res, gate = _res_gate(1000, n, dtype, gpu, 91)
    want = res + gate * y
    so = _lib.require()
    prob = _lib.GemmProblem(q.data_ptr(), q.stride(0), w.data_ptr(), w.stride(0), sx.data_ptr(), sw.data_ptr(),
                            bias.data_ptr(), res.data_ptr(), n, 1000)
    gt = _lib.GemmGate(res.data_ptr(), n, gate.data_ptr())
    rc = so.dc_w8a8_gemm_grouped_gated(ctypes.byref(prob), ctypes.byref(gt), 1, n, k, _lib.BF16, _lib.BF16,
                                       _lib.stream_ptr(gpu))
    assert rc == 0, so.dc_last_error()
    assert torch.equal(res, want)
    wide = torch.randn(1000, 2 * n, device=gpu).to(dtype)
    out = _int8._gemm_grouped([(q, w, sx, sw, bias)], dtype, [(wide[:, 64:64 + n], gate)])[0]
    assert torch.equal(out, wide[:, 64:64 + n] + gate * y)


def test_matmul_quantized_gated_layers(gpu):
    """The layer-level helper: fused (grouped pair; one layer whose plan is
    the DMA-fed kernel) and fallback (a plan that is not) all equal the
    reference's x + gate * layer(x') torch ops, with FLUX's [B, L, N]
    residual and [B, 1, N] gate."""
    torch.manual_seed(5)
    bf = torch.bfloat16
    la = _int8.Int8Linear.from_linear(nn.Linear(3072, 3072).to(gpu).to(bf), 256)
    lb = _int8.Int8Linear.from_linear(nn.Linear(3072, 3072).to(gpu).to(bf), 256)
    xa, xb = torch.randn(1, 4096, 3072, device=gpu).to(bf), torch.randn(1, 512, 3072, device=gpu).to(bf)
    ra, rb = torch.randn(1, 4096, 3072, device=gpu).to(bf), torch.randn(1, 512, 3072, device=gpu).to(bf)
    ga, gb = torch.randn(1, 1, 3072, device=gpu).to(bf), torch.randn(1, 1, 3072, device=gpu).to(bf)
    qa = _int8.quantize_activation(xa.reshape(-1, 3072), 256)
    qb = _int8.quantize_activation(xb.reshape(-1, 3072), 256)
    assert _int8.gemm_group_plan([4096, 512], 3072, 3072) or \
        torch.cuda.get_device_properties(gpu).multi_processor_count != 256
    ya, yb = _int8.matmul_quantized_gated([(la, *qa, ra, ga), (lb, *qb, rb, gb)], bf)
    assert torch.equal(ya.view(ra.shape), ra + ga * la(xa)) and torch.equal(yb.view(rb.shape), rb + gb * lb(xb))
    # one layer: FLUX's linear2 shape, whose plan is the DMA-fed kernel (fused),
    # and the 512-row text layer, whose plan is not (GEMM, then torch ops)
    lc = _int8.Int8Linear.from_linear(nn.Linear(15360, 3072).to(gpu).to(bf), 256)
    xc = torch.randn(1, 4608, 15360, device=gpu).to(bf)
    rc, gc = torch.randn(1, 4608, 3072, device=gpu).to(bf), torch.randn(1, 1, 3072, device=gpu).to(bf)
    if torch.cuda.get_device_properties(gpu).multi_processor_count == 256:
        assert _int8.gemm_plan(4608, 3072, 15360) == "dma_256x256" and _int8.gemm_plan(512, 3072, 3072) != "dma_256x256"
    qc = _int8.quantize_activation(xc.reshape(-1, 15360), 256)
    (y1,) = _int8.matmul_quantized_gated([(lc, *qc, rc, gc)], bf)
    assert torch.equal(y1.view(rc.shape), rc + gc * lc(xc))
    (y2,) = _int8.matmul_quantized_gated([(lb, *qb, rb, gb)], bf)
    assert torch.equal(y2.view(rb.shape), rb + gb * lb(xb))
    # a gate per sample (B = 2) is not one row: the torch ops, same values
    x2, r2 = torch.randn(2, 256, 3072, device=gpu).to(bf), torch.randn(2, 256, 3072, device=gpu).to(bf)
    g2 = torch.randn(2, 1, 3072, device=gpu).to(bf)
    q2 = _int8.quantize_activation(x2.reshape(-1, 3072), 256)
    (y3,) = _int8.matmul_quantized_gated([(la, *q2, r2, g2)], bf)
    assert torch.equal(y3.view(r2.shape), r2 + g2 * la(x2))


# Problems of whole 256 x 256 tiles with 16-bit outputs that take several
# rounds of DMA-fed workgroups, whole and ragged: 992 tiles end on a short
# round, 756 leave 12 CUs one tile fewer; 768 tiles of K = 3072 are FLUX's
# image MLP up.
MULTI_ROUND = [(4096, 15872, 512), (2304, 21504, 512), (4096, 12288, 3072)]


def _int32_then_rescale(q, w, sx, sw, bias, dtype):
    """The same GEMM as an int32 product followed by dc_rescale: the fused
    epilogue's contract (reference ``_int8.py:313-323``)."""
    return _int8.rescale(_int8.int_mm(q, w), sx, sw, bias, dtype)


@pytest.mark.parametrize("mnk", MULTI_ROUND)
@pytest.mark.parametrize("dtype,bias_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, None),
                                              (torch.float16, torch.float32)])
def test_multi_round_gemm_bit_exact(gpu, mnk, dtype, bias_dtype):
    """Several rounds of 256 x 256 tiles: bit for bit the int32 product +
    rescale, the first rows the oracle, and the same bits on every call."""
    m, n, k = mnk
    q, w, sx, sw = _qw(m, n, k, 21)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(21)) * 0.5).to(bias_dtype) \
        if bias_dtype is not None else None
    rows = 96   # a slice of rows against the oracle (the whole product is minutes of CPU)
    ref = OG.rescale(OG.int_mm(q[:rows].numpy(), w.numpy()), sx[:rows].numpy(), sw.numpy(),
                     np32(bias) if bias is not None else None, DT[dtype])
    q, w, sx, sw = q.to(gpu), w.to(gpu), sx.to(gpu), sw.to(gpu)
    bias = bias.to(gpu) if bias is not None else None
    if torch.cuda.get_device_properties(gpu).multi_processor_count == 256:
        assert _int8.gemm_plan(m, n, k) == "dma_256x256"
    y = _gemm_unsplit(q, w, sx, sw, bias, dtype)
    assert np.array_equal(np32(y[:rows]).view(np.uint32), ref.view(np.uint32))
    assert torch.equal(y, _int32_then_rescale(q, w, sx, sw, bias, dtype))
    for _ in range(3):
        assert torch.equal(_gemm_unsplit(q, w, sx, sw, bias, dtype), y)


@pytest.mark.parametrize("ms,n,k,dtype,bias_dtype", [([4096, 512], 9216, 3072, torch.bfloat16, torch.bfloat16),
                                                     ([1024, 4096, 512], 4096, 512, torch.float16, None),
                                                     ([512, 2048], 32768, 768, torch.bfloat16, torch.float32)])
def test_multi_round_grouped_gemm_bit_exact(gpu, ms, n, k, dtype, bias_dtype):
    """Grouped launches of more than one round (FLUX's img + txt qkv is 648
    tiles): every problem equals its int32 product + rescale bit for bit;
    the first rows of the first problem equal the oracle."""
    items = []
    for i, m in enumerate(ms):
        q, w, sx, sw = _qw(m, n, k, 30 + i)
        b = (torch.randn(n, generator=torch.Generator().manual_seed(35 + i)) * 0.5).to(bias_dtype) \
            if bias_dtype is not None else None
        items.append((q, w, sx, sw, b))
    q, w, sx, sw, b = items[0]
    ref = OG.rescale(OG.int_mm(q[:64].numpy(), w.numpy()), sx[:64].numpy(), sw.numpy(),
                     np32(b) if b is not None else None, DT[dtype])
    items = [tuple(t.to(gpu) if t is not None else None for t in it) for it in items]
    outs = _int8._gemm_grouped(items, dtype)
    assert np.array_equal(np32(outs[0][:64]).view(np.uint32), ref.view(np.uint32))
    for (q, w, sx, sw, b), out in zip(items, outs):
        assert torch.equal(out, _int32_then_rescale(q, w, sx, sw, b, dtype))
    assert all(torch.equal(a, c) for a, c in zip(_int8._gemm_grouped(items, dtype), outs))


# The DMA-fed kernel's tiles at whole and ragged edges, with fewer k stages
# than the ring holds, as many, and one or two more; the last ones leave K % 64
# or its depth to the register-staged kernel. The tile each case runs on is the
# one before it in the list (256 CUs).
DMA_EDGES = [("dma_64x64", [(1, 8, 128), (64, 64, 256), (65, 130, 384), (154, 2560, 512), (129, 513, 128)]),
             ("dma_64x128", [(512, 3071, 640), (500, 3072, 1280), (1000, 2048, 256)]),
             ("dma_128x128_8w", [(1025, 2049, 384), (2048, 1281, 512)]),
             ("dma_128x128", [(2047, 3840, 128), (2000, 3840, 384), (7904, 1920, 640), (2560, 16384, 256),
                              (2500, 16380, 384)]),
             ("dma_192x256", [(4096, 3072, 1024), (4095, 3001, 384)]),
             ("dma_256x256", [(2304, 6144, 1024), (2500, 6140, 1536)]),
             ("dma_128x128_k64", [(1, 4, 64), (130, 260, 192), (8192, 1280, 320), (3000, 1284, 576), (100, 100, 960)]),
             ("128x128", [(257, 300, 1088), (300, 200, 48)])]


@pytest.mark.parametrize("mnk,kernel", [(mnk, kernel) for kernel, shapes in DMA_EDGES for mnk in shapes])
def test_dma_tiles_bit_exact(gpu, mnk, kernel):
    """Every tile and edge against the vendor's int32 product and the rescale
    expression in torch ops, from operands that are slices of wider rows
    (strides above K) into an output of every type."""
    m, n, k = mnk
    if torch.cuda.get_device_properties(gpu).multi_processor_count == 256:
        assert _int8.gemm_kernel(m, n, k, k + 32, k + 32) == (kernel, 1)
    g = torch.Generator(device=gpu).manual_seed(m * 7 + n + k)
    wide = k + 32
    q = torch.randint(-128, 128, (m, wide), generator=g, device=gpu, dtype=torch.int8)[:, 16:16 + k]
    w = torch.randint(-128, 128, (n, wide), generator=g, device=gpu, dtype=torch.int8)[:, 16:16 + k]
    sx, sw = (torch.rand(i, generator=g, device=gpu) * 1e-3 for i in (m, n))
    bias = torch.randn(n, generator=g, device=gpu)
    # the vendor product needs M > 16 and sizes that are multiples of 8
    mp, np_ = (max(m, 32) + 7) // 8 * 8, (n + 7) // 8 * 8
    qp, wp = torch.zeros(mp, k, device=gpu, dtype=torch.int8), torch.zeros(np_, k, device=gpu, dtype=torch.int8)
    qp[:m], wp[:n] = q, w
    acc = torch._int_mm(qp, wp.t())[:m, :n]
    assert torch.equal(_int8._gemm(q, w, None, None, None, torch.int32), acc)
    for dtype, b in ((torch.bfloat16, bias.bfloat16()), (torch.float16, None), (torch.float32, bias)):
        y = (acc.float() * (sx.unsqueeze(-1) * sw)).to(dtype)
        if b is not None:
            y = y + b.to(dtype)
        assert torch.equal(_int8._gemm(q, w, sx, sw, b, dtype), y), dtype


@pytest.mark.parametrize("mnk", [(64, 3072, 12288), (100, 3069, 8192), (1, 16, 8704), (256, 3072, 15360)])
def test_dma_split_k_bit_exact(gpu, mnk):
    """Few rows over a deep K: the k slices (in the workspace the library asks
    for) equal the unsplit call."""
    m, n, k = mnk
    q, w, sx, sw = (t.to(gpu) for t in _qw(m, n, k, 17))
    bias = torch.randn(n, device=gpu).bfloat16()
    assert _lib.require().dc_w8a8_gemm_workspace_bytes(m, n, k, k, k) >= 4 * m * n * 4
    for dtype, b in ((torch.bfloat16, bias), (torch.float32, None)):
        assert torch.equal(_int8._gemm(q, w, sx, sw, b, dtype), _gemm_unsplit(q, w, sx, sw, b, dtype))


@pytest.mark.parametrize("shape,n,group,dtype,bias", [
    ((154, 2048), 2560, 256, torch.float16, None), ((2, 77, 768), 640, 256, torch.bfloat16, torch.float32),
    ((1, 320), 4, 0, torch.float32, torch.float32), ((320,), 17, 0, torch.float16, torch.float16),
    ((64, 12288), 3072, 256, torch.bfloat16, torch.bfloat16), ((3, 0, 256), 64, 256, torch.float16, None),
    ((33, 48), 100, 0, torch.float16, torch.float16)])
def test_linear_one_call_equals_two(gpu, shape, n, group, dtype, bias):
    """Int8Linear.forward (one library call) against quantize_activation and
    matmul_quantized, on whole and strided inputs and strided weights."""
    k = shape[-1]
    torch.manual_seed(n)
    m = _int8.Int8Linear(k, n, bias=bias is not None, group=group, device=gpu)
    m.weight.copy_(torch.randint(-127, 128, (n, k), device=gpu))
    m.scale_bits.copy_((torch.rand(n, device=gpu) * 1e-3).view(torch.int32))
    if bias is not None:
        m.bias = nn.Parameter(torch.randn(n, device=gpu).to(bias), requires_grad=False)
    x = torch.randn(*shape, device=gpu).to(dtype)
    wide = torch.randn(*shape[:-1], k + 16, device=gpu).to(dtype)
    odd = torch.randn(*shape[:-1], k + 1, device=gpu).to(dtype)
    for xi in (x, wide[..., 8:8 + k], odd[..., :k], torch.stack((x, x), -1)[..., 0]):
        q, s = _int8.quantize_activation(xi.reshape(-1, k), group)
        want = m.matmul_quantized(q, s, dtype).view(*xi.shape[:-1], n)
        y = m(xi)
        assert y.shape == want.shape and y.dtype == dtype and torch.equal(y, want)
    store = torch.empty(n, k + 64, device=gpu, dtype=torch.int8)
    store[:, 32:32 + k] = m.weight
    want = m(x)
    m.weight = store[:, 32:32 + k]
    assert torch.equal(m(x), want)


def test_linear_one_call_refusals(gpu):
    """What the two calls refuse, the one call refuses: a width that is not
    the layer's, a scratch too small, a bias of another type."""
    m = _int8.Int8Linear(256, 64, group=256, device=gpu)
    with pytest.raises((RuntimeError, ValueError)):
        m(torch.randn(4, 512, device=gpu).half())
    so = _lib.require()
    x, w = torch.randn(4, 256, device=gpu).half(), torch.zeros(64, 256, device=gpu, dtype=torch.int8)
    sw, out, scratch = torch.ones(64, device=gpu), torch.empty(4, 64, device=gpu).half(), \
        torch.empty(4096, device=gpu, dtype=torch.uint8)
    need = so.dc_w8a8_linear_scratch_bytes(4, 64, 256, 256)
    args = lambda k, out_dt, nb: (x.data_ptr(), _lib.F16, 4, k, 256, 256, w.data_ptr(), 256, sw.data_ptr(), None,
                                  _lib.NONE, out.data_ptr(), out_dt, 64, 64, scratch.data_ptr(), nb,
                                  _lib.stream_ptr(gpu))
    assert so.dc_w8a8_linear(*args(256, _lib.F16, need)) == 0
    assert so.dc_w8a8_linear(*args(256, _lib.F16, need - 1)) != 0
    assert so.dc_w8a8_linear(*args(250, _lib.F16, 4096)) != 0
    assert so.dc_w8a8_linear(*args(256, _lib.I32, 4096)) != 0
    m.bias = nn.Parameter(torch.zeros(64, device=gpu, dtype=torch.float64), requires_grad=False)
    with pytest.raises(TypeError):
        m(x)


@pytest.mark.parametrize("k,group", [(256, 256), (512, 0), (48, 0)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_one_row_of_any_row_stride(gpu, k, group, dtype):
    """A [1, K] input is taken whatever its row stride (a transposed column's
    is 1, an expanded vector's may be anything below K, an odd-width buffer's
    is misaligned), by the layer and by the two calls alike."""
    m = _int8.Int8Linear(k, 64, group=group, device=gpu)
    m.weight.copy_(torch.randint(-127, 128, (64, k), device=gpu))
    m.scale_bits.copy_((torch.rand(64, device=gpu) * 1e-3).view(torch.int32))
    x = torch.randn(1, k, device=gpu).to(dtype)
    wide = torch.zeros(3, k + 1, device=gpu, dtype=dtype)
    wide[0, :k] = x[0]
    want = m(x)
    for xi in (x.t().contiguous().t(), wide[:1, :k], torch.as_strided(x.clone(), (1, k), (0, 1)), x[0],
               wide[None, :1, :k]):
        assert torch.equal(m(xi).reshape(1, -1), want)
        q, s = _int8.quantize_activation(xi.reshape(-1, k) if xi.dim() != 2 else xi, group)
        assert torch.equal(m.matmul_quantized(q, s, dtype), want)


def test_forward_runs_an_overridden_matmul(gpu, monkeypatch):
    """A forward goes through a subclass's or a patched matmul_quantized, and
    through a patched quantize_activation."""
    class Doubled(_int8.Int8Linear):
        def matmul_quantized(self, q, s, dtype):
            return super().matmul_quantized(q, s, dtype) * 2

    m, sub = _int8.Int8Linear(256, 64, device=gpu), Doubled(256, 64, device=gpu)
    for layer in (m, sub):
        layer.weight.copy_(torch.arange(64 * 256, device=gpu).view(64, 256) % 255 - 127)
        layer.scale_bits.copy_(torch.full((64,), 1e-3, device=gpu).view(torch.int32))
    x = torch.randn(5, 256, device=gpu).half()
    assert torch.equal(sub(x), m(x) * 2)
    seen = []
    real = _int8.quantize_activation
    monkeypatch.setattr(_int8, "quantize_activation", lambda t, g: (seen.append(t.shape), real(t, g))[1])
    want = sub(x)
    assert torch.equal(m(x) * 2, want) and seen == [(5, 256)] * 2
