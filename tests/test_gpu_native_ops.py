"""The native operators (libdopt_torch.so, csrc/torch_ops.cpp) against the Python implementations
they replace in the dispatcher (act_lib.py, bn_lib.py, which call the same C ABI through ctypes):
every output bit for bit on the same inputs, the in-place running statistics included, and the
same error classes (ValueError for bad bits, RuntimeError for mismatched sizes). The operators'
numerics are pinned against the CPU oracle by the other GPU tests, which now run through these
kernels."""
import os

import pytest
import torch

import deep_optimization_amd  # noqa: F401
from deep_optimization_amd import _lib, _native, act_lib, bn_lib

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not os.path.exists(_native.LIB_PATH), reason="libdopt_torch.so not built")]
DEV = "cuda"
ops = torch.ops.act_lib


def same(a, b):
    if isinstance(a, torch.Tensor):
        assert a.dtype == b.dtype and a.shape == b.shape, (a.dtype, b.dtype, a.shape, b.shape)
        assert torch.equal(a.view(torch.uint8) if a.is_floating_point() else a,
                           b.view(torch.uint8) if b.is_floating_point() else b)
    elif isinstance(a, (tuple, list)):
        assert len(a) == len(b)
        for x, y in zip(a, b):
            same(x, y)
    else:
        assert a == b, (a, b)


def rnd(shape, seed, dtype=torch.bfloat16, scale=2.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(shape, generator=g, device=DEV) * scale).to(dtype)


@pytest.mark.parametrize("rounding", [0, 1, 2])
@pytest.mark.parametrize("bits", [1, 2, 4, 8])
def test_quant_pack_and_dequant(bits, rounding):
    x = rnd((3, 40, 256), bits + 10 * rounding)
    noise = torch.rand((3, 40, 256), generator=torch.Generator(device=DEV).manual_seed(1), device=DEV)
    args = (bits, 256, True, 2.5, True, rounding, noise if rounding == 1 else None, 7, 3, torch.float32)
    got, want = ops.quant_pack(x, *args), act_lib._quant_pack(x, *args)
    same(got, want)
    for dt in (torch.bfloat16, torch.float32):
        same(ops.dequant_unpack(*got, bits, 256, dt), act_lib._dequant_unpack(*got, bits, 256, dt))


@pytest.mark.parametrize("bits", [1, 2, 4, 8])
def test_tile_ops(bits):
    x = rnd((2, 8, 32, 48), bits, dtype=torch.float32)
    args = (bits, 256, False, 0.0, False, 0, None, 0, 0, torch.bfloat16)
    got, want = ops.quant_pack_tiles(x, *args), act_lib._quant_pack_tiles(x, *args)
    same(got, want)
    same(ops.dequant_unpack_tiles(*got, bits, 256, 2, 8, 32, 48, torch.bfloat16),
         act_lib._dequant_unpack_tiles(*got, bits, 256, 2, 8, 32, 48, torch.bfloat16))


@pytest.mark.parametrize("avg_alam,alam_bits", [(False, 0), (True, 2), (True, 4)])
def test_reference_schema_ops(avg_alam, alam_bits):
    x = rnd((4, 12, 256), alam_bits + 3)
    got = ops.quant_pack_triton(x, 2, 256, avg_alam, alam_bits, True, 3.0)
    want = act_lib._quant_pack_triton(x, 2, 256, avg_alam, alam_bits, True, 3.0)
    same(got, want)
    same(ops.dequant_unpack_triton(*got, 2, 256, avg_alam, alam_bits),
         act_lib._dequant_unpack_triton(*got, 2, 256, avg_alam, alam_bits))


@pytest.mark.parametrize("relu6", [False, True])
@pytest.mark.parametrize("bits", [1, 2])
def test_relu_ops(bits, relu6):
    x = rnd((4, 16, 14, 14), bits + 2 * relu6, scale=4.0)
    got = ops.relu_fwd_fused_pack(x, not relu6, relu6, bits, 64)
    want = act_lib._relu_fwd_fused_pack(x, not relu6, relu6, bits, 64)
    same(got, want)
    dy = rnd(x.shape, 9, dtype=torch.float32)
    same(ops.relu_bwd_fused_unpack(got[1], dy, bits, got[2], got[3], 64),
         act_lib._relu_bwd_fused_unpack(got[1], dy, bits, got[2], got[3], 64))


@pytest.mark.parametrize("kind", [_lib.BN_QUANT, _lib.BN_RELU_QUANT, _lib.BN_RELU6_QUANT])
@pytest.mark.parametrize("stats", ["f32", "none", "bf16"])
def test_batchnorm_layer_ops(kind, stats):
    N, C, H, W = 8, 32, 28, 28
    x = rnd((N, C, H, W), kind, scale=1.5)
    w = torch.rand(C, device=DEV) + 0.5
    b = torch.randn(C, device=DEV)
    if stats == "none":
        rm_a = rv_a = rm_b = rv_b = torch.empty(0, device=DEV)
    else:
        dt = torch.float32 if stats == "f32" else torch.bfloat16
        rm_a, rv_a = torch.randn(C, device=DEV).to(dt), (torch.rand(C, device=DEV) + 0.5).to(dt)
        rm_b, rv_b = rm_a.clone(), rv_a.clone()
    got = ops.bn_train_fwd(x, w, b, rm_a, rv_a, 0.1, 256, 2, kind)
    want = bn_lib._bn_train_fwd(x, w, b, rm_b, rv_b, 0.1, 256, 2, kind)
    same(got, want)
    same((rm_a, rv_a), (rm_b, rv_b))
    y, packed, rp, scale, xmin, mean, var = got
    dy = rnd(y.shape, 5)
    relu_packed = rp if kind != _lib.BN_QUANT else None
    same(ops.bn_train_bwd(packed, relu_packed, dy, scale, xmin, w, var, 256, 2, kind),
         bn_lib._bn_train_bwd(packed, relu_packed, dy, scale, xmin, w, var, 256, 2, kind))


def test_error_classes():
    x = torch.zeros(1, 1, 256, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(ValueError):
        ops.quant_pack(x, 3, 256, False, 0.0, False, 0, None, 0, 0, torch.float32)
    with pytest.raises(ValueError):
        ops.quant_pack_triton(x, 5, 256, False, 0, False, 0.0)
    with pytest.raises(RuntimeError, match="shape"):
        ops.quant_pack(x, 2, 128, False, 0.0, False, 0, None, 0, 0, torch.float32)
    with pytest.raises(RuntimeError, match="noise"):
        ops.quant_pack(x, 2, 256, False, 0.0, False, 1, None, 0, 0, torch.float32)
    with pytest.raises(RuntimeError, match="alam_bits"):
        ops.quant_pack_triton(x, 2, 256, True, 3, False, 0.0)
    p, s, m = ops.quant_pack(x, 2, 256, False, 0.0, False, 0, None, 0, 0, torch.float32)
    with pytest.raises(RuntimeError, match="packed holds"):
        ops.dequant_unpack(p[:, :8], s, m, 2, 256, torch.bfloat16)
    with pytest.raises(RuntimeError, match="one per channel"):
        X = torch.zeros(2, 4, 8, 8, device=DEV)
        ops.bn_train_fwd(X, torch.ones(3, device=DEV), torch.zeros(4, device=DEV), torch.empty(0, device=DEV),
                         torch.empty(0, device=DEV), 0.1, 128, 2, _lib.BN_QUANT)
    with pytest.raises(RuntimeError, match="relu"):
        ops.relu_fwd_fused_pack(torch.zeros(2, 64, device=DEV), False, False, 1, 64)


def planes(kind, x, w):
    """the layouts fp8_linear takes in place and packs: [rows, K] row major, a column-major view, a misaligned slice"""
    K = x.shape[1]
    if kind == "row":
        return x.contiguous(), w.contiguous().t()
    if kind == "col":
        return x.t().contiguous().t(), w.t().contiguous()
    return x[:, 3:K - 2], w[:, 3:K - 2].t()


@pytest.mark.parametrize("kind", ["row", "col", "slice"])
@pytest.mark.parametrize("M,N,K", [(1, 8, 16), (5, 130, 250), (129, 64, 512), (0, 64, 64), (64, 0, 64)])
def test_fp8_ops(M, N, K, kind):
    a, b = planes(kind, rnd((M, K), 1).to(torch.float8_e4m3fn), rnd((N, K), 2).to(torch.float8_e4m3fn))
    same(ops.fp8_linear(a, b, 0.125), act_lib._fp8_linear(a, b, 0.125))
    if K % 16 == 0 and kind == "row":
        same(ops.fp8_gemm_nt(a, b.t(), 0.125), act_lib._fp8_gemm_nt(a, b.t(), 0.125))


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(8, 16, 5), (264, 520, 333), (256, 512, 700), (768, 256, 0)])
def test_dw_gemm_any(M, N, K, out_dtype):
    """... and, with both feature counts multiples of 256, dw_gemm on the same x_hat."""
    from deep_optimization_amd import dw_lib

    dy, x = rnd((K, M), 1), rnd((K, N), 2)
    for bias in (True, False):
        got = ops.dw_gemm_any(dy, x, bias, out_dtype)
        same(got, dw_lib._dw_gemm_any(dy, x, bias, out_dtype))
        if M % 256 == 0 and N % 256 == 0:
            same(got, dw_lib._dw_gemm(dy, x, None, None, None, N, 0, 0, bias, out_dtype))
    same(ops.dw_gemm_any(dy.t().contiguous().t(), x, True, out_dtype), ops.dw_gemm_any(dy, x, True, out_dtype))


@pytest.mark.parametrize("shape,g", [((2, 8, 32, 48), 256), ((2, 16, 14, 14), 64), ((4, 12, 256), 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_silu_and_gelu_ops(shape, g, dtype):
    for bits in (1, 2, 4, 8):
        x, dy = rnd(shape, bits, dtype), rnd(shape, bits + 9, dtype)
        for alam in ((False, 0), (True, 1)):
            got = ops.silu_fwd_quan_pack(x, bits, g, *alam, False)
            same(got, act_lib._silu_fwd_quan_pack(x, bits, g, *alam, False))
            y, packed, scale, xmin, N, G, nh, nw, pe, re = got
            bwd = (packed, dy, scale, xmin, bits, N, G, g, False, nh, nw, pe, re, *alam)
            same(ops.silu_bwd_fused_dequan_unpack(*bwd), act_lib._silu_bwd_fused_dequan_unpack(*bwd))
            same(ops.silu_bwd_fused_dequan_unpack(packed, dy.transpose(-1, -2).contiguous().transpose(-1, -2), *bwd[2:]),
                 act_lib._silu_bwd_fused_dequan_unpack(*bwd))
        y, packed, scale, xmin, N, G = ops.gelu_fwd_fused_quan_pack(x, bits, g)
        bwd = (packed, dy, scale, xmin, bits, N, G, g)
        same(ops.gelu_bwd_fused_dequan_unpack(*bwd), act_lib._gelu_bwd_fused_dequan_unpack(*bwd))


@pytest.mark.parametrize("name,args,error", [
    ("silu_fwd_quan_pack", ((4, 8, 256), 3, 256, False, 0, False), ValueError),
    ("silu_fwd_quan_pack", ((4, 8, 256), 2, 256, True, 2, False), NotImplementedError),
    ("silu_fwd_quan_pack", ((4, 8, 256), 2, 192, False, 0, False), RuntimeError),
    ("silu_fwd_quan_pack", ((4, 8, 32, 32), 2, 130, False, 0, False), RuntimeError),
    ("silu_fwd_quan_pack", ((4, 8, 33, 33), 2, 130, False, 0, False), RuntimeError),
])
def test_silu_errors(name, args, error):
    """the classes that the Python implementations raise, on calls that the checks before any launch refuse"""
    x = rnd(args[0], 1)
    for f in (getattr(ops, name), getattr(act_lib, "_" + name)):
        with pytest.raises(error):
            f(x, *args[1:])


def test_refused_operands():
    a8, b8 = (rnd((64, 32), i).to(torch.float8_e4m3fn) for i in (1, 2))
    x = rnd((64, 32), 3)
    packed, s = torch.zeros((8, 16), dtype=torch.int32, device=DEV), torch.ones(8, device=DEV)
    from deep_optimization_amd import dw_lib

    bad = [(ops.fp8_linear, act_lib._fp8_linear, (a8, b8, 1.0)), (ops.fp8_linear, act_lib._fp8_linear, (x, a8.t(), 1.0)),
           (ops.fp8_gemm_nt, act_lib._fp8_gemm_nt, (a8, b8.t(), 1.0)),
           (ops.fp8_gemm_nt, act_lib._fp8_gemm_nt, (a8[:, :24], b8[:, :24], 1.0)),
           (ops.dw_gemm_any, dw_lib._dw_gemm_any, (x.float(), x, True, torch.float32)),
           (ops.dw_gemm_any, dw_lib._dw_gemm_any, (x, x[:32], True, torch.float32)),
           (ops.dw_gemm_any, dw_lib._dw_gemm_any, (x, x, True, torch.float16)),
           (ops.dw_gemm_any, dw_lib._dw_gemm_any, (x, x[:, :12], True, torch.float32)),
           (ops.gelu_bwd_fused_dequan_unpack, act_lib._gelu_bwd_fused_dequan_unpack, (packed, x, s, s, 2, 4, 4, 256)),
           (ops.gelu_bwd_fused_dequan_unpack, act_lib._gelu_bwd_fused_dequan_unpack,
            (packed, x, s, s.bfloat16(), 2, 4, 2, 256))]
    for native, python, args in bad:
        for f in (native, python):
            with pytest.raises(RuntimeError):
                f(*args)


@pytest.mark.parametrize("bits", [1, 2, 4, 8])
@pytest.mark.parametrize("g", [64, 128, 256, 512, 1024])
@pytest.mark.parametrize("N,G", [(1, 1), (3, 7), (5, 67)])
def test_cast_quant_pack(bits, g, N, G):
    """One call equals the cast followed by quant_pack, bit for bit, and the Python implementation: values over the
    whole exponent range, constant groups, infinities, NaN and signed zeros among them."""
    x = rnd((N, G, g), bits + g, dtype=torch.float32)
    x[0, 0, ::3] *= 1e-30
    x[-1, -1] = 1.5
    if N > 1:
        x[1, 0, 5], x[1, 1, 7], x[1, 2, 9] = float("inf"), float("-inf"), float("nan")
        x[1, 3, ::2], x[1, 4] = -0.0, 3.4e38
        x[2, 0] = torch.exp2(torch.linspace(-140.0, 120.0, g, device=DEV))
    for clamp, squash, sdt in ((True, True, torch.bfloat16), (False, True, torch.float32), (True, False, torch.bfloat16),
                               (False, False, torch.float32)):
        got = ops.cast_quant_pack(x, bits, g, clamp, 2.5, squash, sdt)
        same(got, act_lib._cast_quant_pack(x, bits, g, clamp, 2.5, squash, sdt))
        x16 = x.to(torch.bfloat16)
        nan = x16.isnan()
        assert torch.equal(nan, got[0].isnan())
        same(got[0].masked_fill(nan, 0.0), x16.masked_fill(nan, 0.0))
        want = ops.quant_pack(x16, bits, g, clamp, 2.5, squash, 0, None, 0, 0, sdt)
        for i, (a, b) in enumerate(zip(got[1:], want)):
            if i == 0:
                same(a, b)
            else:  # a group of NaN: whatever its NaN's bits
                assert torch.equal(a.isnan(), b.isnan())
                same(torch.nan_to_num(a, 0.0), torch.nan_to_num(b, 0.0))


@pytest.mark.parametrize("shape,bits", [((4, 50, 384), 2), ((5, 768), 1), ((3, 7, 128), 8), ((3, 7, 100), 2)])
def test_linear_layer_fp32_input(shape, bits):
    """The compressed Linear layer on an fp32 input under autocast (one kernel casts and quantizes; a padded one casts
    first) saves and returns what it does on the input cast beforehand; a transposed input too."""
    from deep_optimization_amd.controller import layer_group_meta
    from deep_optimization_amd.modules.ops import _DOLinear

    meta = {"l": {"bits": bits, "pack_only": False, "AVG_ALAM": False, "ALAM_BITS": 0, "DIVISION": None,
                  **layer_group_meta(shape, bits)}}
    w = rnd((256, shape[-1]), 5, torch.float32)
    bias = rnd((256,), 6, torch.float32)
    base = rnd(shape, 7, torch.float32)
    if len(shape) == 3:
        views = (base, base.transpose(0, 1).contiguous().transpose(0, 1))
    else:
        views = (base, base.t().contiguous().t())
    for view in views:
        out = []
        for x in (view.to(torch.bfloat16), view):  # (the cast keeps the strides, and with them the product's kernel)
            x = x.detach().requires_grad_(True)
            wi, bi = w.clone().requires_grad_(True), bias.clone().requires_grad_(True)
            with torch.autocast("cuda", dtype=torch.bfloat16):
                y = _DOLinear.apply(x, wi, 3.0, "l", meta, None, bi)
            y.backward(rnd(y.shape, 8))
            out.append(tuple(t.detach().contiguous() for t in (y, x.grad.float(), wi.grad, bi.grad)))
        same(out[1], out[0])
