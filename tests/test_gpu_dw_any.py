"""The weight-gradient GEMM at ragged shapes: dopt_dw_gemm_any / act_lib::dw_gemm_any (any K, M and N
multiples of 8), the ragged instances behind act_lib::dw_gemm, and the Linear layer's route to them.

Bar: as for dw_gemm, |err| <= 1e-4 of the sum of the terms' magnitudes against float64 (fp32 accumulation);
bit-equal to dw_gemm where both take a shape; nothing outside the operands read, nothing outside the
results written.
"""
import pytest
import torch

import deep_optimization_amd  # noqa: F401
from deep_optimization_amd import _lib
from deep_optimization_amd.controller import layer_group_meta
from deep_optimization_amd.layers import DOLinear

pytestmark = pytest.mark.gpu
DEV = "cuda"
ops = torch.ops.act_lib

# tile edges (128, 256), one column chunk, K around a slab (32), a 64-token split unit, several splits
SHAPES = [(8, 8, 1), (8, 264, 31), (64, 64, 33), (120, 136, 63), (128, 128, 64), (136, 248, 65), (256, 320, 100),
          (384, 192, 999), (1000, 504, 1537), (248, 2056, 130), (1288, 1544, 200), (2056, 2104, 97), (768, 768, 985),
          (3072, 2816, 45), (192, 192, 9001)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("pad", [0, 16])
def test_ragged_shapes(M, N, K, pad):
    """Rows past K and the columns past M and N hold NaN; the results sit between sentinels."""
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    dy = torch.full((K + 2, M + pad), float("nan"), device=DEV, dtype=torch.bfloat16)
    x = torch.full((K + 2, N + pad), float("nan"), device=DEV, dtype=torch.bfloat16)
    dy[:K, :M] = torch.randn((K, M), generator=g, device=DEV).to(torch.bfloat16)
    x[:K, :N] = (torch.randn((K, N), generator=g, device=DEV) * 2).to(torch.bfloat16)
    L = _lib.lib()
    n = L.dopt_dw_gemm_any_workspace_floats(M, N, K)
    st = torch.cuda.current_stream().cuda_stream
    a, b = dy[:K, :M].double(), x[:K, :N].double()
    ref, mag = a.t() @ b, a.abs().t() @ b.abs()
    for f32, with_db in ((True, True), (True, False), (False, True)):
        ws = torch.full((n + 64,), 7.0, device=DEV)
        out = torch.full((M * N + 64,), 7.0, device=DEV, dtype=torch.float32 if f32 else torch.bfloat16)
        db = torch.full((M + 64,), 7.0, device=DEV)
        dw = out[32:32 + M * N]
        rc = L.dopt_dw_gemm_any(dy.data_ptr(), M + pad, x.data_ptr(), N + pad, M, N, K, ws.data_ptr(),
                                dw.data_ptr() if f32 else None, None if f32 else dw.data_ptr(),
                                db.data_ptr() if with_db else None, st)
        _lib.check(rc, "dw_gemm_any")
        err = (dw.view(M, N).double() - ref).abs()
        bar = 1e-4 * mag + 1e-6 + (0 if f32 else 2 ** -8 * ref.abs())
        assert bool((err <= bar).all()), float((err / (mag + 1e-30)).max())
        if with_db:
            assert bool(((db[:M].double() - a.sum(0)).abs() <= 1e-4 * a.abs().sum(0) + 1e-6).all())
        assert bool((out[:32] == 7).all()) and bool((out[32 + M * N:] == 7).all()) and bool((ws[n:] == 7).all())
        assert bool((db[M if with_db else 0:] == 7).all())


# one split (the last two: several), whole and ragged tiles of every shape
@pytest.mark.parametrize("M,N,K", [(8, 8, 1), (136, 248, 20), (264, 136, 40), (1288, 1544, 97), (2056, 2104, 65),
                                   (4096, 4096, 64), (1024, 768, 32), (384, 192, 999), (768, 768, 985)])
def test_bf16_result(M, N, K):
    """The bf16 result is the fp32 one rounded, asked for alone or beside it; with one split it is written at once
    and the workspace stays as it was."""
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    dy = torch.randn((K, M), generator=g, device=DEV).to(torch.bfloat16)
    x = torch.randn((K, N), generator=g, device=DEV).to(torch.bfloat16)
    L = _lib.lib()
    n = max(L.dopt_dw_gemm_any_workspace_floats(M, N, K), 4)
    got = {}
    for f32, b16 in ((True, False), (False, True), (True, True)):
        ws = torch.full((n,), 7.0, device=DEV)
        out32 = torch.full((M * N + 8,), 7.0, device=DEV)
        out16 = torch.full((M * N + 8,), 7.0, device=DEV, dtype=torch.bfloat16)
        db = torch.full((M + 8,), 7.0, device=DEV)
        rc = L.dopt_dw_gemm_any(dy.data_ptr(), M, x.data_ptr(), N, M, N, K, ws.data_ptr(), out32.data_ptr() if f32 else None,
                                out16.data_ptr() if b16 else None, db.data_ptr(), torch.cuda.current_stream().cuda_stream)
        _lib.check(rc, "dw_gemm_any")
        got[f32, b16] = out32, out16, db
        assert bool((out32[M * N if f32 else 0:] == 7).all()) and bool((out16[M * N if b16 else 0:] == 7).all())
        assert bool((db[M:] == 7).all()) and torch.equal(db, got[True, False][2])
        if K <= 97:
            assert bool((ws == 7).all())
    want = got[True, False][0][:M * N]
    assert torch.equal(got[True, True][0][:M * N], want)
    for key in ((False, True), (True, True)):
        assert torch.equal(got[key][1][:M * N], want.to(torch.bfloat16))
    assert torch.equal(ops.dw_gemm_any(dy, x, False, torch.bfloat16)[0].view(-1), want.to(torch.bfloat16))  # without db


@pytest.mark.parametrize("M,N,K", [(256, 256, 777), (512, 768, 2048), (768, 768, 985), (1024, 1280, 333), (256, 512, 64)])
def test_equals_dw_gemm(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(K)
    dy = torch.randn((K, M), generator=g, device=DEV).to(torch.bfloat16)
    x = torch.randn((K, N), generator=g, device=DEV).to(torch.bfloat16)
    for dt in (torch.float32, torch.bfloat16):
        got, want = ops.dw_gemm_any(dy, x, True, dt), ops.dw_gemm(dy, x, None, None, None, N, 0, 0, True, dt)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def test_refused():
    x = torch.zeros((16, 12), device=DEV, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="multiples of 8"):
        ops.dw_gemm_any(x, x, False, torch.float32)
    with pytest.raises(RuntimeError, match="bf16"):
        ops.dw_gemm_any(x.float(), x, False, torch.float32)
    dw, db = ops.dw_gemm_any(torch.empty((0, 64), device=DEV, dtype=torch.bfloat16),
                             torch.empty((0, 24), device=DEV, dtype=torch.bfloat16), True, torch.float32)
    assert dw.shape == (64, 24) and not dw.any() and not db.any()


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("fin,fout,tokens", [(192, 576, 197), (320, 1280, 1111), (384, 200, 50), (36, 100, 40)])
def test_linear_layer_gradients(fin, fout, tokens, bias):
    """The layer's gradients against float64 of what it saved, for feature counts of every route (multiples of 8, and
    ones no kernel takes)."""
    torch.manual_seed(fin + tokens)
    shape = (4, tokens, fin)
    meta = {"l": {"bits": 2, "pack_only": False, "AVG_ALAM": False, "ALAM_BITS": 0, "DIVISION": None, **layer_group_meta(shape, 2)}}
    layer = DOLinear(fin, fout, target_name="l", meta=meta, bias=bias, device=DEV).train()
    x = torch.randn(shape, device=DEV, requires_grad=True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = layer(x)
    dy = torch.randn_like(y)
    y.backward(dy)
    from deep_optimization_amd.modules.module_utils import unified_dequantize, unified_quantize
    q, q_meta, _ = unified_quantize(x.detach().to(torch.bfloat16), None, "l", meta, clamp=True, clamp_alpha=3.0)
    xh = unified_dequantize(q, q_meta, None).reshape(-1, fin).double()
    dyd = dy.reshape(-1, fout).double()
    ref = dyd.t() @ xh
    assert layer.weight.grad.dtype == torch.float32
    assert float((layer.weight.grad.double() - ref).norm() / ref.norm()) <= 5e-3
    if bias:
        assert float((layer.bias.grad.double() - dyd.sum(0)).norm() / dyd.sum(0).norm()) <= 5e-3
