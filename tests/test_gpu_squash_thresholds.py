"""The squashed nearest quantizer of bf16 inputs at 1 and 2 bits (threshold codes on the bf16 grid,
csrc/quant_pack.h: squash16_pass) against the per-element form of the same arithmetic, bit for bit.

The per-element form is what the same operator runs on fp32 inputs: on the same values (bf16 widened
exactly) it must give the same words, scale and min. No tolerance.
"""
import pytest
import torch

import deep_optimization_amd  # noqa: F401

pytestmark = pytest.mark.gpu
DEV = "cuda"
ops = torch.ops.act_lib
INF = float("inf")


def every_bf16():
    bits = torch.arange(1 << 16, device=DEV, dtype=torch.int32)
    return (bits << 16).view(torch.float32)


def test_squash_is_non_decreasing_on_the_bf16_grid():
    """The premise of the thresholds: the squash as the kernels evaluate it, over every bf16 value from
    -inf to inf (a group of 64 equal values stores it as its min)."""
    v = every_bf16()
    v = v[~v.isnan()].sort().values
    x = v.to(torch.bfloat16).view(-1, 1, 1).expand(-1, 1, 64).contiguous()
    _, _, mn = ops.quant_pack(x.float(), 2, 64, False, 0.0, True, 0, None, 0, 0, torch.float32)
    assert bool((mn.flatten().diff() >= 0).all())


def test_squash_is_non_decreasing_around_the_grid():
    """... and over the clamp's alpha, which may lie between two grid values: the 16 fp32 values on either side of every
    finite bf16 value, and runs of consecutive ones where the squash bends and saturates. (All fp32 values from -3.4e38
    to 3.4e38 were checked once, 4.28e9 pairs of neighbours.)"""
    grid = torch.arange(0, 0x7F80, device=DEV, dtype=torch.int32) << 16
    near = (grid[:, None] + torch.arange(-16, 17, device=DEV, dtype=torch.int32)).flatten().clamp_min(0)
    runs = [torch.arange(1 << 18, device=DEV, dtype=torch.int32) + torch.tensor(at, device=DEV).view(torch.int32)
            for at in (1e-4, 0.099, 0.5, 2.69, 2.999, 4.0, 8.0)]
    for bits in (near, *runs):
        v = bits.view(torch.float32)
        for x in (v, -v.flip(0)):
            x = x.view(-1, 1, 1).expand(-1, 1, 64).contiguous()
            _, _, mn = ops.quant_pack(x, 2, 64, False, 0.0, True, 0, None, 0, 0, torch.float32)
            assert bool((mn.flatten().diff() >= 0).all())


def cases(kind, n, g, gen):
    x = torch.randn((n, g), generator=gen, device=DEV)
    if kind == "relu":
        return x.abs_()
    if kind == "wide":  # far into the squash's saturation, and groups that lie wholly in it
        return x * 6 + 4 * torch.randn((n, 1), generator=gen, device=DEV)
    if kind == "scales":  # groups from 1e-6 to 1e3, some around zero, some away from it
        s = 10.0 ** (torch.rand((n, 1), generator=gen, device=DEV) * 9 - 6)
        return x * s + torch.randint(-2, 3, (n, 1), generator=gen, device=DEV) * s * 3
    if kind == "few":  # few distinct values: ties and boundaries on the values themselves
        return torch.randint(-3, 4, (n, g), generator=gen, device=DEV) / 4.0
    if kind == "constant":
        return x[:, :1].expand(n, g).clone()
    if kind == "special":
        x = x.flatten()
        at = torch.randint(0, x.numel(), (x.numel() // 40,), generator=gen, device=DEV)
        pick = torch.tensor([INF, -INF, float("nan"), 0.0, -0.0, 3.0, -3.0, 1e-39, 3e38], device=DEV)
        x[at] = pick[torch.randint(0, 9, at.shape, generator=gen, device=DEV)]
        x = x.view(n, g)
        x[::7] = x[::7].nan_to_num(0.0)
        return x
    return x


@pytest.mark.parametrize("kind", ["normal", "relu", "wide", "scales", "few", "constant", "special"])
@pytest.mark.parametrize("g", [64, 128, 256, 512, 1024])
@pytest.mark.parametrize("bits", [1, 2])
def test_equals_the_per_element_form(bits, g, kind):
    gen = torch.Generator(device=DEV).manual_seed(bits * 1000 + g)
    n = 4096 + 37  # whole and partial waves
    x = cases(kind, n, g, gen).to(torch.bfloat16).view(1, n, g)
    for clamp, alpha in ((True, 3.0), (False, 0.0), (True, 0.5), (True, 0.0)):
        for meta in (torch.float32, torch.bfloat16):
            args = (bits, g, clamp, alpha, True, 0, None, 0, 0, meta)
            got, want = ops.quant_pack(x, *args), ops.quant_pack(x.float(), *args)
            for a, b, what in zip(got, want, ("words", "scale", "min")):
                same = (a == b) | (a.isnan() & b.isnan()) if a.is_floating_point() else a == b
                assert bool(same.all()), (what, clamp, alpha, meta, int((~same).sum()))


@pytest.mark.parametrize("n", [1, 2, 3, 9, 257])
@pytest.mark.parametrize("bits,g,hw", [(1, 64, (8, 24)), (2, 64, (16, 8)), (1, 256, (32, 16)), (2, 256, (16, 48)), (2, 1024, (32, 64))])
def test_tiles_and_small_counts(bits, g, hw, n):
    gen = torch.Generator(device=DEV).manual_seed(n)
    x = torch.randn((n, 3, *hw), generator=gen, device=DEV).to(torch.bfloat16)
    args = (bits, g, True, 3.0, True, 0, None, 0, 0, torch.float32)
    for got, want in zip(ops.quant_pack_tiles(x, *args), ops.quant_pack_tiles(x.float(), *args)):
        assert torch.equal(got, want)


@pytest.mark.parametrize("g,hw,n", [(256, (16, 48), 461), (1024, (32, 64), 175)])
def test_tiles_of_many_groups(g, hw, n):
    """2 bits and groups of 256 and more take the thresholds above 2^20 elements only: the tile layout there, with a
    partial wave, and flat groups on both sides of the line."""
    gen = torch.Generator(device=DEV).manual_seed(n)
    args = (2, g, True, 3.0, True, 0, None, 0, 0, torch.float32)
    x = torch.randn((n, 3, *hw), generator=gen, device=DEV).to(torch.bfloat16)
    assert x.numel() > 1 << 20
    for got, want in zip(ops.quant_pack_tiles(x, *args), ops.quant_pack_tiles(x.float(), *args)):
        assert torch.equal(got, want)
    for groups in ((1 << 20) // g - 1, (1 << 20) // g, (1 << 20) // g + 1):
        x = torch.randn((1, groups, g), generator=gen, device=DEV).to(torch.bfloat16)
        for got, want in zip(ops.quant_pack(x, *args), ops.quant_pack(x.float(), *args)):
            assert torch.equal(got, want)


@pytest.mark.parametrize("alpha", [2.7, 3.0000002, 2.9999998, 0.1, 1e-3, 4.3, 1e-30, 100.1, INF])
@pytest.mark.parametrize("bits", [1, 2])
def test_alpha_between_grid_values(bits, alpha):
    """An alpha that is no bf16 value, a few fp32 steps from one, tiny, in the saturation, or infinite."""
    gen = torch.Generator(device=DEV).manual_seed(int(alpha * 1000) if alpha < INF else 1)
    for kind in ("normal", "wide", "scales", "special"):
        x = cases(kind, 4096 + 37, 256, gen).to(torch.bfloat16).view(1, -1, 256)
        args = (bits, 256, True, alpha, True, 0, None, 0, 0, torch.float32)
        for a, b in zip(ops.quant_pack(x, *args), ops.quant_pack(x.float(), *args)):
            same = (a == b) | (a.isnan() & b.isnan()) if a.is_floating_point() else a == b
            assert bool(same.all()), (kind, int((~same).sum()))
