"""The long-batch transform kernels (qs_linear_rows.hip) against fp64 dense and
against the per-row kernels of shorter batches: row counts around their
thresholds and tiles, odd factors, partial slice groups, dtypes, both sign
formats, bias, strided inputs and outputs."""
import numpy as np
import pytest
import torch

from test_gpu_rht import dense_T

pytestmark = pytest.mark.gpu


def layer(dev, m, n, seed, bias):
    from quipsharp_amd.quantize import PackedCodes
    g = torch.Generator().manual_seed(seed)
    codes = torch.randint(0, 65536, (m, n // 8), generator=g)
    sign = lambda k: (torch.randint(0, 2, (k,), generator=g) * 2 - 1).float()
    b = torch.randn(m, generator=g) if bias else None
    packed = PackedCodes(codes.to(dev), m, n, [0])
    return packed, sign(m), sign(n), b, codes


def dense64(x, codes, su, sv, scale, bias, dev):
    from quipsharp_amd.codebooks.e8p import _decode
    W = _decode(codes.to(dev).unsqueeze(0), [0], [1.0]).reshape(su.numel(), sv.numel()).double() * scale
    Tn, Tm = (torch.from_numpy(dense_T(k)).to(dev) for k in (sv.numel(), su.numel()))
    y = ((x.double() * sv.to(dev).double()) @ Tn.T @ W.T) @ Tm.T * su.to(dev).double()
    return y if bias is None else y + bias.to(dev).double()


@pytest.mark.parametrize("m,n", [(256, 256), (512, 3584), (768, 4096), (2560, 4352), (256, 11008), (13312, 512),
                                 (18944, 256), (25600, 512)])
@pytest.mark.parametrize("B", [159, 160, 163, 320, 337])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_long_batches_match_dense(dev, m, n, B, dtype):
    from quipsharp_amd.quantize import forward_packed, pack_signs
    packed, su, sv, bias, codes = layer(dev, m, n, B + m, B % 2 == 0)
    x = torch.randn(B, n, generator=torch.Generator().manual_seed(B)).to(dev).to(dtype)
    x[3] *= 900.0
    args = (1.0, 0.0, 0.0135, None if bias is None else bias.to(dev))
    y = forward_packed(x, packed, su.to(dev), sv.to(dev), *args, out_dtype=torch.float32)
    want = dense64(x, codes, su, sv, 0.0135, bias, dev)
    # fp16 operand: 2^-11 per element at most, ~2.2e-4 of a row's norm
    rel = ((y.double() - want).norm(dim=1) / want.norm(dim=1)).max().item()
    assert rel < 1e-3, rel
    # the same rows in a batch below the threshold (the per-row kernels)
    short = forward_packed(x[:100].contiguous(), packed, su.to(dev), sv.to(dev), *args, out_dtype=torch.float32)
    rel = ((y[:100] - short).norm(dim=1) / short.norm(dim=1)).max().item()
    assert rel < 5e-4, rel
    if m <= 12288 and n <= 12288:  # packed bits: the same bits out
        bits = forward_packed(x, packed, pack_signs(su.to(dev)), pack_signs(sv.to(dev)), *args, out_dtype=torch.float32)
        assert torch.equal(bits, y)


@pytest.mark.parametrize("m,n", [(13312, 512), (512, 3584)])
def test_strides_dtypes_and_row_isolation(dev, m, n):
    from quipsharp_amd.quantize import forward_packed, forward_packed_group
    B = 341
    packed, su, sv, bias, codes = layer(dev, m, n, 5, True)
    su, sv, bias = su.to(dev), sv.to(dev), bias.to(dev)
    args = (packed, su, sv, 1.0, 0.0, 0.0135, bias)
    x = torch.randn(B, n, device=dev).bfloat16()
    y = forward_packed(x, *args)
    wide = torch.zeros(B, n + 24, device=dev).bfloat16()
    wide[:, 8:8 + n] = x
    assert torch.equal(forward_packed(wide[:, 8:8 + n], *args), y)  # rows on 16 bytes, longer stride
    odd = torch.zeros(B, n + 3, device=dev).bfloat16()
    odd[:, 1:1 + n] = x  # rows off 16 bytes: other kernels, the same result to fp16 rounding
    assert ((forward_packed(odd[:, 1:1 + n], *args).float() - y.float()).norm() / y.float().norm()).item() < 3e-3
    for dt in (torch.float16, torch.float32):
        z = forward_packed(x, *args, out_dtype=dt)
        assert ((z.float() - y.float()).norm() / y.float().norm()).item() < 4e-3
    out = torch.full((B, m + 5), 7.0, device=dev).bfloat16()
    forward_packed(x, *args, out=out[:, 2:2 + m])  # rows off 16 bytes: element stores
    assert torch.equal(out[:, 2:2 + m], y) and (out[:, :2] == 7).all() and (out[:, 2 + m:] == 7).all()
    bad = x.clone()
    bad[7] = float("inf")
    bad[200, 5] = float("nan")
    keep = [i for i in range(B) if i not in (7, 200)]
    assert torch.equal(forward_packed(bad, *args)[keep], y[keep])
    a, b = forward_packed_group(x, [args, args])
    if m > 12288:  # one GEMM launch each: bit-identical
        assert torch.equal(a, y)
    assert torch.equal(a, b)
    zero = forward_packed(x, packed, su * 0, sv * 0, 1.0, 0.0, 0.0135, bias)  # signs of a layer not loaded yet
    assert torch.equal(zero, bias.bfloat16().expand(B, m))


@pytest.mark.parametrize("m,B,has_bias", [(16384, 320, True), (32768, 323, False), (18944, 600, False)])
def test_output_factors_that_are_not_signs(dev, m, B, has_bias):
    """su of other values than +-1 (powers of two: the product is exact), read
    as they are instead of as bits."""
    from quipsharp_amd.quantize import forward_packed
    packed, su, sv, bias, _ = layer(dev, m, 256, m, has_bias)
    su, sv = su.to(dev), sv.to(dev)
    x = torch.randn(B, 256, generator=torch.Generator().manual_seed(B)).to(dev)
    factor = torch.ones(m, device=dev)
    factor[5::97] = 4.0
    args = (1.0, 0.0, 0.0135)
    plain = forward_packed(x, packed, su, sv, *args)
    assert torch.equal(forward_packed(x, packed, su * factor, sv, *args), plain * factor)
    if has_bias:
        b = bias.to(dev).float()
        odd = torch.empty(m + 1, device=dev)[1:].copy_(b)  # off 16 bytes
        want = forward_packed(x, packed, su, sv, *args, bias=b)
        assert torch.equal(forward_packed(x, packed, su, sv, *args, bias=odd), want)
        assert (want - (plain + b)).abs().max() <= 1e-5 * want.abs().max()


def test_group_of_different_long_outputs_equals_single_calls(dev):
    from quipsharp_amd.quantize import forward_packed, forward_packed_group
    lins = []
    for m in (13312, 32768, 14336):
        packed, su, sv, _, _ = layer(dev, m, 256, m, False)
        lins.append((packed, su.to(dev), sv.to(dev), 1.0, 0.0, 0.0135, None))
    x = torch.randn(331, 256, generator=torch.Generator().manual_seed(1)).to(dev)
    for lin, y in zip(lins, forward_packed_group(x, lins)):
        assert torch.equal(y, forward_packed(x, *lin))


def structured_T(v):
    """T along the last dim of fp64 v (the rows of a dense_T product, for long rows)."""
    n = v.shape[-1]
    L = n & -n
    p = n // L
    z, h = v.reshape(-1, p, L), 1
    while h < L:
        z = z.reshape(-1, p, L // (2 * h), 2, h)
        z = torch.stack([z[..., 0, :] + z[..., 1, :], z[..., 0, :] - z[..., 1, :]], -2)
        h *= 2
    z = z.reshape(-1, p, L) / L ** 0.5
    i = torch.arange(p, device=v.device, dtype=torch.float64)
    a = 2 * torch.pi * ((i[:, None] * i) % p) / p
    return ((a.cos() + a.sin()) / p ** 0.5 @ z).reshape(v.shape)


@pytest.mark.parametrize("n,B", [(512, 256), (512, 257), (3584, 256), (3584, 257), (11008, 256), (11008, 257),
                                 (14336, 160)])
@pytest.mark.parametrize("dtype,size", [(torch.bfloat16, 1.0), (torch.float16, 1.0), (torch.float16, 3e4),
                                        (torch.float32, 1.0)])
def test_input_factors_that_are_not_signs(dev, n, B, dtype, size):
    """sv of other values than +-1 on both sides of the thresholds: the products
    keep two 16-bit planes, and those beyond fp16's range stay finite."""
    from quipsharp_amd.codebooks.e8p import _decode
    from quipsharp_amd.quantize import forward_packed
    m = 256
    packed, su, sv, _, codes = layer(dev, m, n, n, False)
    su, sv = su.to(dev), sv.to(dev) * torch.linspace(1.03, 2.33, n, device=dev)
    x = (torch.randn(B, n, generator=torch.Generator().manual_seed(B)).clamp_(-2, 2) * size).to(dev).to(dtype)
    y = forward_packed(x, packed, su, sv, 1.0, 0.0, 0.0135, out_dtype=torch.float32)
    W = _decode(codes.to(dev).unsqueeze(0), [0], [1.0]).reshape(m, n).double()
    want = structured_T(structured_T(x.double() * sv.double()) @ W.T * 0.0135) * su.double()
    # the fp16 operand's 2.2e-4 of a row's norm; one 16-bit plane of bf16 products would leave 2e-3
    rel = ((y.double() - want).norm(dim=1) / want.norm(dim=1)).max().item()
    assert rel < 1e-3, rel


@pytest.mark.parametrize("n", [17408, 18944, 25600, 32768])
def test_long_fp32_rows_are_transformed_in_fp32(dev, n):
    """fp32 activations beyond 16384 columns: a long batch's rows are those of a shorter one."""
    from quipsharp_amd.quantize import forward_packed
    packed, su, sv, _, _ = layer(dev, 256, n, n, False)
    args = (packed, su.to(dev), sv.to(dev), 1.0, 0.0, 0.0135)
    x = torch.randn(160, n, generator=torch.Generator().manual_seed(n)).to(dev)
    assert torch.equal(forward_packed(x, *args)[:159], forward_packed(x[:159].contiguous(), *args))


@pytest.mark.parametrize("m,n", [(512, 3584), (768, 4096), (256, 11008)])
@pytest.mark.parametrize("B", [256, 257, 259])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_threshold_up_to_12288_columns(dev, m, n, B, dtype):
    test_long_batches_match_dense(dev, m, n, B, dtype)
