"""The decode-in-the-loop GEMM (17 or more rows) at the edges of its splits:
rows around the 16-row tiles of each compiled width, weight rows off the
128-row work-group, one slice, linears of different sizes in one launch."""
import numpy as np
import pytest
import torch

from test_gpu_linear import REL_TOL, dense_forward, rel_err, run

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


# activation tiles per work-group 2, 3, 4, 6, 8 with the last tile full, of one
# row or clamped; with two stages also several work-group columns, unevenly filled
@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("m,n,B", [(272, 256, 17), (1024, 512, 32), (400, 1280, 33), (512, 256, 48), (16, 512, 49),
                                   (4096, 768, 64), (656, 512, 65), (1024, 256, 96), (128, 2560, 97), (784, 512, 128),
                                   (256, 512, 145), (512, 256, 289)])
def test_split_edges_vs_dense_fp64(dev, m, n, B, two):
    print(f"case: wide split m={m} n={n} B={B} two={two}", flush=True)
    rng = np.random.default_rng(m + n + B + two)
    c0 = rng.integers(0, 65536, (m, n // 8))
    c1 = rng.integers(0, 256, (m, n // 8)) if two else None
    su, sv = rng.choice([-1.0, 1.0], m), rng.choice([-1.0, 1.0], n)
    x = rng.standard_normal((B, n)).astype(np.float32)
    s0, s1 = (0.93, 0.41) if two else (1.0, 0.0)
    y, _ = run(dev, x, c0, c1, s0, s1, su, sv, 0.0135)
    want = dense_forward(x, c0, c1, s0, s1, su, sv, 0.0135)
    assert rel_err(y.cpu().numpy(), want) < REL_TOL
    # every row on its own as well: a lost or repeated tile is not averaged away
    rows = np.linalg.norm(y.cpu().numpy() - want, axis=1) / np.linalg.norm(want, axis=1)
    assert rows.max() < 2 * REL_TOL, (int(rows.argmax()), rows.max())


@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("B", [17, 60, 100])
def test_linears_of_a_shared_launch_equal_their_own(dev, B, two):
    from quipsharp_amd.quantize import PackedCodes, forward_packed, forward_packed_group
    n, sizes = 1024, [2048, 16, 400, 1024]
    rng = np.random.default_rng(B)
    t = lambda a: torch.from_numpy(np.asarray(a, dtype=np.float32)).to(dev)  # noqa: E731
    sv = t(rng.choice([-1.0, 1.0], n))
    lins = []
    for m in sizes:
        c = [rng.integers(0, 65536, (m, n // 8)), rng.integers(0, 256, (m, n // 8))][:2 if two else 1]
        packed = PackedCodes(torch.from_numpy(np.stack(c)).to(dev), m, n, [0, 1][:len(c)])
        lins.append((packed, t(rng.choice([-1.0, 1.0], m)), sv, 0.95, 0.5 if two else 0.0, 0.01, None))
    x = t(rng.standard_normal((B, n)))
    for lin, y in zip(lins, forward_packed_group(x, lins)):
        assert torch.equal(y, forward_packed(x, *lin))


# both sides of the line between the two GEMM kernels: 2^24 weights from 65 rows on
@pytest.mark.parametrize("m,n", [(4096, 4096), (4224, 4096), (5632, 3072), (1088, 25600)])
@pytest.mark.parametrize("B", [64, 65, 97, 128, 129])
def test_kernel_line_vs_dense_fp64(dev, m, n, B):
    from test_gpu_rows import structured_T

    from quipsharp_amd.codebooks.e8p import _decode
    from quipsharp_amd.quantize import PackedCodes, forward_packed
    g = torch.Generator().manual_seed(m + B)
    codes = torch.randint(0, 65536, (m, n // 8), generator=g)
    sign = lambda k: (torch.randint(0, 2, (k,), generator=g) * 2 - 1).float().to(dev)  # noqa: E731
    su, sv = sign(m), sign(n)
    x = torch.randn(B, n, generator=g).to(dev)
    y = forward_packed(x, PackedCodes(codes.to(dev), m, n, [0]), su, sv, 1.0, 0.0, 0.0135)
    W = _decode(codes.to(dev).unsqueeze(0), [0], [1.0]).reshape(m, n).double()
    want = structured_T(structured_T(x.double() * sv.double()) @ W.T * 0.0135) * su.double()
    rows = (y.double() - want).norm(dim=1) / want.norm(dim=1)
    assert rows.max() < REL_TOL, (int(rows.argmax()), rows.max().item())


@pytest.mark.parametrize("B", [65, 128])
def test_group_on_both_sides_of_the_line_equals_single_calls(dev, B):
    from quipsharp_amd.quantize import PackedCodes, forward_packed, forward_packed_group
    n, g = 4096, torch.Generator().manual_seed(B)
    sign = lambda k: (torch.randint(0, 2, (k,), generator=g) * 2 - 1).float().to(dev)  # noqa: E731
    lins = []
    for m in (4352, 1024, 4352, 4096):
        codes = torch.randint(0, 65536, (m, n // 8), generator=g)
        lins.append((PackedCodes(codes.to(dev), m, n, [0]), sign(m), sign(n), 1.0, 0.0, 0.0135, None))
    x = torch.randn(B, n, generator=g).to(dev).bfloat16()
    for lin, y in zip(lins, forward_packed_group(x, lins)):
        assert torch.equal(y, forward_packed(x, *lin))
