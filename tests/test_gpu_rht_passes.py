"""The transform kernels at the edges of their splits: rows that share a
work-group (with a last one that is not full), every depth of round and of
column pass, odd factors around the eight-output tiles, in place and not,
few rows (several work-groups per row), unaligned rows and inner sizes off
the wave width -- bit for bit against the oracle's Walsh-Hadamard stages, and
within fp32 rounding of the dense fp64 matrix with an odd factor."""
import numpy as np
import pytest
import torch

from oracle import cref
from test_gpu_rht import dense_T

pytestmark = pytest.mark.gpu


def run(dev, x, outer, n, inner, pre=None, pre_inner=None, post=None, in_place=False, offset=0):
    from quipsharp_amd import _lib
    from quipsharp_amd.hadamard import hartley_matrix, kron_factor
    p, _ = kron_factor(n)
    buf = torch.zeros(x.size + offset, device=dev)
    buf[offset:] = torch.from_numpy(x.reshape(-1)).to(dev)
    out = buf if in_place else torch.zeros(x.size + offset, device=dev)
    t = lambda a: None if a is None else torch.from_numpy(a).to(dev)
    ts = [t(pre), t(pre_inner), t(post)]
    K = hartley_matrix(p, dev) if p > 1 else None
    _lib.check(_lib.lib().qs_rht_f32(buf.data_ptr() + 4 * offset, out.data_ptr() + 4 * offset, outer, n, inner,
                                     *[_lib.ptr(a) for a in ts], p, _lib.ptr(K), _lib.stream_of(buf)))
    return out[offset:].cpu().numpy().reshape(x.shape)


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("outer,n", [(1, 1), (5, 2), (700, 8), (1025, 16), (130, 32), (9, 512), (5, 1024), (3, 2048),
                                     (2, 8192), (1, 32768)])
def test_rows_bit_exact(dev, outer, n, in_place):
    rng = np.random.default_rng(n + outer)
    x = rng.standard_normal((outer, n)).astype(np.float32)
    pre, post = (rng.choice([-1.0, 1.0], n).astype(np.float32) for _ in range(2))
    for offset in (0, 1):
        y = run(dev, x, outer, n, 1, pre=pre, post=post, in_place=in_place, offset=offset)
        assert np.array_equal(y, cref.fwht(x * pre, 1) * post)


@pytest.mark.parametrize("outer,n,inner", [(1, 2, 64), (2, 16, 65), (1, 128, 300), (3, 256, 7), (1, 2048, 257),
                                           (1, 8192, 70), (2, 16384, 3)])
def test_columns_bit_exact(dev, outer, n, inner):
    rng = np.random.default_rng(n + inner)
    x = rng.standard_normal((outer, n, inner)).astype(np.float32)
    pre, post = (rng.choice([-1.0, 1.0], n).astype(np.float32) for _ in range(2))
    ri = rng.choice([-1.0, 1.0], inner).astype(np.float32)
    want = cref.fwht(x * pre[:, None] * ri, 1) * post[:, None]
    for in_place in (False, True):
        assert np.array_equal(run(dev, x, outer, n, inner, pre, ri, post, in_place), want)


@pytest.mark.parametrize("n", [3, 5 * 16, 7 * 32, 7 * 64, 9 * 128, 15 * 256, 43 * 256, 63 * 512, 17 * 1024])
@pytest.mark.parametrize("outer,inner", [(1, 1), (4, 1), (300, 1), (1, 70), (2, 5)])
def test_odd_factors_match_the_dense_matrix(dev, n, outer, inner):
    rng = np.random.default_rng(n)
    x = rng.standard_normal((outer, n, inner)).astype(np.float32)
    post = rng.choice([-1.0, 1.0], n).astype(np.float32)
    L = n & -n
    p = n // L
    # H_L over b in the oracle's fp32 stages (bit-exact, tested above), K_p over a in fp64
    K = dense_T(p) if p > 1 else np.ones((1, 1))
    h = cref.fwht(x.reshape(outer, p, L, inner), 2).astype(np.float64)
    want = np.einsum("ac,ocbi->oabi", K, h).reshape(outer, n, inner) * post[:, None]
    for in_place in (False, True):
        y = run(dev, x, outer, n, inner, post=post, in_place=in_place)
        # p FMAs of fp32 values, K rounded to fp32: (p + 1) 2^-24 of sum |K||h|, far above the error seen
        bound = (p + 1) * 2.0 ** -24 * np.einsum("ac,ocbi->oabi", np.abs(K), np.abs(h)).reshape(outer, n, inner)
        assert (np.abs(y - want) <= bound + 1e-30).all()
