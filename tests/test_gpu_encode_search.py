"""The encode kernels' sorted search and its exhaustive fallback on the GPU,
bit for bit against the CPU oracle: both kernels (16 lanes per vector up to
16384 vectors, one vector per lane beyond) at their edges, with inputs whose
winners are certain, near-ties and exact ties; and the refinement's chunk
kernel at both work-group sizes."""
import numpy as np
import pytest
import torch

from oracle import cref
from test_e8_search import inputs

pytestmark = pytest.mark.gpu


def encode(x, kinds, scales, dev):
    from quipsharp_amd.codebooks.e8p import _encode
    vals, codes = _encode(torch.from_numpy(x).to(dev), kinds, scales)
    return vals.cpu().numpy(), codes.cpu().numpy()


@pytest.mark.parametrize("n", [1, 3, 5, 16384, 16385, 16640, 33000])
@pytest.mark.parametrize("kinds,scales", [([0], [1.0]), ([1], [1.0]), ([0, 1], [0.95, 0.55]), ([0, 0], [0.95, 0.28]),
                                          ([0, 1, 0, 1], [1.1, 0.5, 0.3, 0.2])])
def test_encode_matches_the_oracle(dev, n, kinds, scales):
    x = inputs("gauss1.2", np.random.default_rng(n), n).astype(np.float32)
    want, codes = cref.rvq_encode(x, kinds, scales)
    got, gcodes = encode(x, kinds, scales, dev)
    assert np.array_equal(gcodes, np.stack([np.asarray(c) for c in codes]))
    assert np.array_equal(got, want)


@pytest.mark.parametrize("kind", ["codewords", "midpoints", "grid", "sparse", "wide", "gauss6"])
@pytest.mark.parametrize("n", [1000, 20000])
def test_ties_and_large_inputs_match_the_oracle(dev, kind, n):
    x = inputs(kind, np.random.default_rng(n), n).astype(np.float32)
    x[::97] = 0.0
    for kinds, scales in (([0], [1.0]), ([1], [1.0]), ([0, 1], [0.95, 0.55])):
        want, codes = cref.rvq_encode(x, kinds, scales)
        got, gcodes = encode(x, kinds, scales, dev)
        assert np.array_equal(gcodes, np.stack([np.asarray(c) for c in codes]))
        assert np.array_equal(got, want)


def test_unaligned_rows_match(dev):
    """Row strides and offsets off 16 bytes (dword accesses)."""
    from quipsharp_amd import _lib
    rng = np.random.default_rng(3)
    for n in (40, 20000):
        buf = torch.from_numpy(rng.standard_normal((n, 11)).astype(np.float32)).to(dev)
        out = torch.zeros(n, 9, device=dev)
        codes = torch.zeros(n, dtype=torch.int32, device=dev)
        L = _lib.lib()
        _lib.check(L.qs_rvq_encode(buf.data_ptr() + 4, 11, n, 1, _lib.int_array([0]), _lib.float_array([1.0]), 1.0, 1.0,
                                   out.data_ptr() + 4, 9, codes.data_ptr(), 4, n, 1, _lib.stream_of(buf)))
        x = buf.cpu().numpy()[:, 1:9].copy()
        want, wc = cref.e8p_encode(x)
        got = out.cpu().numpy().reshape(-1)[1:1 + 9 * n - 1]
        got = np.stack([got[9 * i:9 * i + 8] for i in range(n)])
        assert np.array_equal(got, want) and np.array_equal(codes.cpu().numpy(), wc)


@pytest.mark.parametrize("m,nb,kinds,scales", [(4100, 16, [0], [1.0]), (4129, 5, [0, 1], [0.95, 0.55])])
def test_chunk_rows_do_not_depend_on_the_work_group(dev, m, nb, kinds, scales):
    """More than 4096 rows run 32 to a work-group; each row as in a launch of
    its own few rows (16 to a work-group)."""
    from quipsharp_amd import _lib
    L = _lib.lib()
    n, c0 = 256, 7
    T = n // 8
    torch.manual_seed(m)
    W, E = torch.randn(m, n, device=dev), 0.3 * torch.randn(m, n, device=dev)
    Wq, P = torch.randn(m, n, device=dev), 0.1 * torch.randn(m, 8 * nb, device=dev)
    H = torch.eye(n, device=dev) + 0.02 * torch.randn(n, n, device=dev)
    D = (torch.eye(8, device=dev) + 0.02 * torch.randn(T, 8, 8, device=dev)).contiguous()
    kc, sc = _lib.int_array(kinds), _lib.float_array(scales)

    def run(rows):
        wq, e = Wq[rows].clone(), E[rows].clone()
        w, p = W[rows].contiguous(), P[rows].contiguous()
        r = w.shape[0]
        codes = torch.full((len(kinds), r, T), -1, dtype=torch.int64, device=dev)
        _lib.check(L.qs_ldlq_chunk(w.data_ptr(), n, wq.data_ptr(), n, e.data_ptr(), n, p.data_ptr(), 8 * nb,
                                   H.data_ptr() + 8 * c0 * n * 4, n, D.data_ptr(), c0, nb, r, len(kinds), kc, sc,
                                   codes.data_ptr(), 8, r * T, T, _lib.stream_of(w)))
        return wq, e, codes

    whole = run(slice(0, m))
    untouched = [i for i in range(n) if not 8 * c0 <= i < 8 * (c0 + nb)]
    assert torch.equal(whole[0][:, untouched], Wq[:, untouched]) and torch.equal(whole[1][:, untouched], E[:, untouched])
    for rows in (slice(0, 1), slice(5, 24), slice(4060, m), slice(m - 3, m)):
        part = run(rows)
        assert torch.equal(part[0], whole[0][rows]) and torch.equal(part[1], whole[1][rows])
        assert torch.equal(part[2], whole[2][:, rows])
    assert (whole[2][:, :, c0:c0 + nb] >= 0).all() and (whole[2][:, :, :c0] == -1).all()
