"""reconstruct_weight / reconstruct_hessian multiply by the signs as torch would:
with the signs' gradients, tangents and dtype."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def pieces(dev, m, n):
    from quipsharp_amd.incoherence import IncoherenceSigns, reconstruct_weight
    g = torch.Generator().manual_seed(m + n)
    what = torch.randn(m, n, generator=g).to(dev)
    sign = lambda k: (torch.randint(0, 2, (k,), generator=g) * 2 - 1).float().to(dev)
    one = lambda k: torch.ones(k, device=dev)
    plain = reconstruct_weight(what, IncoherenceSigns(one(m), one(n)))
    return what, sign(m), sign(n), plain


@pytest.mark.parametrize("m,n", [(32, 64), (48, 1024), (256, 24)])
def test_gradients_of_the_signs(dev, m, n):
    from quipsharp_amd.incoherence import IncoherenceSigns, reconstruct_hessian, reconstruct_weight
    what, su, sv, plain = pieces(dev, m, n)
    weight = torch.randn(m, n, generator=torch.Generator().manual_seed(1)).to(dev)
    a, b = su.clone().requires_grad_(), sv.clone().requires_grad_()
    out = reconstruct_weight(what, IncoherenceSigns(a, b))
    assert torch.equal(out, plain * su[:, None] * sv)  # +-1: exact
    (out * weight).sum().backward()
    for got, want in ((a.grad, (plain * weight * sv).sum(1)), (b.grad, (plain * weight * su[:, None]).sum(0))):
        assert (got - want).norm() <= 1e-5 * want.norm()
    assert not reconstruct_weight(what, IncoherenceSigns(su, sv)).requires_grad
    c = sv.clone().requires_grad_()
    assert reconstruct_hessian(torch.eye(n, device=dev), IncoherenceSigns(su, c)).requires_grad


def test_dtypes_tangents_and_batches_of_the_signs(dev):
    from quipsharp_amd.incoherence import IncoherenceSigns, reconstruct_weight
    what, su, sv, plain = pieces(dev, 64, 96)
    want = plain * su[:, None] * sv
    for left, right, dtype in ((su.double(), sv, torch.float64), (su, sv.double(), torch.float64),
                               (su.half(), sv.bfloat16(), torch.float32)):
        out = reconstruct_weight(what, IncoherenceSigns(left, right))
        assert out.dtype == dtype and torch.equal(out, want.to(dtype))
    third = su.double() / 3  # not rounded to fp32
    assert torch.equal(reconstruct_weight(what, IncoherenceSigns(third, sv)), plain * third[:, None] * sv)
    fw = torch.autograd.forward_ad
    with fw.dual_level():
        out = reconstruct_weight(what, IncoherenceSigns(fw.make_dual(su, 2 * su), sv))
        assert torch.equal(fw.unpack_dual(out).tangent, 2 * want)
    each = torch.func.vmap(lambda s: reconstruct_weight(what, IncoherenceSigns(s, sv)))(torch.stack([su, -su]))
    assert torch.equal(each, torch.stack([want, -want]))
