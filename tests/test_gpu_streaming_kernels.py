"""Kernels that move rows between layouts 16 bytes at a time: sizes around a workgroup's share, and arrays that do not start at
a multiple of 16 bytes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _tensor(shape, gen, offset):
    """Normal values in memory that starts `offset` floats behind a multiple of 16 bytes."""
    room = torch.empty(int(np.prod(shape)) + offset, device=DEV)
    t = room[offset:].view(shape)
    return t.copy_(torch.randn(*shape, generator=gen, device=DEV))


@pytest.mark.parametrize("rest", (1, 2, 3, 8, 14, 15, 16))
@pytest.mark.parametrize("offset", (0, 1))
def test_sh_rows_are_joined_and_split_bit_for_bit(rest, offset):
    from retinags_amd import _host
    gen = torch.Generator(device=DEV).manual_seed(rest)
    for n in (1, 2, 127, 128, 129, 1021):
        dc, more = _tensor((n, 1, 3), gen, offset), _tensor((n, rest, 3), gen, offset)
        small = [torch.randn(n, k, generator=gen, device=DEV) for k in (3, 4, 1)]
        leaves = [t.requires_grad_(True) for t in (dc, more, *small)]
        shs = _host.activate(*leaves, 0)[0]
        assert torch.equal(shs.detach(), torch.cat((dc, more), dim=1).detach())
        upstream = torch.randn(n, 1 + rest, 3, generator=gen, device=DEV)
        d_dc, d_more = torch.autograd.grad([shs], leaves[:2], [upstream])
        assert torch.equal(d_dc, upstream[:, :1]) and torch.equal(d_more, upstream[:, 1:])


@pytest.mark.parametrize("n", (1, 1023, 1024, 1025, 4097))
def test_activated_values_at_the_edges_of_a_workgroup(n):
    """Every row against torch's expressions in 64 bits: a library exp, division and square root differ by a few units in
    the last place (2^-23 each), so 1e-6 relative leaves room for eight of them."""
    from retinags_amd import _host
    gen = torch.Generator(device=DEV).manual_seed(n)
    features = torch.randn(n, 1, 3, generator=gen, device=DEV), torch.randn(n, 15, 3, generator=gen, device=DEV)
    small = [torch.randn(n, k, generator=gen, device=DEV) for k in (3, 4, 1)]
    leaves = [t.requires_grad_(True) for t in (*features, *small)]
    outs = _host.activate(*leaves, 0)[1:]
    upstream = [torch.randn_like(o) for o in outs]
    grads = torch.autograd.grad(outs, leaves[2:], upstream)
    wide = [t.detach().double().requires_grad_(True) for t in small]
    want = [torch.exp(wide[0]), torch.nn.functional.normalize(wide[1]), torch.sigmoid(wide[2])]
    want_grads = torch.autograd.grad(want, wide, [u.double() for u in upstream])
    for got, ref in zip(outs, want):
        assert torch.allclose(got.double(), ref, rtol=1e-6, atol=0)
    for got, ref in zip(grads, want_grads):
        # (the quaternion's gradient is a difference of terms as large as the upstream gradient)
        assert float((got.double() - ref).norm() / ref.norm()) < 2e-6
