"""Router with six chunks requested up front (bf16, H >= 768 in chunks of 128, 128 to 4096 tokens): rows at the ends of that range and of
a workgroup's 16 tokens, chunk counts of one ring, one more and two, few experts; the same bits as calls of 64 tokens, which the two-stage
kernel takes (both add up a dot product in the same order), and the selection of the oracle from the kernel's own logits."""
import numpy as np
import pytest
import torch

from bibo_amd import ops
from oracle import bibo_moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("H", [640, 768, 896, 1536, 1664])
@pytest.mark.parametrize("T,E,k", [(127, 64, 6), (128, 64, 6), (131, 3, 2), (1000, 9, 2), (4096, 64, 8), (4097, 33, 4)])
def test_ring(H, T, E, k):
    g = torch.Generator().manual_seed(H + T)
    x = torch.randn(T, H, generator=g).bfloat16()
    wr = (torch.randn(E, H, generator=g) * 0.1).bfloat16()
    bias = torch.rand(E, generator=g) * 0.02 - 0.01
    xd, wd, bd = x.to(DEV), wr.to(DEV), bias.to(DEV)
    idx, w, logits, _ = (t if t is None else t.cpu() for t in ops.router_fwd(xd, wd, bd, k, "sum", want_logits=True))
    for t0 in range(0, T, 64):
        part = ops.router_fwd(xd[t0:t0 + 64], wd, bd, k, "sum", want_logits=True)
        for whole, few in zip((idx, w, logits), part):
            assert torch.equal(whole[t0:t0 + 64], few.cpu())
    # H products of fp32 sums: |error| <= H * 2^-24 * sum |x w|, times 2 for the matrix unit's own order
    bound = (x.double().abs() @ wr.double().abs().t()) * H * 2.0 ** -23
    assert bool(((logits.double() - x.double() @ wr.double().t()).abs() <= bound).all())
    oi, ow, _ = O.route_from_logits(logits.numpy(), bias.numpy(), k, "sum")
    assert np.array_equal(idx.numpy(), oi) and np.array_equal(w.numpy(), ow)


@pytest.mark.parametrize("H", [128, 640, 768, 896, 1024])
@pytest.mark.parametrize("T,E,k", [(127, 9, 2), (128, 64, 6), (1000, 64, 6), (4096, 64, 8), (4097, 33, 4), (8192, 64, 6), (8197, 64, 6)])
def test_behind_the_norm(H, T, E, k):
    """The same kernel shapes with the RMSNorm in front: the bits of the norm and the router on their own."""
    g = torch.Generator().manual_seed(H + T)
    I = 128
    x = torch.randn(T, H, generator=g).bfloat16().to(DEV)
    nw = (torch.rand(H, generator=g) + 0.5).to(DEV)
    wr = (torch.randn(E, H, generator=g) * 0.1).bfloat16().to(DEV)
    bias = (torch.rand(E, generator=g) * 0.02 - 0.01).to(DEV)
    gu = (torch.randn(E, 2 * I, H, generator=g) * 0.05).bfloat16().to(DEV)
    dn = (torch.randn(E, H, I, generator=g) * 0.05).bfloat16().to(DEV)
    th = torch.zeros(E, device=DEV)
    got = ops.ffn_forward(x, nw, 1e-6, wr, bias, gu, dn, th, k, want_routing=True)
    xn = ops.rmsnorm_fwd(x, nw, 1e-6)
    idx, w, _, _ = ops.router_fwd(xn, wr, bias, k, "sum")
    assert torch.equal(got[1], idx) and torch.equal(got[2], w)
    out = ops.moe_forward(xn, wr, bias, gu, dn, th, k)[0]
    assert float((got[0].double() - (x.double() + out.double())).abs().max()) <= 2.0 ** -7 * float((x.double() + out.double()).abs().max())
