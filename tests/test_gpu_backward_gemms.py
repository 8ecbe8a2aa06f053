"""The three products of the backward pass that share a launch (dx of every slot, dW_gate_up, dW_down), on 128-row tiles and on 256-row ones
(experts of 192 rows and more, several rounds of workgroups), over the widths their workgroups divide into; against autograd in fp32."""
import pytest
import torch

from bibo_amd import ops
from oracle import bibo_moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _reference(x, d, idx, w, wgu, wd, theta):
    x, wgu, wd = (t.float().requires_grad_() for t in (x, wgu, wd))
    I = wd.shape[2]
    out = torch.zeros(x.shape, device=x.device)
    for e in range(wgu.shape[0]):
        t, j = (idx == e).nonzero(as_tuple=True)
        g, u = (x[t] @ wgu[e].T).split(I, -1)
        r = (g.pow(2).mean(-1, keepdim=True) + 1e-6).sqrt()
        h = r ** torch.sigmoid(theta[e]) * torch.nn.functional.silu(g / r) * u
        out = out.index_add(0, t, (h @ wd[e].T) * w[t, j][:, None])
    out.backward(d.float())
    return x.grad, wgu.grad, wd.grad


@pytest.mark.parametrize("T,H,I,E,k", [(100, 384, 128, 3, 2), (400, 256, 384, 5, 2), (700, 640, 256, 4, 1), (300, 768, 512, 9, 2),      # 128 rows
                                       (10000, 640, 128, 4, 2), (24000, 768, 384, 4, 2), (24000, 512, 256, 5, 2), (8100, 1024, 512, 4, 2),
                                       (10000, 640, 384, 4, 2)])                                                                     # 256 rows
def test_products(T, H, I, E, k):
    p = O.make_inputs(T=8, H=H, E=E, k=k, I=I, theta="normal", seed=T)
    g = torch.Generator().manual_seed(T)
    x, d = (torch.randn(T, H, generator=g).bfloat16().to(DEV) for _ in range(2))
    hot = torch.rand(T, E, generator=g) + torch.linspace(0, 0.3, E)              # ragged: the last experts hold more rows
    idx = hot.topk(k, -1).indices.sort(-1).values.to(torch.int32).to(DEV)
    w = torch.rand(T, k, generator=g).to(DEV)
    wgu, wd, theta = (p[n].to(DEV) for n in ("w_gate_up", "w_down", "theta"))
    dx, _, dgu, ddn = ops.experts_backward(x, d, idx, w, wgu, wd, theta)[:4]
    for name, a, ref in zip(("dx", "dW_gate_up", "dW_down"), (dx, dgu, ddn), _reference(x, d, idx, w, wgu, wd, theta)):
        assert float((a.float() - ref).norm() / ref.norm()) <= 1e-2, name
        assert float((a.float() - ref).abs().max() / ref.abs().max()) <= 2e-2, name
