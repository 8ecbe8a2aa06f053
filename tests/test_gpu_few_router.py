"""One launch for a token's routing and its experts' gate/up pass: the routing of the router's own launch, and the same bits token by token
as in a call of several, whose workgroups take several blocks of rows; every chunk count of a row, few and many experts, experts of a width no workgroup divides, +/-Identity."""
import pytest
import torch

from bibo_amd import ops

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("H", [128, 256, 384, 512, 640, 768, 896, 1024])
@pytest.mark.parametrize("Eg,pairs,k,I", [(64, 0, 6, 384), (62, 1, 6, 384), (64, 0, 8, 512), (5, 0, 2, 488), (1, 1, 3, 504)])
def test_token_by_token(H, Eg, pairs, k, I):
    g = torch.Generator().manual_seed(H + I)
    T, E = 48 // k, Eg + 2 * pairs
    x = torch.randn(T, H, generator=g).bfloat16().to(DEV)
    args = [t.to(DEV) for t in ((torch.randn(E, H, generator=g) * 0.1).bfloat16(), torch.rand(E, generator=g) * 0.02 - 0.01,
                                (torch.randn(Eg, 2 * I, H, generator=g) * 0.05).bfloat16(),
                                (torch.randn(Eg, H, I, generator=g) * 0.05).bfloat16(), torch.randn(Eg, generator=g))]
    kw = dict(n_pos=pairs, n_neg=pairs, want_routing=True, want_logits=True)
    whole = ops.moe_forward(x, *args, k, **kw)
    alone = ops.router_fwd(x, args[0], args[1], k, "sum", want_logits=True)
    for i, ref in zip((1, 2, 4), alone):
        assert torch.equal(whole[i], ref)
    for t in range(T):
        one = ops.moe_forward(x[t:t + 1], *args, k, want_counts=t % 2 == 1, **kw)
        for i in (0, 1, 2, 4):
            assert torch.equal(one[i], whole[i][t:t + 1])
        if t % 2 == 1:
            assert torch.equal(one[3], torch.bincount(one[1].flatten().long(), minlength=E).int())
    # behind the norm: the bits of the norm, the layer and the sum on their own
    nw = (torch.rand(H, generator=g) + 0.5).to(DEV)
    kw = dict(n_pos=pairs, n_neg=pairs)
    xn = ops.rmsnorm_fwd(x, nw, 1e-6)
    seam = ops.ffn_forward(x, nw, 1e-6, *args, k, want_routing=True, residual=False, **kw)
    ref = ops.moe_forward(xn, *args, k, want_routing=True, **kw)
    for a, b in zip(seam[:3], ref[:3]):
        assert torch.equal(a, b)
