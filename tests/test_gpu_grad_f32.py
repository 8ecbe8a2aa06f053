"""BIBO_FLAG_GRAD_F32: under bf16 autocast the gradients of fp32 master weights are the kernels' fp32 sums; rounded to bf16
they are the gradients a layer with bf16 weights of the same values gets, bit for bit."""
import pytest
import torch

import bibo_amd

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("T,H,I,E,k,pairs,hot", [(1, 128, 128, 8, 2, 0, 0), (700, 256, 384, 16, 4, 1, 0), (3000, 256, 128, 16, 2, 0, 1),
                                                 (900, 768, 512, 4, 2, 0, 0),                      # 256-row tiles
                                                 (50, 72, 36, 6, 2, 1, 0), (40, 66, 34, 6, 2, 0, 0)])   # generic family
@pytest.mark.parametrize("keep", [True, False])
def test_fp32_gradients_round_to_the_bf16_ones(T, H, I, E, k, pairs, hot, keep):
    torch.manual_seed(T + H)
    cfg = bibo_amd.BiBoMoEConfig(hidden_size=H, moe_intermediate_size=I, num_routed_experts=E, num_experts_per_tok=k,
                                 special_expert_pairs=pairs, bias_update_factor=0.0)
    low = bibo_amd.BiBoMoELayer(cfg).to(DEV)
    with torch.no_grad():
        low.experts.radial_theta.normal_(0, 0.5)
        low.gate.bias[:hot] = 2.0
    for p in (low.gate.gate_proj.weight, low.experts.gate_up_proj, low.experts.down_proj):
        p.data = p.data.bfloat16()
    master = bibo_amd.BiBoMoELayer(cfg).to(DEV)
    master.load_state_dict(low.state_dict())                       # fp32 copies of the same bf16 values
    low.keep_activations = master.keep_activations = keep
    x = torch.randn(1, T, H, device=DEV).bfloat16()
    d = torch.randn(1, T, H, device=DEV).bfloat16()
    xs = [x.clone().requires_grad_(), x.clone().requires_grad_()]
    out = low(xs[0])
    with torch.autocast("cuda", dtype=torch.bfloat16):
        out2 = master(xs[1])
    assert torch.equal(out, out2)
    out.backward(d)
    out2.backward(d)
    assert torch.equal(xs[0].grad, xs[1].grad)
    for (n, a), b in zip(low.named_parameters(), master.parameters()):
        if a.requires_grad:
            assert b.grad.dtype == torch.float32 and torch.equal(a.grad, b.grad.to(a.grad.dtype)), n
            if a.dtype == torch.bfloat16:
                assert not torch.equal(a.grad.float(), b.grad), n      # more than the bf16 gradient widened
