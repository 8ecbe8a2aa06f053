"""Training forwards that keep routing, permutation and, on the fp32 tile kernels, pre-activations for their backward pass, for the shapes the
fused kernel does not take: the same outputs and gradients, bit for bit, as a backward pass that computes them again, and again from the
same graph."""
import pytest
import torch

import bibo_amd
from bibo_amd import _lib as L

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
F32, BF16 = torch.float32, torch.bfloat16

CASES = [  # dtype, T, H, I, E, k, pairs
    (F32, 777, 192, 88, 16, 3, 0),      # fp32 tiles
    (F32, 130, 64, 512, 9, 2, 1),       # 2 I > H, +/-Identity experts: rows without pre-activations
    (F32, 4100, 256, 128, 4, 2, 0),     # tall tiles
    (F32, 17, 64, 32, 8, 3, 0),         # 51 slots, the fewest on tiles
    (F32, 16, 64, 32, 8, 3, 0),         # 48: few-token kernels, no pre-activations
    (F32, 1, 64, 32, 8, 3, 0),
    (F32, 60, 50, 30, 5, 2, 1),         # no tile divides it: a workgroup per row
    (BF16, 200, 200, 72, 8, 2, 0),      # bf16 on fp32 tiles
    (BF16, 40, 256, 512, 8, 2, 0),      # I = 512: streaming, then tiles cut by columns, one round of tiles and several
    (BF16, 300, 256, 512, 8, 2, 1),
    (BF16, 300, 1024, 512, 8, 2, 0),    # whose workgroups find their rows themselves
    (BF16, 1500, 256, 512, 8, 4, 0),
    (BF16, 9000, 128, 512, 40, 4, 0),
]


def _train(layer, x, d_out, twice=False):
    x.grad = None
    layer.zero_grad(set_to_none=True)
    out = layer(x)
    out.backward(d_out, retain_graph=twice)
    grads = lambda: [x.grad.clone(), *(p.grad.clone() for p in layer.parameters() if p.grad is not None)]
    first = grads()
    if twice:
        x.grad = None
        layer.zero_grad(set_to_none=True)
        layer(torch.randn_like(x)).sum().backward()          # somebody else's pass over the same workspace
        x.grad = None
        layer.zero_grad(set_to_none=True)
        out.backward(d_out)
        for a, b in zip(first, grads()):
            assert torch.equal(a, b)
    return [out.detach(), *first, layer.gate.bias.detach().clone()]


@pytest.mark.parametrize("dtype,T,H,I,E,k,pairs", CASES)
def test_kept_state(dtype, T, H, I, E, k, pairs):
    res = []
    for keep in (True, False):
        torch.manual_seed(T)
        cfg = bibo_amd.BiBoMoEConfig(hidden_size=H, moe_intermediate_size=I, num_routed_experts=E, num_experts_per_tok=k,
                                     special_expert_pairs=pairs)
        layer = bibo_amd.BiBoMoELayer(cfg).to(DEV).train()
        for p in (layer.gate.gate_proj.weight, layer.experts.gate_up_proj, layer.experts.down_proj):
            p.data = (torch.randn(p.shape, device=DEV) * 0.1).to(dtype)
        layer.keep_activations = keep
        x = torch.randn(1, T, H, device=DEV).to(dtype).requires_grad_()
        res.append(_train(layer, x, torch.randn(1, T, H, device=DEV).to(dtype), twice=keep)[:-1])
    assert len(res[0]) == len(res[1]) == 6
    for a, b in zip(*res):
        assert torch.equal(a, b)
    assert float(res[0][1].float().abs().max()) > 0


def test_which_shapes_keep_what():
    import ctypes
    n = ctypes.c_size_t(0)

    def size(flags, *dims):
        sh = L.Shape(*dims)
        sh.flags = flags
        rc = L.lib().bibo_moe_train_state_bytes(ctypes.byref(sh), ctypes.byref(n))
        return n.value if rc == 0 else rc

    tiles, rows, wide = (777, 192, 16, 3, 88, L.DTYPE_F32), (60, 50, 5, 2, 30, L.DTYPE_F32), (1500, 256, 8, 4, 512, L.DTYPE_BF16)
    for dims in (tiles, rows, wide):
        assert size(0, *dims) == -6
    assert L.FLAG_KEEP_ANY == 32
    assert size(32, *tiles) >= 777 * 3 * (2 * 88 * 4 + 16)
    assert 0 < size(32, *rows) < 60 * 2 * 2 * 30 * 4 + 8192
    assert 0 < size(32, *wide) < 1500 * 4 * 2 * 512
    fused = (1500, 256, 8, 4, 256, L.DTYPE_BF16)
    assert size(32, *fused) == size(0, *fused)
