"""The three products of the backward pass that share a launch (dx of every slot, dW_gate_up, dW_down), on 128-row tiles and on 256-row ones
(experts of 128 rows and more on average, several rounds of workgroups), over the widths their workgroups divide into; against autograd in fp32."""
import ctypes

import pytest
import torch

from bibo_amd import _lib as L
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


def _weight_grads_f32(x, d, idx, w, wgu, wd, theta):
    """Both weight gradients of bibo_moe_experts_backward in fp32, as for the masters of mixed-precision training."""
    (T, H), (E, _, I), k = x.shape, wd.shape, idx.shape[1]
    sh = L.Shape(T, H, E, k, I, 0, 0, 0, 0, L.FLAG_GRAD_F32)
    need = ctypes.c_size_t(0)
    L.check(L.lib().bibo_moe_backward_workspace_bytes(ctypes.byref(sh), ctypes.byref(need)), "bytes")
    ws = torch.empty(need.value + 256, dtype=torch.uint8, device=DEV)
    dx, dw, dth = torch.empty_like(x), torch.empty_like(w), torch.empty_like(theta)
    dgu, ddn = (torch.empty(t.shape, dtype=torch.float32, device=DEV) for t in (wgu, wd))
    ptr = [ctypes.c_void_p(t.data_ptr()) for t in (x, d, idx, w, wgu, wd, theta)]
    out = [ctypes.c_void_p(t.data_ptr()) for t in (dx, dw, dgu, ddn, dth)]
    L.check(L.lib().bibo_moe_experts_backward(*ptr, ctypes.byref(sh), *out, ctypes.c_void_p((ws.data_ptr() + 255) & ~255), need.value,
                                              ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "bibo_moe_experts_backward")
    return dx, None, dgu, ddn


# An expert's rows are a loop over stages of 32 in rings of four (128-row tiles) or three (256-row ones): no stage, less than a ring, every
# remainder, and last stages of one row and of all but one.
@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("H,I,counts", [(256, 128, [0, 1, 2, 31, 32, 33, 63, 64, 65, 96, 97, 127, 128, 129, 159, 161, 225, 256]),
                                        (768, 384, [0, 1, 33] + [193 + 5 * i for i in range(61)]),
                                        (512, 256, [0, 1, 255, 256, 257] + [98 + i for i in range(59)]),       # 128 rows and more on average
                                        (512, 256, [0, 1, 255, 256, 257] + [96 + i for i in range(59)]),       # and less
                                        # 128-row tiles of dW_down (H no multiple of 256) beside 256-row ones of the others: three stages behind
                                        # the last full ring of four, the loads of their row indices gone
                                        (640, 128, [65 + i for i in range(32)] + [193 + i for i in range(32)]),
                                        (640, 256, [65 + i for i in range(32)] + [193 + i for i in range(32)]),
                                        (384, 384, [65 + i for i in range(32)] + [193 + i for i in range(32)]),
                                        (384, 256, [193 + i for i in range(32)] + [321 + i for i in range(32)]),
                                        # two stages, fewer than a ring of three: in whole experts and in the last chunk of cut ones
                                        (768, 384, [33 + i for i in range(32)] + [545 + i for i in range(32)])])
def test_rows_of_an_expert(H, I, counts, f32):
    E, T = len(counts), sum(counts)
    p = O.make_inputs(T=8, H=H, E=E, k=1, I=I, theta="normal", seed=E)
    g = torch.Generator().manual_seed(E)
    x, d = (torch.randn(T, H, generator=g).bfloat16().to(DEV) for _ in range(2))
    idx = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=g)].to(torch.int32)[:, None].to(DEV)
    w = torch.rand(T, 1, generator=g).to(DEV)
    wgu, wd, theta = (p[n].to(DEV) for n in ("w_gate_up", "w_down", "theta"))
    dx, _, dgu, ddn = (_weight_grads_f32 if f32 else ops.experts_backward)(x, d, idx, w, wgu, wd, theta)[:4]
    for name, a, ref in zip(("dx", "dW_gate_up", "dW_down"), (dx, dgu, ddn), _reference(x, d, idx, w, wgu, wd, theta)):
        assert float((a.float() - ref).norm() / ref.norm()) <= 1e-2, name
        if name == "dx":
            continue
        for e in range(E):          # an expert at a time: a row too many or too few of one does not drown in the others
            assert float((a[e].float() - ref[e]).norm()) <= 2e-2 * float(ref[e].norm()) + 1e-6, (name, e, counts[e])


def test_weight_gradients_of_4_gib():
    """One expert whose fp32 gate/up gradient holds 2^32 bytes: offsets into it do not fit 32 bits."""
    T, H, E, I = 40, 1 << 20, 1, 512
    g = torch.Generator(device=DEV).manual_seed(1)
    rand = lambda *shape: torch.randn(*shape, generator=g, device=DEV, dtype=torch.bfloat16)
    try:
        x, d, wgu, wd = rand(T, H), rand(T, H), rand(E, 2 * I, H) * 1e-3, rand(E, H, I) * 1e-3
        idx, w = torch.zeros(T, 1, dtype=torch.int32, device=DEV), torch.rand(T, 1, generator=g, device=DEV)
        theta = torch.zeros(E, device=DEV)
        dx, _, dgu, ddn = _weight_grads_f32(x, d, idx, w, wgu, wd, theta)
        assert dgu.numel() * dgu.element_size() >= 2 ** 32
        for name, a, ref in zip(("dx", "dW_gate_up", "dW_down"), (dx, dgu, ddn), _reference(x, d, idx, w, wgu, wd, theta)):
            assert float((a.float() - ref).norm() / ref.norm()) <= 1e-2, name
    finally:
        torch.cuda.empty_cache()
