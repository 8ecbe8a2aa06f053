"""The fp32 tile kernels of the generic family (tile_f32.h) at the edges of their tiles: row counts around 16 and 64 per
expert, widths below, at and past 64 columns, contractions that end inside a step of 32, widths that are no multiples of
four (the row kernels), +/-Identity experts; forward and backward against the fp64 oracle."""
import numpy as np
import pytest
import torch

from bibo_amd import ops
from oracle import bibo_moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _rel(a, ref):
    return float((a.double().cpu() - ref.double()).abs().max() / ref.double().abs().max().clamp_min(1e-30))


# the same with more than 96 rows per expert on average, where the 64-row tiles run in both directions
TALL = [(130, 100, 1, 0, 1, 28), (194, 68, 2, 0, 1, 36), (200, 132, 1, 1, 2, 64), (449, 64, 4, 0, 1, 128), (400, 260, 2, 1, 3, 132)]


@pytest.mark.parametrize("T,H,Eg,pairs,k,I", TALL)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_tall_tile_edges(T, H, Eg, pairs, k, I, dtype):
    test_tile_edges(T, H, Eg, pairs, k, I, dtype)


@pytest.mark.parametrize("T,H,Eg,pairs,k,I", [(1, 64, 8, 0, 2, 32), (12, 68, 2, 0, 2, 36), (24, 132, 4, 0, 2, 64), (63, 100, 2, 0, 1, 28),
                                              (65, 64, 1, 1, 2, 64), (129, 192, 14, 1, 3, 88), (200, 66, 4, 0, 2, 33),
                                              (17, 260, 64, 0, 8, 132), (300, 516, 5, 2, 4, 260)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_tile_edges(T, H, Eg, pairs, k, I, dtype):
    E = Eg + 2 * pairs
    p = O.make_inputs(T=T, H=H, E=Eg, k=min(k, Eg), I=I, theta="normal", seed=T + H, dtype=dtype)
    g = torch.Generator().manual_seed(T)
    p["w_router"] = (torch.randn(E, H, generator=g) * 0.1).to(dtype)
    p["bias"] = torch.rand(E, generator=g) * 0.02 - 0.01
    d_out = torch.randn(T, H, generator=g).to(dtype)
    args = [p[n].to(DEV) for n in ("w_router", "bias", "w_gate_up", "w_down", "theta")]
    kw = dict(n_pos=pairs, n_neg=pairs)
    out, idx, w, counts, logits = ops.moe_forward(p["x"].to(DEV), *args, k, want_routing=True, want_counts=True, want_logits=True, **kw)
    got = ops.moe_backward(p["x"].to(DEV), d_out.to(DEV), *args, k, want_dw=True, **kw)
    torch.cuda.synchronize()
    idx, w = idx.cpu().numpy(), w.cpu().numpy()
    lg = p["x"].double() @ p["w_router"].double().t()
    assert _rel(logits, lg) <= 1e-5
    ri, rw = O.route_from_logits(logits.cpu().numpy(), p["bias"].numpy(), k)[:2]
    assert np.array_equal(ri, idx) and np.array_equal(rw, w)
    assert np.array_equal(np.bincount(ri.ravel(), minlength=E), counts.cpu().numpy())
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    ref = O.experts_forward(p["x"], idx, w, p["w_gate_up"], p["w_down"], p["theta"], dtype=torch.float64, **kw)
    assert _rel(out, ref) <= tol
    grads = O.moe_backward(p["x"], p["w_router"], p["w_gate_up"], p["w_down"], p["theta"], idx, d_out, **kw)
    # one token: a single cancelling dot product decides a tensor's largest entry
    for name, a in zip(("x", "w_router", "w_gate_up", "w_down", "theta", "w"), got):
        assert _rel(a, grads[name]) <= (tol if T > 1 else 4 * tol), name


@pytest.mark.parametrize("H,I", [(736, 304), (768, 280), (768, 288), (576, 88)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_half_filled_tiles_repeat(H, I, dtype):
    """32 rows of 64-row tiles, contractions of odd and even numbers of steps: the waves without rows must not bring in what their registers
    held.  Bit for bit what the same tokens give where every wave has rows, whatever ran before."""
    E, T = 16, 1024
    p = O.make_inputs(T=T, H=H, E=E, k=1, I=I, theta="normal", seed=I, dtype=dtype)
    g = torch.Generator().manual_seed(H)
    x, d = p["x"].to(DEV), torch.randn(T, H, generator=g).to(dtype).to(DEV)
    idx = (torch.arange(T) % E).to(torch.int32)[:, None].to(DEV)
    w = torch.rand(T, 1, generator=g).to(DEV)
    wgu, wd, theta = (p[n].to(DEV) for n in ("w_gate_up", "w_down", "theta"))
    run = lambda n: (ops.experts_fwd(x[:n], idx[:n], w[:n], wgu, wd, theta)[0], ops.experts_backward(x[:n], d[:n], idx[:n], w[:n], wgu, wd, theta)[0])
    full = run(T)
    for i in range(6):
        dirt = torch.full((2048, 2048), (float("nan"), float("inf"), 1.0)[i % 3], device=DEV, dtype=(torch.float32, torch.bfloat16)[i % 2])
        dirt @ dirt
        for name, a, b in zip(("out", "d_x"), run(T // 2), full):
            assert torch.equal(a, b[:T // 2]), (name, i)
