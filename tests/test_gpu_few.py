"""The few-token kernels (experts_few.hip) at the edges of their range: one slot to kFewSlots, widths that end inside a
lane's granules, experts shared by several slots, padded indices, +/-Identity experts, residuals; against the fp64 oracle."""
import numpy as np
import pytest
import torch

from bibo_amd import ops
from oracle import bibo_moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _rel(a, ref):
    return float((a.double().cpu() - ref.double()).abs().max() / ref.double().abs().max().clamp_min(1e-30))


@pytest.mark.parametrize("T,H,Eg,pairs,k,I", [(1, 8, 1, 0, 1, 8), (1, 768, 64, 0, 6, 384), (8, 1024, 64, 0, 6, 512), (6, 136, 9, 1, 8, 88),
                                              (48, 256, 3, 0, 1, 128), (3, 1016, 5, 2, 4, 504), (5, 520, 62, 1, 6, 264)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("act", ["radial", "silu"])
def test_few_tokens(T, H, Eg, pairs, k, I, dtype, act):
    E = Eg + 2 * pairs
    p = O.make_inputs(T=T, H=H, E=Eg, k=min(k, Eg), I=I, theta="normal", seed=T + H, dtype=dtype)
    g = torch.Generator().manual_seed(T)
    p["w_router"] = (torch.randn(E, H, generator=g) * 0.1).to(dtype)
    p["bias"] = torch.rand(E, generator=g) * 0.02 - 0.01
    args = [p[n].to(DEV) for n in ("w_router", "bias", "w_gate_up", "w_down", "theta")]
    kw = dict(n_pos=pairs, n_neg=pairs, act=act)
    out, idx, w, counts, logits = ops.moe_forward(p["x"].to(DEV), *args, k, want_routing=True, want_counts=True, want_logits=True, **kw)
    torch.cuda.synchronize()
    idx, w = idx.cpu().numpy(), w.cpu().numpy()
    ri, rw = O.route_from_logits(logits.cpu().numpy(), p["bias"].numpy(), k)[:2]
    assert np.array_equal(ri, idx) and np.array_equal(rw, w)
    assert np.array_equal(np.bincount(ri.ravel(), minlength=E), counts.cpu().numpy())
    ref = O.experts_forward(p["x"], idx, w, p["w_gate_up"], p["w_down"], p["theta"], dtype=torch.float64, **kw)
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    assert _rel(out, ref) <= tol
    # the seam: rmsnorm in front, another tensor added behind
    nw, res = torch.rand(H, generator=g) + 0.5, torch.randn(T, H, generator=g).to(dtype)
    seam = ops.ffn_forward(p["x"].to(DEV), nw.to(DEV), 1e-6, *args, k, residual=res.to(DEV), want_routing=True, **kw)
    xn = ops.rmsnorm_fwd(p["x"].to(DEV), nw.to(DEV), 1e-6).cpu()
    blk = O.experts_forward(xn, seam[1].cpu().numpy(), seam[2].cpu().numpy(), p["w_gate_up"], p["w_down"], p["theta"],
                            dtype=torch.float64, **kw)
    assert _rel(seam[0], blk + res.double()) <= tol
    # a caller's indices: every slot on one expert, one slot padded
    idx1 = np.full((T, k), Eg - 1, np.int32)
    idx1[0, k - 1] = -1
    got, _ = ops.experts_fwd(p["x"].to(DEV), torch.from_numpy(idx1).to(DEV), torch.from_numpy(w).to(DEV), *args[2:], **kw)
    torch.cuda.synchronize()
    w1 = w.copy()
    w1[0, k - 1] = 0.0
    ref = O.experts_forward(p["x"], np.full((T, k), Eg - 1, np.int32), w1, p["w_gate_up"], p["w_down"], p["theta"], dtype=torch.float64, **kw)
    assert float((got.double().cpu() - ref.double()).abs().max()) <= tol * max(float(ref.abs().max()), 1e-3)
