"""Calls that leave the streaming kernels for tiles keep their fp32 rows between the experts and the combine: the output is what one gets by
rounding the activations and the sum, and nothing else, to bf16.  Fused and cut tiles, every width of a column block, +/-Identity experts,
the seam, a caller's own routing."""
import numpy as np
import pytest
import torch

from bibo_amd import ops
from oracle import bibo_moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _rows_in_64_bits(x, idx, w, gu, dn, th):
    out = torch.zeros(x.shape, dtype=torch.float64)
    for e in range(gu.shape[0]):
        t, j = np.nonzero(idx == e)
        if len(t) == 0:
            continue
        h = O.expert_hidden(x[t].double(), gu[e].double(), th[e].double()).bfloat16().double()
        out.index_add_(0, torch.from_numpy(t), h @ dn[e].double().T * w[t, j].double()[:, None])
    return out


# An activation whose fp32 value lies within its error, 1e-6, of the middle of two bf16 numbers, 2^-8 apart, goes to the other one: about 1 in
# 2000 of k I, one or two a token, each moving an output by 2^-9 of one of k I terms, 2^-9 / sqrt(k I) of it.  That takes one output in
# 20 sqrt(k I) / 2 across a middle, below 1 %; with 16-bit rows two outputs in five differ (one expert per token: none, the sum is the row).
@pytest.mark.parametrize("T,H,I,E,k", [(250, 512, 256, 64, 6), (200, 512, 256, 64, 6), (250, 512, 128, 64, 6), (220, 384, 256, 64, 4),
                                       (1000, 128, 128, 48, 1), (150, 512, 384, 64, 6), (120, 512, 512, 64, 8), (190, 384, 384, 32, 4),
                                       (130, 1024, 512, 64, 8), (60, 1024, 512, 16, 4), (66, 1024, 512, 9, 2), (130, 640, 512, 64, 6)])
def test_only_activations_and_sums_are_rounded(T, H, I, E, k):
    p = O.make_inputs(T=T, H=H, E=E, k=k, I=I, theta="normal", bias="uniform", seed=T + I)
    assert T * k > (704 if H <= 512 and I <= 512 else 11 * E) and ops.select_algo(T, H, E, k, I) == "stream"
    args = [p[n].to(DEV) for n in ("w_router", "bias", "w_gate_up", "w_down", "theta")]
    x = p["x"].to(DEV)
    out, idx, w, _, _ = ops.moe_forward(x, *args, k, want_routing=True)
    ref = _rows_in_64_bits(p["x"], idx.cpu().numpy(), w.cpu(), p["w_gate_up"], p["w_down"], p["theta"])
    assert float((out.cpu() != ref.bfloat16()).double().mean()) < 0.02
    # with a permutation of the rows, and a caller's indices
    assert torch.equal(ops.moe_forward(x, *args, k, want_counts=True)[0], out)
    assert torch.equal(ops.experts_fwd(x, idx, w, *args[2:])[0], out)


def test_identity_and_seam():
    T, H, I, Eg, k = 240, 512, 256, 62, 6
    p = O.make_inputs(T=T, H=H, E=Eg + 2, k=k, I=I, theta="normal", bias="uniform", seed=3)
    gu, dn, th = p["w_gate_up"][:Eg], p["w_down"][:Eg], p["theta"][:Eg]
    p["bias"][[0, 62, 63]] = 2.0
    args = [t.to(DEV) for t in (p["w_router"], p["bias"], gu, dn, th)]
    nw = torch.rand(H, generator=torch.Generator().manual_seed(1)) + 0.5
    h = p["x"].to(DEV)
    kw = dict(n_pos=1, n_neg=1, want_routing=True)
    seam, idx, w = ops.ffn_forward(h, nw.to(DEV), 1e-6, *args, k, **kw)[:3]
    xn = ops.rmsnorm_fwd(h, nw.to(DEV), 1e-6)
    i, wc, xc = idx.cpu().numpy(), w.cpu(), xn.cpu()
    ref = _rows_in_64_bits(xc, i, wc, gu, dn, th)
    for e, sign in ((Eg, 1), (Eg + 1, -1)):
        t, j = np.nonzero(i == e)
        assert len(t) == T
        ref[t] += sign * wc[t, j].double()[:, None] * xc[t].double()
    assert float((seam.cpu() != (ref + p["x"].double()).bfloat16()).double().mean()) < 0.02
