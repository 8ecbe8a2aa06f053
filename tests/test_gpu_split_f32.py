"""The fp32 products on bf16 matrix instructions (three bf16 parts per number): tiles of 64 and 128 rows at their edges, contractions with
and without a partial step, both directions; numbers that bf16 rounds to infinity; infinities and NaNs; against the oracle in float64."""
import numpy as np
import pytest
import torch

from bibo_amd import ops
from oracle import bibo_moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
NAMES = ("w_router", "bias", "w_gate_up", "w_down", "theta")


def _rel(a, ref):
    return float((a.double().cpu() - ref.double()).norm() / ref.double().norm())


def _inputs(H, I, rows, seed):
    E, T = len(rows), sum(rows)
    p = O.make_inputs(T=T, H=H, E=E, k=1, I=I, theta="normal", seed=seed, dtype=torch.float32)
    idx = np.repeat(np.arange(E, dtype=np.int32), rows)
    np.random.default_rng(seed).shuffle(idx)
    w = np.random.default_rng(seed + 1).random((T, 1)).astype(np.float32)
    return p, idx.reshape(T, 1), w


def _forward(p, idx, w, act="radial"):
    return ops.experts_fwd(p["x"].to(DEV), torch.from_numpy(idx).to(DEV), torch.from_numpy(w).to(DEV),
                           *(p[n].to(DEV) for n in ("w_gate_up", "w_down", "theta")), act=act)[0]


# 64 x 64 tiles while 128 x 128 ones are fewer than 128, which the second list is not; a result is up to 1000 / 32 sums rounded to 2^-24,
# of which each can be off by the 2-norm bound 2^-24 sqrt(steps) < 4e-7; three of them follow one another
@pytest.mark.parametrize("H,I", [(512, 256), (516, 260), (1000, 504), (640, 36)])
@pytest.mark.parametrize("rows", [(63, 64, 65, 129, 0, 1, 400, 500), (127, 128, 129, 1, 0, 1000, 2000, 900)])
def test_forward(H, I, rows):
    p, idx, w = _inputs(H, I, rows, H + I)
    ref = O.experts_forward(p["x"], idx, w, p["w_gate_up"], p["w_down"], p["theta"], dtype=torch.float64)
    assert _rel(_forward(p, idx, w), ref) <= 1.2e-6


@pytest.mark.parametrize("T,H,I,E,k", [(300, 64, 32, 4, 2), (777, 192, 88, 16, 3), (500, 516, 260, 8, 2), (1200, 640, 256, 9, 2), (40, 1000, 504, 8, 1)])
def test_backward(T, H, I, E, k):
    p = O.make_inputs(T=T, H=H, E=E, k=k, I=I, bias="uniform", theta="normal", seed=T, dtype=torch.float32)
    d = torch.randn(T, H, generator=torch.Generator().manual_seed(T))
    args = [p[n].to(DEV) for n in NAMES]
    got = ops.moe_backward(p["x"].to(DEV), d.to(DEV), *args, k)
    idx = ops.moe_forward(p["x"].to(DEV), *args, k, want_routing=True)[1].cpu().numpy()
    ref = O.moe_backward(p["x"], p["w_router"], p["w_gate_up"], p["w_down"], p["theta"], idx, d)
    for name, a in zip(("x", "w_router", "w_gate_up", "w_down"), got):
        assert _rel(a, ref[name]) <= 2e-6, name


@pytest.mark.parametrize("rows", [(400, 800), (2000, 2400)])
def test_numbers_that_bf16_rounds_to_infinity(rows):
    """3.4e38 is finite in fp32 and infinite in bf16; the weights it meets are small enough for a finite sum."""
    p, idx, w = _inputs(1024, 512, rows, 5)
    p["x"][7::50, 3] = 3.4e38
    p["w_gate_up"][:, :, 3] = torch.randn(2, 1024, generator=torch.Generator().manual_seed(1)) * 1e-38
    ref = O.experts_forward(p["x"], idx, w, p["w_gate_up"], p["w_down"], p["theta"], dtype=torch.float64)
    got = _forward(p, idx, w)
    assert torch.isfinite(got).all() and _rel(got, ref) <= 1.2e-6


@pytest.mark.parametrize("rows", [(400, 800), (2000, 2400)])
def test_infinities_and_nans_stay_where_they_are(rows):
    """An infinity in a row of d makes its row of dW_down infinite, not NaN; NaN spreads over what it is multiplied with and no further."""
    p, idx, w = _inputs(1024, 512, rows, 6)
    T = sum(rows)
    d = torch.randn(T, 1024, generator=torch.Generator().manual_seed(2))
    a, b = int(np.flatnonzero(idx[:, 0] == 0)[0]), int(np.flatnonzero(idx[:, 0] == 1)[0])
    d[a, 5], d[b, 900] = float("inf"), float("nan")
    dx, _, dgu, ddn = ops.experts_backward(p["x"].to(DEV), d.to(DEV), torch.from_numpy(idx).to(DEV), torch.from_numpy(w).to(DEV),
                                           *(p[n].to(DEV) for n in ("w_gate_up", "w_down", "theta")))[:4]
    ddn = ddn.cpu()
    assert torch.isinf(ddn[0, 5]).all() and torch.isnan(ddn[1, 900]).all()
    bad = torch.zeros(2, 1024, dtype=torch.bool)
    bad[0, 5] = bad[1, 900] = True
    assert torch.equal(~torch.isfinite(ddn).all(-1), bad)
    rest = torch.ones(T, dtype=torch.bool)
    rest[[a, b]] = False
    assert torch.isfinite(dx.cpu()[rest]).all() and not torch.isfinite(dx.cpu()[[a, b]]).any()
    x = p["x"].clone()
    x[a, 1] = float("nan")
    out = _forward({**p, "x": x}, idx, w).cpu()
    assert torch.isnan(out[a]).all() and torch.isfinite(out[rest]).all()


# bf16 ends at 2^-133, so a number below 2^-110 is not the sum of three bf16 parts.  2^-118 loses bits from 2^-15 of it down, 2^-130 is a
# subnormal itself.  The results are in the usual range, or as far above 2^-149 as their bound needs
@pytest.mark.parametrize("e", [112, 118, 130])
@pytest.mark.parametrize("rows", [(400, 800), (2000, 2400)])
def test_small_numbers(rows, e):
    p, idx, w = _inputs(516, 260, rows, 7)
    p["x"] *= 2.0 ** (e - 8)
    p["w_gate_up"] *= 2.0 ** -e
    ref = O.experts_forward(p["x"], idx, w, p["w_gate_up"], p["w_down"], p["theta"], dtype=torch.float64)
    assert _rel(_forward(p, idx, w), ref) <= 1.2e-6
    p, idx, w = _inputs(516, 260, rows, 8)
    p["w_down"] *= 2.0 ** -min(e, 118)
    ref = O.experts_forward(p["x"], idx, w, p["w_gate_up"], p["w_down"], p["theta"], dtype=torch.float64)
    assert _rel(_forward(p, idx, w), ref) <= 1.2e-6


@pytest.mark.parametrize("T,H,I,E,k", [(777, 192, 88, 16, 3), (1200, 640, 256, 9, 2)])
def test_small_gradients(T, H, I, E, k):
    p = O.make_inputs(T=T, H=H, E=E, k=k, I=I, bias="uniform", theta="normal", seed=T, dtype=torch.float32)
    d = torch.randn(T, H, generator=torch.Generator().manual_seed(T)) * 2.0 ** -112
    args = [p[n].to(DEV) for n in NAMES]
    got = ops.moe_backward(p["x"].to(DEV), d.to(DEV), *args, k)
    idx = ops.moe_forward(p["x"].to(DEV), *args, k, want_routing=True)[1].cpu().numpy()
    ref = O.moe_backward(p["x"], p["w_router"], p["w_gate_up"], p["w_down"], p["theta"], idx, d)
    for name, a in zip(("x", "w_router", "w_gate_up", "w_down"), got):
        assert _rel(a, ref[name]) <= 2e-6, name


# The mean of n independent errors of either sign lies within 5 of their root mean square / sqrt(n).  (The rows' own errors reach a result
# through weights of either sign, so they count as independent.)  Even numbers of steps of 32: an odd one leaves the share of one step.
@pytest.mark.parametrize("H,I", [(512, 256), (1024, 512), (64, 64)])
@pytest.mark.parametrize("rows", [(400, 800), (2000, 2400)])
def test_errors_have_no_sign(H, I, rows):
    p, idx, w = _inputs(H, I, rows, 9)
    ref = O.experts_forward(p["x"], idx, w, p["w_gate_up"], p["w_down"], p["theta"], dtype=torch.float64)
    err = _forward(p, idx, w).double().cpu() - ref
    assert abs(float(err.mean())) <= 5 * float(err.pow(2).mean() / err.numel()) ** 0.5


@pytest.mark.parametrize("T,H,I,E,k", [(800, 512, 400, 16, 2), (1200, 640, 256, 9, 2)])
def test_errors_of_weight_gradients_have_no_sign(T, H, I, E, k):
    """Experts have any number of steps here, and an odd one leaves the share of one: where its 24 roundings cut off 0.12 of a last place,
    and the others round to 0.29, less than 1 / 50 of the spread stays in the mean."""
    p = O.make_inputs(T=T, H=H, E=E, k=k, I=I, bias="uniform", theta="normal", seed=T, dtype=torch.float32)
    d = torch.randn(T, H, generator=torch.Generator().manual_seed(T))
    args = [p[n].to(DEV) for n in NAMES]
    got = ops.moe_backward(p["x"].to(DEV), d.to(DEV), *args, k)
    idx = ops.moe_forward(p["x"].to(DEV), *args, k, want_routing=True)[1].cpu().numpy()
    ref = O.moe_backward(p["x"], p["w_router"], p["w_gate_up"], p["w_down"], p["theta"], idx, d)
    for name, a in zip(("w_gate_up", "w_down"), got[2:4]):
        err = a.double().cpu() - ref[name]
        assert abs(float(err.mean())) <= float(err.pow(2).mean()) ** 0.5 / 50, name
