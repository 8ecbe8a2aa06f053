"""The fused kernel of I = 512 with more than 8192 slots: output blocks of every width and the ends of its tile heights, with idle experts;
against the fp32 oracle and against the first rows alone, which the kernel for fewer slots takes."""
import numpy as np
import pytest
import torch

from bibo_amd import ops
from oracle import bibo_moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")

ROWS = {
    "one slot more than the limit": [1161, 0, 1025, 1023, 1024, 1026, 1434, 1500],
    "one block each": [128] * 63 + [130],
    "ragged": [0, 1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 1400, 7] * 4,
    "one expert": [0, 16385, 0],
}


@pytest.mark.parametrize("H", [128, 256, 384, 640, 768])
@pytest.mark.parametrize("name", ROWS)
def test_many_slots(H, name):
    rows, I = ROWS[name], 512
    E, T = len(rows), sum(rows)
    assert T > 8192
    p = O.make_inputs(T=T, H=H, E=E, k=1, I=I, theta="normal", seed=H + I)
    idx = np.repeat(np.arange(E, dtype=np.int32), rows)
    np.random.default_rng(I).shuffle(idx)
    idx, w = idx.reshape(T, 1), np.random.default_rng(H).random((T, 1)).astype(np.float32)

    def run(keep):
        args = [p["x"][keep].to(DEV), torch.from_numpy(idx[keep]).to(DEV), torch.from_numpy(w[keep]).to(DEV),
                *(p[n].to(DEV) for n in ("w_gate_up", "w_down", "theta"))]
        return ops.experts_fwd(*args, algo="auto")[0].float().cpu()

    got, few = run(slice(None)), run(slice(0, 1500))
    ref = O.experts_forward(p["x"], idx, w, p["w_gate_up"], p["w_down"], p["theta"]).float()
    top = float(ref.abs().max())
    assert float((got - ref).abs().max()) <= 2e-2 * top
    # sums in another order: an activation and an output may round to the neighbouring bf16 value, 2^-7 of the value each
    assert float((few - got[:1500]).abs().max()) <= 2 * 2.0 ** -7 * top


@pytest.mark.parametrize("act", ["radial", "tanh", "silu"])
@pytest.mark.parametrize("T,H,E,k,n_pos,n_neg", [(1201, 1024, 62, 8, 1, 1), (1500, 256, 9, 6, 0, 0), (4100, 384, 3, 2, 0, 1)])
def test_what_a_call_may_hold(T, H, E, k, n_pos, n_neg, act):
    """Every activation, several experts per token, +/-Identity experts and slots without an expert; each token on its own, so that a wrong
    row of one does not drown in the others."""
    I, Et = 512, E + n_pos + n_neg
    assert T * k > 8192
    p = O.make_inputs(T=T, H=H, E=E, k=k, I=I, theta="normal", seed=T)
    rng = np.random.default_rng(T)
    idx = np.argsort(rng.random((T, Et)) + np.linspace(0, 0.2, Et), axis=1)[:, :k].astype(np.int32)
    w = rng.random((T, k)).astype(np.float32)
    w_of, bad = w.copy(), idx.copy()
    for rows, j, e in ((slice(0, None, 3), 1, Et), (slice(1, None, 5), 0, -1), (slice(T - 1, T), slice(None), Et + 7)):
        bad[rows, j], w_of[rows, j] = e, 0.0
    ops.workspace(DEV, 64 << 20).fill_(0x7f)                  # an unwritten slot row does not pass by luck
    out, counts = ops.experts_fwd(p["x"].to(DEV), torch.from_numpy(bad).to(DEV), torch.from_numpy(w).to(DEV),
                                  *(p[n].to(DEV) for n in ("w_gate_up", "w_down", "theta")), want_counts=True, n_pos=n_pos, n_neg=n_neg, act=act)
    got = out.float().cpu()
    ref = O.experts_forward(p["x"], idx, w_of, p["w_gate_up"], p["w_down"], p["theta"], n_pos=n_pos, n_neg=n_neg, act=act).float()
    assert np.array_equal(counts.cpu().numpy(), np.bincount(bad[(bad >= 0) & (bad < Et)], minlength=Et))
    assert float((got - ref).abs().max()) <= 2e-2 * float(ref.abs().max())
    # per token: activation, slot row and output are rounded to bf16, up to 2^-9 each and independent: 3.4e-3 of a slot, and of the sum of k
    # independent ones; six times that, for slots that cancel
    size = ref.norm(dim=1) + 1e-3 * float(ref.norm(dim=1).max())
    assert float(((got - ref).norm(dim=1) / size).max()) <= 2e-2
    assert not got[T - 1].any()                                # no expert at all


def test_x_of_almost_4_gib():
    """Rows of x beyond byte 0xff000000, the last tokens among them: the requests behind the last K step lie past x whatever its size.  A
    row's sums do not depend on its tile, so the ends of the call are the same bits as those tokens alone."""
    H, I, E, part = 1024, 512, 8, 9000
    T = 0xff000000 // (2 * H) + 3
    p = O.make_inputs(T=8, H=H, E=E, k=1, I=I, theta="normal", seed=5)
    wgu, wd, theta = (p[n].to(DEV) for n in ("w_gate_up", "w_down", "theta"))
    g = torch.Generator(device=DEV).manual_seed(6)
    try:
        x = torch.randn(T, H, generator=g, device=DEV, dtype=torch.bfloat16)
        idx = torch.randint(E, (T, 1), generator=g, device=DEV, dtype=torch.int32)
        w = torch.rand(T, 1, generator=g, device=DEV)
        out = ops.experts_fwd(x, idx, w, wgu, wd, theta)[0]
        for a in (0, T // 2, T - part):
            few = slice(a, a + part)
            assert torch.equal(ops.experts_fwd(x[few], idx[few], w[few], wgu, wd, theta)[0], out[few]), a
        tail = slice(T - 64, T)
        ref = O.experts_forward(x[tail].cpu(), idx[tail].cpu(), w[tail].cpu(), p["w_gate_up"], p["w_down"], p["theta"]).float()
        assert float((out[tail].float().cpu() - ref).abs().max()) <= 2e-2 * float(ref.abs().max())
    finally:
        ops._workspaces.clear()                      # 4 GB of workspace: not kept for the tests that follow
        torch.cuda.empty_cache()
