"""Calls of more than one round of tiles whose experts' rows are cut into tiles of two heights: rows per expert at the edges of the rule, hot and
idle experts among them; against the fp32 oracle, and the same bits as a call of one round."""
import numpy as np
import pytest
import torch

from bibo_amd import ops
from oracle import bibo_moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")

# rows per expert, 64 experts.  128-row tiles:
ROWS = {
    "two rounds": [768] * 32 + [769] * 32,               # 3.25 blocks a tile: 8 of 3, or 7 of 3 and one of 4
    "two rounds, 2.25 blocks": [560] * 64,                                  # 18 blocks in 8 tiles
    "two rounds, idle experts": [1120, 1121, 1, 0, 31, 1500, 1100, 1152] * 8,
    "two rounds, 3.5 blocks": [870] * 64,                                   # 28 blocks in 8 tiles
    "three rounds": [1170] * 32 + [1160, 1180] * 16,                        # 37 blocks in 12 tiles
    "four rounds": [1540] * 60 + [0, 33, 3000, 1540],                       # 49 blocks in 16 tiles
    "four rounds, hot experts": [16384] * 4 + [540] * 60,                   # 512 blocks in 158 tiles, 17 in 6
    "one height": [1500] * 64,                                              # 47 blocks in 12 tiles, three full rounds
    "one expert": [65536 + 100] + [0] * 63,
}


def _check(rows, H, I, algo):
    E, T = len(rows), sum(rows)
    p = O.make_inputs(T=T, H=H, E=E, k=1, I=I, theta="normal", seed=T)
    idx = np.repeat(np.arange(E, dtype=np.int32), rows)
    np.random.default_rng(T).shuffle(idx)
    idx, w = idx.reshape(T, 1), np.random.default_rng(T + 1).random((T, 1)).astype(np.float32)

    def run(keep=slice(None)):
        args = [p["x"][keep].to(DEV), torch.from_numpy(idx[keep]).to(DEV), torch.from_numpy(w[keep]).to(DEV),
                *(p[n].to(DEV) for n in ("w_gate_up", "w_down", "theta"))]
        return ops.experts_fwd(*args, algo=algo)[0].float().cpu()

    got = run()
    ref = O.experts_forward(p["x"], idx, w, p["w_gate_up"], p["w_down"], p["theta"]).float()
    scale = ref.abs().max()
    assert float((got - ref).abs().max() / scale) <= 2e-2
    # a row that a wrong map would leave out or take from elsewhere is off by its own size: no row may be
    assert float(((got - ref).norm(dim=1) / ref.norm(dim=1).clamp_min(1e-3 * float(scale))).max()) <= 0.1
    return run, got


@pytest.mark.parametrize("H,I", [(128, 128), (128, 256), (128, 384)])      # one height; two from two rounds on; from three on
@pytest.mark.parametrize("name", ROWS)
def test_two_heights(name, H, I):
    run, got = _check(ROWS[name], H, I, "fused")
    few = slice(100, 1500)
    assert torch.equal(run(few), got[few])


@pytest.mark.parametrize("rows", [[375] * 64, [300, 260, 1, 0, 64, 700, 33, 320] * 8, [256] * 60 + [257, 0, 3000, 1000]])
def test_two_heights_at_wide_experts(rows):
    """I = 512: tiles of 32 and 64 rows within a call of two rounds."""
    _check(rows, 128, 512, "auto")
