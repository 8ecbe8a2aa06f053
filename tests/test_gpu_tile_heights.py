"""Tile heights of the fused kernel (32, 64, 96 or 128 rows, the lowest that fit the rounds of 256 tiles that the tallest take): rows per
expert at the edges of every height and of a round, idle experts among them; against the fp32 oracle, and the same bits whatever height
a row's tile has."""
import numpy as np
import pytest
import torch

from bibo_amd import ops
from oracle import bibo_moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _inputs(H, I, rows, seed):
    E, T = len(rows), sum(rows)
    p = O.make_inputs(T=T, H=H, E=E, k=1, I=I, theta="normal", seed=seed)
    idx = np.repeat(np.arange(E, dtype=np.int32), rows)
    np.random.default_rng(seed).shuffle(idx)
    w = np.random.default_rng(seed + 1).random((T, 1)).astype(np.float32)
    return p, idx.reshape(T, 1), w


def _run(p, idx, w, algo, keep=slice(None)):
    args = [p["x"][keep].to(DEV), torch.from_numpy(idx[keep]).to(DEV), torch.from_numpy(w[keep]).to(DEV),
            *(p[n].to(DEV) for n in ("w_gate_up", "w_down", "theta"))]
    return ops.experts_fwd(*args, algo=algo)[0]


# lists of rows per expert: 64 experts; the tallest tiles take one round of 256 unless said otherwise
ROWS = {
    "one block each": [128] * 64,                               # 256 tiles of 32 rows: a full round
    "one row over": [128] * 63 + [129],                         # 257 of 32 do not fit: 64 rows
    "two blocks": [256] * 64,
    "two blocks, one row over": [256] * 60 + [257, 0, 1, 510],
    "three blocks": [384] * 63 + [383],
    "four blocks": [512] * 64,
    "a row into the second round": [512] * 63 + [513],          # 257 of 128: two rounds, filled by 64-row and one-block tiles
    "two rounds of 96": [768] * 60 + [1, 33, 0, 700],
    "ragged": [0, 1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 1000, 7] * 4,
}


@pytest.mark.parametrize("H,I", [(128, 128), (256, 256), (384, 384)])
@pytest.mark.parametrize("name", ROWS)
def test_heights(H, I, name):
    p, idx, w = _inputs(H, I, ROWS[name], 3 + H)
    got = _run(p, idx, w, "fused").float().cpu()
    ref = O.experts_forward(p["x"], idx, w, p["w_gate_up"], p["w_down"], p["theta"])
    assert float((got - ref.float()).abs().max() / ref.float().abs().max()) <= 2e-2
    # the first 1500 rows alone: 32-row tiles, another place in them and another order of the column blocks; the same sums
    few = slice(0, 1500)
    assert torch.equal(_run(p, idx, w, "fused", few).float().cpu(), got[few])


@pytest.mark.parametrize("rows", [[1] * 5, [64] * 64, [65] * 64, [128] * 64, [256] * 64, [257] * 64, [0, 700, 3, 64]])
def test_heights_at_wide_experts(rows):
    """I = 512: tiles of 32 or 64 rows, four column blocks."""
    p, idx, w = _inputs(128, 512, rows, 11)
    got = _run(p, idx, w, "auto").float().cpu()
    ref = O.experts_forward(p["x"], idx, w, p["w_gate_up"], p["w_down"], p["theta"])
    assert float((got - ref.float()).abs().max() / ref.float().abs().max()) <= 2e-2
