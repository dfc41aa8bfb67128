"""Dense int8/fp8 attention whose last key tile is partial (GPU): the keys past the end take no
part in the output, the row sum or the max, at every position the end can have in a tile."""
import numpy as np
import pytest
import torch

import oracle as O
from mod_dit_amd import ops
from q8_contract import check_q8_model
from test_gpu_q8 import _check_lse, _z_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("S", [1, 63, 65, 95, 96, 97, 127, 129, 641])
@pytest.mark.parametrize("scale,shift", [(1.0, 0.0), (4.0, 3.0), (1e-3, 0.0)])
def test_partial_last_tile(S, D, scale, shift):
    """Wide scores with a large K offset, ordinary ones, and scores near 0 (where each key past
    the end would weigh as much as a real one)."""
    g = torch.Generator().manual_seed(S + D)
    q, k, v = (torch.randn((1, 2, S, D), generator=g) for _ in range(3))
    q, k, v = (t.to(torch.bfloat16).cuda() for t in (q * scale, k * scale + shift, v))
    qz = ops.quantize_qkv(q, k, v)
    out, lse = ops.flash_fwd_q8(qz)
    _, ref_lse = check_q8_model(out[0], _z_np(qz), tag=f"S={S} D={D} scale={scale}")
    _check_lse(lse[0], ref_lse, f"S={S} D={D} scale={scale}", 2e-4)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("S", [65, 257, 1000])
@pytest.mark.parametrize("qval", [4.0, 30.0, 60.0, 100.0])
def test_partial_last_tile_under_negative_rows(S, D, qval):
    """Rows whose int8 scores are all negative: a wide channel sets the K step, on which +0.03
    rounds to 0 and -0.034 to -1. A key past the end (score 0) would outweigh every real one."""
    g = torch.Generator().manual_seed(S + D)
    q = torch.full((1, 2, S, D), qval)
    q[..., 0] = 0.0
    q[:, 1] *= torch.linspace(0.25, 1.0, S)[None, :, None]
    rank = torch.rand((1, 2, S, D), generator=g).argsort(dim=2)  # per channel: 17 in 32 positive
    k = torch.where(rank < round(S * 0.034 / 0.064), 0.03, -0.034)
    k[..., 0] = 8.0 - 16.0 * (torch.arange(S) % 2)
    v = torch.randn((1, 2, S, D), generator=g)
    q, k, v = (t.to(torch.bfloat16).cuda() for t in (q, k, v))
    qz = ops.quantize_qkv(q, k, v)
    z = _z_np(qz)
    s = z["q8"].astype(np.int64) @ z["k8"].astype(np.int64).transpose(0, 2, 1)
    assert (s.max(axis=-1) < 0).mean() > 0.9
    out, lse = ops.flash_fwd_q8(qz)
    _, ref_lse = check_q8_model(out[0], z, tag=f"S={S} D={D} q={qval}")
    _check_lse(lse[0], ref_lse, f"S={S} D={D} q={qval}", 2e-4)
