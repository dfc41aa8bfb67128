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
