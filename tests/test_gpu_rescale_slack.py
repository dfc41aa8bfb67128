"""How far a row's largest weight may lie above the running max it is taken against (GPU): a
weight of 1 is exact in bf16 and fp16, any other is rounded once."""
import pytest
import torch

from mod_dit_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (128, torch.bfloat16), (64, torch.float16)])
@pytest.mark.parametrize("kind", ["dense", "sparse", "split"])
def test_largest_weight_is_exact_from_the_slack_on(D, dtype, kind):
    """One key, 6 to 8 log2 units above the others, in the last tile: its weight must be exact,
    which leaves the other keys' rounding and the output's."""
    S, H = (4096, 1) if kind == "split" else (320, 2)
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11  # unit roundoff
    rise = torch.linspace(6.02, 8.0, 128).repeat(-(-S // 128))[:S]   # by query, log2 units
    q, k = (torch.zeros((1, H, S, D)) for _ in range(2))
    q[..., 0] = rise * D ** 0.5 / 1.4426950408889634
    k[..., S - 7, 0] = 1.0
    k[..., 1] = -64.0                                                # others: weight 2^-92
    q[..., 1] = D ** 0.5
    k[..., 5, 1] = k[..., S - 7, 1] = 0.0                            # key 5 sets the first max: 0
    g = torch.Generator().manual_seed(D)
    v = torch.randn((1, H, S, D), generator=g)
    q, k, v = (t.to(dtype).cuda() for t in (q, k, v))
    if kind == "sparse":
        n = S // 64
        tiles = ops.mask_to_tiles(torch.ones((H, n, n), dtype=torch.bool, device="cuda"), 64)
        out, _ = ops.block_sparse_fwd(q, k, v, tiles)
    else:
        out, _ = ops.flash_fwd(q, k, v)
    s = q.double() @ k.double().transpose(2, 3).contiguous() * D ** -0.5
    p = torch.softmax(s, dim=-1)
    ref = p @ v.double()
    # key 5's weight rounded (2^-6 to 2^-8 of the largest), fp32 sums, the output rounded
    lim = eps * (p[..., 5:6] * v[..., 5:6, :].double().abs() + ref.abs()) * 1.001 + 1e-5
    worst = ((out.double() - ref).abs() / lim).max().item()
    print(f"{kind} D={D} {dtype}: worst element at {worst:.3f} of its bound", flush=True)
    assert worst <= 1.0
