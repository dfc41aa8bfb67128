"""Attention tiles whose weights are taken against an older running max (GPU): scores that
climb, fall and jump along the keys, so that tiles land on both sides of the rescale limit,
and non-finite scores, against fp64 attention."""
import pytest
import torch

from mod_dit_amd import ops

pytestmark = pytest.mark.gpu


def _inputs(S, D, dtype, profile, seed=0):
    """q, k, v (1,2,S,D) with scores = profile(key) * (0..2, by query) + noise."""
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn((1, 2, S, D), generator=g) for _ in range(3))
    q[..., 0] = torch.linspace(0, 2, S) * D ** 0.5
    k[..., 0] = profile
    return (t.to(dtype).cuda() for t in (q, k, v))


def _profiles(S):
    t = torch.arange(S).float()
    yield "climbs past the limit", t * (100.0 / S)
    yield "climbs by less than the limit per tile", t * (30.0 / S)
    yield "falls", 60.0 - t * (120.0 / S)
    yield "jumps once", (t >= S // 2 + 5).float() * 80.0 - 40.0
    yield "one high key per tile", ((t % 64) == 63).float() * (t / 64).clamp(max=20)
    yield "flat at the limit of bf16's reach", torch.where(t < 64, -44.0, 44.0)


@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (128, torch.float16), (128, torch.bfloat16)])
@pytest.mark.parametrize("S", [192, 1000])
def test_against_fp64(D, dtype, S):
    eps = 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12
    for name, profile in _profiles(S):
        q, k, v = _inputs(S, D, dtype, profile)
        s = q.double() @ k.double().transpose(2, 3).contiguous() * D ** -0.5
        ref_lse = torch.logsumexp(s, dim=-1)
        ref = torch.softmax(s, dim=-1) @ v.double()
        n = -(-S // 64)
        tiles = ops.mask_to_tiles(torch.ones((2, n, n), dtype=torch.bool, device="cuda"), 64,
                                  union_rows=False)
        for out, lse in (ops.flash_fwd(q, k, v), ops.block_sparse_fwd(q, k, v, tiles, return_lse=True)):
            # P rounded once (relative eps), the output once; scores in fp32: |s| < 2^8 with D
            # products each rounded, 2^-13 absolute
            lim = 2 * eps * (v.abs().max().double() + ref.abs()) + 2.0 ** -12 * v.abs().max().double()
            assert ((out.double() - ref).abs() <= lim).all(), name
            assert ((lse.double() - ref_lse).abs() <= 2.0 ** -12).all(), name


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_non_finite_scores(dtype):
    """A NaN key poisons the rows that see it, an infinite one its rows too (inf - inf in the
    softmax), -inf scores weigh nothing: wherever the key lies."""
    S, D = 320, 64
    for at in (3, 70, 200, 319):
        for value in (float("nan"), float("inf"), float("-inf")):
            q, k, v = _inputs(S, D, dtype, torch.zeros(S))
            q = q.abs()
            k = k.clone()
            k[0, 0, at, 1] = value
            out, lse = ops.flash_fwd(q, k, v)
            clean, clean_lse = ops.flash_fwd(q[:, 1:], k[:, 1:], v[:, 1:])
            assert torch.equal(out[:, 1:], clean) and torch.equal(lse[:, 1:], clean_lse)
            if value == float("-inf"):
                s = q[:, :1].double() @ k[:, :1].double().transpose(2, 3).contiguous() * D ** -0.5
                ref = torch.softmax(s, dim=-1) @ v[:, :1].double()
                assert ((out[:, :1].double() - ref).abs() <= 0.05).all()
            else:
                assert torch.isnan(out[:, :1]).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_whose_first_tiles_weigh_nothing(dtype):
    """Every score of the first two tiles is -inf: the max is still -inf when the loop's own
    tiles begin."""
    S, D = 512, 128
    q, k, v = _inputs(S, D, dtype, torch.zeros(S))
    q = q.abs()
    k = k.clone()
    k[:, :, :128, 5] = float("-inf")
    out, lse = ops.flash_fwd(q, k, v)
    ref, ref_lse = ops.flash_fwd(q, k[:, :, 128:], v[:, :, 128:])
    assert ((out.double() - ref.double()).abs() <= 2.0 ** -7 * v.abs().max().double()).all()
    assert ((lse - ref_lse).abs() <= 1e-4).all()
