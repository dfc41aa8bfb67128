"""Split key ranges (GPU): launches with few query tiles run several workgroups per tile and
combine fp32 partial results; checked against the unsplit launch and fp64 attention."""
import pytest
import torch

import mod_dit_amd as md
from mod_dit_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _qkv(B, H, Sq, Skv, D, dtype, nhd, seed=0):
    g = torch.Generator().manual_seed(seed)

    def one(S):
        shape = (B, S, H, D) if nhd else (B, H, S, D)
        t = torch.randn(shape, generator=g).to(dtype).cuda()
        return t.transpose(1, 2) if nhd else t

    return one(Sq), one(Skv), one(Skv)


def _check(q, k, v, run, monkeypatch, mask=None):
    """run(): (O, LSE). Its split result against the same call without a workspace, and
    against fp64 attention under the token mask."""
    out, lse = run()
    with monkeypatch.context() as mp:
        mp.setattr(ops, "_workspace", lambda nbytes, device: (None, 0))
        plain, plain_lse = run()
    s = q.double() @ k.double().transpose(2, 3).contiguous() * q.shape[-1] ** -0.5
    if mask is not None:
        s = s.masked_fill(~mask, float("-inf"))
    ref_lse = torch.logsumexp(s, dim=-1)
    ref = torch.softmax(s, dim=-1).nan_to_num(0.0) @ v.double()
    # each side rounds P (relative 2^-9 in bf16) against its own running max and the output
    # once: |dO| <= 2 * 2^-9 * sum p|v| + 2 * 2^-9 |o|, with sum p|v| <= max |v|
    eps = 2.0 ** -9 if q.dtype == torch.bfloat16 else 2.0 ** -12
    lim = 2 * eps * (v.abs().max().double() + plain.abs().double())
    assert ((out.double() - plain.double()).abs() <= lim).all()
    assert ((out.double() - ref).abs() <= lim + 1e-5).all()
    # LSE: fp32 sums of at most 2^13 terms and one rounding of a value below 2^5
    dead = torch.isinf(ref_lse)
    assert torch.equal(torch.isinf(lse), dead) and torch.equal(torch.isinf(plain_lse), dead)
    assert ((lse.double() - ref_lse)[~dead].abs() <= 2.0 ** -13).all()
    again, _ = run()
    assert torch.equal(out, again)


@pytest.mark.parametrize("B,H,Sq,Skv,D,dtype,nhd", [
    (1, 1, 1, 1023, 64, torch.bfloat16, False),     # the fewest key tiles that split, one row
    (1, 2, 129, 4097, 128, torch.bfloat16, True),   # one row past a tile, one key past a tile
    (1, 3, 255, 2048, 64, torch.float16, False),
    (2, 2, 640, 1999, 128, torch.float16, True),
    (1, 1, 128, 8192, 128, torch.bfloat16, False),  # many pieces of one tile
])
def test_dense_split(B, H, Sq, Skv, D, dtype, nhd, monkeypatch):
    assert _lib.load().moddit_flash_fwd_workspace_bytes(B, H, Sq, Skv, D) > 0
    q, k, v = _qkv(B, H, Sq, Skv, D, dtype, nhd)
    _check(q, k, v, lambda: ops.flash_fwd(q, k, v), monkeypatch)


@pytest.mark.parametrize("H,S,D,dtype,block,origin,union", [
    (2, 4096, 64, torch.bfloat16, 64, 0, False),
    (1, 4096 + 37, 128, torch.float16, 64, -27, True),   # shifted grid, ragged end
    (2, 4096 + 90, 64, torch.float16, 64, -38, False),
    (1, 6016, 128, torch.bfloat16, 128, 0, True),
])
def test_sparse_split(H, S, D, dtype, block, origin, union, monkeypatch):
    g = torch.Generator().manual_seed(3)
    nb = -(-(S - origin) // block)
    mask = torch.rand((H, nb, nb), generator=g) < 0.15
    mask[:, nb // 2:nb // 2 + 2] = False   # rows without any key: zeros, LSE -inf
    mask[:, 1, :] = False
    mask[:, 1, 2] = True                   # fewer tiles than pieces
    mask = mask.cuda()
    tiles = ops.mask_to_tiles(mask, block, union_rows=union, grid_origin=origin)
    assert _lib.load().moddit_block_sparse_fwd_workspace_bytes(1, H, S, D, tiles.cap, origin) > 0
    q, k, v = _qkv(1, H, S, S, D, dtype, False, seed=1)
    run = mask
    if union and block == 64:
        pair = torch.arange(nb, device="cuda") // 2 * 2
        run = mask[:, pair] | mask[:, (pair + 1).clamp(max=nb - 1)]
    at = (torch.arange(S, device="cuda") - origin) // block
    token = run[:, at][:, :, at][None]
    _check(q, k, v, lambda: ops.block_sparse_fwd(q, k, v, tiles, return_lse=True), monkeypatch, token)


def test_large_launches_do_not_split():
    lib = _lib.load()
    assert lib.moddit_flash_fwd_workspace_bytes(1, 24, 115200, 115200, 128) == 0
    assert lib.moddit_block_sparse_fwd_workspace_bytes(1, 48, 17776, 64, 279, -30) == 0


def test_split_replays_in_a_graph():
    q, k, v = _qkv(1, 2, 256, 4096, 128, torch.bfloat16, False)
    want, _ = ops.flash_fwd(q, k, v)
    out = torch.empty_like(want)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        ops.flash_fwd(q, k, v, return_lse=False, out=out)
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ops.flash_fwd(q, k, v, return_lse=False, out=out)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        ops.flash_fwd(k, q, v[:, :, :256])


@pytest.mark.parametrize("op", ["flash_fwd", "block_sparse_fwd"])
def test_the_library_decides_what_splits(op, monkeypatch):
    """The workspace of a call is what the library asks for, at every size."""
    lib = _lib.load()
    name = f"moddit_{op}_workspace_bytes"
    asked = []
    monkeypatch.setattr(lib, name, lambda *sizes: 4096)
    monkeypatch.setattr(ops, "_workspace", lambda nbytes, device: asked.append(nbytes) or (None, 0))
    q, k, v = _qkv(1, 1, 128, 128, 64, torch.bfloat16, False)
    tiles = ops.mask_to_tiles(torch.ones((1, 2, 2), dtype=torch.bool, device="cuda"), 64)
    ops._split_bytes.cache_clear()
    try:
        getattr(ops, op)(*((q, k, v) if op == "flash_fwd" else (q, k, v, tiles)))
    finally:
        ops._split_bytes.cache_clear()
    assert asked == [4096]


def test_without_memory_for_scratch(monkeypatch):
    """A call whose scratch cannot be had warns and returns the unsplit launch's result."""
    q, k, v = _qkv(1, 2, 256, 4096, 128, torch.bfloat16, False)
    with monkeypatch.context() as mp:
        mp.setattr(ops, "_workspace", lambda nbytes, device: (None, 0))
        plain, plain_lse = ops.flash_fwd(q, k, v)
    split, _ = ops.flash_fwd(q, k, v)
    assert not torch.equal(split, plain)
    real = torch.empty

    def empty(*size, **kw):
        if kw.get("dtype") == torch.uint8:
            raise torch.cuda.OutOfMemoryError("no scratch")
        return real(*size, **kw)

    monkeypatch.setattr(torch, "empty", empty)
    with pytest.warns(RuntimeWarning, match="scratch"):
        out, lse = ops.flash_fwd(q, k, v)
    assert torch.equal(out, plain) and torch.equal(lse, plain_lse)
