"""Tile lists of caller masks and rows of generated masks at the sizes where the kernels'
widths end (GPU): odd column counts, strided views, several passes, cut key-tile limits."""
import numpy as np
import pytest
import torch

from mod_dit_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _lists(mask, block, union, kv_tiles):
    """Entries per (head, 128-row tile), straight from the definition."""
    H, rows, cols = mask.shape
    per_tile, per_col = (2, 1) if block == 64 else (1, 2)
    out = []
    for h in range(H):
        for t in range(-(-rows // per_tile)):
            r = mask[h, t * per_tile:(t + 1) * per_tile]
            want = []
            for j in range(cols):
                if not r[:, j].any():
                    continue
                bits = 3 if union or block == 128 else int(r[0, j]) | (int(r[1, j]) << 1 if len(r) > 1 else 0)
                want += [(kt << 2) | bits for kt in range(j * per_col, (j + 1) * per_col) if kt < kv_tiles]
            out.append(want)
    return out


@pytest.mark.parametrize("H,rows,cols,block,union,kv_tiles,pad", [
    (1, 1, 1, 64, False, 1, 0),
    (2, 3, 7, 64, False, 7, 0),        # below one lane's columns, odd rows
    (2, 9, 513, 64, False, 500, 0),    # one column past a pass, limit inside it
    (1, 4, 1031, 64, True, 1031, 5),   # strided rows at odd addresses
    (2, 5, 67, 128, False, 91, 0),     # limit in the middle of a column's two tiles
    (1, 3, 520, 128, True, 1040, 3),
    (3, 2, 40, 64, False, 0, 0),       # every tile dropped
])
def test_tiles_from_mask(H, rows, cols, block, union, kv_tiles, pad):
    rng = np.random.default_rng(rows * cols)
    full = torch.from_numpy(rng.random((H, rows + 1, cols + pad)) < 0.4).cuda()
    mask = full[:, 1:, pad:]  # a view whose rows start anywhere
    tiles = ops.mask_to_tiles(mask, block, union_rows=union, kv_tiles=kv_tiles)
    counts, entries = tiles.counts.cpu().numpy(), tiles.entries.cpu().numpy()
    want = _lists(mask.cpu().numpy(), block, union, kv_tiles)
    nq = counts.shape[1]
    for i, w in enumerate(want):
        h, t = divmod(i, nq)
        assert counts[h, t] == len(w)
        assert entries[h, t, :counts[h, t]].tolist() == w


def test_any_nonzero_byte_is_true():
    rng = np.random.default_rng(1)
    raw = torch.from_numpy(rng.integers(0, 256, (1, 4, 21), dtype=np.uint8) * (rng.random((1, 4, 21)) < 0.5).astype(np.uint8)).cuda()
    a = ops.mask_to_tiles(raw.view(torch.bool), 64, union_rows=False)
    b = ops.mask_to_tiles(raw != 0, 64, union_rows=False)
    assert torch.equal(a.counts, b.counts)
    for t in range(a.n_qtiles):
        n = int(a.counts[0, t])
        assert torch.equal(a.entries[0, t, :n], b.entries[0, t, :n])


@pytest.mark.parametrize("n,layout,text", [
    (5, _lib.LAYOUT_WAN, 0), (64, _lib.LAYOUT_WAN, 0), (275, _lib.LAYOUT_COGVIDEOX, 4),
    (2053, _lib.LAYOUT_WAN, 0), (2050, _lib.LAYOUT_HUNYUAN, 3)])
def test_generated_rows(n, layout, text):
    """Every byte of the mask, rows starting at any address, and its lists."""
    nb, H, bpf = n + text, 2, max(1, n // 5)
    rng = np.random.default_rng(n)
    k = max(1, n // 4)
    sel = np.stack([np.sort(rng.choice(3 * n - 1, k, replace=False)) for _ in range(H)])
    mode = torch.tensor([0, 1], dtype=torch.uint8, device="cuda")
    mask, tiles = ops.mask_from_lines(torch.from_numpy(sel).int().cuda(), mode, n=n,
                                      blocks_per_frame=bpf, layout=layout, nb=nb, text_blocks=text,
                                      block_size=64, union_rows=False)
    i = np.arange(n)
    lo = text if layout == _lib.LAYOUT_COGVIDEOX else 0
    want = np.ones((H, nb, nb), dtype=bool)
    for h in range(H):
        line = np.zeros(3 * n - 1, dtype=bool)
        line[sel[h]] = True
        v = line[:n][None, :] | line[n:][i[None, :] - i[:, None] + n - 1]
        if h == 1:
            v = v | (i[None, :] // bpf == i[:, None] // bpf)
        want[h, lo:lo + n, lo:lo + n] = v
    assert np.array_equal(mask.cpu().numpy(), want)
    again = ops.mask_to_tiles(mask, 64, union_rows=False)
    assert torch.equal(tiles.counts, again.counts)
    idx = torch.arange(tiles.cap, device="cuda") < tiles.counts[..., None]
    assert torch.equal(tiles.entries[idx], again.entries[idx])
