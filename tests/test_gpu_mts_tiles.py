"""M^T S at the edges of the kernel's tiles and in both tile heights (GPU), against exact
sums: any fp16 values, rows at any address, single-column to several-tile maps."""
import numpy as np
import pytest
import torch

import mod_dit_amd as md
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,n,bpf", [
    (1, 1, 1), (2, 3, 2), (1, 7, 3), (3, 9, 4),       # less than one lane's columns, one more
    (7, 1, 1), (1, 2, 1), (1, 3, 2), (8, 1, 1),       # 7 and 4 cells in all, 9, 8
    (1, 8, 3), (24, 16, 5), (1, 22, 4), (1, 23, 4),   # every row's load passes the map's end
    (2, 63, 8), (1, 65, 64), (1, 257, 30),            # one row past a short / a tall tile
    (1, 511, 60), (2, 513, 60), (1, 1025, 1025),      # one column past a strip
    (150, 513, 40),                                   # enough tiles for the tall form
])
def test_exact_sums(H, n, bpf):
    rng = np.random.default_rng(n * 7 + H)
    bits = rng.integers(0, 0x7c00, (H, n, n), dtype=np.uint16) | (rng.integers(0, 2, (H, n, n), dtype=np.uint16) << 15)
    S = bits.view(np.float16)  # every finite value, both signs, subnormals
    got = md.compute_mts(torch.from_numpy(S).cuda(), bpf).cpu().numpy()
    pick = [0, H - 1]
    assert np.array_equal(got[pick], O.mts_exact(S[pick], bpf))


@pytest.mark.parametrize("offset", [1, 3])
def test_map_at_any_address(offset):
    """A map whose first cell is only 2-byte aligned and ends with its allocation."""
    n, bpf = 70, 9
    rng = np.random.default_rng(offset)
    flat = torch.from_numpy(rng.random(offset + n * n).astype(np.float16)).cuda()
    S = flat[offset:].view(1, n, n)
    assert S.data_ptr() % 16
    assert np.array_equal(md.compute_mts(S, bpf).cpu().numpy(), O.mts_exact(S.cpu().numpy(), bpf))


def test_non_finite_cells_reach_their_lines_only():
    n, bpf = 600, 50
    S = torch.zeros((1, n, n), dtype=torch.float16)
    S[0, 100, 520] = float("inf")
    S[0, 30, 31] = float("nan")
    S[0, 599, 0] = -float("inf")
    got = md.compute_mts(S.cuda(), bpf).cpu()[0]
    nd = 2 * n - 1
    want = torch.zeros(3 * n)
    for r, c in ((100, 520), (30, 31), (599, 0)):
        want[c - r + n - 1] += S[0, r, c].float()
        want[nd + c] += S[0, r, c].float()
        if r // bpf == c // bpf:
            want[-1] += S[0, r, c].float()
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))


def test_small_maps_are_not_read_cell_by_cell():
    """Every load of a 16 x 16 map passes its end, hardly one of a 64 x 64 map (measured 1.05
    of its time; 1.35 cell by cell)."""
    def us(n):
        S = torch.rand((24, n, n), device="cuda").half()
        md.compute_mts(S, 4)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(20):
                md.compute_mts(S, 4)
        start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        times = []
        for _ in range(9):
            start.record()
            graph.replay()
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end) * 50)
        return sorted(times)[4]

    small, large = us(16), us(64)
    print(f"{small:.1f} us at 16 blocks, {large:.1f} us at 64", flush=True)
    assert small <= 1.2 * large
