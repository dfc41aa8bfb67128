"""Times of bf16/fp16 attention calls relative to each other, in one process (GPU): what
the scores' spread may cost."""
import pytest
import torch

from mod_dit_amd import ops

pytestmark = pytest.mark.gpu


def _us(run, reps=20):
    """Median of nine timings of `reps` calls each, in microseconds a call."""
    start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    run()
    times = []
    for _ in range(9):
        start.record()
        for _ in range(reps):
            run()
        end.record()
        end.synchronize()
        times.append(start.elapsed_time(end) * 1e3 / reps)
    return sorted(times)[4]


def _qkv(H, S, D, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(0)
    q, k, v = (torch.randn((1, H, S, D), generator=g, device="cuda") for _ in range(3))
    return (q * scale).to(torch.bfloat16), k.to(torch.bfloat16), v.to(torch.bfloat16)


@pytest.mark.parametrize("H,S,D", [(48, 1577, 64), (24, 1577, 128), (24, 4096, 128)])
def test_peaked_rows_cost_no_second_sweep(H, S, D):
    """Scores of standard deviation 16 move the running max on many tiles: such a tile costs a
    rescale of O, not its products again (measured 1.06-1.14 of flat rows' time; 1.38-1.56
    where it did)."""
    flat, peaked = (_qkv(H, S, D, scale) for scale in (1.0, 16.0))
    t0, t1 = (_us(lambda: ops.flash_fwd(*x, return_lse=False)) for x in (flat, peaked))
    print(f"H={H} S={S} D={D}: {t0:.1f} us flat, {t1:.1f} us peaked", flush=True)
    assert t1 <= 1.25 * t0, (t0, t1)

