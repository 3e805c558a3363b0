"""The mask scan (mask_interval, and the range and chunk skipping of the masked attention): rows that start 16-byte aligned
and rows that start anywhere before a 16-byte boundary (the positions before it and the last few take loads of their own),
capacities around the sizes of a lane's load, a wave's and a workgroup's and of the skip map's blocks, single kept
positions at their edges, both mask types."""
import numpy as np
import pytest
import torch

from breeze_tts_2_flash_amd import gqa_decode_masked, mask_interval
from oracle.attention import decode_attention

pytestmark = pytest.mark.gpu

NEG = float(torch.finfo(torch.bfloat16).min)
CAPS = [1, 3, 4, 7, 8, 9, 63, 64, 65, 511, 512, 513, 1023, 1024, 1025, 2047, 2048, 2049, 2056, 4100, 8192, 8199, 20001]


def place(m, dtype, device, aligned):
    """The rows of m as a device tensor whose rows all start 16-byte aligned, or none of them."""
    pitch = (m.shape[1] + 15) // 8 * 8
    t = torch.full((m.shape[0], pitch + 8), NEG, dtype=dtype, device=device)
    v = t[:, 0 if aligned else 1:][:, :m.shape[1]]
    v.copy_(torch.from_numpy(m))
    return v


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("cap", CAPS)
def test_single_positions_and_intervals(device, dtype, aligned, cap):
    edges = {0, 1, 7, 8, 63, 64, 511, 512, 1023, 1024, 2047, 2048, 8191, 8192, cap // 2, cap - 8, cap - 2, cap - 1}
    edges = sorted(e for e in edges if 0 <= e < cap)
    rows = [(e, e + 1) for e in edges] + [(0, 0), (0, cap)] + [(a, b + 1) for a, b in zip(edges, edges[2:])]
    m = np.full((len(rows), cap), NEG, dtype=np.float32)
    for i, (a, b) in enumerate(rows):
        m[i, a:b] = np.linspace(-2.0, 2.0, b - a)
        if b - a > 3:
            m[i, a + 1:a + 1 + (b - a - 2) // 2] = -np.inf
    lens, starts = mask_interval(place(m, dtype, device, aligned), cap)
    torch.cuda.synchronize()
    assert [tuple(r) for r in zip(starts.tolist(), lens.tolist())] == rows


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("cap", [70, 2047, 2304, 8199, 131073, 140005, 270001])  # blocks of 64, 128 and 256 positions
def test_chunks_are_skipped_or_kept(device, dtype, aligned, cap):
    """Attended positions are few and far apart, so most chunks are skipped; a position whose block went unrecorded would
    be missing from the result."""
    rng = np.random.default_rng(cap)
    B, NH, NKV, D = 3, 4, 2, 64
    m = np.full((B, cap), -np.inf, dtype=np.float32)
    for b in range(B):
        keep = np.unique(np.concatenate([rng.integers(0, cap, 6), [cap - 1 - b, b]]))
        m[b, keep] = rng.uniform(-1, 1, keep.size)
    q, k, v = (torch.from_numpy(rng.standard_normal(s).astype(np.float32)).bfloat16()
               for s in ((B, NH, D), (B, NKV, cap, D), (B, NKV, cap, D)))
    mask = place(m, dtype, device, aligned)
    ref = decode_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), np.full(B, cap), D ** -0.5,
                           mask=mask.float().cpu().numpy())
    for splits in (0, 7):
        out = gqa_decode_masked(q.to(device), k.to(device), v.to(device), mask, D ** -0.5, num_splits=splits)
        got = out.float().cpu().numpy()
        assert (np.abs(got - ref) <= 2e-3 + 1e-2 * np.abs(ref)).all(), (cap, splits)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("cap", [1, 3, 6, 8, 13, 71, 2055, 131080])
def test_every_row_start(device, dtype, cap):
    """Rows that start 0 .. 7 elements past a 16-byte boundary: one kept position at either end, at the first boundary and
    around the first two blocks' edges, alone in its row (interval), and all of them together (chunk skipping)."""
    esize = torch.tensor([], dtype=dtype).element_size()
    for off in range(16 // esize):
        head = -off % (16 // esize)
        at = sorted({p for p in (0, head - 1, head, head + 63, head + 64, 63, 64, 127, 128, cap - 2, cap - 1) if 0 <= p < cap})
        pitch = (cap + 31) // 16 * 16
        rows = torch.full((len(at) + 1, pitch), NEG, dtype=dtype, device=device)
        m = rows[:, off:off + cap]
        for i, p in enumerate(at):
            m[i, p] = m[-1, p] = 0.5
        lens, starts = mask_interval(m, cap)
        torch.cuda.synchronize()
        want = [(p, p + 1) for p in at] + [(at[0], at[-1] + 1)]
        assert [tuple(r) for r in zip(starts.tolist(), lens.tolist())] == want, off
        if cap > 2055:
            continue
        g = torch.Generator().manual_seed(off)
        q, k, v = (torch.randn(s, generator=g).bfloat16() for s in ((1, 4, 64), (1, 2, cap, 64), (1, 2, cap, 64)))
        ref = decode_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), np.full(1, cap), 0.125,
                               mask=m[-1:].float().cpu().numpy())
        for splits in (0, 9):
            out = gqa_decode_masked(q.to(device), k.to(device), v.to(device), m[-1:], 0.125, num_splits=splits)
            assert (np.abs(out.float().cpu().numpy() - ref) <= 2e-3 + 1e-2 * np.abs(ref)).all(), (off, splits)
