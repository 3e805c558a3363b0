"""The matrix-core tiles of the split kernel (groups of 4 and 8 q heads) where they can go wrong: lengths around the wave's
16 and the workgroup's 64 and 128 positions, non-zero starts, probabilities whose low bits decide the result, infinite
and NaN values of V, and the fused step's slot at the edges of a tile."""
import numpy as np
import pytest
import torch

from breeze_tts_2_flash_amd import gqa_decode, gqa_decode_fused, gqa_decode_masked
from tests.test_gpu_parity import assert_close, oracle, rand_case

pytestmark = pytest.mark.gpu

GROUPS = [(8, 2), (8, 1), (32, 4)]  # q heads, kv heads
EDGES = [1, 4, 15, 16, 17, 33, 63, 64, 65, 127, 128, 129, 191, 193, 255, 256, 300]


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("NH,NKV", GROUPS)
@pytest.mark.parametrize("splits", [1, 3])
def test_lengths_around_the_tiles(device, D, NH, NKV, splits):
    starts = [(3 * i) % 7 for i in range(len(EDGES))]
    lens = [n + s for n, s in zip(EDGES, starts)]
    w, st = rand_case(NH + D + splits, len(EDGES), NH, NKV, D, 320, lens, starts=starts)
    for b, (s, e) in enumerate(zip(starts, lens)):  # nothing outside the range reaches the output
        w.k[b, :, :s] = w.v[b, :, :s] = float("nan")
        w.k[b, :, e:] = w.v[b, :, e:] = float("nan")
    g = w.to(device)
    out = gqa_decode(g.q, g.k, g.v, g.seq_lens, g.scale, kv_start=st.to(device), num_splits=splits)
    torch.cuda.synchronize()
    assert_close(out.float().cpu().numpy(), oracle(w, kv_start=starts), f"D={D} G={NH // NKV} splits={splits}")


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("cap", [1, 17, 32, 33])
def test_one_short_split_of_a_group_of_four(device, D, cap):
    """One split of at most 32 positions takes the vector path, 33 the matrix tiles; a max_seq_len below the capacity
    counts, and lengths beyond it stay right."""
    lens = list(range(1, cap + 1))
    w, _ = rand_case(cap + D, cap, 8, 2, D, cap, lens)
    ref = oracle(w)
    for b, n in enumerate(lens):
        w.k[b, :, n:] = w.v[b, :, n:] = float("nan")
    g = w.to(device)
    for msl in (0, 7):
        for combine in ("auto", "kernel"):
            out = gqa_decode(g.q, g.k, g.v, g.seq_lens, g.scale, num_splits=1, max_seq_len=msl, combine=combine)
            torch.cuda.synchronize()
            assert_close(out.float().cpu().numpy(), ref, f"D={D} cap={cap} max_seq_len={msl} {combine}")


@pytest.mark.parametrize("NH,NKV", GROUPS)
def test_probabilities_keep_their_low_bits(device, NH, NKV):
    """V is +1 at one position and -1 at another whose score differs by d: the result tanh(d / 2) is the difference of
    two probabilities near 1/2, of the order of their 12th bit and below, rounded to bf16 (2^-9 relative; 24-bit
    probabilities add at most 2^-23 / d, 16-bit ones 2^-17 / d)."""
    D = 128
    for d in (2.0 ** -10, 2.0 ** -12):
        for a, b in ((0, 1), (3, 40), (16, 63)):
            q = torch.zeros(1, NH, D, dtype=torch.bfloat16, device=device)
            q[:, :, 5] = 1
            k = torch.zeros(1, NKV, 64, D, dtype=torch.bfloat16, device=device)
            v = torch.zeros_like(k)
            k[:, :, :, 5] = -100.0
            k[:, :, a, 5], k[:, :, b, 5] = d, 0.0
            v[:, :, a], v[:, :, b] = 1.0, -1.0
            lens = torch.tensor([64], dtype=torch.int32, device=device)
            out = gqa_decode(q, k, v, lens, 1.0, num_splits=1).float()  # (short rows otherwise take the wave kernel)
            want = float(np.tanh(d / 2))
            assert (out - want).abs().max().item() <= want * 2.0 ** -8 + 2.0 ** -23, (d, a, b)


@pytest.mark.parametrize("NH,NKV", [(4, 4)] + GROUPS)
def test_non_finite_values_of_v(device, NH, NKV):
    """An infinite V at an attended position gives an infinity of its sign in its dim and leaves the other dims alone,
    NaN gives NaN, as the vector path does; the position that holds it may carry any probability that is not 0."""
    D, cap = 128, 200
    w, _ = rand_case(5, 1, NH, NKV, D, cap, [cap])
    base = oracle(w)
    w.v[0, :, 7, 3], w.v[0, :, 150, 40], w.v[0, :, 63, 100] = float("inf"), -float("inf"), float("nan")
    g = w.to(device)
    for splits in (1, 3):
        out = gqa_decode(g.q, g.k, g.v, g.seq_lens, g.scale, num_splits=splits).float().cpu().numpy()
        assert np.isposinf(out[0, :, 3]).all() and np.isneginf(out[0, :, 40]).all() and np.isnan(out[0, :, 100]).all()
        rest = [d for d in range(D) if d not in (3, 40, 100)]
        assert_close(out[:, :, rest], base[:, :, rest], f"splits={splits}")


@pytest.mark.parametrize("NH,NKV", GROUPS)
def test_masked_positions_hide_non_finite_values(device, NH, NKV):
    D, cap = 64, 150
    w, _ = rand_case(6, 2, NH, NKV, D, cap, [cap, cap])
    mask = torch.zeros(2, 1, 1, cap)
    holes = [1, 15, 16, 64, 77, 148]
    mask[..., holes] = float("-inf")
    ref = oracle(w, mask=mask[:, 0, 0].numpy())
    w.k[:, :, holes], w.v[:, :, holes] = float("nan"), float("inf")
    g = w.to(device)
    for dtype in (torch.float32, torch.bfloat16):
        out = gqa_decode_masked(g.q, g.k, g.v, mask.to(device, dtype), g.scale)
        torch.cuda.synchronize()
        assert_close(out.float().cpu().numpy(), ref, str(dtype))


@pytest.mark.parametrize("NH,NKV", GROUPS)
@pytest.mark.parametrize("pos", [0, 15, 16, 63, 64, 127, 128, 199])
def test_fused_slot_at_the_edges_of_a_tile(device, NH, NKV, pos):
    from oracle.attention import interval_mask
    from tests.test_gpu_fused import bits, check_against_oracle, make_step, tens

    s = make_step(pos + NH, NH=NH, NKV=NKV, cap=200, pos=pos)
    lens, starts = [pos + 1, 200], [0, min(pos, 3)]
    mask = torch.cat([interval_mask([a], e - 1, 200) for a, e in zip(starts, lens)]).to(device)
    ranges = [dict(mask=mask)]  # G = 4 with lengths runs on the vector path
    if NH // NKV == 8:
        ranges.append(dict(seq_lens=torch.tensor(lens, dtype=torch.int32, device=device),
                           kv_start=torch.tensor(starts, dtype=torch.int32, device=device)))
    for kw in ranges:
        for splits in (1, 2):
            kc, vc = tens(s["kc"], device), tens(s["vc"], device)
            out = gqa_decode_fused(tens(s["qkv"], device), tens(s["qn"], device), tens(s["kn"], device), 1e-6,
                                   tens(s["cos"], device), tens(s["sin"], device), kc, vc,
                                   torch.tensor([pos], device=device), 128 ** -0.5, num_splits=splits, **kw)
            torch.cuda.synchronize()
            check_against_oracle(s, pos, lens, starts, out.float().cpu().numpy(), bits(kc), bits(vc),
                                 f"pos={pos} splits={splits} {list(kw)}")
