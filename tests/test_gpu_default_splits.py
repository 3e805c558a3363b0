"""The default split count on each branch of its rule (one round of workgroups, two or three rounds for a server's batch,
the merge-batch limit, rows short enough for one split), against the oracle, and the bound by which the static scratch
refuses sizes, which does not follow the tuning. The counts are those of a 256-CU device."""
import pytest
import torch

from breeze_tts_2_flash_amd import default_splits, gqa_decode, gqa_decode_fused, workspace_bytes
from tests.test_gpu_parity import assert_close, oracle, rand_case
from tests.test_zz_no_alloc import BZ_ERR_SCRATCH, noalloc

pytestmark = pytest.mark.gpu

# rows, q heads, kv heads, head_dim, capacity, splits
CASES = [
    (2, 16, 8, 128, 2048, 16),    # one round: 256 workgroups
    (3, 16, 8, 128, 2000, 10),    # one round, rounded down: 240
    (1, 8, 1, 128, 1000, 16),     # the merge batch bounds a single unit
    (1, 8, 1, 128, 1300, 21),     # ... a second batch for chunks of 64 positions, none of 65
    (1, 16, 8, 128, 1500, 24),
    (1, 8, 1, 128, 1087, 16),     # ... but no second batch for less than 17 whole chunks
    (1, 8, 1, 128, 8450, 34),     # ... chunks of 256 positions, none of 257
    (1, 8, 1, 128, 4000, 32),     # ... two batches
    (1, 8, 1, 128, 9000, 36),     # ... more for chunks of 256 positions
    (1, 8, 1, 64, 9000, 32),      # (512 at head_dim 64)
    (4, 16, 8, 128, 1024, 8),     # a batch of short rows stays at one round
    (16, 16, 8, 128, 2048, 4),    # two rounds
    (12, 8, 8, 64, 2048, 8),      # three rounds divide the row better
    (16, 16, 8, 128, 256, 1),     # half of the CUs taken by the rows alone, 128 KB a row: no split
    (15, 16, 8, 128, 256, 2),     # just below half of the CUs
    (16, 16, 8, 128, 264, 2),     # just above 128 KB
    (33, 8, 8, 64, 600, 2),       # more units than CUs
]


@pytest.mark.parametrize("B,NH,NKV,D,cap,splits", CASES)
def test_default_split_count(device, B, NH, NKV, D, cap, splits):
    if torch.cuda.get_device_properties(device).multi_processor_count == 256:
        assert default_splits(B, NKV, D, cap) == splits
    lens = [cap - (37 * b) % cap if b % 3 else cap for b in range(B)]
    starts = [min(5 * b, n) for b, n in enumerate(lens)]
    w, st = rand_case(B + cap, B, NH, NKV, D, cap, lens, starts=starts)
    g = w.to(device)
    out = gqa_decode(g.q, g.k, g.v, g.seq_lens, g.scale, kv_start=st.to(device))
    torch.cuda.synchronize()
    assert_close(out.float().cpu().numpy(), oracle(w, kv_start=starts), f"B={B} NKV={NKV} cap={cap}")


def test_static_scratch_refuses_by_the_largest_default(device):
    """2 rows x 8 kv heads x 8 q heads over 32768 slots: one split per 256 positions is 8.5 MB of partials, refused
    although the default count is lower; an explicit count that fits is taken."""
    q = torch.zeros(2, 64, 128, dtype=torch.bfloat16, device=device)
    kv = torch.zeros(2, 8, 32768, 128, dtype=torch.bfloat16, device=device)
    lens = torch.zeros(2, dtype=torch.int32, device=device)
    assert default_splits(2, 8, 128, 32768) < 128
    rc, _ = noalloc(q, kv, kv, lens, 0.125)
    assert rc == BZ_ERR_SCRATCH
    rc, _ = noalloc(q, kv, kv, lens, 0.125, num_splits=16)
    torch.cuda.synchronize()
    assert rc == 0


@pytest.mark.parametrize("B,NKV,G,cap", [(1, 1, 2, 4000), (1, 4, 4, 4096), (2, 8, 4, 2048), (4, 8, 2, 3000), (5, 2, 4, 1024),
                                         (1, 4, 1, 5000)])
def test_fused_default_is_the_queried_count(device, B, NKV, G, cap):
    """bz_gqa_decode_default_splits is what num_splits = 0 takes in the fused call as well: a workspace sized for that count
    serves it, and its outputs equal the explicit count's bit for bit."""
    from tests.test_gpu_fused import make_step, tens

    splits = default_splits(B, NKV, 128, cap)
    ws = torch.zeros(workspace_bytes(B, NKV * G, NKV, 128, cap, splits), dtype=torch.uint8, device=device)
    s = make_step(cap, B=B, NH=NKV * G, NKV=NKV, cap=cap, pos=cap - 5)
    lens = torch.full((B,), cap - 4, dtype=torch.int32, device=device)
    outs = []
    for n in (0, splits):
        outs.append(gqa_decode_fused(*(tens(s[k], device) for k in ("qkv", "qn", "kn")), 1e-6, tens(s["cos"], device),
                                     tens(s["sin"], device), tens(s["kc"], device), tens(s["vc"], device),
                                     torch.tensor([cap - 5], device=device), 128 ** -0.5, seq_lens=lens, num_splits=n,
                                     workspace=ws))
    torch.cuda.synchronize()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
