"""The merge of the split partials around its batches of 16 splits, for every column layout (q heads per kv head x
head_dim): the split counts on each side of a batch, against the oracle; both merge modes bit for bit."""
import pytest
import torch

from breeze_tts_2_flash_amd import gqa_decode
from tests.test_gpu_parity import assert_close, oracle, rand_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("G", [1, 2, 4, 8])
def test_split_counts_around_the_batches(device, D, G):
    cap = 8192 if D == 64 else 4096  # up to 128 splits of the smallest chunk
    w, _ = rand_case(D + G, 2, 2 * G, 2, D, cap, [cap, cap - 45])
    ref = oracle(w)
    g = w.to(device)
    for splits in (2, 3, 15, 16, 17, 31, 32, 33, 47, 48, 49, 64, 65, 128):
        out = gqa_decode(g.q, g.k, g.v, g.seq_lens, g.scale, num_splits=splits)
        two = gqa_decode(g.q, g.k, g.v, g.seq_lens, g.scale, num_splits=splits, combine="kernel")
        torch.cuda.synchronize()
        assert_close(out.float().cpu().numpy(), ref, f"D={D} G={G} splits={splits}")
        assert torch.equal(out.view(torch.int16), two.view(torch.int16)), f"D={D} G={G} splits={splits}"
