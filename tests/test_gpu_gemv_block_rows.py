"""The block-ordered GEMV (256 threads for 1024 < k <= 2048 and three or four rows of x, 768 for 4096 < k <= 6144) where it
can go wrong: k on each side of its ranges, k that leaves lanes idle, both row counts per workgroup with a ragged last
workgroup, segments that end inside a workgroup. Against the GEMV oracle, with its tolerance."""
import numpy as np
import pytest
import torch

from breeze_tts_2_flash_amd import gemv_gateup, gemv_resid, gemv_seg
from oracle.bf16 import f32_to_bf16
from oracle.gemv import gemv as gemv_ref
from tests.test_gpu_gemv import assert_gemv_close, dev_bf16 as dev, host_bits, rand_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [3, 4])
@pytest.mark.parametrize("K,N", [(1032, 4093), (2048, 1), (2040, 6), (1544, 515), (2048, 4099), (1032, 6150)])
def test_gateup(device, M, K, N):
    rng = np.random.default_rng(M * K + N)
    x, nw = rand_bits(rng, M, K), f32_to_bf16((1 + 0.2 * rng.standard_normal(K)).astype(np.float32))
    wg, wu = (rand_bits(rng, N, K, scale=K ** -0.5) for _ in range(2))
    y = torch.empty(M, N, dtype=torch.bfloat16, device=device)
    gemv_gateup(dev(x, device), dev(nw, device), 1e-6, dev(wg, device), dev(wu, device), y)
    torch.cuda.synchronize()
    assert_gemv_close(host_bits(y), gemv_ref(x, [wg, wu], nw, 1e-6, epilogue="silu_mul"), f"gateup M={M} K={K} N={N}")


@pytest.mark.parametrize("M", [3, 4])
@pytest.mark.parametrize("K,ns", [(1032, (13, 7, 30)), (2048, (9, 1, 6)), (1096, (1, 0, 0))])
def test_segments_and_residual(device, M, K, ns):
    rng = np.random.default_rng(M * K + sum(ns))
    N = sum(ns)
    x, nw = rand_bits(rng, M, K), f32_to_bf16((1 + 0.2 * rng.standard_normal(K)).astype(np.float32))
    W, res = [rand_bits(rng, n, K, scale=K ** -0.5) for n in ns], rand_bits(rng, M, N)
    y = torch.empty(M, N, dtype=torch.bfloat16, device=device)
    gemv_seg(dev(x, device), dev(nw, device), 1e-6, *(dev(w, device) for w in W), y)
    torch.cuda.synchronize()
    assert_gemv_close(host_bits(y), gemv_ref(x, [w for w in W if w.shape[0]], nw, 1e-6), f"seg M={M} K={K} ns={ns}")
    w = np.concatenate(W)
    gemv_resid(dev(x, device), dev(w, device), dev(res, device), y)
    torch.cuda.synchronize()
    assert_gemv_close(host_bits(y), gemv_ref(x, [w], epilogue="residual", res_bits=res), f"resid M={M} K={K} N={N}")


@pytest.mark.parametrize("M", [1, 2, 4])
@pytest.mark.parametrize("K,N", [(4104, 1), (6144, 1022), (4960, 1027), (4104, 2051), (5000, 3073)])
def test_long_rows(device, M, K, N):
    rng = np.random.default_rng(M * K + N)
    x, w, res = rand_bits(rng, M, K), rand_bits(rng, N, K, scale=K ** -0.5), rand_bits(rng, M, N)
    y = torch.empty(M, N, dtype=torch.bfloat16, device=device)
    gemv_resid(dev(x, device), dev(w, device), dev(res, device), y)
    torch.cuda.synchronize()
    assert_gemv_close(host_bits(y), gemv_ref(x, [w], epilogue="residual", res_bits=res), f"resid M={M} K={K} N={N}")
