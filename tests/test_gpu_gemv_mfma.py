"""The MFMA GEMV kernel (gemv_mfma_kernel) where it can go wrong: k on each side of its range (2048 < k <= 4096), its waves'
chunks (128) and its tile counts (1024), rows that are not whole quads, segments that end inside a quad, each tiling of
quads per workgroup, rows of x apart, and infinite weights next to a row's end; and the sizes around it that stay on the
other kernels (k 2048, some SiLU * up sizes at one or two rows of x, the residual). Against the GEMV oracle, with its
tolerance."""
import numpy as np
import pytest
import torch

from breeze_tts_2_flash_amd import gemv_gateup, gemv_resid, gemv_seg
from oracle.bf16 import f32_to_bf16
from oracle.gemv import gemv as gemv_ref
from tests.test_gpu_gemv import assert_gemv_close, dev_bf16 as dev, host_bits, rand_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N", [(3, 2048, 2050), (3, 2056, 515), (3, 3072, 70), (1, 2056, 33), (2, 2176, 1100),
                                   (4, 3072, 514), (2, 3080, 130), (1, 4096, 2052), (4, 4088, 1026),
                                   # four quads a workgroup (256 CUs): one round, its edge, many rounds, the last ragged
                                   (2, 2056, 2046), (4, 2304, 1031), (1, 2816, 2043), (3, 3584, 6913), (2, 4096, 8199),
                                   (4, 3080, 5001),
                                   # two quads: a grid just past a round of four; the LDS kernel's sizes between
                                   (2, 2304, 3001), (4, 3328, 2307), (1, 3328, 3331), (2, 3840, 6917), (1, 4096, 1283)])
def test_gateup(device, M, K, N):
    rng = np.random.default_rng(M * K + N)
    x, nw = rand_bits(rng, M, K), f32_to_bf16((1 + 0.2 * rng.standard_normal(K)).astype(np.float32))
    wg, wu = (rand_bits(rng, N, K, scale=K ** -0.5) for _ in range(2))
    y = torch.empty(M, N, dtype=torch.bfloat16, device=device)
    gemv_gateup(dev(x, device), dev(nw, device), 1e-6, dev(wg, device), dev(wu, device), y)
    torch.cuda.synchronize()
    assert_gemv_close(host_bits(y), gemv_ref(x, [wg, wu], nw, 1e-6, epilogue="silu_mul"), f"gateup M={M} K={K} N={N}")


@pytest.mark.parametrize("norm", [True, False])
@pytest.mark.parametrize("M,K,ns", [(3, 2048, (1030, 513, 517)), (4, 2056, (13, 7, 30)),
                                    (3, 3000, (5, 1, 2)), (4, 4096, (1024, 512, 512)), (3, 4096, (1, 0, 0)),
                                    # four quads a workgroup, ragged segments: one round, two and a half past k = 3072
                                    (4, 2056, (1030, 513, 517)), (3, 3072, (2049, 1022, 1001)), (3, 3584, (5121, 2563, 2553)),
                                    (4, 2560, (2001, 1603, 1602)),  # two quads
                                    # one quad a workgroup in a full round, two where those would be more
                                    (4, 2560, (1000, 11, 9)), (3, 3584, (513, 258, 262))])
def test_segments(device, M, K, ns, norm):
    rng = np.random.default_rng(M * K + sum(ns))
    x = rand_bits(rng, M, K)
    nw = f32_to_bf16((1 + 0.2 * rng.standard_normal(K)).astype(np.float32)) if norm else None
    W = [rand_bits(rng, n, K, scale=K ** -0.5) for n in ns]
    y = torch.empty(M, sum(ns), dtype=torch.bfloat16, device=device)
    gemv_seg(dev(x, device), None if nw is None else dev(nw, device), 1e-6, *(dev(w, device) for w in W), y)
    torch.cuda.synchronize()
    assert_gemv_close(host_bits(y), gemv_ref(x, [w for w in W if w.shape[0]], nw, 1e-6), f"seg M={M} K={K} ns={ns}")


@pytest.mark.parametrize("M,K,N", [(3, 2056, 203), (4, 4096, 2060)])
def test_rows_apart(device, M, K, N):
    """Rows of x and y that do not follow one another."""
    rng = np.random.default_rng(K + N)
    x, nw = rand_bits(rng, M, K), f32_to_bf16((1 + 0.2 * rng.standard_normal(K)).astype(np.float32))
    wg, wu = (rand_bits(rng, N, K, scale=K ** -0.5) for _ in range(2))
    xs = torch.full((M, K + 64), float("nan"), dtype=torch.bfloat16, device=device)[:, :K]
    xs.copy_(dev(x, device))
    ys = torch.full((M, N + 5), 7.0, dtype=torch.bfloat16, device=device)
    gemv_gateup(xs, dev(nw, device), 1e-6, dev(wg, device), dev(wu, device), ys[:, :N])
    torch.cuda.synchronize()
    assert_gemv_close(host_bits(ys[:, :N].contiguous()), gemv_ref(x, [wg, wu], nw, 1e-6, epilogue="silu_mul"), f"M={M} K={K}")
    assert (ys[:, N:] == 7.0).all()


@pytest.mark.parametrize("K,N", [(2056, 1), (2176, 1023), (3072, 2050), (4096, 4099)])
def test_residual(device, K, N):  # on the kernel with x in LDS
    rng = np.random.default_rng(K + N)
    x, w, res = rand_bits(rng, 3, K), rand_bits(rng, N, K, scale=K ** -0.5), rand_bits(rng, 3, N)
    y = torch.empty(3, N, dtype=torch.bfloat16, device=device)
    xs = torch.zeros(3, K + 64, dtype=torch.bfloat16, device=device)[:, :K]  # rows of x apart
    xs.copy_(dev(x, device))
    gemv_resid(xs, dev(w, device), dev(res, device), y)
    torch.cuda.synchronize()
    assert_gemv_close(host_bits(y), gemv_ref(x, [w], epilogue="residual", res_bits=res), f"resid K={K} N={N}")


def test_infinite_weights_stay_in_their_row(device):
    """k = 2056 ends inside a chunk: the lanes past it must not read the next row."""
    M, K, N = 4, 2056, 40
    gen = torch.Generator().manual_seed(3)
    x, w = torch.randn(M, K, generator=gen).bfloat16(), torch.randn(N, K, generator=gen).bfloat16()
    w[1::2, :8] = float("inf")
    e = torch.empty(0, K, dtype=torch.bfloat16, device=device)
    y = gemv_seg(x.to(device), None, 0.0, w.to(device), e, e, torch.empty(M, N, dtype=torch.bfloat16, device=device))
    torch.cuda.synchronize()
    assert torch.isfinite(y[:, 0::2].float()).all() and not torch.isfinite(y[:, 1::2].float()).any()
