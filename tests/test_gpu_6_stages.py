"""GPU parity of every workgroup tile for each small number of K steps, with operand rows on 128-byte lines and off them:
fragments are held for one stage or two in turn, fetched ahead of the stage they belong to, so that the first, the last and
an odd number of stages are where the order can go wrong."""
import pytest
import torch

from gpu_util import BF16, F16, TORCH_DTYPE, max_rel_err, seeded

pytestmark = pytest.mark.gpu

TILES = [  # reorder tile, M, N       workgroup tile
    (128, 128, 128, 256),           # 32x32
    (128, 128, 128, 3072),          # 64x32
    (256, 128, 256, 2944),          # 64x64
    (128, 128, 384, 3200),          # 64x96
    (128, 128, 512, 3456),          # 64x128
    (128, 128, 1408, 1536),         # 96x128
    (128, 128, 2560, 1280),         # 128x128
    (128, 128, 1920, 2560),         # 128x160
    (128, 128, 1280, 4096),         # 128x192
    (128, 128, 3968, 1920),         # 128x256
    (256, 128, 3840, 1920),         # 256x128
    (128, 256, 4096, 4096),         # 256x256
]


@pytest.mark.parametrize("K", [8, 64, 72, 128, 136, 192, 256, 264, 320, 392, 512, 648])
@pytest.mark.parametrize("bm,bn,M,N", TILES)
def test_stages(fo, bm, bn, M, N, K):
    dtype = F16 if K % 64 else BF16
    algo = fo._capi.find_algo(bm, bn, swizzle=4)
    A, _ = seeded((M, K), dtype, M + K)
    B, _ = seeded((N, K), dtype, N + K, scale=K ** -0.5)
    C = torch.full((M, N), float("nan"), device="cuda", dtype=TORCH_DTYPE[dtype])
    fo.ops.gemm(A, B, C, algo)
    # one rounding to 16 bits: 2^-11 of the value (fp16), 2^-9 (bf16), sums in 32 bits in another order behind it
    assert max_rel_err(C.float(), A.float() @ B.float().T) <= 1e-2
