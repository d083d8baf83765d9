"""Calls on two streams whose last wave is summed by the GEMM itself: product, accumulator, this rank's rows, counters and
normalised rows against their definitions, at the partitions and storage orders where the rule changes sides."""
import numpy as np
import pytest
import torch

from gpu_util import BF16, F16, TORCH_DTYPE, seeded

pytestmark = pytest.mark.gpu
EPS = 1e-6


def _setup(fo, dtype, bm, bn, M, N, K, cseg, order):
    algo = fo._capi.find_algo(bm, bn, swizzle=4)
    TM, TN = M // bm, N // bn
    T = TM * TN
    assert sum(cseg) == T
    A, _ = seeded((M, K), dtype, M + K)
    B, _ = seeded((N, K), dtype, N + K, scale=K ** -0.5)
    before, _ = seeded((M * N,), dtype, 17)
    plain = torch.empty(M, N, device="cuda", dtype=TORCH_DTYPE[dtype])
    fo.ops.gemm(A, B, plain, algo)
    if order == "schedule":
        RA = fo.layout.reorder_indices(T, fo._capi.schedule_order(algo, M, N), device="cuda").reshape(TM, TN)
    else:  # any: the last slots belong to tiles of every wave
        RA = torch.from_numpy(np.random.default_rng(K).permutation(T).astype(np.int32)).reshape(TM, TN).cuda()
    cs = torch.tensor(cseg, dtype=torch.int32)
    MM = torch.zeros(fo.layout.counter_size(len(cseg), TM, TN), dtype=torch.int32, device="cuda")
    ov = fo.ops.Overlap()
    ov.set_schedule(in_stream_below_flop=0)  # two streams, however short
    ov.set_fused_consumer(0)                 # per-wave launches, however many groups
    return algo, A, B, before, plain, RA, cs, cs.cuda(), MM, ov


# 256x256 tiles of 128x128 reorder tiles: 8192x4096 is two whole waves of 1024 slots, 4096x7168 one and three quarters
@pytest.mark.parametrize("dtype,bm,bn,M,N,K,cseg,order", [
    (F16, 128, 128, 8192, 4096, 72, [1024, 1024], "schedule"),             # groups end with waves
    (BF16, 128, 128, 8192, 4096, 64, [2048], "schedule"),                  # one group over both
    (F16, 128, 128, 8192, 4096, 200, [700, 700, 648], "schedule"),         # the last begins in the last wave, the second before it
    (F16, 128, 128, 8192, 4096, 136, [1023, 2, 1023], "schedule"),         # one slot of a group on either side
    (BF16, 128, 256, 4096, 7168, 328, [400, 496], "schedule"),             # a partial last wave
    (F16, 256, 128, 8192, 4096, 72, [512, 300, 212], "any"),
    (BF16, 128, 128, 8192, 4096, 72, [1500, 548], "any"),
])
@pytest.mark.parametrize("norm", [False, True])
def test_allreduce(fo, dtype, bm, bn, M, N, K, cseg, order, norm):
    algo, A, B, before, plain, RA, cs, cs_gpu, MM, ov = _setup(fo, dtype, bm, bn, M, N, K, cseg, order)
    td = TORCH_DTYPE[dtype]
    gamma = (1 + 0.01 * torch.randn(N, generator=torch.Generator().manual_seed(3))).to(td).cuda()
    acc = before.clone()
    ov.set_accumulator(acc)
    RA_cpu = RA.cpu()
    want_y = torch.empty(M, N, device="cuda", dtype=td)
    for rep in range(2):
        C = torch.full((M * N,), float("nan"), device="cuda", dtype=td)
        Y = torch.full((M, N), float("nan"), device="cuda", dtype=td)
        was = acc.clone()
        if norm:
            ov.gemm_allreduce_rmsnorm_overlap(A, B, C, MM, RA, RA_cpu, 1, cs, cs_gpu, algo, Y, gamma, eps=EPS)
        else:
            ov.gemm_allreduce_overlap(A, B, C, MM, RA, 1, cs, cs_gpu, algo)
        torch.cuda.synchronize()
        assert ov.status() == 0
        assert torch.equal(fo.layout.unpermute(C, M, N, bm, bn, RA), plain)
        assert torch.equal(acc, (was.float() + C.float()).to(td))
        assert (MM == 0).all()
        if norm:
            fo.ops.reorder_rmsnorm_rows(C.view(M, N), want_y, gamma, 0, M, bm, bn, 1, RA, eps=EPS)  # the kernel that the call uses
            torch.cuda.synchronize()
            assert torch.equal(Y, want_y)
    ov.close()


@pytest.mark.parametrize("dtype,bm,bn,M,N,K,cseg,order,W", [
    (F16, 128, 128, 8192, 4096, 72, [512] * 4, "schedule", 8),             # the last two groups are the last wave
    (BF16, 128, 128, 8192, 4096, 136, [1024, 200, 824], "schedule", 2),
    (F16, 128, 128, 8192, 4096, 72, [1000, 1048], "schedule", 4),          # the last begins in the wave before: as ever
    (BF16, 256, 128, 8192, 4096, 64, [512, 512], "any", 8),
    (F16, 128, 256, 4096, 7168, 200, [512, 300, 84], "schedule", 4),       # a partial last wave
])
@pytest.mark.parametrize("own", [False, True])
def test_reduce_scatter(fo, dtype, bm, bn, M, N, K, cseg, order, W, own):
    algo, A, B, before, plain, RA, cs, cs_gpu, MM, ov = _setup(fo, dtype, bm, bn, M, N, K, cseg, order)
    td = TORCH_DTYPE[dtype]
    rank = W - 1
    ov.close()
    ov = fo.ops.Overlap(rank=rank, world=W)
    ov.set_schedule(in_stream_below_flop=0)
    ov.set_fused_consumer(0)
    RE = fo.layout.generate_row_mapping(M, N, bm, bn, cseg, W)
    acc = before.clone()
    ov.set_accumulator(acc)
    C = torch.full((M * N,), float("nan"), device="cuda", dtype=td)
    D = torch.full((M // W * N,), float("nan"), device="cuda", dtype=td) if own else None
    ov.gemm_reducescatter_overlap(A, B, C, D, MM, RA, RE, 1, cs, cs_gpu, algo)
    torch.cuda.synchronize()
    assert ov.status() == 0 and (MM == 0).all()
    assert torch.equal(fo.layout.unpermute(C, M, N, bm, bn, RA, RE=RE), plain)
    rows, seg = C.view(-1, bn), M * N // bn // W
    want, mine, first = torch.empty_like(rows), [], 0
    for n in cseg:
        chunk = rows[first:first + n * bm].view(W, n * bm // W, bn)
        for q in range(W):
            want[q * seg + first // W:q * seg + (first + n * bm) // W] = chunk[q]
        mine.append(chunk[rank])
        first += n * bm
    assert torch.equal(acc, (before.float() + want.reshape(-1).float()).to(td))
    if own:
        assert torch.equal(D.view(-1, bn), torch.cat(mine))
    ov.close()
