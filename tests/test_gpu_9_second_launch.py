"""Launches without counters whose last round of 256x256 tiles goes to a second launch, in each tile that it may have (64x64,
64x128, 128x128, 128x256), with every epilogue, its positions inside of the matrix and half outside at both edges: all tiles sum a product
in the same order, so the whole product must have the bits of its slices of 512 rows, which are single rounds of small tiles.  That the
second launch is there, and in which tile, is asserted."""
import numpy as np
import pytest
import torch

from gpu_util import TORCH_DTYPE, seeded
from second_launch_cases import CASES, FORMS, expected, planned

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in c[:6]))
def test_second_launch(fo, case):
    dtype, bm, bn, M, N, K = case[:6]
    ops, layout, td = fo.ops, fo.layout, TORCH_DTYPE[dtype]
    algo = fo._capi.find_algo(bm, bn, swizzle=4)
    TM, TN = M // bm, N // bn
    T, W, rank = TM * TN, 4, 2
    A, _ = seeded((M, K), dtype, M + K)
    B, _ = seeded((N, K), dtype, N + K, scale=K ** -0.5)
    before, _ = seeded((M * N,), dtype, 7)
    for form in FORMS:
        _, second, edges = planned(case, form, A.data_ptr(), B.data_ptr())
        assert (second, edges) == (expected(case, form), case[7] if second else "")
    want = torch.full((M, N), float("nan"), device="cuda", dtype=td)
    for row in range(0, M, 512):
        ops.gemm(A[row:row + 512], B, want[row:row + 512], algo)
    plain = torch.full((M, N), float("nan"), device="cuda", dtype=td)
    ops.gemm(A, B, plain, algo)
    assert torch.equal(plain, want)

    ov = ops.Overlap(rank=rank, world=W)
    ov.set_schedule(in_stream_below_flop=1e15)
    acc = before.clone()
    ov.set_accumulator(acc)
    C = torch.full((M, N), float("nan"), device="cuda", dtype=td)
    ov.gemm_allreduce(A, B, C, algo)
    torch.cuda.synchronize()
    assert torch.equal(C, want) and torch.equal(acc, (before.float() + C.view(-1).float()).to(td))

    cseg = [T // 3, T - T // 3]
    RA = torch.from_numpy(np.random.default_rng(M + N).permutation(T).astype(np.int32)).reshape(TM, TN).cuda()
    cs_cpu = torch.tensor(cseg, dtype=torch.int32)
    cs_gpu = cs_cpu.cuda()
    MM = torch.zeros(layout.counter_size(len(cseg), TM, TN), dtype=torch.int32, device="cuda")
    RE = layout.generate_row_mapping(M, N, bm, bn, cseg, W)
    for with_acc in (True, False):
        acc = before.clone()
        ov.set_accumulator(acc if with_acc else None)
        C = torch.full((M * N,), float("nan"), device="cuda", dtype=td)
        ov.gemm_allreduce_overlap(A, B, C, MM, RA, 1, cs_cpu, cs_gpu, algo)
        torch.cuda.synchronize()
        assert torch.equal(layout.unpermute(C, M, N, bm, bn, RA), want)
        if with_acc:
            assert torch.equal(acc, (before.float() + C.float()).to(td))

        acc = before.clone()
        ov.set_accumulator(acc if with_acc else None)
        C.fill_(float("nan"))
        D = torch.full((M // W, N), float("nan"), device="cuda", dtype=td)
        ov.gemm_reducescatter_overlap(A, B, C, D, MM, RA, RE, 1, cs_cpu, cs_gpu, algo)
        torch.cuda.synchronize()
        assert torch.equal(layout.unpermute(C, M, N, bm, bn, RA, RE=RE), want)
        rows, seg = C.view(-1, bn), M * N // bn // W
        summed, own, first = torch.empty_like(rows), [], 0
        for n in cseg:
            chunk = rows[first:first + n * bm].view(W, n * bm // W, bn)
            for q in range(W):
                summed[q * seg + first // W:q * seg + (first + n * bm) // W] = chunk[q]
            own.append(chunk[rank])
            first += n * bm
        assert torch.equal(D.view(-1, bn), torch.cat(own))
        if with_acc:
            assert torch.equal(acc, (before.float() + summed.reshape(-1).float()).to(td))
    assert (MM == 0).all()
    ov.close()
