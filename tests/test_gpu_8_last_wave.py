"""Calls on two streams whose last wave is summed by the GEMM itself: product, accumulator, this rank's rows, counters and
normalised rows against their definitions, at the partitions and storage orders where the rule changes sides; and what
automatic mode keeps on one stream against what two streams leave.  Every route gives the same bits: which one a call takes
is asked of the planners that the calls decide with."""
import numpy as np
import pytest
import torch

from gpu_util import BF16, F16, TORCH_DTYPE, planned_route, seeded

pytestmark = pytest.mark.gpu
EPS = 1e-6
TWO_STREAMS = dict(in_stream_below_flop=0, fused_from_groups=1 << 20)  # however short, and launches per wave however many groups


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
    ov.set_schedule(**TWO_STREAMS)
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
    per_wave = 256 * (256 // bm) * (256 // bn)
    first = (sum(cseg) - 1) // per_wave * per_wave
    across = first not in np.cumsum(cseg)  # groups across waves: the call that also normalises leaves the GEMM its sums then
    last_begins = sum(cseg) if norm and not across else first
    for rep in range(2):
        C = torch.full((M * N,), float("nan"), device="cuda", dtype=td)
        Y = torch.full((M, N), float("nan"), device="cuda", dtype=td)
        was = acc.clone()
        rows = (Y, gamma) if norm else (None, None)
        assert planned_route(fo, ov, dtype, A, B, C, cseg, algo, 1, *rows) == last_begins
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
    (BF16, 128, 128, 8192, 4096, 136, [4] * 512, "schedule", 8),           # more groups than their sizes are held in registers
    (F16, 128, 128, 8192, 4096, 72, [1024] + [1, 3] * 256, "any", 2),
])
@pytest.mark.parametrize("own", [False, True])
def test_reduce_scatter(fo, dtype, bm, bn, M, N, K, cseg, order, W, own):
    algo, A, B, before, plain, RA, cs, cs_gpu, MM, ov = _setup(fo, dtype, bm, bn, M, N, K, cseg, order)
    td = TORCH_DTYPE[dtype]
    rank = W - 1
    ov.close()
    ov = fo.ops.Overlap(rank=rank, world=W)
    ov.set_schedule(**TWO_STREAMS)
    RE = fo.layout.generate_row_mapping(M, N, bm, bn, cseg, W)
    acc = before.clone()
    ov.set_accumulator(acc)
    C = torch.full((M * N,), float("nan"), device="cuda", dtype=td)
    D = torch.full((M // W * N,), float("nan"), device="cuda", dtype=td) if own else None
    per_wave = 256 * (256 // bm) * (256 // bn)
    first = (sum(cseg) - 1) // per_wave * per_wave
    route = planned_route(fo, ov, dtype, A, B, C, cseg, algo, D=D, scatter=True)
    assert route == (first if first in np.cumsum(cseg) else sum(cseg))
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


@pytest.mark.parametrize("dtype,bm,bn,M,N,K,cseg,order,W", [
    (F16, 128, 128, 8192, 4096, 72, [512] * 4, "schedule", 8),
    (BF16, 256, 128, 8192, 4096, 136, [512, 512], "any", 2),
    (F16, 128, 256, 4096, 7168, 200, [512, 300, 84], "schedule", 4),
    (BF16, 128, 128, 8192, 4096, 64, [4] * 512, "schedule", 8),            # groups beyond the registers again
])
def test_reduce_scatter_rows_without_accumulator(fo, dtype, bm, bn, M, N, K, cseg, order, W):
    """The same without an accumulator: this rank's rows of the last wave are the GEMM's too."""
    algo, A, B, before, plain, RA, cs, cs_gpu, MM, ov = _setup(fo, dtype, bm, bn, M, N, K, cseg, order)
    ov.close()
    rank = 0
    ov = fo.ops.Overlap(rank=rank, world=W)
    ov.set_schedule(**TWO_STREAMS)
    RE = fo.layout.generate_row_mapping(M, N, bm, bn, cseg, W)
    td = TORCH_DTYPE[dtype]
    for rep in range(2):
        C = torch.full((M * N,), float("nan"), device="cuda", dtype=td)
        D = torch.full((M // W * N,), float("nan"), device="cuda", dtype=td)
        first = 256 * (256 // bm) * (256 // bn)  # two waves
        assert planned_route(fo, ov, dtype, A, B, C, cseg, algo, D=D, scatter=True) == first
        ov.gemm_reducescatter_overlap(A, B, C, D, MM, RA, RE, 1, cs, cs_gpu, algo)
        torch.cuda.synchronize()
        assert ov.status() == 0 and (MM == 0).all()
        assert torch.equal(fo.layout.unpermute(C, M, N, bm, bn, RA, RE=RE), plain)
        rows, mine, first = C.view(-1, bn), [], 0
        for n in cseg:
            mine.append(rows[first:first + n * bm].view(W, n * bm // W, bn)[rank])
            first += n * bm
        assert torch.equal(D.view(-1, bn), torch.cat(mine))
    ov.close()


@pytest.mark.parametrize("dtype,bm,bn,M,N,K,groups,order,rldn", [
    (F16, 128, 128, 4096, 4096, 2048, 4, "schedule", 1),      # one round
    (BF16, 128, 256, 4096, 4096, 2104, 20, "any", 2),         # one round, more groups than per-wave launches are made for
    (F16, 128, 128, 8192, 4096, 1032, 3, "schedule", 1),      # two waves of whole rows, groups across them
    (BF16, 256, 128, 6144, 6144, 1024, 5, "any", 1),          # two waves and a quarter, not whole rows
    (F16, 128, 128, 8192, 8192, 520, 700, "schedule", 2),     # four waves, very many groups
])
@pytest.mark.parametrize("norm", [False, True])
def test_automatic_choice_against_two_streams(fo, dtype, bm, bn, M, N, K, groups, order, rldn, norm):
    """What automatic mode does on one stream and what two streams leave: the same product, accumulator, counters and rows."""
    T = (M // bm) * (N // bn)
    cuts = [T * g // groups for g in range(groups + 1)]
    cseg = [b - a for a, b in zip(cuts, cuts[1:])]
    algo, A, B, before, plain, RA, cs, cs_gpu, MM, ov = _setup(fo, dtype, bm, bn, M, N, K, cseg, order)
    ov.set_schedule()
    td = TORCH_DTYPE[dtype]
    gamma = (1 + 0.01 * torch.randn(N, generator=torch.Generator().manual_seed(5))).to(td).cuda()
    RA_cpu = RA.cpu()
    left = []
    for fused in (-1, 0):
        ov.set_fused_consumer(fused)
        acc = before.clone()
        C = torch.full((M * N,), float("nan"), device="cuda", dtype=td)
        Y = torch.full((M, N), float("nan"), device="cuda", dtype=td)
        ov.set_accumulator(acc)
        rows = (Y, gamma) if norm else (None, None)
        assert planned_route(fo, ov, dtype, A, B, C, cseg, algo, rldn, *rows) == (0 if fused < 0 else T)
        for rep in range(2):
            if norm:
                ov.gemm_allreduce_rmsnorm_overlap(A, B, C, MM, RA, RA_cpu, rldn, cs, cs_gpu, algo, Y, gamma, eps=EPS)
            else:
                ov.gemm_allreduce_overlap(A, B, C, MM, RA, rldn, cs, cs_gpu, algo)
        torch.cuda.synchronize()
        assert ov.status() == 0 and (MM == 0).all()
        left.append((C, acc, Y))
    assert torch.equal(fo.layout.unpermute(left[0][0], M, N, bm, bn, RA, rLDN=rldn), plain)
    assert torch.equal(left[0][0], left[1][0])
    assert torch.equal(left[0][1], left[1][1])
    if norm:
        assert torch.equal(left[0][2], left[1][2])
    ov.close()


@pytest.mark.parametrize("dtype,bm,bn,M,N,K,cseg,W", [
    (F16, 128, 128, 4096, 4096, 2056, [256] * 4, 8),          # one round; without an accumulator two streams all the same
    (F16, 128, 128, 3328, 4096, 2504, [208] * 4, 8),          # five sixths of one
    (BF16, 256, 128, 4096, 8192, 2048, [50] * 20 + [24], 4),  # two waves, more groups than per-wave launches are made for
    (F16, 128, 128, 4224, 7168, 1032, [500, 700, 648], 2),    # rows that 256 does not divide
])
@pytest.mark.parametrize("with_acc", [True, False])
def test_automatic_choice_of_a_reduce_scatter(fo, dtype, bm, bn, M, N, K, cseg, W, with_acc):
    """The same for a reduce-scatter: product, accumulator, this rank's rows and counters."""
    rank = W - 1
    algo, A, B, before, plain, RA, cs, cs_gpu, MM, ov = _setup(fo, dtype, bm, bn, M, N, K, cseg, "schedule")
    ov.close()
    ov = fo.ops.Overlap(rank=rank, world=W)
    RE = fo.layout.generate_row_mapping(M, N, bm, bn, cseg, W)
    left = []
    for fused in (-1, 0):
        ov.set_fused_consumer(fused)
        acc = before.clone()
        ov.set_accumulator(acc if with_acc else None)
        C = torch.full((M * N,), float("nan"), device="cuda", dtype=TORCH_DTYPE[dtype])
        D = torch.full((M // W * N,), float("nan"), device="cuda", dtype=TORCH_DTYPE[dtype])
        one_stream = fused < 0 and (with_acc or M != 4096 or N != 4096)
        assert planned_route(fo, ov, dtype, A, B, C, cseg, algo, D=D, scatter=True) == (0 if one_stream else sum(cseg))
        for rep in range(2):
            ov.gemm_reducescatter_overlap(A, B, C, D, MM, RA, RE, 1, cs, cs_gpu, algo)
        torch.cuda.synchronize()
        assert ov.status() == 0 and (MM == 0).all()
        left.append((C, acc, D))
    assert torch.equal(fo.layout.unpermute(left[0][0], M, N, bm, bn, RA, RE=RE), plain)
    for one, two in zip(*left):
        assert torch.equal(one, two)
    ov.close()


@pytest.mark.parametrize("call,cseg", [
    ("allreduce", [700, 700, 648]),
    ("norm", [2048]),
    ("reducescatter", [512] * 4),
    ("reducescatter without accumulator", [512] * 4),
])
def test_captured_in_a_hip_graph(fo, call, cseg):
    """A call whose last wave the GEMM sums, captured once and replayed with other operands and eager work between the replays."""
    dtype, bm, bn, M, N, K, W = F16, 128, 128, 8192, 4096, 200, 8
    td, scatter, with_acc = TORCH_DTYPE[dtype], call.startswith("reducescatter"), "without" not in call
    algo, A, B, before, plain, RA, cs, cs_gpu, MM, ov = _setup(fo, dtype, bm, bn, M, N, K, cseg, "schedule")
    ov.close()
    gamma = (1 + 0.01 * torch.randn(N, generator=torch.Generator().manual_seed(7))).to(td).cuda()
    RA_cpu, RE = RA.cpu(), fo.layout.generate_row_mapping(M, N, bm, bn, cseg, W) if scatter else None
    C, acc = torch.empty(M * N, device="cuda", dtype=td), before.clone()
    D, Y, want_y = (torch.empty(r, N, device="cuda", dtype=td) for r in (M // W, M, M))
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        ov = fo.ops.Overlap(rank=W - 1, world=W) if scatter else fo.ops.Overlap()
        ov.set_schedule(**TWO_STREAMS)
        ov.set_accumulator(acc if with_acc else None)

        def step():
            if scatter:
                ov.gemm_reducescatter_overlap(A, B, C, D, MM, RA, RE, 1, cs, cs_gpu, algo)
            elif call == "norm":
                ov.gemm_allreduce_rmsnorm_overlap(A, B, C, MM, RA, RA_cpu, 1, cs, cs_gpu, algo, Y, gamma, eps=EPS)
            else:
                ov.gemm_allreduce_overlap(A, B, C, MM, RA, 1, cs, cs_gpu, algo)

        step()  # one-time kernel attribute set-up
    torch.cuda.synchronize()
    rows = (Y, gamma) if call == "norm" else (None, None)
    assert planned_route(fo, ov, dtype, A, B, C, cseg, algo, 1, *rows, D=D, scatter=scatter) == 1024
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        step()
    torch.cuda.synchronize()
    acc.copy_(before)
    A0 = A.clone()
    for rep in range(4):
        A.copy_((A0 * (0.5 + 0.25 * rep)).roll(rep * 11, dims=1))
        C.fill_(float("nan"))
        Y.fill_(float("nan"))
        D.fill_(float("nan"))
        was = acc.clone()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        fo.ops.gemm(A, B, plain, algo)
        torch.cuda.synchronize()
        assert torch.equal(fo.layout.unpermute(C, M, N, bm, bn, RA, RE=RE), plain), f"replay {rep}"
        if scatter:
            view, seg = C.view(-1, bn), M * N // bn // W
            want, mine, first = torch.empty_like(view), [], 0
            for n in cseg:
                chunk = view[first:first + n * bm].view(W, n * bm // W, bn)
                want.view(W, seg, bn)[:, first // W:(first + n * bm) // W] = chunk
                mine.append(chunk[W - 1])
                first += n * bm
            assert torch.equal(D.view(-1, bn), torch.cat(mine)), f"replay {rep}"
        else:
            want = C
        if with_acc:
            assert torch.equal(acc, (was.float() + want.reshape(-1).float()).to(td)), f"replay {rep}"
        if call == "norm":
            fo.ops.reorder_rmsnorm_rows(C.view(M, N), want_y, gamma, 0, M, bm, bn, 1, RA, eps=EPS)
            torch.cuda.synchronize()
            assert torch.equal(Y, want_y), f"replay {rep}"
        assert (MM == 0).all() and ov.status() == 0
    ov.close()
