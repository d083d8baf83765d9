"""GPU parity of every workgroup tile of the GEMM at the sizes where it can go wrong: tiles moved back at the end of
a dimension, tiles that lie across two reorder tiles, partial last K steps, one K step, the second launch over the
last wave's positions.  The plain product against torch in fp32; the reordered store (row-mapped as well) bit for
bit against the plain product through the inverse permutation; counters and stamps exact."""
import numpy as np
import pytest
import torch

from gpu_util import BF16, F16, TORCH_DTYPE, max_rel_err, seeded

pytestmark = pytest.mark.gpu

CASES = [  # dtype, reorder tile, M, N, K                workgroup tile
    (F16, 128, 128, 128, 256, 8),                      # 32x32, one chunk of K
    (BF16, 128, 256, 256, 1024, 1544),                 # 32x32, parts of a 128x256 reorder tile, counted behind the launch
    (BF16, 128, 128, 128, 1024, 1000),                 # 32x32, accumulator no larger than an allocation's granule
    (F16, 128, 128, 128, 3072, 136),                   # 64x32
    (BF16, 256, 128, 256, 2944, 1672),                 # 64x64
    (F16, 128, 128, 384, 3200, 200),                   # 64x96, across reorder tiles and moved back along N
    (BF16, 128, 256, 256, 5632, 1608),                 # 64x96 over 256-wide reorder tiles
    (F16, 128, 128, 512, 3456, 1600),                  # 64x128
    (BF16, 128, 128, 1408, 1536, 328),                 # 96x128, moved back along M
    (F16, 256, 128, 1536, 1408, 1544),                 # 96x128 over 256-high reorder tiles
    (F16, 128, 128, 2560, 1280, 64),                   # 128x128, one K step
    (BF16, 128, 128, 1920, 2560, 136),                 # 128x160
    (F16, 256, 128, 2048, 2432, 1600),                 # 128x160, half of each 256-high reorder tile, moved back along N
    (F16, 128, 128, 3968, 1920, 72),                   # two rounds of 128x128
    (BF16, 256, 128, 3840, 1920, 192),                 # 256x128
    (F16, 128, 128, 4224, 3200, 136),                  # 256x256, half a tile left along both
    (BF16, 128, 256, 4224, 3328, 72),                  # 256x256, half a tile left along M
    (BF16, 128, 128, 4224, 4352, 264),                 # 256x256 and a second launch for the last wave
    (F16, 128, 128, 1280, 4096, 192),                  # 128x192, operand rows on 128-byte lines
    (BF16, 256, 128, 2048, 2816, 64),                  # 128x192 over 256-high reorder tiles
    (F16, 128, 128, 3968, 1920, 128),                  # 128x256, the same
    (F16, 128, 128, 2048, 4224, 136),                  # two rounds of 128x160; 256x256 with counters
    (BF16, 128, 256, 2048, 4608, 1600),                # the same over 256-wide reorder tiles, on lines
    (BF16, 256, 128, 2304, 4096, 72),                  # the same over 256-high ones
    (BF16, 128, 128, 1792, 4608, 72),                  # two rounds of 128x128
    (F16, 128, 128, 3456, 4864, 64),                   # three rounds of 128x192
]


@pytest.mark.parametrize("dtype,bm,bn,M,N,K", CASES)
def test_workgroup_tiles(fo, dtype, bm, bn, M, N, K):
    ops, layout, td = fo.ops, fo.layout, TORCH_DTYPE[dtype]
    algo = fo._capi.find_algo(bm, bn, swizzle=4)
    TM, TN = M // bm, N // bn
    T = TM * TN
    A, _ = seeded((M, K), dtype, M + K)
    B, _ = seeded((N, K), dtype, N + K, scale=K ** -0.5)
    plain = torch.full((M, N), float("nan"), device="cuda", dtype=td)
    ops.gemm(A, B, plain, algo)
    assert max_rel_err(plain.float(), A.float() @ B.float().T) <= 1e-2
    rng = np.random.default_rng(M + N)
    RA = torch.from_numpy(rng.permutation(T).astype(np.int32)).reshape(TM, TN).cuda()
    cseg = [T] if T < 3 else [1, T // 2, T - 1 - T // 2]
    cs_cpu = torch.tensor(cseg, dtype=torch.int32)
    cs_gpu = cs_cpu.cuda()
    RE = layout.generate_row_mapping(M, N, bm, bn, cseg, 2)
    Cp = torch.empty(M * N, device="cuda", dtype=td)

    def check(what, RE=None, rLDN=1):
        torch.cuda.synchronize()
        assert torch.equal(layout.unpermute(Cp, M, N, bm, bn, RA, rLDN=rLDN, RE=RE), plain), what
        Cp.fill_(float("nan"))

    Cp.fill_(float("nan"))
    # with counters
    MM = torch.zeros(layout.counter_size(len(cseg), TM, TN), dtype=torch.int32, device="cuda")
    for re, rldn in ((None, 1), (RE, 1), (None, 2 if T % 2 == 0 else 1)):
        ops.gemm_signal(A, B, Cp, MM, RA, cs_gpu, algo, rLDN=rldn, RE=re)
        check("signalled", re, rldn)
        assert MM[:len(cseg)].tolist() == cseg and (MM[len(cseg):] == 0).all()
        MM.zero_()
    if len(cseg) <= TN - 1:  # monitor: its order counter lives at MM[TN - 1]
        MMm = torch.zeros(layout.counter_size(len(cseg), TM, TN, True), dtype=torch.int32, device="cuda")
        ops.gemm_signal(A, B, Cp, MMm, RA, cs_gpu, algo, monitor=True)
        check("monitored")
        mm = MMm.cpu()
        assert mm[:len(cseg)].tolist() == cseg and mm[TN - 1] == T
        assert sorted(mm[TN:TN + T].tolist()) == list(range(T))
    # without (a call that stays on one stream)
    ov = ops.Overlap(world=2)
    ov.set_schedule(in_stream_below_flop=1e15)
    ov.gemm_allreduce_overlap(A, B, Cp, MM, RA, 1, cs_cpu, cs_gpu, algo)
    check("on one stream")
    D = torch.empty(M // 2, N, device="cuda", dtype=td)
    ov.gemm_reducescatter_overlap(A, B, Cp, D, MM, RA, RE, 1, cs_cpu, cs_gpu, algo)
    torch.cuda.synchronize()
    assert torch.equal(layout.unpermute(D.reshape(-1), M // 2, N, bm // 2, bn, RA), plain[0::2])
    check("on one stream, row-mapped", RE)
    assert (MM == 0).all()
    ov.close()


@pytest.mark.parametrize("dtype,bm,bn,M,N,K", CASES)
def test_accumulating_epilogue(fo, dtype, bm, bn, M, N, K):
    """A call on one stream with an accumulator attached: same product, and the accumulator the once-rounded sum."""
    ops, layout, td = fo.ops, fo.layout, TORCH_DTYPE[dtype]
    algo = fo._capi.find_algo(bm, bn, swizzle=4)
    TM, TN = M // bm, N // bn
    T = TM * TN
    A, _ = seeded((M, K), dtype, M + K)
    B, _ = seeded((N, K), dtype, N + K, scale=K ** -0.5)
    before, _ = seeded((M, N), dtype, 7)
    acc = before.clone()
    plain, C = (torch.full((M, N), float("nan"), device="cuda", dtype=td) for _ in range(2))
    ops.gemm(A, B, plain, algo)
    ov = ops.Overlap()
    ov.set_schedule(in_stream_below_flop=1e15)
    ov.set_accumulator(acc)
    ov.gemm_allreduce(A, B, C, algo)
    torch.cuda.synchronize()
    assert torch.equal(C, plain)
    assert torch.equal(acc, (before.float() + plain.float()).to(td))
    RA = torch.from_numpy(np.random.default_rng(M + N).permutation(T).astype(np.int32)).reshape(TM, TN).cuda()
    cs_cpu = torch.tensor([T], dtype=torch.int32)
    MM = torch.zeros(layout.counter_size(1, TM, TN), dtype=torch.int32, device="cuda")
    for rldn in (1, 2 if T % 2 == 0 else 1):
        C.fill_(float("nan"))
        acc.copy_(before)
        ov.gemm_allreduce_overlap(A, B, C, MM, RA, rldn, cs_cpu, cs_cpu.cuda(), algo)
        torch.cuda.synchronize()
        assert torch.equal(layout.unpermute(C, M, N, bm, bn, RA, rLDN=rldn), plain)
        assert torch.equal(acc.reshape(-1), (before.float() + C.float()).to(td).reshape(-1))
    assert (MM == 0).all()
    ov.close()


@pytest.mark.parametrize("dtype,bm,bn,M,N,K", CASES)
@pytest.mark.parametrize("W", [1, 8])
def test_reduce_scatter_epilogue(fo, dtype, bm, bn, M, N, K, W):
    """A reduce-scatter on one stream, with and without an accumulator: product, this rank's rows and the
    accumulator's W segments against the definition, group by group."""
    ops, layout, td = fo.ops, fo.layout, TORCH_DTYPE[dtype]
    algo = fo._capi.find_algo(bm, bn, swizzle=4)
    TM, TN = M // bm, N // bn
    T = TM * TN
    A, _ = seeded((M, K), dtype, M + K)
    B, _ = seeded((N, K), dtype, N + K, scale=K ** -0.5)
    before, _ = seeded((M * N,), dtype, 7)
    acc = before.clone()
    plain = torch.empty(M, N, device="cuda", dtype=td)
    ops.gemm(A, B, plain, algo)
    cseg = [T] if T < 3 else [1, T // 2, T - 1 - T // 2]
    if T > 600:
        cseg = [1] * 300 + [T - 300]  # more groups than the 256x256 kernel holds in registers
    RA = torch.from_numpy(np.random.default_rng(M + N).permutation(T).astype(np.int32)).reshape(TM, TN).cuda()
    RE = layout.generate_row_mapping(M, N, bm, bn, cseg, W)
    cs_cpu = torch.tensor(cseg, dtype=torch.int32)
    MM = torch.zeros(layout.counter_size(len(cseg), TM, TN), dtype=torch.int32, device="cuda")
    rank = W - 1
    ov = ops.Overlap(rank=rank, world=W)
    ov.set_schedule(in_stream_below_flop=1e15)
    for with_acc in (True, False):
        ov.set_accumulator(acc if with_acc else None)
        C = torch.full((M * N,), float("nan"), device="cuda", dtype=td)
        D = torch.full((M // W, N), float("nan"), device="cuda", dtype=td)
        ov.gemm_reducescatter_overlap(A, B, C, D, MM, RA, RE, 1, cs_cpu, cs_cpu.cuda(), algo)
        torch.cuda.synchronize()
        assert torch.equal(layout.unpermute(C, M, N, bm, bn, RA, RE=RE), plain)
        rows, seg = C.view(-1, bn), M * N // bn // W
        want, own = torch.empty_like(rows), []
        first = 0
        for n in cseg:
            chunk = rows[first:first + n * bm].view(W, n * bm // W, bn)
            for q in range(W):
                want[q * seg + first // W:q * seg + (first + n * bm) // W] = chunk[q]
            own.append(chunk[rank])
            first += n * bm
        assert torch.equal(D.view(-1, bn), torch.cat(own))
        if with_acc:
            assert torch.equal(acc, (before.float() + want.reshape(-1).float()).to(td))
    assert (MM == 0).all()
    ov.close()


LINES = [  # dtype, reorder tile, M, N, K       workgroup tile; K / 8 odd, even, a multiple of four; one to many K steps
    (F16, 128, 128, 128, 1024, 8),           # 32x32
    (BF16, 128, 128, 128, 1024, 1000),
    (F16, 128, 128, 128, 3072, 1112),        # 64x32
    (BF16, 128, 128, 256, 3072, 144),        # 64x64, one step and a part
    (F16, 128, 256, 256, 3072, 1064),
    (BF16, 128, 128, 384, 3200, 72),         # 64x96
    (F16, 128, 128, 384, 3200, 1120),
    (F16, 128, 128, 512, 3456, 456),         # 64x128
    (BF16, 256, 128, 512, 3456, 1656),
    (BF16, 128, 128, 1408, 1536, 184),       # 96x128
    (F16, 128, 128, 2560, 1280, 40),         # 128x128
    (F16, 128, 128, 2560, 1280, 1096),
]


@pytest.mark.parametrize("dtype,bm,bn,M,N,K", LINES)
def test_operand_rows_off_the_line(fo, dtype, bm, bn, M, N, K):
    """Operand rows that begin anywhere in a 128-byte line, by the leading dimension and by the operand's own address: every
    product is summed in the same order, so each result is that of the operands padded with zero columns to whole lines,
    bit for bit, whatever stands in memory around them."""
    ops, td = fo.ops, TORCH_DTYPE[dtype]
    algo = fo._capi.find_algo(bm, bn, swizzle=4)
    A, _ = seeded((M, K), dtype, M + K)
    B, _ = seeded((N, K), dtype, N + K, scale=K ** -0.5)
    before, _ = seeded((M, N), dtype, 7)
    Kp = -(-K // 64) * 64
    Ap, Bp = (torch.nn.functional.pad(t, (0, Kp - K)) for t in (A, B))
    want = torch.empty(M, N, device="cuda", dtype=td)
    ops.gemm(Ap, Bp, want, algo)
    assert max_rel_err(want.float(), A.float() @ B.float().T) <= 1e-2

    def placed(t, columns):  # t, that many columns behind a line's start, with NaN on both sides
        room = torch.full((t.numel() + 128,), float("nan"), device="cuda", dtype=td)
        view = room[columns:columns + t.numel()].view_as(t)
        view.copy_(t)
        return view

    ov = ops.Overlap()
    for a_columns, b_columns in ((64, 64), (72, 64), (88, 120)):
        a, b = placed(A, a_columns), placed(B, b_columns)
        C = torch.full((M, N), float("nan"), device="cuda", dtype=td)
        ops.gemm(a, b, C, algo)
        torch.cuda.synchronize()
        assert torch.equal(C, want), (a_columns, b_columns)
        acc = before.clone()
        C.fill_(float("nan"))
        ov.set_accumulator(acc)
        ov.gemm_allreduce(a, b, C, algo)
        torch.cuda.synchronize()
        assert torch.equal(C, want) and torch.equal(acc, (before.float() + want.float()).to(td))
    ov.close()


@pytest.mark.parametrize("alias", ["C", "A"])
def test_accumulator_in_an_operand_or_the_product(fo, alias):
    """An accumulator that shares memory with an operand or with the product is updated behind the GEMM, not by it."""
    ops, M, N = fo.ops, 256, 512
    algo = fo._capi.find_algo(128, 128, swizzle=4)
    A, _ = seeded((M, N), F16, 1)
    B, _ = seeded((N, N), F16, 2, scale=N ** -0.5)
    plain = torch.empty(M, N, device="cuda", dtype=torch.float16)
    ops.gemm(A, B, plain, algo)
    cs = torch.tensor([M // 128 * (N // 128)], dtype=torch.int32)
    RA = torch.arange(int(cs[0]), dtype=torch.int32, device="cuda").reshape(M // 128, N // 128)
    MM = torch.zeros(fo.layout.counter_size(1, M // 128, N // 128), dtype=torch.int32, device="cuda")
    RE = fo.layout.generate_row_mapping(M, N, 128, 128, [int(cs[0])], 1)
    for call in ("serial", "overlap", "scatter"):
        C = torch.empty_like(plain)
        a = A.clone()
        acc = C if alias == "C" else a
        D = torch.empty_like(plain)
        ov = ops.Overlap()
        ov.set_accumulator(acc)
        if call == "serial":
            ov.gemm_allreduce(a, B, C, algo)
        elif call == "overlap":
            ov.gemm_allreduce_overlap(a, B, C, MM, RA, 1, cs, cs.cuda(), algo)
        else:
            ov.gemm_reducescatter_overlap(a, B, C, D, MM, RA, RE, 1, cs, cs.cuda(), algo)
        torch.cuda.synchronize()
        if alias == "A":
            product = C
            want = (A.float().reshape(-1) + C.float().reshape(-1)).half()
        else:
            product = C / 2  # exact: the product added to itself
            want = C.reshape(-1)
        product = product.reshape(-1) if call == "serial" else fo.layout.unpermute(
            product.reshape(-1), M, N, 128, 128, RA, RE=RE if call == "scatter" else None)
        assert torch.equal(product.reshape(-1), plain.reshape(-1)), call
        assert torch.equal(acc.reshape(-1), want), call
        ov.close()


@pytest.mark.parametrize("groups", [16, 17, 300])
def test_reduce_scatter_without_accumulator_by_groups(fo, groups):
    """Both sides of the group count from which a long reduce-scatter without an accumulator stays on one stream."""
    ops, M, N, K, W, bm = fo.ops, 4352, 4352, 2048, 4, 128   # more than 6.4e10 flop, 289 tiles of 256x256
    algo = fo._capi.find_algo(bm, 128, swizzle=4)
    TM, TN = M // bm, N // 128
    T = TM * TN
    A, _ = seeded((M, K), F16, 1)
    B, _ = seeded((N, K), F16, 2, scale=K ** -0.5)
    plain = torch.empty(M, N, device="cuda", dtype=torch.float16)
    ops.gemm(A, B, plain, algo)
    cseg = [1] * (groups - 1) + [T - groups + 1]
    RA = torch.from_numpy(np.random.default_rng(3).permutation(T).astype(np.int32)).reshape(TM, TN).cuda()
    RE = fo.layout.generate_row_mapping(M, N, bm, 128, cseg, W)
    cs_cpu = torch.tensor(cseg, dtype=torch.int32)
    MM = torch.zeros(fo.layout.counter_size(groups, TM, TN), dtype=torch.int32, device="cuda")
    ov = ops.Overlap(rank=1, world=W)
    C = torch.full((M * N,), float("nan"), device="cuda", dtype=torch.float16)
    D = torch.full((M // W, N), float("nan"), device="cuda", dtype=torch.float16)
    ov.gemm_reducescatter_overlap(A, B, C, D, MM, RA, RE, 1, cs_cpu, cs_cpu.cuda(), algo)
    torch.cuda.synchronize()
    assert torch.equal(fo.layout.unpermute(C, M, N, bm, 128, RA, RE=RE), plain)
    rows, own, first = C.view(-1, 128), [], 0
    for n in cseg:
        own.append(rows[first:first + n * bm].view(W, n * bm // W, 128)[1])
        first += n * bm
    assert torch.equal(D.view(-1, 128), torch.cat(own))
    assert (MM == 0).all() and ov.status() == 0
    ov.close()


@pytest.mark.parametrize("bm,bn,M,N", [
    (128, 128, 4224, 4352),  # 256 divides N only
    (128, 256, 4224, 4352),
    (256, 128, 4352, 4224),  # 256 divides M only
    (128, 128, 2432, 7040),  # neither
    (128, 128, 8064, 4096),  # a last round that is nearly full
    (128, 128, 4096, 6144),  # 256x256 tiles: a round and a half
    (128, 256, 8192, 4096),  # 256x256 tiles: two rounds of whole rows
])
def test_counted_launch_walks_the_reported_order(fo, bm, bn, M, N):
    """What a consumer waits for group by group completes in the order that it was told: with the slots in the order of
    fo_schedule_order, workgroup w stamps the tiles of positions w, w + 256, ... one after the other."""
    ops, K = fo.ops, 128
    algo = fo._capi.find_algo(bm, bn, swizzle=4)
    TM, TN = M // bm, N // bn
    T = TM * TN
    per = (256 // bm) * (256 // bn) if M % 256 == 0 and N % 256 == 0 else 1
    A, _ = seeded((M, K), F16, 1)
    B, _ = seeded((N, K), F16, 2, scale=K ** -0.5)
    C = torch.empty(M * N, device="cuda", dtype=torch.float16)
    RA = fo.layout.reorder_indices(T, fo._capi.schedule_order(algo, M, N)).reshape(TM, TN)
    for RE in (None, fo.layout.generate_row_mapping(M, N, bm, bn, [T], 2)):
        MM = torch.zeros(fo.layout.counter_size(1, TM, TN, True), dtype=torch.int32, device="cuda")
        ops.gemm_signal(A, B, C, MM, RA, torch.tensor([T], dtype=torch.int32, device="cuda"), algo, monitor=True, RE=RE)
        stamps = MM[TN:TN + T].cpu()
        assert sorted(stamps.tolist()) == list(range(T))
        rounds = stamps.reshape(-1, per)
        assert (rounds[:-256].amax(dim=1) < rounds[256:].amin(dim=1)).all()
    assert fo._capi.wave_tiles(algo, M, N) == 256 * per


@pytest.mark.parametrize("M,N,K", [(4224, 4352, 2048), (8064, 8064, 4096)])  # 7.5e10 and 5.3e11 flop
@pytest.mark.parametrize("with_acc", [True, False])
@pytest.mark.parametrize("W", [1, 4])
@pytest.mark.parametrize("groups", [5, 9])
def test_reduce_scatter_that_256_does_not_divide(fo, M, N, K, with_acc, W, groups):
    """Both sides of the size and the group count from which such a call leaves sums and copies to launches behind the GEMM."""
    ops, bm = fo.ops, 128
    algo = fo._capi.find_algo(bm, 128, swizzle=4)
    TM, TN = M // bm, N // 128
    T = TM * TN
    A, _ = seeded((M, K), F16, 1)
    B, _ = seeded((N, K), F16, 2, scale=K ** -0.5)
    plain = torch.empty(M, N, device="cuda", dtype=torch.float16)
    ops.gemm(A, B, plain, algo)
    cseg = [T // groups] * (groups - 1) + [T - T // groups * (groups - 1)]
    RA = fo.layout.reorder_indices(T, fo._capi.schedule_order(algo, M, N)).reshape(TM, TN)
    RE = fo.layout.generate_row_mapping(M, N, bm, 128, cseg, W)
    cs_cpu = torch.tensor(cseg, dtype=torch.int32)
    MM = torch.zeros(fo.layout.counter_size(groups, TM, TN), dtype=torch.int32, device="cuda")
    before, _ = seeded((M * N,), F16, 7)
    acc = before.clone()
    ov = ops.Overlap(rank=W - 1, world=W)
    ov.set_accumulator(acc if with_acc else None)
    C = torch.full((M * N,), float("nan"), device="cuda", dtype=torch.float16)
    D = torch.full((M // W, N), float("nan"), device="cuda", dtype=torch.float16)
    ov.gemm_reducescatter_overlap(A, B, C, D, MM, RA, RE, 1, cs_cpu, cs_cpu.cuda(), algo)
    torch.cuda.synchronize()
    assert torch.equal(fo.layout.unpermute(C, M, N, bm, 128, RA, RE=RE), plain)
    rows, seg, own, first = C.view(-1, 128), M * N // 128 // W, [], 0
    want = torch.empty_like(rows)
    for n in cseg:
        chunk = rows[first:first + n * bm].view(W, n * bm // W, 128)
        for q in range(W):
            want[q * seg + first // W:q * seg + (first + n * bm) // W] = chunk[q]
        own.append(chunk[W - 1])
        first += n * bm
    assert torch.equal(D.view(-1, 128), torch.cat(own))
    if with_acc:
        assert torch.equal(acc, (before.float() + want.reshape(-1).float()).half())
    assert (MM == 0).all() and ov.status() == 0
    ov.close()


@pytest.mark.parametrize("bm,bn,M,N,K", [(128, 128, 512, 4096, 2048), (128, 256, 256, 8192, 1544), (256, 128, 512, 4096, 1536)])
def test_monitor_stamps_of_one_round_are_measured(fo, bm, bn, M, N, K):
    """Products that a launch without the monitor computes in parts of reorder tiles: the stamps are the order in which
    the launch completed the tiles (the eight XCDs interleave them), not the tiles' own order."""
    ops, T = fo.ops, (M // bm) * (N // bn)
    algo = fo._capi.find_algo(bm, bn, swizzle=4)
    TN = N // bn
    A, _ = seeded((M, K), F16, 1)
    B, _ = seeded((N, K), F16, 2, scale=K ** -0.5)
    C = torch.empty(M * N, device="cuda", dtype=torch.float16)
    RA = torch.arange(T, dtype=torch.int32, device="cuda").reshape(M // bm, TN)
    MM = torch.zeros(fo.layout.counter_size(1, M // bm, TN, True), dtype=torch.int32, device="cuda")
    ops.gemm_signal(A, B, C, MM, RA, torch.tensor([T], dtype=torch.int32, device="cuda"), algo, monitor=True)
    stamps = MM[TN:TN + T].tolist()
    assert MM[0] == T and MM[TN - 1] == T and sorted(stamps) == list(range(T))
    assert stamps != list(range(T))


@pytest.mark.parametrize("dtype,bm,bn,M,N,K", [
    (F16, 128, 128, 4096, 4096, 256),     # 256x256, four K steps: the accumulator is read in the epilogue
    (F16, 128, 128, 4096, 4096, 320),     # five: requested in the first four, one step left
    (BF16, 128, 256, 4096, 4096, 360),    # six, the last one partial
    (BF16, 128, 256, 4224, 7168, 384),    # half a tile left along M, a workgroup's second tile
    (F16, 128, 128, 4224, 7296, 520),     # half a tile left along both
])
def test_accumulator_requested_during_the_product(fo, dtype, bm, bn, M, N, K):
    """The 256x256 kernel asks for the accumulator's values while it multiplies: sums of every element once rounded, none of
    another's, over reordered and plain stores."""
    ops, layout, td = fo.ops, fo.layout, TORCH_DTYPE[dtype]
    algo = fo._capi.find_algo(bm, bn, swizzle=4)
    TM, TN = M // bm, N // bn
    A, _ = seeded((M, K), dtype, M + K)
    B, _ = seeded((N, K), dtype, N + K, scale=K ** -0.5)
    before, _ = seeded((M, N), dtype, 11)
    acc = before.clone()
    plain, C = (torch.full((M, N), float("nan"), device="cuda", dtype=td) for _ in range(2))
    ops.gemm(A, B, plain, algo)
    ov = ops.Overlap()
    ov.set_schedule(in_stream_below_flop=1e15)
    ov.set_accumulator(acc)
    ov.gemm_allreduce(A, B, C, algo)
    torch.cuda.synchronize()
    assert torch.equal(C, plain)
    assert torch.equal(acc, (before.float() + plain.float()).to(td))
    RA = torch.from_numpy(np.random.default_rng(K).permutation(TM * TN).astype(np.int32)).reshape(TM, TN).cuda()
    cs = torch.tensor([TM * TN], dtype=torch.int32)
    MM = torch.zeros(layout.counter_size(1, TM, TN), dtype=torch.int32, device="cuda")
    C.fill_(float("nan"))
    acc.copy_(before)
    ov.gemm_allreduce_overlap(A, B, C, MM, RA, 1, cs, cs.cuda(), algo)
    torch.cuda.synchronize()
    assert torch.equal(layout.unpermute(C, M, N, bm, bn, RA), plain)
    assert torch.equal(acc.reshape(-1), (before.float() + C.float()).to(td).reshape(-1))
    ov.close()


@pytest.mark.parametrize("dtype,bm,bn,M,N,K", [
    (BF16, 128, 128, 1152, 5120, 8),      # one chunk of K; the last tile moved back along N, tiles across reorder tiles
    (F16, 128, 128, 1152, 5120, 72),      # fewer K steps than stages
    (BF16, 128, 128, 1152, 5120, 1720),
    (F16, 128, 256, 1536, 3840, 1112),    # whole tiles along N, 256-wide reorder tiles
    (BF16, 256, 128, 1536, 3712, 456),    # 256-high reorder tiles
    (F16, 128, 128, 1792, 6912, 712),     # more than one round
])
def test_whole_lines_in_128x192_tiles(fo, dtype, bm, bn, M, N, K):
    """The 128x192 tile whose loads are whole lines: plain, reordered without and with an accumulator, and row-mapped (which it
    is not built for), each the product of the operands padded to whole lines, bit for bit."""
    ops, layout, td = fo.ops, fo.layout, TORCH_DTYPE[dtype]
    algo = fo._capi.find_algo(bm, bn, swizzle=4)
    TM, TN = M // bm, N // bn
    T = TM * TN
    A, _ = seeded((M, K), dtype, M + K)
    B, _ = seeded((N, K), dtype, N + K, scale=K ** -0.5)
    before, _ = seeded((M, N), dtype, 13)
    pad = -K % 64
    want, C = (torch.full((M, N), float("nan"), device="cuda", dtype=td) for _ in range(2))
    ops.gemm(*(torch.nn.functional.pad(t, (0, pad)) for t in (A, B)), want, algo)
    assert max_rel_err(want.float(), A.float() @ B.float().T) <= 1e-2
    ops.gemm(A, B, C, algo)
    torch.cuda.synchronize()
    assert torch.equal(C, want)
    RA = torch.from_numpy(np.random.default_rng(K).permutation(T).astype(np.int32)).reshape(TM, TN).cuda()
    cs = torch.tensor([T], dtype=torch.int32)
    RE = layout.generate_row_mapping(M, N, bm, bn, [T], 2)
    MM = torch.zeros(layout.counter_size(1, TM, TN), dtype=torch.int32, device="cuda")
    D = torch.empty(M // 2, N, device="cuda", dtype=td)
    acc = before.clone()
    ov = ops.Overlap(world=2)
    ov.set_schedule(in_stream_below_flop=1e15)
    for rldn in (1, 2 if T % 2 == 0 else 1):
        C.fill_(float("nan"))
        ov.gemm_allreduce_overlap(A, B, C, MM, RA, rldn, cs, cs.cuda(), algo)
        torch.cuda.synchronize()
        assert torch.equal(layout.unpermute(C, M, N, bm, bn, RA, rLDN=rldn), want)
    C.fill_(float("nan"))
    ov.gemm_reducescatter_overlap(A, B, C, D, MM, RA, RE, 1, cs, cs.cuda(), algo)
    torch.cuda.synchronize()
    assert torch.equal(layout.unpermute(C, M, N, bm, bn, RA, RE=RE), want)
    ov.set_accumulator(acc)
    C.fill_(float("nan"))
    ov.gemm_allreduce_overlap(A, B, C, MM, RA, 1, cs, cs.cuda(), algo)
    torch.cuda.synchronize()
    assert torch.equal(layout.unpermute(C, M, N, bm, bn, RA), want)
    assert torch.equal(acc.reshape(-1), (before.float() + C.float()).to(td).reshape(-1))
    assert (MM == 0).all()
    ov.close()


@pytest.mark.parametrize("dtype,bm,bn,M,N,K", [
    (F16, 128, 128, 8064, 4224, 8),        # half a tile left along both, one K step, a workgroup's tiles half and whole in turn
    (BF16, 128, 128, 8064, 4224, 200),
    (F16, 128, 256, 4224, 7168, 648),      # along M
    (BF16, 256, 128, 4096, 7296, 128),     # along N, rows on the lines
])
def test_repeated_halves_are_not_multiplied(fo, dtype, bm, bn, M, N, K):
    """256x256 tiles with half a tile left: the wavefronts of the half that another tile computes bring operands only.  Plain
    and reordered without counters, against the launch with counters (other tiles) bit for bit."""
    ops, layout, td = fo.ops, fo.layout, TORCH_DTYPE[dtype]
    algo = fo._capi.find_algo(bm, bn, swizzle=4)
    TM, TN = M // bm, N // bn
    T = TM * TN
    A, _ = seeded((M, K), dtype, M + K)
    B, _ = seeded((N, K), dtype, N + K, scale=K ** -0.5)
    RA = torch.from_numpy(np.random.default_rng(K).permutation(T).astype(np.int32)).reshape(TM, TN).cuda()
    cs = torch.tensor([T], dtype=torch.int32)
    MM = torch.zeros(layout.counter_size(1, TM, TN), dtype=torch.int32, device="cuda")
    Cp = torch.full((M * N,), float("nan"), device="cuda", dtype=td)
    ops.gemm_signal(A, B, Cp, MM, RA, cs.cuda(), algo)
    torch.cuda.synchronize()
    want = layout.unpermute(Cp, M, N, bm, bn, RA)
    assert MM[0] == T
    MM.zero_()
    plain = torch.full((M, N), float("nan"), device="cuda", dtype=td)
    ops.gemm(A, B, plain, algo)
    torch.cuda.synchronize()
    assert torch.equal(plain, want)
    assert max_rel_err(plain.float(), A.float() @ B.float().T) <= 1e-2
    ov = ops.Overlap()
    for rldn in (1, 2 if T % 2 == 0 else 1):
        Cp.fill_(float("nan"))
        ov.gemm_allreduce_overlap(A, B, Cp, MM, RA, rldn, cs, cs.cuda(), algo)
        torch.cuda.synchronize()
        assert torch.equal(layout.unpermute(Cp, M, N, bm, bn, RA, rLDN=rldn), want)
    assert (MM == 0).all()
    ov.close()


@pytest.mark.parametrize("N,settings", [
    (32768, dict(in_stream_below_flop=1e15)),                         # one stream: rows of 17.8 million elements
    (16384, dict(in_stream_below_flop=0, fused_from_groups=1 << 20)),  # two: 8.9 million
])
def test_accumulator_rows_longer_than_a_buffer_range(fo, N, settings):
    """An output view as wide as all tiles side by side: a 128x128 block of the accumulator then spans more than 31 bits, and its
    old values are read with whole addresses, or left to the consumer."""
    ops, td, M, K, bm, bn = fo.ops, TORCH_DTYPE[F16], 69632, 640, 128, 128
    algo = fo._capi.find_algo(bm, bn, swizzle=4)
    TM, TN = M // bm, N // bn
    T = TM * TN
    g = torch.Generator(device="cuda").manual_seed(5)
    A = torch.randn(M, K, generator=g, device="cuda", dtype=td)
    B = torch.randn(N, K, generator=g, device="cuda", dtype=td) * K ** -0.5
    before = torch.randn(M * N, generator=g, device="cuda", dtype=td)
    plain, C, acc = torch.empty(M, N, device="cuda", dtype=td), torch.empty(M * N, device="cuda", dtype=td), before.clone()
    ops.gemm(A, B, plain, algo)
    RA = torch.arange(T, dtype=torch.int32, device="cuda").reshape(TM, TN)
    cs = torch.tensor([T], dtype=torch.int32)
    MM = torch.zeros(fo.layout.counter_size(1, TM, TN), dtype=torch.int32, device="cuda")
    ov = ops.Overlap()
    ov.set_schedule(**settings)
    ov.set_accumulator(acc)
    ov.gemm_allreduce_overlap(A, B, C, MM, RA, T, cs, cs.cuda(), algo)
    torch.cuda.synchronize()
    assert ov.status() == 0 and (MM == 0).all()
    step = TM // 8
    for t in range(0, TM, step):  # tile rows, all rows of a tile
        got = C.view(bm, TM, TN, bn)[:, t:t + step].permute(1, 0, 2, 3)
        assert torch.equal(got, plain.view(TM, bm, TN, bn)[t:t + step])
    step = M * N // 16
    for i in range(0, M * N, step):
        assert torch.equal(acc[i:i + step], (before[i:i + step].float() + C[i:i + step].float()).to(td))
    ov.close()
