"""GPU parity of the kernel that updates the accumulator and normalises the same rows: batches that are whole tile rows and
batches that are not, rows that fill the workgroup's lanes and rows that do not, one batch and several.  Everything the
call leaves is compared bit for bit with the separate calls (see _run_both)."""
import numpy as np
import pytest
import torch

from gpu_util import BF16, F16, TORCH_DTYPE, planned_route, seeded
from test_gpu_3_norm_overlap import _run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("bm,bn,M,N,cseg", [
    (128, 128, 8192, 4096, [512] * 4),               # two waves of whole rows
    (128, 128, 8192, 4096, [100, 412, 512, 1024]),   # groups that end inside rows
    (128, 256, 8192, 8192, [256] * 8),               # four waves, two groups each
    (256, 128, 4096, 8192, [1024]),                  # one group
    (128, 256, 256, 6144, [48]),                     # three chunks a lane
    (128, 128, 256, 1920, [10, 20]),                 # one chunk, lanes left over
    (128, 128, 384, 4224, [33, 66]),                 # three chunks, most of the third beyond the row
    (128, 256, 128, 256, [1]),                       # one tile
    (128, 128, 128, 1024, [8]),                      # the shortest rows, one tile row
])
def test_rows_are_consumed_and_normalised(fo, dtype, bm, bn, M, N, cseg):
    _run_both(fo, dtype, bm, bn, M, N, 72, cseg, 0, seed=700)


@pytest.mark.parametrize("dtype", [F16, BF16])
def test_rows_in_another_order(fo, dtype):
    """Whole rows in an order of their own, and rows spread over two batches."""
    bm, bn, M, N = 128, 128, 8192, 4096
    TM, TN = M // bm, N // bn
    rng = np.random.default_rng(3)
    rows = [t for half in (0, 1) for tm in rng.permutation(TM // 2) + half * (TM // 2) for t in rng.permutation(TN) + tm * TN]
    _run_both(fo, dtype, bm, bn, M, N, 64, [TM * TN // 2] * 2, 0, seed=710, hint=[int(t) for t in rows])
    spread = rng.permutation(TM * TN)
    _run_both(fo, dtype, bm, bn, M, N, 64, [TM * TN // 2] * 2, 0, seed=711, hint=[int(t) for t in spread])


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("bm,bn,M,N", [(96, 128, 192, 1024), (1, 64, 5, 320), (16, 256, 48, 2048), (24, 32, 72, 96)])
def test_tile_heights(fo, dtype, bm, bn, M, N):
    """Tile heights that are powers of two (shifts) and that are not (divisions), against the plain rows: the same bits."""
    td = TORCH_DTYPE[dtype]
    T = (M // bm) * (N // bn)
    hint = [int(t) for t in np.random.default_rng(5).permutation(T)]
    RA = fo.layout.reorder_indices(T, hint, device="cuda").reshape(M // bm, N // bn)
    g = torch.Generator(device="cuda").manual_seed(6)
    C = torch.randn(M, N, device="cuda", generator=g).to(td)
    W = torch.randn(N, device="cuda", generator=g).to(td)
    Y, Z = torch.empty_like(C), torch.empty_like(C)
    fo.ops.reorder_rmsnorm_rows(C, Y, W, 0, M, bm, bn, 1, RA, eps=1e-6)
    plain = fo.layout.unpermute(C, M, N, bm, bn, RA).contiguous()
    fo.ops.reorder_rmsnorm_rows(plain, Z, W, 0, M, 1, 8, 1, None, eps=1e-6)
    torch.cuda.synchronize()
    assert torch.equal(Y, Z)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("M,N", [(2176, 4224), (2304, 7168), (2176, 4096)])
def test_many_wide_rows(fo, dtype, M, N):
    """More rows than get a workgroup each, on both sides of the width from which they are a workgroup's anyhow: at most two
    units in the last place from a sum in 64 bits (one for each of the two roundings, neither of which can be off by more)."""
    td, bn = TORCH_DTYPE[dtype], 128
    g = torch.Generator(device="cuda").manual_seed(8)
    C = torch.randn(M, N, device="cuda", generator=g).to(td)
    W = torch.randn(N, device="cuda", generator=g).to(td)
    T = (M // 128) * (N // bn)
    RA = fo.layout.reorder_indices(T, [int(t) for t in np.random.default_rng(9).permutation(T)], device="cuda").reshape(M // 128, N // bn)
    Y = torch.empty_like(C)
    fo.ops.reorder_rmsnorm(C, Y, W, 128, bn, 1, RA, eps=1e-6)
    x = fo.layout.unpermute(C, M, N, 128, bn, RA).double()
    want = x * torch.rsqrt(x.pow(2).mean(1, keepdim=True) + 1e-6) * W.double()
    ulp = 2.0 ** -10 if dtype == F16 else 2.0 ** -7
    torch.cuda.synchronize()
    assert ((Y.double() - want).abs() <= 2 * ulp * want.abs() + 2.0 ** -23).all()


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("rows_behind", [0, 256])
@pytest.mark.parametrize("settings", [dict(), dict(in_stream_below_flop=0)])
def test_rows_over_the_product(fo, dtype, rows_behind, settings):
    """Normalised rows written over the product: the accumulator takes the product and none of them.  One batch, tile rows in
    reverse order, so that most rows are written where another one's product lies (which rows then come out is nobody's
    promise: they are not looked at), and four times as many workgroups of rows as the GPU holds at once."""
    bm, bn, M, N, K = 128, 128, 8192, 4096, 72
    td, TM, TN = TORCH_DTYPE[dtype], M // bm, N // bn
    algo = fo._capi.find_algo(bm, bn, swizzle=4)
    hint = [tm * TN + tn for tm in reversed(range(TM)) for tn in range(TN)]
    RA = fo.layout.reorder_indices(TM * TN, hint, device="cuda").reshape(TM, TN)
    A, _ = seeded((M, K), dtype, 1)
    B, _ = seeded((N, K), dtype, 2, scale=K ** -0.5)
    before, _ = seeded((M * N,), dtype, 3)
    gamma = torch.ones(N, device="cuda", dtype=td)
    cs = torch.tensor([TM * TN], dtype=torch.int32)
    MM = torch.zeros(fo.layout.counter_size(1, TM, TN), dtype=torch.int32, device="cuda")
    ov = fo.ops.Overlap()
    ov.set_fused_consumer(-1 if settings else 0)  # launches per wave, by choice and always
    ov.set_schedule(**settings)
    product, want = torch.empty(M * N, device="cuda", dtype=td), before.clone()
    ov.set_accumulator(want)
    ov.gemm_allreduce_overlap(A, B, product, MM, RA, 1, cs, cs.cuda(), algo)
    room = torch.empty((M + rows_behind) * N, device="cuda", dtype=td)
    C, Y, acc = room[:M * N], room[rows_behind * N:].view(M, N), before.clone()
    ov.set_accumulator(acc)
    # on one stream, consumer and rows one behind the other: the rows of a last wave that the GEMM sums are behind the GEMM only
    assert planned_route(fo, ov, dtype, A, B, C, [TM * TN], algo, 1, Y, gamma) == TM * TN
    ov.gemm_allreduce_rmsnorm_overlap(A, B, C, MM, RA, RA.cpu(), 1, cs, cs.cuda(), algo, Y, gamma, eps=1e-6)
    torch.cuda.synchronize()
    assert torch.equal(acc, want) and torch.equal(want, (before.float() + product.float()).to(td))
    assert (MM == 0).all() and ov.status() == 0
    ov.close()
