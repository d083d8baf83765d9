"""Which stream an overlapped call takes and which sums its GEMM does itself, by the planners that the calls decide with: on both
sides of every line, without a GPU (256 CUs are assumed).  Buffers are addresses only."""
import ctypes

import pytest

from flashoverlap_amd import _capi

BUFFER = 1 << 40  # buffers lie this far apart


class Handle:
    def __init__(self, rank=0, world=1, fused=-1, in_stream_below_flop=-1.0, fused_from_groups=-1, link=0.0):
        L = _capi.lib()
        self._h = ctypes.c_void_p()
        assert L.fo_overlap_create(ctypes.byref(self._h)) == 0
        assert L.fo_overlap_set_world(self._h, rank, world) == 0
        assert L.fo_overlap_set_fused_consumer(self._h, fused) == 0
        assert L.fo_overlap_set_schedule(self._h, in_stream_below_flop, fused_from_groups) == 0
        assert L.fo_overlap_set_link_rate(self._h, link) == 0

    def __enter__(self):
        return self

    def __exit__(self, *_):
        _capi.lib().fo_overlap_destroy(self._h)

    def _common(self, M, N, bm, bn, cseg, acc):
        L = _capi.lib()
        assert L.fo_overlap_set_accumulator(self._h, acc, M * N if acc else 0) == 0
        T = (M // bm) * (N // bn)
        if isinstance(cseg, int):
            cseg = [T * (g + 1) // cseg - T * g // cseg for g in range(cseg)]
        return T, (ctypes.c_int32 * len(cseg))(*cseg), len(cseg), min(T, 256 * (256 // bm) * (256 // bn)), _capi.find_algo(bm, bn, swizzle=4)

    def allreduce(self, M, N, K, cseg, bm=128, bn=128, acc=4 * BUFFER, norm=False, Y=5 * BUFFER, Wt=6 * BUFFER, rldn=1, monitor=0,
                  C=3 * BUFFER):
        _, arr, G, wave, algo = self._common(M, N, bm, bn, cseg, acc)
        return _capi.lib().fo_overlap_plan_allreduce(self._h, M, N, K, BUFFER, 2 * BUFFER, C, Y if norm else None,
                                                     Wt if norm else None, rldn, arr, G, wave, algo, monitor)

    def reducescatter(self, M, N, K, cseg, bm=128, bn=128, acc=4 * BUFFER, D=5 * BUFFER, rldn=1, monitor=0):
        _, arr, G, wave, algo = self._common(M, N, bm, bn, cseg, acc)
        return _capi.lib().fo_overlap_plan_reducescatter(self._h, M, N, K, BUFFER, 2 * BUFFER, 3 * BUFFER, D, rldn, arr, G, wave,
                                                         algo, monitor)


ONE = 0        # everything on the GEMM stream
REFUSED = -2


def two(M, N, bm=128, bn=128):  # two streams, every sum by the consumer
    return (M // bm) * (N // bn)


@pytest.mark.parametrize("M,N,K,cseg,kw,want", [
    (4096, 4096, 4096, 4, {}, ONE),                                  # one round
    (4096, 4352, 4096, 4, dict(acc=None, norm=True), two(4096, 4352)),  # sixteen tiles more, nothing to sum
    (4096, 4096, 4096, 4, dict(monitor=1), two(4096, 4096)),
    (8192, 8192, 4096, 4, dict(acc=None), ONE),                      # neither sums nor rows
    (8192, 8192, 4096, 4, dict(acc=None, norm=True), two(8192, 8192)),
    (8192, 8192, 4096, 4, {}, ONE),                                  # without the normalisation up to four waves
    (8192, 10240, 4096, 5, {}, 4096),                                # five: the last one's sums by the GEMM
    (16384, 8192, 4096, 8, {}, 7 * 1024),
    (8192, 8192, 4096, 16, dict(norm=True), two(8192, 8192)),        # waves of whole rows, groups that end with them
    (8192, 8192, 4096, 17, dict(norm=True), ONE),                    # more groups than are launched one by one
    (8192, 8192, 632, 4, dict(norm=True), ONE),
    (8192, 8192, 640, 4, dict(norm=True), two(8192, 8192)),
    (8192, 8192, 4096, 3, dict(norm=True), 3 * 1024),                # groups across waves
    (8192, 4096, 3576, 2, dict(norm=True), ONE),                     # two waves
    (8192, 4096, 3584, 2, dict(norm=True), two(8192, 4096)),
    (8192, 4096, 3584, 1, dict(norm=True), 1024),
    (5120, 8192, 4096, 4, dict(norm=True), ONE),                     # waves that are not whole rows
    (8064, 8192, 4096, 4, dict(norm=True), ONE),                     # rows that 256 does not divide
    (8192, 8192, 4096, 3, dict(norm=True, acc=4 * BUFFER + 8), REFUSED),  # an accumulator that no launch takes
    (8192, 10240, 4096, 5, dict(acc=3 * BUFFER), two(8192, 10240)),  # the accumulator is the product
    (8192, 10240, 4096, 5, dict(monitor=1), two(8192, 10240)),
    (8192, 8192, 4096, 3, dict(norm=True, Y=4 * BUFFER), two(8192, 8192)),        # rows over the accumulator
])
def test_route_of_an_allreduce(M, N, K, cseg, kw, want):
    with Handle() as h:
        assert h.allreduce(M, N, K, cseg, **kw) == want


@pytest.mark.parametrize("M,N,rldn,in_range", [
    (337 * 256, 49 * 256, 66052, True),   # rows of the view of 8454656 elements: the last that fit
    (272 * 256, 64 * 256, 69632, False),  # 8912896
    (272 * 256, 64 * 256, 1, True),
])
def test_rows_of_the_view_longer_than_a_buffer_range(M, N, rldn, in_range):
    """The GEMM reads the accumulator of a 128x128 block through one 31-bit buffer range: what does not fit is the consumer's."""
    assert (((127 * rldn * 128 + 128) * 2) < 1 << 31) == in_range
    with Handle() as h:
        assert (h.allreduce(M, N, 264, 1, rldn=rldn) < two(M, N)) == in_range


@pytest.mark.parametrize("offset", [0, 256 * 4096 * 2, 8192 * 4096 * 2 - 16, -8192 * 4096 * 2 + 16])
@pytest.mark.parametrize("settings", [dict(), dict(fused=0)])
def test_rows_over_the_product_follow_its_consumer(settings, offset):
    """Rows that share memory with the product, behind it on one stream: a consumer on the other that had yet to read the first
    wave's slots would add rows to the accumulator."""
    with Handle(**settings) as h:
        assert h.allreduce(8192, 4096, 4096, 1, norm=True, Y=3 * BUFFER + offset) == two(8192, 4096)


@pytest.mark.parametrize("Y", [BUFFER, 2 * BUFFER, 4 * BUFFER - 16])
def test_rows_over_the_operands_follow_the_gemm(Y):
    """One group: its rows follow the whole GEMM, also where its first waves complete some of them."""
    with Handle() as h:
        assert h.allreduce(8192, 4096, 4096, 1, norm=True, Y=Y) == two(8192, 4096)


@pytest.mark.parametrize("settings", [dict(in_stream_below_flop=0, fused_from_groups=1 << 20), dict(link=100.0)])
@pytest.mark.parametrize("M,N,cseg,tile,first", [
    (8192, 4096, [1024, 1024], (128, 128), 1024),
    (8192, 4096, [700, 700, 648], (128, 128), 1024),
    (4096, 7168, [400, 496], (128, 256), 512),
    (8192, 8192, 700, (128, 128), 3072),
    (4096, 4096, 4, (128, 128), 1024),      # one wave has no last one: every slot is the consumer's
    (8064, 8192, 4, (128, 128), 63 * 64),   # counted in the Algo's own tile
])
def test_two_streams_asked_for(settings, M, N, cseg, tile, first):
    with Handle(**settings) as h:
        got = h.allreduce(M, N, 72, cseg, *tile)
        assert got == (two(M, N, *tile) if "link" in settings else first)


@pytest.mark.parametrize("M,N,K,cseg,W,kw,want", [
    (4096, 4096, 4096, 4, 8, {}, ONE),                                 # one round, with an accumulator
    (4096, 4096, 4096, 4, 8, dict(acc=None), two(4096, 4096)),         # without one: up to five sixths of a round
    (3328, 4096, 4096, 4, 8, dict(acc=None), ONE),
    (8192, 4096, 4096, 8, 8, {}, 1024),                                # the last four groups are the last wave
    (8192, 4096, 4096, 1, 8, {}, two(8192, 4096)),                     # the last group begins before it
    (8192, 4096, 4096, 16, 8, dict(acc=None), 1024),
    (8192, 4096, 4096, 17, 8, dict(acc=None), ONE),
    (8192, 4096, 4096, 17, 8, {}, ONE),
    (8192, 4096, 4096, 8, 8, dict(acc=None, D=None), two(8192, 4096)),
    (8192, 4096, 4096, 8, 1, {}, two(8192, 4096)),                     # one rank
    (8192, 4096, 4096, 8, 8, dict(rldn=2), two(8192, 4096)),           # ranks that do not own whole rows
    (8192, 4096, 4096, 17, 8, dict(rldn=2), two(8192, 4096)),
    (8192, 4096, 4096, 8, 8, dict(D=4 * BUFFER), two(8192, 4096)),     # rows over the accumulator
    (8064, 8192, 4096, 4, 8, {}, ONE),                                 # rows that 256 does not divide
    (8192, 4096, 4096, 8, 8, dict(monitor=1), two(8192, 4096)),
])
def test_route_of_a_reduce_scatter(M, N, K, cseg, W, kw, want):
    with Handle(rank=W - 1, world=W) as h:
        assert h.reducescatter(M, N, K, cseg, **kw) == want


@pytest.mark.parametrize("M,N,cseg", [(8192, 4096, [1024, 1024]), (8192, 8192, 3), (8192, 4096, 700), (128, 1024, 1), (8064, 8192, 4)])
def test_launches_per_group_asked_for_are_all_there(M, N, cseg):
    """set_fused_consumer(0): every slot is counted, waited for and summed on the second stream."""
    with Handle(fused=0) as h:
        assert h.allreduce(M, N, 4096, cseg) == h.allreduce(M, N, 4096, cseg, norm=True) == two(M, N)
    with Handle(world=8, fused=0) as h:
        assert h.reducescatter(M, N, 4096, cseg) == h.reducescatter(M, N, 4096, cseg, acc=None) == two(M, N)


def test_a_planner_refuses_what_the_calls_refuse():
    with Handle() as h:
        for call in (h.allreduce, h.reducescatter):
            assert call(4096, 4096, 4096, [1000]) < 0          # groups that do not cover the tiles
            assert call(4096, 4096, 0, 4) < 0
            assert call(4096, 4096, 4096, 4, rldn=3) < 0
            assert call(4000, 4096, 4096, 4) < 0
    assert _capi.lib().fo_overlap_plan_allreduce(None, 1, 1, 1, 0, 0, 0, 0, 0, 1, None, 0, 0, 0, 0) < 0
