"""Which launches a GEMM is made of, by the planner that the launches decide with, without a GPU (256 CUs are assumed).  Operands are
addresses only."""
import pytest

from flashoverlap_amd import _capi
from second_launch_cases import CASES, FORMS, LINE, expected, planned


def plan(M, N, K, form="reordered", bm=128, bn=128, counts=False, off=0):
    """(tile), or (tile, second launch's tile), of a launch; form: what its epilogue does; off: bytes between operands and line."""
    epilogue = 0 if form in ("plain", "acc") else 2 if form.startswith("ranks") else 1
    p = _capi.gemm_plan(_capi.find_algo(bm, bn, swizzle=4), M, N, K, epilogue, counts, form.endswith("acc"), LINE + off, LINE + off)
    return (p["tile"], p["second_tile"]) if p["second"] else (p["tile"],)


# Rows that are an odd multiple of 64 bytes apart: every other one begins on a 128-byte line, but none does where the operands'
# bases are off by 16 bytes.  256x256 tiles, which cannot load whole lines, then take longer (us, whole passes in these tiles -> in
# 128x192 tiles, bases off by 16 bytes): 209.5 -> 173.0, 127.3 -> 111.7, 161.6 -> 144.0.
@pytest.mark.parametrize("form,bm,bn,M,N,K", [
    ("reordered", 256, 128, 5888, 3072, 5216),
    ("acc", 128, 128, 6912, 3072, 1824),
    ("reordered acc", 256, 128, 6144, 2688, 3808),
])
def test_rows_off_the_lines_by_their_base_address(form, bm, bn, M, N, K):
    assert plan(M, N, K, form, bm, bn)[0] == (256, 256)
    assert plan(M, N, K, form, bm, bn, off=64)[0] == (256, 256)  # still every other row
    assert plan(M, N, K, form, bm, bn, off=16) == ((128, 192),)


# What an estimate with other constants had given to larger tiles (us, whole passes in those -> in these): 169 -> 138, 73.7 -> 67.1,
# 30.9 -> 28.7, 72.4 -> 70.4, 66.9 -> 60.0, 24.7 -> 20.3, 143 -> 125; the last with operands off the lines, 209 -> 173.
@pytest.mark.parametrize("form,bm,bn,M,N,K,off,tile", [
    ("reordered", 128, 256, 6144, 2048, 5544, 0, (128, 128)),
    ("reordered acc", 256, 128, 5120, 3200, 1232, 0, (128, 128)),
    ("reordered acc", 128, 128, 6912, 1152, 936, 0, (128, 128)),
    ("reordered acc", 128, 128, 3456, 7936, 376, 0, (128, 128)),
    ("reordered acc", 128, 128, 5120, 4224, 488, 0, (128, 128)),
    ("reordered acc", 128, 128, 4864, 1664, 304, 0, (128, 128)),
    ("ranks", 128, 256, 3072, 3840, 5144, 0, (128, 128)),
    ("reordered", 256, 128, 5888, 3072, 5216, 16, (128, 192)),
])
def test_smaller_tiles_where_they_are_faster(form, bm, bn, M, N, K, off, tile):
    assert plan(M, N, K, form, bm, bn, off=off) == (tile,)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in c[:6]))
def test_second_launches_are_what_their_cases_say(case, form):
    _, second, edges = planned(case, form)
    assert (second, edges) == (expected(case, form), case[7] if second else "")


def test_each_second_launch_is_in_some_case_with_each_epilogue_and_edge():
    seen = {(form, *planned(case, form)[1:]) for case in CASES for form in FORMS}
    for form in FORMS:
        for tile in ((64, 64), (64, 128), (128, 128), (128, 256)):
            assert (form, tile, "MN") in seen


def test_plan_refuses_what_no_launch_takes():
    algo = _capi.find_algo(128, 128, swizzle=4)
    for bad in ((algo, 128, 128, 0), (algo, 128, 128, 12), (algo, 100, 128, 64), (-1, 128, 128, 64)):
        with pytest.raises(_capi.FlashOverlapError):
            _capi.gemm_plan(*bad)
    with pytest.raises(_capi.FlashOverlapError):
        _capi.gemm_plan(algo, 128, 128, 64, epilogue=1, counts=True, acc=True)
    with pytest.raises(_capi.FlashOverlapError):
        _capi.gemm_plan(algo, 128, 128, 64, epilogue=3)
