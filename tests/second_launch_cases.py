"""Launches without counters whose last round of 256x256 tiles goes to a second launch: the cases of test_gpu_9_second_launch.py and
what the planner says of them, which test_plan_cpu.py asserts without a GPU."""
from flashoverlap_amd import _capi

F16, BF16 = 0, 1
LINE = 1 << 20  # an address on a 128-byte line

# What the epilogue of a launch does: (epilogue, whether it adds to an accumulator) of gemm_plan.
FORMS = {"plain": (0, False), "plain acc": (0, True), "reordered": (1, False), "reordered acc": (1, True),
         "ranks": (2, False), "ranks acc": (2, True)}

S64, S64W, S128, S256 = (64, 64), (64, 128), (128, 128), (128, 256)
# dtype, reorder tile, M, N, K; the second launch's tile without and with an accumulator, over ranks without and with one (None: one
# launch); where second-launch positions lie half outside of the matrix.
CASES = [
    (F16, 128, 128, 4352, 4096, 1536, (S64, S64, S64, S64), ""),
    (BF16, 256, 128, 4352, 4096, 2048, (S64, S64, S64, S64), ""),      # two or four of its tiles in a reorder tile
    (BF16, 128, 128, 4224, 4096, 1032, (None, None, S64, S64), "M"),  # rows off the lines
    (F16, 128, 256, 4352, 4352, 1536, (S128, S128, S128, S128), ""),
    (F16, 128, 128, 4608, 4608, 3000, (S256, None, S256, S256), ""),   # rows off the lines
    # each tile with each epilogue, at both edges of the matrix
    (F16, 128, 128, 3456, 4736, 1536, (S64, S64, S64, S64), "MN"),
    (BF16, 128, 128, 3200, 5248, 1536, (S64W, S64W, S64W, S64W), "MN"),
    (BF16, 128, 128, 6272, 2944, 1536, (S128, S128, S128, S128), "MN"),
    (F16, 128, 128, 4224, 4992, 520, (S256, None, S256, S256), "MN"),
    (BF16, 128, 128, 5504, 3712, 4608, (S256, S256, S256, S256), "MN"),
]


def expected(case, form):
    """The second launch's tile, or None."""
    epilogue, acc = FORMS[form]
    return case[6][(2 if epilogue == 2 else 0) + acc]


def planned(case, form, A=LINE, B=LINE):
    """(the main launch's tile, the second launch's tile or None, the edges at which its positions lie half outside: "M", "N")."""
    _, bm, bn, M, N, K = case[:6]
    epilogue, acc = FORMS[form]
    p = _capi.gemm_plan(_capi.find_algo(bm, bn, swizzle=4), M, N, K, epilogue, False, acc, A, B)
    if not p["second"]:
        return p["tile"], None, ""
    assert p["tile"] == (256, 256)
    grid_m, grid_n = -(-M // 256), -(-N // 256)
    assert p["count"] + p["second"] == grid_m * grid_n
    edges = ""
    if M % 256 or N % 256:  # the raster is then panels of p["panel"] tile rows, an eighth of its walk to each XCD
        at = [position(t, grid_m, grid_n, p["panel"]) for t in range(p["count"], grid_m * grid_n)]
        edges = ("M" if M % 256 and any(m == grid_m - 1 for m, _ in at) else "") + \
                ("N" if N % 256 and any(n == grid_n - 1 for _, n in at) else "")
    return p["tile"], p["second_tile"], edges


def position(t, grid_m, grid_n, panel):
    nt = grid_m * grid_n
    x = t % 8
    v = x * (nt // 8) + min(x, nt % 8) + t // 8
    first = v // (panel * grid_n) * panel
    inside, rows = v - first * grid_n, min(panel, grid_m - first)
    return first + inside % rows, inside // rows
