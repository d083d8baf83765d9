"""The launch arguments: what the host packs into the smaller tiles' 112 bytes and into the words in front of the 256x256
tile's, and the raster walks that read them, against the launch as it is described (host code of the library's own header, built for the CPU)."""
import subprocess

import pytest

from flashoverlap_amd import build

PROGRAM = r"""
#include "fo_gemm_common.h"
#include <cstdio>
using namespace fo_gemm_dev;
static long bad = 0, seen = 0, walked = 0;
static void compare(const GemmArgs &a, int mode) {
    const TileArgs t = TileArgs::of(a, 17, mode);
    const bool general = t.bits & TileArgs::GENERAL;
    bad += t.A != a.A || t.B != a.B || t.C != a.C || t.M != a.M || t.N != a.N || t.K != a.K || t.RA != a.RA || t.RE != a.RE ||
           t.cseg != a.cseg || t.G != a.G || t.stride != 17 || fo_tile_count(t) != a.count;
    if (mode == MODE_ACC || mode == MODE_RS) bad += t.ACC != a.ACC;
    else bad += t.MM != a.MM;
    if (mode == MODE_RS) {
        const int w = 1 << (t.bits >> TileArgs::RANKS & 15), wide = t.bits & TileArgs::WIDE ? 256 : 128;
        bad += t.OWN != a.OWN || w != a.W || (int)(t.bits >> TileArgs::RANK & 255) != a.rank || (t.M / w) * (t.N / wide) != a.seg_rows;
    } else {
        bad += t.rLDN != a.rLDN;
    }
    bad += (t.bits & TileArgs::TALL ? 256 : 128) != a.BM || (t.bits & TileArgs::WIDE ? 256 : 128) != a.BN;
    bad += !!(t.bits & TileArgs::MONITOR) != !!a.monitor || !!(t.bits & TileArgs::QUIET) != !!a.quiet;
    const int step = a.count > 3000 ? a.count / 1500 : 1;
    for (int u = 0; u < a.count; u += step) {
        int m, n, pm, pn;
        fo_tile_of(t, u, &m, &n);
        fo_unit_to_tile(u, a.first, a.sub_m, a.sub_n, a.grid_m, a.grid_n, a.panel, a.xcd_remap, &pm, &pn);
        bad += m != pm || n != pn;
        walked += !general;
    }
    GemmArgs h = a;
    h.half = (mode & 3) | (a.quiet ? 4 : 0);
    const Front256 f = Front256::of(h);
    bad += f.A != a.A || f.B != a.B || f.K != a.K || f.count != a.count || (int)(f.bits >> 3) != h.half;
    const int positions = a.grid_m * a.grid_n;
    for (int u = 0; u < positions; u += positions > 3000 ? positions / 1500 : 1) {
        int m, n, pm, pn;
        fo_tile_of(f, u, &m, &n);
        fo_wg_to_tile(u, a.grid_m, a.grid_n, a.panel, a.xcd_remap, &pm, &pn);
        bad += m != pm || n != pn;
    }
    seen++;
}
int main() {
    GemmArgs a = {};
    static uint16_t x[4];
    static int32_t y[4];
    a.A = x; a.B = x + 1; a.C = x + 2; a.RA = y; a.RE = y + 1; a.cseg = y + 2; a.MM = y + 3;
    const int grids[][2] = {{1, 1}, {1, 9}, {3, 5}, {4, 4}, {7, 37}, {8, 32}, {9, 28}, {17, 29}, {33, 64}, {1, 32767}, {1, 32768}, {300, 300}, {2000, 3}};
    for (int mode = 0; mode <= MODE_RS; mode++)
        for (const auto &g : grids)
            for (int panel : {1, 3, 4, 8, 255, 256})
                for (int remap = 0; remap < 2; remap++)
                    for (int part = 0; part < 4; part++) {
                        if (panel > g[0] && panel > 1) continue;
                        a.grid_m = g[0]; a.grid_n = g[1]; a.panel = panel; a.xcd_remap = remap;
                        const int positions = g[0] * g[1];
                        a.first = part ? positions / 3 : 0;
                        a.sub_m = part & 1 ? 2 << (panel & 1) : 1; a.sub_n = part & 2 ? 4 >> remap : 1;
                        a.count = (positions - a.first) * a.sub_m * a.sub_n;
                        a.BM = part & 2 ? 256 : 128; a.BN = part & 1 ? 256 : 128;
                        a.M = a.grid_m * 256; a.N = a.grid_n * 256; a.K = 8 * panel; a.rLDN = 1 + part; a.G = 5 + part;
                        a.monitor = part & 1; a.quiet = part >> 1;
                        a.ACC = mode == MODE_ACC || (mode == MODE_RS && part & 1) ? x + 3 : nullptr;
                        a.OWN = mode == MODE_RS && part & 2 ? x + 2 : nullptr;
                        for (int w = 1; w <= (mode == MODE_RS ? 128 : 1); w *= 2) {
                            a.W = w; a.rank = w - 1;
                            a.seg_rows = (int)((int64_t)a.M * a.N / a.BN / w);
                            compare(a, mode);
                        }
                    }
    // waves of whole tile rows
    a.grid_m = a.grid_n = 32; a.panel = fo_pack_row_waves(2, 3, 2, 256); a.xcd_remap = 2; a.first = 512; a.count = 512; a.sub_m = a.sub_n = 1;
    a.M = a.N = 8192; a.W = 1; a.rank = 0;
    compare(a, MODE_PLAIN);
    std::printf("%ld %ld %ld\n", bad, seen, walked);
    return 0;
}
"""


def test_packed_arguments_say_what_the_launch_is(tmp_path):
    src = tmp_path / "args.hip"
    src.write_text(PROGRAM)
    flags = [f for f in build.HIP_FLAGS if not f.startswith("--offload-arch") and f not in ("-Xclang", "-target-feature", "-packed-fp32-ops")]
    try:
        subprocess.run([build.HIPCC, "--cuda-host-only"] + flags + [str(src), "-o", str(tmp_path / "args")], check=True, capture_output=True, text=True)
    except FileNotFoundError:
        pytest.skip("no hipcc")
    out = subprocess.run([str(tmp_path / "args")], check=True, capture_output=True, text=True).stdout.split()
    bad, seen, walked = map(int, out)
    assert bad == 0 and seen > 1000 and walked > 100000


NO_STRIDES = r"""
#include "fo_gemm_common.h"
#include <cstdio>
using namespace fo_gemm_dev;
template <typename T> auto has_a(int) -> decltype((void)T::lda, true) { return true; }
template <typename T> bool has_a(...) { return false; }
template <typename T> auto has_b(int) -> decltype((void)T::ldb, true) { return true; }
template <typename T> bool has_b(...) { return false; }
int main() {
    std::printf("%d\n", has_a<GemmArgs>(0) || has_b<GemmArgs>(0) || has_a<TileArgs>(0) || has_b<TileArgs>(0));
    return 0;
}
"""


def test_a_launch_cannot_name_a_row_stride_that_the_kernels_ignore(tmp_path):
    """Both kernels take K as the row stride of A and B: a launch described with another one would read wrong rows."""
    src = tmp_path / "strides.hip"
    src.write_text(NO_STRIDES)
    flags = [f for f in build.HIP_FLAGS if not f.startswith("--offload-arch") and f not in ("-Xclang", "-target-feature", "-packed-fp32-ops")]
    try:
        subprocess.run([build.HIPCC, "--cuda-host-only"] + flags + [str(src), "-o", str(tmp_path / "strides")], check=True, capture_output=True, text=True)
    except FileNotFoundError:
        pytest.skip("no hipcc")
    out = subprocess.run([str(tmp_path / "strides")], check=True, capture_output=True, text=True).stdout.split()
    assert out == ["0"]
