// The instantiations of the smaller-tile GEMM kernel for one type and one epilogue per translation unit: built
// ten times with -DFO_INST_DTYPE={0,1} (fp16, bf16) and -DFO_INST_MODE={0,1,2,3,4} (plain, signal, scatter, accumulating, reduce-scatter epilogue).
#include "fo_gemm_launch.h"
#include "fo_gemm_tile_kernel.h"

#if !defined(FO_INST_DTYPE) || !defined(FO_INST_MODE)
#error "compile with -DFO_INST_DTYPE=0|1 -DFO_INST_MODE=0|1|2|3|4"
#endif

namespace fo_gemm_dev {

#define FO_CAT3_(a, b, c, d) a##b##c##d
#define FO_CAT3(a, b, c, d) FO_CAT3_(a, b, c, d)

#if FO_INST_DTYPE == 0
typedef fo_f16_tag inst_tag;
#else
typedef fo_bf16_tag inst_tag;
#endif

// Columns per stage and slots of each tile: as many operand bytes in flight as 160 KB of LDS hold (96 to 128 KB),
// in steps of 128 columns where a tile's step of 64 is too short to hide a barrier in.
int FO_CAT3(fo_gemm_tile_launch_, FO_INST_DTYPE, _, FO_INST_MODE)(const GemmArgs &a, int tm, int tn, hipStream_t stream,
                                                              int *resident_out, int expect_resident) {
#define FO_TILE(TM_, TN_, BK_, S_) FO_TILE_(TM_, TN_, BK_, S_, false)
#define FO_TILE_(TM_, TN_, BK_, S_, SHIFT_)                                                                                       \
    if (tm == TM_ && tn == TN_)                                                                                          \
        return launch_kernel<TileArgs, FO_INST_MODE, fo_gemm_tile_kernel<inst_tag, TM_, TN_, BK_, S_, FO_INST_MODE, SHIFT_>,                     \
                             tile_smem_bytes<TM_, TN_, BK_, S_>(), kTileThreads>(a, stream, resident_out, expect_resident);
    // Operand rows that do not begin on 128-byte lines: the form that loads whole lines, for the tiles whose stages leave
    // LDS for one more in flight beside the two a step then reads.
    if (!on_lines(a)) {
        FO_TILE_(32, 32, 128, 8, true)
        FO_TILE_(64, 32, 128, 6, true)
        FO_TILE_(64, 64, 128, 4, true)
        FO_TILE_(64, 96, 64, 7, true)
        FO_TILE_(64, 128, 64, 6, true)
        FO_TILE_(96, 128, 64, 5, true)
        FO_TILE_(128, 128, 64, 4, true)
        FO_TILE_(128, 160, 64, 4, true)
        // The whole of a CU's LDS: no consumer that polls could be on the CU beside it, and the row-mapped epilogues' maps do
        // not fit.  Only for what moves no counters (fo_gemm.hip).
#if FO_INST_MODE == 0 || FO_INST_MODE == 3
        FO_TILE_(128, 192, 64, 4, true)
#endif
    }
    FO_TILE(32, 32, 128, 8)
    FO_TILE(64, 32, 128, 6)
    FO_TILE(64, 64, 128, 4)
    FO_TILE(64, 96, 128, 3)
    FO_TILE(64, 128, 128, 3)
    FO_TILE(96, 128, 64, 5)
    FO_TILE(128, 128, 64, 4)
    FO_TILE(128, 160, 64, 4)
    FO_TILE(128, 192, 64, 3)
    FO_TILE(128, 256, 64, 3)
    FO_TILE(256, 128, 64, 3)
#undef FO_TILE
#undef FO_TILE_
    return FO_ERR_ALGO;
}

}  // namespace fo_gemm_dev
