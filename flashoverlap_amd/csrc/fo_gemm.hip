// Host side of the gfx950 MFMA GEMM: picks the workgroup tile for a problem and
// launches it (plain, signal and scatter epilogues).  The device code is in
// fo_gemm256_kernel.h and fo_gemm_tile_kernel.h, whose instantiations are
// compiled in translation units of their own (fo_gemm256_inst.hip, fo_gemm_tile_inst.hip).
#include <atomic>

#include "fo_gemm_launch.h"

int fo_gemm_dev::fo_gemm256_launch(int dtype, int mode, const GemmArgs &a, hipStream_t stream, int *resident_out,
                                   int expect_resident) {
    const int key = (dtype == FO_BF16 ? 8 : 0) + mode;
    switch (key) {
        case 0: return fo_gemm256_launch_0_0(a, stream, resident_out, expect_resident);
        case 1: return fo_gemm256_launch_0_1(a, stream, resident_out, expect_resident);
        case 2: return fo_gemm256_launch_0_2(a, stream, resident_out, expect_resident);
        case 3: return fo_gemm256_launch_0_3(a, stream, resident_out, expect_resident);
        case 4: return fo_gemm256_launch_0_4(a, stream, resident_out, expect_resident);
        case 5: return fo_gemm256_launch_0_5(a, stream, resident_out, expect_resident);
        case 6: return fo_gemm256_launch_0_6(a, stream, resident_out, expect_resident);
        case 7: return fo_gemm256_launch_0_7(a, stream, resident_out, expect_resident);
        case 8: return fo_gemm256_launch_1_0(a, stream, resident_out, expect_resident);
        case 9: return fo_gemm256_launch_1_1(a, stream, resident_out, expect_resident);
        case 10: return fo_gemm256_launch_1_2(a, stream, resident_out, expect_resident);
        case 11: return fo_gemm256_launch_1_3(a, stream, resident_out, expect_resident);
        case 12: return fo_gemm256_launch_1_4(a, stream, resident_out, expect_resident);
        case 13: return fo_gemm256_launch_1_5(a, stream, resident_out, expect_resident);
        case 14: return fo_gemm256_launch_1_6(a, stream, resident_out, expect_resident);
        case 15: return fo_gemm256_launch_1_7(a, stream, resident_out, expect_resident);
    }
    return FO_ERR_ARG;
}

int fo_gemm_dev::fo_gemm_tile_launch(int dtype, int mode, const GemmArgs &a, int tm, int tn, hipStream_t stream,
                                     int *resident_out, int expect_resident) {
    const int key = (dtype == FO_BF16 ? 5 : 0) + mode;
    switch (key) {
        case 0: return fo_gemm_tile_launch_0_0(a, tm, tn, stream, resident_out, expect_resident);
        case 1: return fo_gemm_tile_launch_0_1(a, tm, tn, stream, resident_out, expect_resident);
        case 2: return fo_gemm_tile_launch_0_2(a, tm, tn, stream, resident_out, expect_resident);
        case 3: return fo_gemm_tile_launch_0_3(a, tm, tn, stream, resident_out, expect_resident);
        case 4: return fo_gemm_tile_launch_0_4(a, tm, tn, stream, resident_out, expect_resident);
        case 5: return fo_gemm_tile_launch_1_0(a, tm, tn, stream, resident_out, expect_resident);
        case 6: return fo_gemm_tile_launch_1_1(a, tm, tn, stream, resident_out, expect_resident);
        case 7: return fo_gemm_tile_launch_1_2(a, tm, tn, stream, resident_out, expect_resident);
        case 8: return fo_gemm_tile_launch_1_3(a, tm, tn, stream, resident_out, expect_resident);
        case 9: return fo_gemm_tile_launch_1_4(a, tm, tn, stream, resident_out, expect_resident);
    }
    return FO_ERR_ARG;
}

namespace {

using namespace fo_gemm_dev;

int launch_tile(int dtype, int mode, const GemmArgs &a, int tm, int tn, hipStream_t stream, int *resident_out = nullptr,
                int expect_resident = 0) {
    if (dtype != FO_F16 && dtype != FO_BF16) return FO_ERR_DTYPE;
    if (tm == 256 && tn == 256) return fo_gemm256_launch(dtype, mode, a, stream, resident_out, expect_resident);
    return fo_gemm_tile_launch(dtype, mode, a, tm, tn, stream, resident_out, expect_resident);
}

// How a problem is launched: workgroup tile and raster, and what a second launch computes in a smaller tile.
struct launch_plan {
    int tm, tn;                            // workgroup tile
    int grid_m, grid_n, panel, xcd_remap;  // its raster
    int count;                             // tiles the launch computes
    bool whole;                            // a tile is one or more whole reorder tiles, so the kernel can count them
    int tail, tail_tm, tail_tn;            // raster positions left to the second launch, and its tile
};

// A launch of parts of reorder tiles cannot count them; fo_signal_all_kernel behind it does (about 3 us).  Shorter
// products than this many columns of K are computed in whole reorder tiles instead when counters are wanted, and so is
// whatever the monitor watches: its stamps say in which order the launch completed its tiles.
constexpr int kSignalAfterFromK = 1536;

// What launches without counters of more than one round of 128x160 tiles take, microseconds.  Each round, all CUs busy, has a share
// that goes with K (given at K = 4096: operand rows on 128-byte lines, off them, and off them with a row map, which leaves
// 128x192 no LDS for its line loads; 128x256 and 256x256 have none) and an end that does not: a tile's stores, which nothing of the
// next one runs beside, dearer by a row map, and an accumulator's values and sums.
//
// The constants of both tables and those beside them are the ones that leave least of (r + 4 r r), r the part by which the pass in the tile of
// least estimate is longer than in the best one, over whole passes, GEMM and normalisation, of 8400 products: calls that come here, K =
// 256 to 8192, 500 of them with operands 16 bytes off the lines, each in all tiles, three states in turn, in five runs.
// The pass in the tile of least estimate is longer than in the best one by 0.45 % in the mean and by more than 3 % in one of 20; over 1500
// products that were not fitted by 0.56 % and in one of 15.  (Before, a fit to 2220 products of one box with corrections behind it: 0.71 %
// and one of 11, 0.78 % and one of 10, with operands off the lines 1.1 % and one of 7; estimates in proportion to K: 1.76 % and one of 5.)
// What the former fit had lost came from too dear sums in the smaller tiles, and from counting a 256x256 tile of which half
// repeats its neighbour's as half a tile: us, its choice -> now, 6144x2048x5544 bf16 169 -> 138, 5120x3200x1232 with an accumulator 73.7 ->
// 67.1, 6912x1152x936 30.9 -> 28.7, 3456x7936x376 72.4 -> 70.4; others go the other way, 6400x6528x5840 bf16 424 -> 438,
// 8192x4224x264 with an accumulator 84 -> 98.
struct tile_cost {
    int tm, tn;
    double on_lines, off_lines, mapped;  // at K = 4096
    double end, end_mapped, sums, sums_mapped;
};
constexpr tile_cost kTileCosts[] = {
    {96, 128, 25.3, 25.5, 25, 1.5, 3.0, 1.4, 2.3},     {128, 128, 30.5, 31.5, 30.5, 1.7, 3.4, 1.6, 2.8},
    {128, 160, 35.2, 37, 37, 2.3, 4.0, 2.7, 3.7},      {128, 192, 40.5, 40.5, 52, 3.0, 4.2, 3.0, 4.0},
    {128, 256, 52, 65.5, 64.5, 2.8, 5.1, 3.7, 5.1},    {256, 128, 52, 65.5, 64.5, 2.8, 5.1, 3.7, 5.1},
    {256, 256, 88.5, 106, 104, 4.7, 10.5, 8.9, 10.5}};
// An accumulator's sums in a tile between 128x160 and 256x256 that lies in one reorder tile, or in a product that is not reordered, cost
// that much less: its pieces need one address (each_piece in the kernel).  Without this term the passes above are 0.04 % longer.
constexpr double kOnePiece = 0.4;
constexpr double kLastRound = 0.6;
constexpr double kHalfOffLines = 0.22;  // 256x256, several rounds: of what rows off the lines cost, where every other one lies on one
// Near ties of several rounds go to the 256x256 tiles, which take the least energy: 5248x7936x2496 222 us, in 128x256 232.
constexpr double kLargestTile = 0.98;
// A last round of 256x256 tiles that is at most half full may go to a second launch: its start and end behind the first one's,
// its share of K and an accumulator's sums, for each tile that it may have; from the same passes, which a term for rows off
// the lines or for a row map, or counting only the tiles that lie inside of the matrix, makes no shorter.  (With rem * 16 tiles of 64x64 on a chip that is otherwise idle
// instead of rem * 2 of 128x256: 2944x6144x3848 over four ranks 166 -> 133 us, 7168x4736x7928 616 -> 519, 3072x6400x4936 with an
// accumulator 251 -> 214.)
struct tail_cost {
    int tm, tn;
    double start, at_4096, sums;
};
constexpr tail_cost kTailCosts[] = {{64, 64, 3.7, 18.5, 1.9}, {64, 128, 4.3, 24.5, 2.0}, {128, 128, 5.1, 33, 4.0}, {128, 256, 5.1, 65, 7.9}};
constexpr double kTailLastRound = 0.5;

// Share of an operand's rows that do not begin on a 128-byte line.  Its row stride is a multiple of `step` bytes, a power of two up
// to 128: from a base that is one too, every 128 / step-th row lies on a line, from another one none.
double off_lines_share(const void *base, int K) {
    const unsigned pitch = (unsigned)K * 2 | 128, step = pitch & (0 - pitch);
    return (uintptr_t)base % step ? 1.0 : 1.0 - step / 128.0;
}

// Rounds of `count` tiles: a last one that is not full costs a part of a round and its share of the CUs (fewer active CUs
// share the L2s, HBM and the power limit).
double rounds(long count, long cus, double last) {
    const long full = count / cus, rest = count % cus;
    return full + (rest ? last + (1 - last) * rest / cus : 0.0);
}

// What fits the chip in one round, one tile per CU, takes the smallest tile that does: a smaller tile moves
// more operand bytes per flop (64x64 twice those of 128x128), but it puts the operand paths of CUs to work that a larger
// tile leaves idle, and up to that point a CU's time goes into waiting for its operands.  Measured over
// M = 128..4224, N = 1024..8192, K = 512, 2048, 8192: the rule picks the fastest tile or one within a few percent of it
// (K = 2048, us: 128x4096 64x32 7.3, 64x64 8.1, 128x128 12.8; 512x4096 64x128 11.7, 128x128 13.7, 64x64 16.2; 1024x4096
// 128x128 16.8, 128x256 21.8, 64x128 21.7).
// Up to 128x160 that is so whatever the estimate above says; beyond, it decides, for launches whose order and counters
// nobody waits for.  K = 4096 and 4088, us, against the rule before it (the largest tile that fits, else 256x256 from 60 %
// of the CUs on, else rounds of 128x256): 2048x4224 87.6 -> 64.1 and 117.9 -> 67.9 (two rounds of 128x160), 2048x5120
// 80.5 -> 75.5 and 93.9 -> 77.2, 2304x4096 77.1 -> 68.1 and 80.8 -> 71.8, 3456x4864 124.1 -> 119.7 (three rounds of
// 128x192); one round: 1536x3328 39.4 -> 36.2 and 50.7 -> 38.4 (128x160).
// Launches that move counters (`counted`) want whole reorder tiles, and what takes more than one round is walked in the
// raster that fo_schedule_order reports, tile by tile: a consumer waits for the groups in that order.  A larger tile
// beside the Algo's own would be faster (256x256 with half tiles where 256 does not divide M or N: 97 us a round of four
// times the output against 31), but its workgroups cross the order's XCD ranges, and the first group of such a launch
// was complete in its last round (8064x8192 in four groups: rounds 3, 1, 2, 3 of 0..3).
// M and N need only be multiples of 128: the last tile of a dimension is moved back or, 256x256, repeats half of its
// neighbour.
launch_plan plan_launch(const fo_raster &r, int M, int N, int K, int BM, int BN, bool whole_only, bool counted, double off_lines,
                        bool reordered, bool mapped, bool acc) {
    const bool on_lines = off_lines == 0;
    launch_plan p;
    p.tail = p.tail_tm = p.tail_tn = 0;
    auto set = [&](int tm, int tn) {
        p.tm = tm;
        p.tn = tn;
        p.grid_m = (M + tm - 1) / tm;
        p.grid_n = (N + tn - 1) / tn;
        p.whole = tm % BM == 0 && tn % BN == 0;
        p.count = p.grid_m * p.grid_n;
        p.xcd_remap = p.count >= 16 ? 1 : 0;
    };
    const bool square = r.mtm == 256 && r.mtn == 256;  // what fo_schedule_order assumes
    const long cus = fo_main_tile_resident();
    auto tiles = [&](int tm, int tn) { return (long)((M + tm - 1) / tm) * ((N + tn - 1) / tn); };
    // An XCD's workgroups (every eighth of the launch) take one stretch of panels of eight tile rows: they share operand
    // rows in its L2 both ways.
    auto set_shared = [&](int tm, int tn) {
        set(tm, tn);
        p.panel = p.grid_m < 8 ? p.grid_m : 8;
        // One or two rows left over would be a panel whose XCDs share one operand hardly at all (a block of 32 tiles reads 12
        // panels of operand rows as 8 x 4, 18 as 2 x 16, 33 as 1 x 32): panels of about one height instead, while that panel would be a large part
        // of the raster.  Whole passes of 1600 problems of more than eight tile rows in both: 0.8 % shorter in the mean for 9, 10, 17
        // and 18 rows (1.8 % for 9; 43 of 255 by more than 2 %, 9 longer by that), the same within 0.2 % for 25 and 26 and for other remainders.
        // 640x1024x4408 (10 rows of 64x64) 18.8 -> 18.3 us, 4224x7168x3584 (17 of 256x256) 180.5 -> 177.7, 1152x5120x1720 (9 of 128x192) the same.
        // (From 33 rows on, rasters of many rounds, one or two rows left over would gain 0.6 %; they keep eight.)
        const int panels = (p.grid_m + 7) / 8, left = p.grid_m % 8;
        if (panels > 1 && panels < 4 && (left == 1 || left == 2)) p.panel = (p.grid_m + panels - 1) / panels;
    };
    static const int shapes[][2] = {{32, 32},  {64, 32},   {64, 64},   {64, 96},   {64, 128}, {96, 128},
                                    {128, 128}, {128, 160}, {128, 192}, {128, 256}, {256, 128}};
    for (const auto &s : shapes) {
        if (!counted && s[0] * s[1] > 128 * 160) break;
        if (square || M < s[0] || N < s[1] || tiles(s[0], s[1]) > cus) continue;
        if (whole_only && (s[0] % BM || s[1] % BN)) continue;
        set_shared(s[0], s[1]);
        // of the two largest, the one that holds whole reorder tiles
        if (!p.whole && s[0] == 128 && s[1] == 256 && M >= 256 && tiles(256, 128) <= cus) set_shared(256, 128);
        return p;
    }
    const long nt = tiles(256, 256);
    if (!counted) {
        const int rem = nt > cus && nt % cus * 2 <= cus ? (int)(nt % cus) : 0;  // what a second launch may take
        const double k = K / 4096.0;
        const tile_cost *best = nullptr;
        const tail_cost *best_tail = nullptr;
        double least = 0;
        for (const tile_cost &t : kTileCosts) {
            if (M < t.tm || N < t.tn) continue;
            const bool largest = t.tm * t.tn == 256 * 256;
            const bool rounds_of_largest = nt > cus && largest;
            const double off = ((mapped ? t.mapped : t.off_lines) - t.on_lines) * (rounds_of_largest && off_lines <= 0.5 ? kHalfOffLines : 1.0);
            const bool one_piece = !mapped && !largest && t.tm * t.tn > 128 * 160 && (!reordered || (BM % t.tm == 0 && BN % t.tn == 0));
            const double round = (k * (t.on_lines + (on_lines ? 0 : off)) + (mapped ? t.end_mapped : t.end) +
                                  (!acc ? 0 : mapped ? t.sums_mapped : t.sums - (one_piece ? kOnePiece : 0))) *
                                 (rounds_of_largest ? kLargestTile : 1.0);
            auto offer = [&](double cost, const tail_cost *tail) {
                if (best && cost >= least) return;
                best = &t;
                best_tail = tail;
                least = cost;
            };
            offer(round * rounds(tiles(t.tm, t.tn), cus, kLastRound), nullptr);
            if (t.tm != 256 || t.tn != 256 || !rem) continue;
            for (const tail_cost &u : kTailCosts)
                offer(round * rounds(nt - rem, cus, kLastRound) + u.start +
                          (k * u.at_4096 + (acc ? u.sums : 0)) * rounds((long)rem * (256 / u.tm) * (256 / u.tn), cus, kTailLastRound),
                      &u);
        }
        set_shared(best->tm, best->tn);  // the 96x128 tile at least: M and N are multiples of 128
        if (p.tm == 256 && p.tn == 256) {
            if (best_tail) {
                p.tail = rem;
                p.count -= rem;
                p.tail_tm = best_tail->tm;
                p.tail_tn = best_tail->tn;
            }
            if (square) {
                p.panel = r.panel;
                p.xcd_remap = r.xcd_remap;
            }
        }
        return p;
    }
    set(r.mtm, r.mtn);
    p.panel = r.panel;
    p.xcd_remap = r.xcd_remap;
    if (r.tail_tiles) {
        // 128x128 while one round of them does it, else 128x256 or 256x128
        p.tail = r.tail_tiles;
        p.count -= r.tail_tiles;
        p.tail_tm = BM;
        p.tail_tn = BN;
        if (BM == 128 && BN == 128 && r.tail_tiles * 4 > r.resident && N % 256 == 0) p.tail_tn = 256;
    }
    return p;
}

// The plan of a GEMM whose operands lie at A and B.
launch_plan plan_gemm(const fo_raster &r, const fo_algo_entry &e, int M, int N, int K, const void *A, const void *B, int mode,
                      bool reordered, bool counts, bool monitor, bool acc) {
    return plan_launch(r, M, N, K, e.f[0], e.f[1], counts && (monitor || K < kSignalAfterFromK), counts,
                       (off_lines_share(A, K) + off_lines_share(B, K)) / 2, reordered, mode == MODE_SCATTER || mode == MODE_RS, acc);
}

// Whether a launch that counts can do the sums of its last wave itself (MODE_SIGNAL_SUM, MODE_SCATTER_SUM).
bool last_wave_sums(const launch_plan &p) {
    return p.tm == 256 && p.tn == 256 && !p.tail && p.count > fo_main_tile_resident();
}

// Signals of a launch whose workgroup tiles are parts of reorder tiles: behind it on the stream, everything at once
// (such a launch is a single round of short tiles; its reorder tiles complete together anyway).  MM[g] += cseg[g].
__global__ __launch_bounds__(256) void fo_signal_all_kernel(const int32_t *cseg, int G, int32_t *MM) {
    for (int g = threadIdx.x; g < G; g += 256)
        __hip_atomic_fetch_add(MM + g, cseg[g], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// What the epilogue of a reduce-scatter on one stream does besides storing C (MODE_RS in fo_gemm_common.h).
struct rs_args {
    void *own;
    int W, rank;
};

// What a launch refuses, asked before anything is enqueued.
int check_gemm(int mode, int dtype, int M, int N, int K, int rLDN, const int32_t *cseg, int G, const void *A, const void *B,
               const void *C, const int32_t *MM, const int32_t *RA, const int32_t *RE, int monitor, int algo, bool quiet,
               const void *acc) {
    if (dtype != FO_F16 && dtype != FO_BF16) return FO_ERR_DTYPE;
    const fo_algo_entry *e = fo_algo_lookup(algo);
    if (!e) return FO_ERR_ALGO;
    if (!A || !B || !C || M <= 0 || N <= 0 || K <= 0) return FO_ERR_ARG;
    if (M % e->f[0] || N % e->f[1]) return FO_ERR_SHAPE;
    if (K % 8) return FO_ERR_SHAPE;  // operand rows are fetched in 16-byte chunks
    if (K > (1 << 21)) return FO_ERR_SHAPE;  // 256 operand rows are addressed through one 31-bit buffer range
    // the epilogues assume reorder tiles made of 128 x 128 blocks
    if (e->f[0] % 128 || e->f[1] % 128) return FO_ERR_ALGO;
    if (mode == MODE_ACC && (((uintptr_t)C | (uintptr_t)acc) & 15)) return FO_ERR_SHAPE;  // as the consumer launch would
    if (mode == MODE_PLAIN || (mode == MODE_ACC && !RA)) return FO_OK;
    const int TN = N / e->f[1];
    const long T = (long)(M / e->f[0]) * TN;
    if ((!MM && !quiet) || !RA || !cseg) return FO_ERR_ARG;
    if ((mode == MODE_SCATTER || mode == MODE_RS) && !RE) return FO_ERR_ARG;
    if (rLDN <= 0 || T % rLDN) return FO_ERR_SHAPE;
    if (G <= 0 || G > T) return FO_ERR_SEGMENTS;
    if (monitor && G > TN - 1) return FO_ERR_SEGMENTS;
    return FO_OK;
}

int run_gemm(int mode, int dtype, int M, int N, int K, int rLDN, const int32_t *cseg, int G,
             const void *A, const void *B, void *C, int32_t *MM, const int32_t *RA,
             const int32_t *RE, int monitor, int algo, fo_stream_t stream, bool quiet = false, void *acc = nullptr,
             const rs_args *rs = nullptr, int sum_from = -1) {
    int rc = check_gemm(mode, dtype, M, N, K, rLDN, cseg, G, A, B, C, MM, RA, RE, monitor, algo, quiet, acc);
    if (rc) return rc;
    const fo_algo_entry *e = fo_algo_lookup(algo);
    fo_raster r;
    rc = fo_pick_raster(algo, M, N, &r);
    if (rc) return rc;
    GemmArgs a;
    a.A = static_cast<const uint16_t *>(A);
    a.B = static_cast<const uint16_t *>(B);
    a.C = static_cast<uint16_t *>(C);
    a.ACC = static_cast<uint16_t *>(acc);
    a.M = M; a.N = N; a.K = K;
    a.BM = e->f[0]; a.BN = e->f[1];
    a.TN = N / a.BN;
    a.rLDN = rLDN;
    a.RA = RA; a.RE = RE; a.cseg = cseg; a.G = G; a.MM = MM; a.monitor = monitor;
    a.OWN = static_cast<uint16_t *>(rs ? rs->own : nullptr);
    a.W = rs ? rs->W : 1;
    a.rank = rs ? rs->rank : 0;
    a.seg_rows = (int)((int64_t)M * N / a.BN / a.W);
    const bool counts = (mode == MODE_SIGNAL || mode == MODE_SCATTER) && !quiet;
    const launch_plan plan = plan_gemm(r, *e, M, N, K, A, B, mode, RA != nullptr, counts, monitor, acc != nullptr);
    a.grid_m = plan.grid_m; a.grid_n = plan.grid_n; a.panel = plan.panel; a.xcd_remap = plan.xcd_remap;
    a.first = 0; a.sub_m = a.sub_n = 1;
    a.count = plan.count;
    a.half = (M % 256 ? 1 : 0) | (N % 256 ? 2 : 0) | (mode == MODE_ACC && !fo_block_in_range(RA ? (int64_t)rLDN * a.BN : N) ? 4 : 0);
    // counters the launch cannot move itself are moved behind it
    const bool signal_after = counts && !plan.whole;
    a.quiet = quiet || signal_after ? 1 : 0;
    a.stream_out = (int64_t)M * N * 2 > kStreamOutAboveBytes ? 1 : 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    // The 128x192 tile that loads whole lines takes all of a CU's LDS and is not built for the epilogues that count; the
    // reordered store without counters is the accumulating epilogue without an accumulator.
    if (mode == MODE_SIGNAL && !counts && plan.tm == 128 && plan.tn == 192 && !on_lines(a)) mode = MODE_ACC;
    const bool only_stores = mode == MODE_SIGNAL && !counts && plan.tm == 256 && plan.tn == 256;
    const int tail_mode = mode;  // of the second launch, in a smaller tile
    if (only_stores) mode = MODE_REORDER;
    a.sum_from = sum_from;
    if (sum_from >= 0) {
        if (!last_wave_sums(plan) || monitor || (!acc && (mode != MODE_SCATTER || !a.OWN))) return FO_ERR_STATE;
        mode = mode == MODE_SCATTER ? MODE_SCATTER_SUM : MODE_SIGNAL_SUM;
    }
    // the tail split was computed for that many workgroups of the main launch
    rc = launch_tile(dtype, mode, a, plan.tm, plan.tn, s, nullptr, plan.tail ? fo_main_tile_resident() : 0);
    if (rc) return rc;
    if (signal_after) {
        hipLaunchKernelGGL(fo_signal_all_kernel, dim3(1), dim3(256), 0, s, cseg, G, MM);
        FO_LAUNCH_CHECK();
    }
    if (!plan.tail) return FO_OK;
    // the last, partial wave of 256x256 tiles: the same raster positions in a smaller tile
    GemmArgs t = a;
    t.first = a.count;
    t.sub_m = 256 / plan.tail_tm; t.sub_n = 256 / plan.tail_tn;
    t.count = plan.tail * t.sub_m * t.sub_n;
    return launch_tile(dtype, tail_mode, t, plan.tail_tm, plan.tail_tn, s);
}

}  // namespace

// Workgroups of the 256x256 shape that stay resident on the current device: what the
// raster's tail split is computed from.  All epilogues and both dtypes of that shape use
// the same LDS (one workgroup per CU); the launch checks its own instantiation against
// this number.  Without a usable device (host-only callers asking for the schedule order)
// the answer is MI355X's: 256 CUs, one workgroup each.
int fo_main_tile_resident() {
    const int limit = gemm_cu_limit().load(std::memory_order_relaxed);
    const int no_device = limit > 0 && limit < 256 ? limit / 8 * 8 : 256;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        (void)hipGetLastError();
        return no_device;
    }
    // Asked on every launch: answered from here after the first.  An entry holds the CU limit it was
    // computed under (plus one, in the upper half) and the answer.
    static std::atomic<int> cached[kMaxDevices];
    if (dev >= 0 && dev < kMaxDevices) {
        const int c = cached[dev].load(std::memory_order_relaxed);
        if ((c >> 16) == limit + 1) return c & 0xFFFF;
    }
    GemmArgs a = {};
    a.count = 1 << 30;
    int info[5] = {0, 0, 0, 0, 0};
    if (launch_tile(FO_F16, MODE_SIGNAL, a, 256, 256, nullptr, info) != FO_OK || info[4] <= 0 || info[4] > 0xFFFF) {
        (void)hipGetLastError();
        return no_device;
    }
    if (dev >= 0 && dev < kMaxDevices) cached[dev].store((limit + 1) << 16 | info[4], std::memory_order_relaxed);
    return info[4];
}

// The GEMM launches count on n CUs from here on (n <= 0: on all).  Process-wide, read at every launch;
// the caller changes it only while no schedule order taken under the old value is still in use.
extern "C" int fo_gemm_set_cu_limit(int n) {
    if (n > 0 && n < 8) return FO_ERR_ARG;  // the raster wants a workgroup count that is a multiple of the 8 XCDs
    if (n > 0x7FFE) return FO_ERR_ARG;
    gemm_cu_limit().store(n > 0 ? n : 0, std::memory_order_relaxed);
    return FO_OK;
}

// The reordered (optionally row-mapped) store of the signalling GEMMs without
// their counters, for a caller that orders GEMM and consumer by the stream alone.
int fo_gemm_reordered_quiet(int dtype, int M, int N, int K, int rLDN, const int32_t *cseg_dev, int G,
                            const void *A, const void *B, void *C, const int32_t *RA, const int32_t *RE,
                            int algo, fo_stream_t stream) {
    return run_gemm(RE ? MODE_SCATTER : MODE_SIGNAL, dtype, M, N, K, rLDN, cseg_dev, G, A, B, C, nullptr, RA, RE,
                    0, algo, stream, true);
}

int fo_gemm_signal_check(int dtype, int M, int N, int K, int rLDN, const int32_t *cseg_dev, int G, const void *A, const void *B,
                         const void *C, const int32_t *MM, const int32_t *RA, const int32_t *RE, int monitor, int algo) {
    return check_gemm(RE ? MODE_SCATTER : MODE_SIGNAL, dtype, M, N, K, rLDN, cseg_dev, G, A, B, C, MM, RA, RE, monitor, algo,
                      false, nullptr);
}

int fo_gemm_accumulate(int dtype, int M, int N, int K, int rLDN, const int32_t *cseg_dev, int G, const void *A, const void *B,
                       void *C, void *acc, const int32_t *RA, int algo, fo_stream_t stream) {
    if (!acc) return FO_ERR_ARG;
    return run_gemm(MODE_ACC, dtype, M, N, K, rLDN, cseg_dev, G, A, B, C, nullptr, RA, nullptr, 0, algo, stream, true, acc);
}

int fo_gemm_reduce_scatter(int dtype, int M, int N, int K, const int32_t *cseg_dev, int G, const void *A, const void *B, void *C,
                           void *acc, void *own, const int32_t *RA, const int32_t *RE, int W, int rank, int algo,
                           fo_stream_t stream) {
    const fo_algo_entry *e = fo_algo_lookup(algo);
    if (!e) return FO_ERR_ALGO;
    if (W <= 0 || rank < 0 || rank >= W || e->f[0] % W || (((uintptr_t)C | (uintptr_t)acc | (uintptr_t)own) & 15)) return FO_ERR_ARG;
    const rs_args rs = {own, W, rank};
    return run_gemm(MODE_RS, dtype, M, N, K, 1, cseg_dev, G, A, B, C, nullptr, RA, RE, 0, algo, stream, true, acc, &rs);
}

int fo_gemm_last_wave(int algo, int M, int N, int32_t *first, int32_t *slots) {
    const fo_algo_entry *e = fo_algo_lookup(algo);
    if (!e) return FO_ERR_ALGO;
    fo_raster r;
    int rc = fo_pick_raster(algo, M, N, &r);
    if (rc) return rc;
    const launch_plan plan = plan_launch(r, M, N, 4096, e->f[0], e->f[1], false, true, 0.0, true, false, false);
    const int resident = fo_main_tile_resident();
    *slots = (M / e->f[0]) * (N / e->f[1]);
    *first = last_wave_sums(plan) ? (plan.count - 1) / resident * resident * (256 / e->f[0]) * (256 / e->f[1]) : *slots;
    return FO_OK;
}

int fo_gemm_signal_sums(int dtype, int M, int N, int K, int rLDN, const int32_t *cseg_dev, int G, const void *A, const void *B,
                        void *C, int32_t *MM, const int32_t *RA, const int32_t *RE, void *acc, int sum_from, void *own, int W,
                        int rank, int algo, fo_stream_t stream) {
    const rs_args rs = {own, W, rank};
    return run_gemm(RE ? MODE_SCATTER : MODE_SIGNAL, dtype, M, N, K, rLDN, cseg_dev, G, A, B, C, MM, RA, RE, 0, algo, stream, false,
                    acc, &rs, sum_from);
}

extern "C" int fo_gemm_wave_tiles(int dtype, int algo, int M, int N, int32_t *tiles) {
    if (!tiles) return FO_ERR_ARG;
    const fo_algo_entry *e = fo_algo_lookup(algo);
    if (!e) return FO_ERR_ALGO;
    fo_raster r;
    int rc = fo_pick_raster(algo, M, N, &r);
    if (rc) return rc;
    const launch_plan plan = plan_launch(r, M, N, 4096, e->f[0], e->f[1], false, true, 0.0, true, false, false);
    GemmArgs a = {};
    a.count = plan.count;
    int info[5] = {0, 0, 0, 0, 0};
    rc = launch_tile(dtype, MODE_SIGNAL, a, plan.tm, plan.tn, nullptr, info);
    if (rc) return rc;
    const long all = (long)(M / e->f[0]) * (N / e->f[1]);
    const long wave = (long)info[0] * plan.tm * plan.tn / ((long)e->f[0] * e->f[1]);
    *tiles = (int32_t)(!plan.whole || wave > all ? all : wave);
    return FO_OK;
}

extern "C" int fo_gemm_kernel_info(int dtype, int algo, int M, int N, int epilogue, int32_t info[4]) {
    if (!info) return FO_ERR_ARG;
    fo_raster r;
    int rc = fo_pick_raster(algo, M, N, &r);
    if (rc) return rc;
    const fo_algo_entry *e = fo_algo_lookup(algo);
    const launch_plan plan = plan_launch(r, M, N, 4096, e->f[0], e->f[1], false, epilogue != MODE_PLAIN, 0.0,
                                         epilogue != MODE_PLAIN, epilogue == MODE_SCATTER, false);
    GemmArgs a = {};
    a.count = plan.count;
    int out[5] = {0, 0, 0, 0, 0};
    if (epilogue < MODE_PLAIN || epilogue > MODE_SCATTER) return FO_ERR_ARG;
    rc = launch_tile(dtype, epilogue, a, plan.tm, plan.tn, nullptr, out);
    if (rc) return rc;
    for (int i = 0; i < 4; i++) info[i] = out[i];
    return FO_OK;
}

extern "C" int fo_gemm_plan(int algo, int M, int N, int K, const void *A, const void *B, int epilogue, int counts, int acc,
                            int32_t plan[7]) {
    if (!plan || epilogue < MODE_PLAIN || epilogue > MODE_SCATTER || (counts && (acc || epilogue == MODE_PLAIN))) return FO_ERR_ARG;
    if (K <= 0) return FO_ERR_ARG;
    if (K % 8) return FO_ERR_SHAPE;
    const fo_algo_entry *e = fo_algo_lookup(algo);
    if (!e) return FO_ERR_ALGO;
    if (e->f[0] % 128 || e->f[1] % 128) return FO_ERR_ALGO;
    fo_raster r;
    int rc = fo_pick_raster(algo, M, N, &r);
    if (rc) return rc;
    const launch_plan p = plan_gemm(r, *e, M, N, K, A, B, epilogue, epilogue != MODE_PLAIN, counts != 0, false, acc != 0);
    const int32_t out[7] = {p.tm, p.tn, p.count, p.panel, p.tail, p.tail_tm, p.tail_tn};
    for (int i = 0; i < 7; i++) plan[i] = out[i];
    return FO_OK;
}

extern "C" int fo_gemm(int dtype, int M, int N, int K, const void *A, const void *B, void *C,
                       int algo, fo_stream_t stream) {
    return run_gemm(MODE_PLAIN, dtype, M, N, K, 1, nullptr, 0, A, B, C, nullptr, nullptr, nullptr, 0,
                    algo, stream);
}

extern "C" int fo_gemm_signal(int dtype, int M, int N, int K, int rLDN, const int32_t *cseg_dev,
                              int G, const void *A, const void *B, void *C, int32_t *MM,
                              const int32_t *RA, int monitor, int algo, fo_stream_t stream) {
    return run_gemm(MODE_SIGNAL, dtype, M, N, K, rLDN, cseg_dev, G, A, B, C, MM, RA, nullptr,
                    monitor, algo, stream);
}

extern "C" int fo_gemm_scatter(int dtype, int M, int N, int K, int rLDN, const int32_t *cseg_dev,
                               int G, const void *A, const void *B, void *C, int32_t *MM,
                               const int32_t *RA, const int32_t *RE, int monitor, int algo,
                               fo_stream_t stream) {
    return run_gemm(MODE_SCATTER, dtype, M, N, K, rLDN, cseg_dev, G, A, B, C, MM, RA, RE, monitor,
                    algo, stream);
}
