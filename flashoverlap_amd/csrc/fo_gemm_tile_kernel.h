// The workgroup tiles from 32x32 to 128x256 / 256x128 of the gfx950 MFMA GEMM (plain, signal and scatter
// epilogues): problems that do not fill the chip with 256x256 tiles, the remainder of a last wave of those,
// and sizes that 256 does not divide.  Arguments, raster and epilogue semantics are those of fo_gemm_common.h
// (its reference citations hold here too), and every product is summed in the same order (ascending K,
// 32 columns per MFMA) whatever the tile, so all shapes give the same bits.
//
// What bounds these sizes is not the matrix pipe but getting operands to it: a CU takes at most 64 bytes per clock
// from its L2 (152 GB/s measured on one CU, 130 with all of them loading), returned in order, so that a load
// that misses the L2 holds up the hits behind it, and a wavefront that presents loads faster than they drain
// stands still with its MFMAs behind them.  The workgroup is therefore split in two roles, four wavefronts
// each: loaders, which do nothing but move operand stages HBM/L2 -> LDS (buffer_load_dwordx4 ... lds) up to
// S - 1 stages ahead and may stand still as long as they like, and computing wavefronts, which touch nothing
// but LDS and the matrix pipe.  One barrier per K step (BK columns) says that the step's slot has been read by everyone
// (the loaders refill it next) and that the next stage has landed.
//
// The MFMAs of a step run in strips of two long fragments (those of the operand of which a wavefront holds more) by all
// short ones, all k-steps of an accumulator block in a row and one operand changing from block to block: the order that
// costs least energy (fo_gemm256_kernel.h; these sizes run at 1.65 to 1.9 GHz of 2.4 with random operands and at 2.37 with
// zeros).  Fragment fetches are spread between the MFMAs: issued as one burst, all wavefronts burst together behind the
// barrier and the matrix pipe waits for the LDS.  Two ways to hold fragments:
//   AHEAD: the whole next stage in a second set of registers, fetched from the middle of the step on.  Small wavefront
//     tiles, whose step is too short to hide a fetch in, and the shifted form, whose fetches take longer.
//   otherwise long fragments a strip ahead; a short one is replaced once the last strip is done with it.
// In us against one set of fragments per k-step, fetched a k-step ahead (fp16, GEMM alone): AHEAD 128x1024x8192 15.8 ->
// 12.8, 128x4096x1024 5.4 -> 5.2, 128x4096x4088 12.7 -> 11.7, 384x4096x4088 37.7 -> 30.6, 1152x5120x1720 26.4 -> 25.1;
// strips 1024x4096x2048 18.3 -> 17.8, 1536x3328x4096 37.1 -> 36.6, 1536x4096x4096 69.7 -> 68.0, 1024x8192x2048 30.7 -> 29.9,
// 512x4096x4096 the same.  The other way round: 1024x4096x4088 in strips 34.2 against 33.4, 128x160 tiles hold no second set.
//
// Measured against the kernel this one replaced (loads issued by the computing wavefronts; fp16, GEMM alone,
// operands of three buffer sets in turn, which the memory-side cache holds): 512x4096x4096 39.1 -> 21 us, 256x8192x3584
// 35.5 -> 19.5, 128x4096x1024 10.4 -> 4.5, 128x1024x8192 71 -> 12.5, 2048x4096x4096 62 -> 55.
// None of it is at a unit's limit.  512x4096x4096 on 64x128 tiles (21.0 us): 39 bytes a clock and CU of the 64, matrix pipe
// busy 41 % of the clocks, LDS reads 32 %; with the MFMAs taken out 19.7 of 21.8 us, so what is left is round trips to the
// operands.  With operands that no cache holds (eight sets in turn) the same misses take longer: 28.1 us, 256x8192x3584 19.7
// -> 28.2.  One round of 128x256 tiles (1024x8192x2048, 29.2 us) has the matrix pipe busy for 64 % and LDS reads for 27 %.
//
// SHIFT: operand rows that do not begin on 128-byte lines (K no multiple of 64, or an operand's own address).  A load of
// eight rows x 128 bytes then touches sixteen lines instead of eight, and these sizes slow down by 30 to 40 %.  Shifted,
// the loaders fetch whole lines: row r's stage begins at the line that holds the stage's first column, up to seven chunks
// early, and a computing lane whose chunk lies behind that line's end takes it from the following block (all its
// fragments belong to rows 16 apart, so that is a constant of the lane).  A step thus reads its own stage and the next,
// which costs one stage of the ones in flight; the products and their order are the same.  K = 4088 against 4096 (us):
// 512x4096 30.4 -> 22.6 against 22.2, 1024x4096 41.4 -> 34.5 against 32.5, 128x4096 15.4 -> 13.2 against 12.3.  Both forms
// permute a row's chunks by exclusive or: a fetch takes lanes of two chunk columns in one pass, and with the chunks rotated
// instead half of this form's LDS time was bank conflicts (exclusive or against rotated: 1152x5120x1720 27.8 -> 26.8 us,
// 512x4096x4088 23.3 -> 22.6, 384x4096x4088 39.0 -> 36.9, 128x4096x4088 12.7 -> 12.3).  Tiles with room for three
// stages only (128x256, and 128x192 where a row map takes LDS as well: four stages of it are all a CU has) keep the plain form:
// with both stages of a step awaited, nothing would be in flight.
//
// MODE_ACC, the epilogue of calls that stay on one stream: what the consumer kernel would do behind the GEMM (read C and
// the accumulator, write the accumulator) is done on the tile in LDS.  The loaders, idle by then, request the
// accumulator's values while the last S - 1 stages are multiplied and write the sums; the computing wavefronts store
// C.  Saves the second read of C and a launch.  Whole passes: 512x4096x4096 29.5 -> 28.7 us, 1152x5120x1720
// 42.7 -> 40.7, 1024x8192x2048 49 -> 46.2.
#pragma once

#include <type_traits>

#include "fo_gemm_common.h"

namespace fo_gemm_dev {

template <typename Tag> struct fo_mfma16;
template <> struct fo_mfma16<fo_f16_tag> {
    typedef fo_half8 frag;
    static __device__ __forceinline__ fo_float4v go(frag a, frag b, fo_float4v c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};
template <> struct fo_mfma16<fo_bf16_tag> {
    typedef fo_bf8 frag;
    static __device__ __forceinline__ fo_float4v go(frag a, frag b, fo_float4v c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};

constexpr int kTileLoaders = 4, kTileComputers = 4, kTileThreads = (kTileLoaders + kTileComputers) * 64;

// Columns, in chunks of 8, by which row `row` (0..15) of an operand that begins at `base` lies behind the start of its
// 128-byte line.  The same for rows 8 apart, whatever the leading dimension (a multiple of 8).
__device__ __forceinline__ int row_shift(const uint16_t *base, int ld, int row) {
    return (int)(((uintptr_t)base >> 4) + (unsigned)(row * (ld >> 3))) & 7;
}

// S operand slots; the output tile is staged in the same space once the K loop is done.
template <int TM, int TN, int BK, int S>
constexpr int tile_smem_bytes() {
    return S * (TM + TN) * BK * 2 > TM * (TN + 8) * 2 ? S * (TM + TN) * BK * 2 : TM * (TN + 8) * 2;
}

// What a computing wavefront's K step is made of: FL x FS accumulator blocks, KK k-steps.
template <int FL, int FS, int KK>
struct tile_step {
    static constexpr int NB = FL * FS, LEAD_B = FL % 2 * FS;  // blocks, of those in a first strip of one
    static constexpr int NS = (FL + 1) / 2;                   // strips; an odd one out is a strip of its own, the first
    static constexpr int NF = (FL + FS) * KK, NM = NB * KK;   // fetches of a stage and MFMAs of a step
    // The blocks in their order: strips of two long fragments by all short ones, one operand changing from block to block.
    struct block { int i, j; };
    static constexpr block block_at(int c) {
        if (c < LEAD_B) return block{0, c};
        const int e = c - LEAD_B, j = e % (2 * FS) / 2;
        return block{FL % 2 + e / (2 * FS) * 2 + ((e & 1) ^ (j & 1)), j};
    }
    // The fragments of a stage in the order in which its blocks want them.
    struct fetch { bool is_long; int at, kk; };
    struct fetch_order { fetch nth[NF]; };
    static constexpr fetch_order fetches() {
        fetch_order f{};
        bool have_l[FL] = {}, have_s[FS] = {};
        int n = 0;
        for (int c = 0; c < NB; c++) {
            const block x = block_at(c);
            for (int kk = 0; kk < KK; kk++) {
                if (!have_s[x.j]) f.nth[n++] = fetch{false, x.j, kk};
                if (!have_l[x.i]) f.nth[n++] = fetch{true, x.i, kk};
            }
            have_s[x.j] = have_l[x.i] = true;
        }
        return f;
    }
    // `n` things spread evenly over `span` places: the first one at place w or behind it.
    static constexpr int first_at(int w, int n, int span) {
        const int t = w <= 0 ? 0 : (w * n + span - 1) / span;
        return t < n ? t : n;
    }
};

template <typename Tag, int TM, int TN, int BK, int S, int MODE, bool SHIFT>
__global__ __launch_bounds__(kTileThreads, 2) void fo_gemm_tile_kernel(uint64_t A, uint64_t B, uint64_t M_N,
                                                                          uint64_t K_grid_m, uint64_t grid_n_stride,
                                                                          uint64_t by_panel_rows, uint64_t by_last_bits, TileRest) {
    // The fields of TileArgs that the first operand load needs.
    TileArgs args;
    args.A = (const uint16_t *)(uintptr_t)A;
    args.B = (const uint16_t *)(uintptr_t)B;
    args.M = (int)M_N;
    args.N = (int)(M_N >> 32);
    args.K = (int)K_grid_m;
    args.grid_m = (int)(K_grid_m >> 32);
    args.grid_n = (int)grid_n_stride;
    args.stride = (int)(grid_n_stride >> 32);
    args.by_panel.mul = (uint32_t)by_panel_rows;
    args.by_rows.mul = (uint32_t)(by_panel_rows >> 32);
    args.by_last_rows.mul = (uint32_t)by_last_bits;
    args.bits = (uint32_t)(by_last_bits >> 32);
    typedef fo_elem<Tag> E;
    typedef fo_mfma16<Tag> X;
    typedef typename X::frag frag;
    constexpr int NL = kTileLoaders, KB = BK / 64, KK = BK / 32;  // 64-column blocks and MFMA k-steps per stage
    constexpr int WTM = TM / 2, WTN = TN / 2, FM = WTM / 16, FN = WTN / 16;  // computing wavefronts: 2 x 2
    constexpr int PA = TM / 8 / NL, PB = TN / 8 / NL, P = KB * (PA + PB);    // 1 KiB loads per loader and stage
    constexpr unsigned A_BLK = TM * 128, B_BLK = TN * 128, STAGE = KB * (A_BLK + B_BLK);
    constexpr bool ACC = MODE == MODE_ACC || MODE == MODE_RS, COUNTS = MODE == MODE_SIGNAL || MODE == MODE_SCATTER;
    constexpr bool MAPPED = MODE == MODE_SCATTER || MODE == MODE_RS;
    // Where MODE_ACC also stands for the reordered store without counters (fo_gemm.hip).  (Asked where it need not be, the
    // question waits for an argument in front of the first further load: 1664x4608x904 in 128x128 tiles 27.1 -> 27.6 us.)
    constexpr bool MAY_LACK = MODE == MODE_RS || (SHIFT && TM == 128 && TN == 192);
    // output staging; with an accumulator the computing wavefronts store the tile and the loaders update the accumulator
    constexpr int STORERS = ACC ? kTileComputers * 64 : kTileThreads;
    constexpr int PITCH = TN + 8, CPR = TN / 8, NCH = (TM * CPR + STORERS - 1) / STORERS;
    static_assert(STORERS % CPR || TM * CPR < STORERS || TM * CPR % STORERS == 0, "a piece per thread and step, none behind the tile");
    static_assert(BK % 64 == 0 && TM % 32 == 0 && TN % 32 == 0, "whole 1 KiB loads for every loader");
    // Loads that may be in flight while a K step is multiplied whose successor is to be ready: all stages behind that one
    // or, shifted, behind the first 64 columns of the stage that follows it.
    constexpr int FLIGHT = SHIFT ? (S - 3) * P + (KB - 1) * (P / KB) : (S - 2) * P;
    static_assert(!SHIFT || (S >= 4 && KB <= 2), "a shifted step reads two stages, one more has to be in flight");
    static_assert(S >= 2 && (S - 1) * P < 64 && (!ACC || (S - 3) * P + NCH < 64), "vmcnt range");

    extern __shared__ fo_u32x4 smem[];
    __shared__ int32_t row_map[MAPPED ? 256 : 1];          // where the tile's rows go
    __shared__ int32_t rs_map[MODE == MODE_RS ? 256 : 1];  // and their rows in the accumulator
    const unsigned lds0 = (unsigned)(uintptr_t)FO_LDS_PTR(smem);
    uint16_t *stage = reinterpret_cast<uint16_t *>(smem);  // the output tile, once the K loop is done
    const int tid = threadIdx.x;
    const int wave_id = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool loader = wave_id < NL;
    const int wave = loader ? wave_id : wave_id - NL;
    const int wm = wave >> 1, wn = wave & 1;
    const int KT = (args.K + BK - 1) / BK;

    const int count = fo_tile_count(args);

    // The first tile from position `tile` on.  (One cut from a 256x256 position may lie beyond the matrix.)
    int tile = blockIdx.x, pm = 0, pn = 0;
    auto settle = [&]() __attribute__((always_inline)) {
        while (tile < count) {
            fo_tile_of(args, tile, &pm, &pn);
            pm = __builtin_amdgcn_readfirstlane(pm);
            pn = __builtin_amdgcn_readfirstlane(pn);
            if (__builtin_expect(!(args.bits & TileArgs::GENERAL), 1) || (pm * TM < args.M && pn * TN < args.N)) break;
            tile += args.stride;
        }
    };
    // A loader's part of the tile: load u of a 64-column block brings rows (u * NL + wave) * 8 + lane / 8 of an operand, 128
    // bytes each; LDS slot `lane` of the 1 KiB block is (row lane / 8, chunk lane % 8) and receives chunk phys ^ key(row).
    // Shifted, slot `lane` receives chunk ((phys ^ key(row)) + shift(row)) % 8 of the row's aligned line, so that a
    // column's chunk lies where it would unshifted; what lies before the row's first column or behind its last is
    // requested out of range (zeros).
    fo_srd_t ra = {}, rb = {};
    int a_chunk = 0, b_chunk = 0;
    unsigned lane_row = 0, wave_lds = 0;
    const unsigned row_step = (unsigned)(NL * 8 * args.K * 2);
    // With twelve loads a stage the row offsets no longer fit the scalar registers.
    auto load = [&](fo_srd_t srd, unsigned voff, unsigned row_off, unsigned col_off, unsigned lds_addr) __attribute__((always_inline)) {
        if constexpr (P >= 12)
            dma_buf16_sum(srd, voff, __builtin_amdgcn_readfirstlane(row_off), col_off, lds_addr);
        else
            dma_buf16(srd, voff, __builtin_amdgcn_readfirstlane(row_off + col_off), lds_addr);
    };
    auto request = [&](int kt, unsigned slot_v) __attribute__((always_inline)) {
        const unsigned slot = __builtin_amdgcn_readfirstlane(slot_v);  // uniform by construction; said so for the assembly's operands
#pragma unroll
        for (int kb = 0; kb < KB; kb++) {
            const int col = __builtin_amdgcn_readfirstlane(kt * BK + kb * 64);
            // chunks beyond K (a partial last step, stages behind the last) are requested out of range: zeros
            const unsigned a_off = (SHIFT ? (unsigned)(col + a_chunk * 8) < (unsigned)args.K : a_chunk * 8 < args.K - col) ? lane_row + a_chunk * 16 : 0x80000000u;
            const unsigned b_off = !SHIFT ? a_off : (unsigned)(col + b_chunk * 8) < (unsigned)args.K ? lane_row + b_chunk * 16 : 0x80000000u;
#pragma unroll
            for (int u = 0; u < PB; u++)
                load(rb, b_off, u * row_step, col * 2, wave_lds + slot + KB * A_BLK + kb * B_BLK + u * NL * 1024);
#pragma unroll
            for (int u = 0; u < PA; u++)
                load(ra, a_off, u * row_step, col * 2, wave_lds + slot + kb * A_BLK + u * NL * 1024);
        }
    };
    // Requests the tile's first S - 1 stages.  A launch's first tile is begun in front of everything else in the kernel:
    // every instruction and argument in front of the first load is itself fetched from memory.  With the raster's divisions,
    // the reorder table's entries and what the compiler moves out of the tile loop there, the first load left 2800 to 3900
    // clocks after the kernel's start, now 1200 (us, GEMM alone, plain / reordered: 128x4096x1024 5.1 -> 4.5 / 5.6 -> 4.7,
    // 512x4096x4096 21.6 -> 21.3 / 22.1 -> 21.3, 1024x4096x2048 18.6 -> 18.0 / 19.1 -> 17.8).
    auto begin = [&]() __attribute__((always_inline)) {
        int lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));
        const int m0 = pm * TM + TM > args.M ? args.M - TM : pm * TM, n0 = pn * TN + TN > args.N ? args.N - TN : pn * TN;  // as below
        const int lrow = lane >> 3, lkey = ((wave * 8 + lrow) >> 1) & 7;
        const uint16_t *a0 = args.A + (size_t)m0 * args.K, *b0 = args.B + (size_t)n0 * args.K;
        const int a_shift = SHIFT ? row_shift(a0, args.K, lrow) : 0, b_shift = SHIFT ? row_shift(b0, args.K, lrow) : 0;
        a_chunk = SHIFT ? ((((lane & 7) ^ lkey) + a_shift) & 7) - a_shift : (lane & 7) ^ lkey;
        b_chunk = SHIFT ? ((((lane & 7) ^ lkey) + b_shift) & 7) - b_shift : (lane & 7) ^ lkey;
        constexpr int LEAD = SHIFT ? 128 : 0;  // the range starts a line early: no lane's offset is negative
        lane_row = (unsigned)((wave * 8 + lrow) * args.K * 2 + LEAD);
        ra = fo_make_srd(a0 - LEAD / 2, (unsigned)TM * args.K * 2 + LEAD);
        rb = fo_make_srd(b0 - LEAD / 2, (unsigned)TN * args.K * 2 + LEAD);
        wave_lds = __builtin_amdgcn_readfirstlane(lds0 + wave * 1024);
        asm volatile("" : "+s"(wave_lds));  // the loads' LDS addresses are sums made where they are used
        __builtin_amdgcn_s_setprio(3);
#pragma unroll
        for (int s = 0; s < S - 1; s++) request(s, s * STAGE);
    };
    asm volatile("" : : "s"(args.A), "s"(args.B), "s"(args.bits));  // in registers from here on, not put together again where they are used
    settle();
    if (loader && tile < count) begin();

    // The arguments that are not needed before this point are read from here on, not at the kernel's entry.
    typedef const __attribute__((address_space(4))) TileArgs *args_t;
    args_t rest = (args_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(rest));
    const __attribute__((address_space(4))) TileArgs &p = *rest;

    const uint32_t bits = p.bits;
    const int bm_shift = bits & TileArgs::TALL ? 8 : 7, bn_shift = bits & TileArgs::WIDE ? 8 : 7;  // reorder tiles: 128 or 256 each way
    const int RTN = p.N >> bn_shift;  // reorder tiles along N
    const int log_ranks = bits >> TileArgs::RANKS & 15, ranks = 1 << log_ranks;  // MODE_RS
    const bool reorder = MODE == MODE_ACC ? p.RA != nullptr : MODE != MODE_PLAIN;
    const int rLDN = MODE == MODE_RS ? 1 : p.rLDN;
    const int ldp = reorder ? rLDN << bn_shift : p.N;  // leading dimension of the output view
    const bool signalling = COUNTS && !(bits & TileArgs::QUIET);
    typedef const __attribute__((address_space(4))) int32_t *cptr_t;  // read-only for the whole launch: scalar loads
    const cptr_t RAc = (cptr_t)(uintptr_t)p.RA;

    while (tile < count) {
        // What is computed from the lane is computed for each tile: kept from one to the next, the group search's and the
        // loaders' part of it alone took twenty registers through the K loop.
        int lane = tid & 63;
        asm volatile("" : "+v"(lane));
        // Where the dimension ends inside the tile, the tile is moved back so that all of its operand rows exist; the
        // rows or columns it then shares with its neighbour are neither stored nor counted.
        const int m0 = pm * TM + TM > p.M ? p.M - TM : pm * TM, n0 = pn * TN + TN > p.N ? p.N - TN : pn * TN;
        const int skip_m = pm * TM - m0, skip_n = pn * TN - n0;
        // The tile lies in one reorder tile or in two, one above or beside the other; the second begins at row split_m
        // or column split_n.  r0, r1: their storage slots.
        int r0 = 0, r1 = 0;
        bool two_m = false, two_n = false;
        int split_m = TM, split_n = TN;
        if (reorder) {
            const int tm0 = m0 >> bm_shift, tn0 = n0 >> bn_shift;
            two_m = (m0 + TM - 1) >> bm_shift != tm0;
            two_n = (n0 + TN - 1) >> bn_shift != tn0;
            if (two_m) split_m = ((tm0 + 1) << bm_shift) - m0;
            if (two_n) split_n = ((tn0 + 1) << bn_shift) - n0;
            r0 = RAc[tm0 * RTN + tn0];
            r1 = two_m || two_n ? RAc[(tm0 + two_m) * RTN + tn0 + two_n] : r0;
        }
        int g0 = 0, g1 = 0;  // groups of r0 and r1 (the wavefront that signals)
        // Row and column of the output view at which the tile's row and column 0 are, or would be, in r0 and in r1.
        int row0 = m0, row1 = m0, col0 = n0, col1 = n0;
        auto find_bases = [&]() __attribute__((always_inline)) {
            if (!reorder) return;
            int rldn = rLDN;
            asm volatile("" : "+s"(rldn));  // the divisions by it are done here, not in front of the K loop
            int q0 = r0, q1 = r1;
            if (rldn != 1) {
                q0 /= rldn;
                q1 /= rldn;
            }
            row0 = (q0 << bm_shift) + (m0 & ((1 << bm_shift) - 1));
            row1 = (q1 << bm_shift) + (two_m ? -split_m : m0 & ((1 << bm_shift) - 1));
            col0 = (r0 - q0 * rldn << bn_shift) + (n0 & ((1 << bn_shift) - 1));
            col1 = (r1 - q1 * rldn << bn_shift) + (two_n ? -split_n : n0 & ((1 << bn_shift) - 1));
        };
        // The tile in pieces of 16 bytes: act(u, row, column, address in the view `out`) for thread t's piece u, those
        // to be stored or (EVERY) all of them.  A tile that lies in one reorder tile and is stored whole needs one address
        // per thread, the pieces following at a uniform distance (the general address costs some forty instructions, and
        // a thread has up to sixteen pieces).  (The thread id is laundered so that this is computed here instead of
        // resting in registers across the K loop.)
        const bool simple = !two_m && !two_n && !skip_m && !skip_n && ldp < 1 << 22;
        auto each_piece = [&](int t, uint16_t *out, auto every, auto act) __attribute__((always_inline)) {
            constexpr bool EVERY = decltype(every)::value;
            asm volatile("" : "+v"(t));
            if (EVERY && TM * CPR < STORERS) t %= TM * CPR;  // threads beyond the tile's pieces read some of them again, nothing behind the tile
            if (simple) {
                uint16_t *base = out + (size_t)row0 * ldp + col0;
#pragma unroll
                for (int u = 0; u < NCH; u++) {
                    const bool steps = STORERS % CPR == 0;
                    const int idx = (u * STORERS + t) % (EVERY ? TM * CPR : 1 << 30);
                    const int row = steps ? u * (STORERS / CPR) + t / CPR : idx / CPR, col = (steps ? t : idx) % CPR * 8;
                    const unsigned off = (unsigned)((steps ? t / CPR : row) * ldp + col);
                    if (EVERY || TM * CPR % STORERS == 0 || row < TM)
                        act(u, row, col, base + (steps ? (size_t)(u * (STORERS / CPR)) * ldp : 0) + off);
                }
            } else {
#pragma unroll
                for (int u = 0; u < NCH; u++) {
                    const int idx = (u * STORERS + t) % (EVERY ? TM * CPR : 1 << 30), row = idx / CPR, col = idx % CPR * 8;
                    const bool second = row >= split_m || col >= split_n;
                    if (EVERY || ((TM * CPR % STORERS == 0 || row < TM) && row >= skip_m && col >= skip_n))
                        act(u, row, col, out + (size_t)((second ? row1 : row0) + row) * ldp + (second ? col1 : col0) + col);
                }
            }
        };
        // The same where a map in LDS says which row of the view a row goes to.  Only rows [from, from + rows) of the view
        // exist, and `out` is where the first of them begins; the others' pieces are left out (EVERY: read at row 0).
        auto each_mapped_piece = [&](int t, const int32_t *map, uint16_t *out, auto every, auto act, int from = 0,
                                     int rows = 0x7fffffff) __attribute__((always_inline)) {
            constexpr bool EVERY = decltype(every)::value;
            asm volatile("" : "+v"(t));
#pragma unroll
            for (int u = 0; u < NCH; u++) {
                const int idx = (u * STORERS + t) % (EVERY ? TM * CPR : 1 << 30), row = idx / CPR, col = idx % CPR * 8;
                const bool second = row >= split_m || col >= split_n;
                if (EVERY || ((TM * CPR % STORERS == 0 || row < TM) && row >= skip_m && col >= skip_n)) {
                    const int to = map[two_n && second ? TM + row : row] - from;
                    if (EVERY || (unsigned)to < (unsigned)rows)
                        act(u, row, col, out + (size_t)(to < 0 ? 0 : to) * ldp + (second ? col1 : col0) + col);
                }
                if (u % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // sixteen addresses at once would be too many registers
            }
        };
        auto piece = [&](int row, int col) __attribute__((always_inline)) {
            return *reinterpret_cast<const fo_u32x4 *>(stage + row * PITCH + col);
        };

        if (loader) {
            wait_vmcnt<FLIGHT>();  // what the first step reads has landed (vmcnt retires in issue order)
            __builtin_amdgcn_s_barrier();
            unsigned slot = (S - 1) * STAGE;
            // With an accumulator the steps behind the last request ask for its values instead of further stages: they
            // arrive while the last S - 1 stages are multiplied.
            const bool sums = ACC && (!MAY_LACK || p.ACC);
            const int stages = SHIFT ? KT + 1 : KT;
            // (At least two steps in front of it where the maps are written behind the first: KT > S there, and the second step's
            // barrier publishes rs_map, from which the addresses come.)
            const int fetching = sums ? (stages > S - 1 ? stages - (S - 1) : 0) : KT;
            for (int kt = 0; kt < fetching; kt++) {
                request(kt + S - 1, slot);  // the slot of stage kt - 1, given up at the last barrier
                slot = slot + STAGE == S * STAGE ? 0 : slot + STAGE;
                wait_vmcnt<FLIGHT>();  // what step kt + 1 reads
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
            }
            // The ways with and without an accumulator meet behind the sums, not between request and wait: the compiler took the values
            // for still on their way there, and the rows for this rank waited until the sums had reached memory (whole calls, eight
            // ranks, us: 2048x4096x2048 39.0 -> 37.4, 3456x2176x680 25.2 -> 23.4, 512x4096x1024 bf16 with two 12.3 -> 11.6).
            if (ACC && sums) {
                fo_u32x4 old[ACC ? NCH : 1];  // the accumulator's values
                // every wavefront loads every piece, needed or not: the waits below count
                find_bases();
                if constexpr (MODE == MODE_RS) {
                    each_mapped_piece(wave * 64 + lane, rs_map, p.ACC, std::true_type{},
                                      [&](int u, int, int, uint16_t *at) __attribute__((always_inline)) {
                        old[ACC ? u : 0] = *reinterpret_cast<const fo_u32x4 *>(at);
                    });
                } else {
                    // The addresses first, the loads behind the point where the ways to them meet: with loads on both ways the compiler,
                    // which takes the second for a way that may follow the first, waited there for the registers of the first,
                    // and with them for every operand stage in flight (whole passes, us: 896x3968x4088 by the serial call 33.2 -> 32.2,
                    // 512x4096x1000 13.3 -> 12.8, 7680x2560x368 in 300 groups 52.6 -> 52.1; the others up to 0.7 %).
                    typedef const __attribute__((address_space(1))) fo_u32x4 *global_t;
                    global_t from[ACC ? NCH : 1];
                    each_piece(wave * 64 + lane, p.ACC, std::true_type{}, [&](int u, int, int, uint16_t *at) __attribute__((always_inline)) {
                        from[ACC ? u : 0] = (global_t)(uintptr_t)at;
                    });
#pragma unroll
                    for (int u = 0; u < (ACC ? NCH : 1); u++) asm volatile("" : "+v"(from[u]));
#pragma unroll
                    for (int u = 0; u < (ACC ? NCH : 1); u++) old[u] = *from[u];
                }
                asm volatile("" ::: "memory");
#pragma unroll
                for (int j = 0; j < S - 1; j++) {
                    if (fetching + j < KT) {
                        const int left = FLIGHT - (j + 1) * P;  // the same, with one stage fewer requested each time
                        if (j < S - 2) asm volatile("s_waitcnt vmcnt(%0)" : : "i"(ACC ? (left > 0 ? left : 0) + NCH : 0) : "memory");
                        __builtin_amdgcn_s_barrier();
                        asm volatile("" ::: "memory");
                    }
                }
                wait_vmcnt<ACC ? NCH : 0>();
                __builtin_amdgcn_s_barrier();  // every fragment has been fetched
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_barrier();  // the tile has been staged
                asm volatile("" ::: "memory");
                // All of them are awaited, those of pieces that are not stored too: one left pending would be waited
                // for in the next tile's K loop, with everything else in flight.
#pragma unroll
                for (int u = 0; u < (ACC ? NCH : 1); u++) asm volatile("" : "+v"(old[u]));
                auto add = [&](int u, int row, int col, uint16_t *at) __attribute__((always_inline)) {
                    store16_write_through(at, fo_add8<Tag>(old[ACC ? u : 0], piece(row, col)));
                };
                if constexpr (MODE == MODE_RS)
                    each_mapped_piece(wave * 64 + lane, rs_map, p.ACC, std::false_type{}, add);
                else
                    each_piece(wave * 64 + lane, p.ACC, std::false_type{}, add);
            } else {
                wait_vmcnt<0>();  // nothing lands in the space the output is staged in
                __builtin_amdgcn_s_barrier();  // every fragment has been fetched
                asm volatile("" ::: "memory");
                if (ACC) {
                    __builtin_amdgcn_s_barrier();  // the tile has been staged
                    asm volatile("" ::: "memory");
                }
            }
            if constexpr (ACC) {
                if (MODE == MODE_RS && p.OWN) {
                    find_bases();
                    each_mapped_piece(wave * 64 + lane, rs_map, p.OWN, std::false_type{},
                                      [&](int, int row, int col, uint16_t *at) __attribute__((always_inline)) {
                        store16_write_through(at, piece(row, col));
                    }, (int)(bits >> TileArgs::RANK & 255) * ((p.M >> log_ranks) * RTN), (p.M >> log_ranks) * RTN);
                }
            }
        } else {
            fo_float4v acc[FM][FN];
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++) acc[i][j] = fo_float4v{0.f, 0.f, 0.f, 0.f};
            // Fragment addressing: lane l supplies row l & 15, k-chunk l >> 4 of a 16x32 block.  The operand of which a
            // wavefront holds more fragments is the long one: a k-step goes through it fragment by fragment (a "row"),
            // each with all fragments of the short one.
            constexpr bool LONG_B = FN > FM;
            constexpr int FL = LONG_B ? FN : FM, FS = LONG_B ? FM : FN;
            constexpr unsigned L_BLK = LONG_B ? B_BLK : A_BLK, S_BLK = LONG_B ? A_BLK : B_BLK;
            const int frow = lane & 15, fk = lane >> 4, key = (frow >> 1) & 7;
            const unsigned la = lds0 + (unsigned)((wm * WTM + frow) * 8 + (fk ^ key)) * 16;
            const unsigned lb = lds0 + KB * A_BLK + (unsigned)((wn * WTN + frow) * 8 + (fk ^ key)) * 16;
            const unsigned l_lds = LONG_B ? lb : la, s_lds = LONG_B ? la : lb;
            typedef const __attribute__((address_space(3))) frag *lds_frag_t;
            typedef tile_step<FL, FS, KK> T;
            constexpr int NS = T::NS, NB = T::NB, NF = T::NF, NM = T::NM;
            // (Up to 224 registers in all, and a consumer's wavefront still fits on the SIMD beside this kernel's two.)
            constexpr bool AHEAD = (SHIFT || FL < 4) && (2 * KK * (FL + FS) + FL * FS) * 4 <= 192;
            static_assert(AHEAD || (FL >= 4 && FS >= 2), "a strip in front of the last one fetches the last short fragment");
            constexpr int LSETS = AHEAD ? 2 : NS % 2 ? NS : 2;  // AHEAD: one per stage, else one per strip
            frag lf[LSETS][AHEAD ? FL : 2][KK], sf[AHEAD ? 2 : 1][FS][KK];
            // Shifted: column chunk c of a 64-column block lies c + shift chunks behind the start of the row's line, that is
            // in the following block from 8 on (all rows of a lane have the same shift: they are 16 apart).
            int l_shift = 0, s_shift = 0;
            if (SHIFT) {
                const int a_shift = row_shift(p.A + (size_t)m0 * p.K, p.K, frow), b_shift = row_shift(p.B + (size_t)n0 * p.K, p.K, frow);
                l_shift = fk + (LONG_B ? b_shift : a_shift);
                s_shift = fk + (LONG_B ? a_shift : b_shift);
            }
            auto block_of = [&](int kk, unsigned slot, unsigned next, unsigned blk, int shift) __attribute__((always_inline)) {
                const unsigned here = slot + (kk >> 1) * blk, behind = (kk >> 1) + 1 < KB ? here + blk : next;
                return SHIFT && shift + (kk & 1) * 4 >= 8 ? behind : here;
            };
            // Fragment i, k-step kk of the stage in `slot` (and, shifted, of the one in `next`).
            auto fetch_l = [&](frag &to, int i, int kk, unsigned slot, unsigned next) __attribute__((always_inline)) {
                const unsigned at = (l_lds + block_of(kk, slot, next, L_BLK, l_shift)) ^ ((kk & 1) * 64);
                to = ((lds_frag_t)(uintptr_t)at)[i * 128];
            };
            auto fetch_s = [&](frag &to, int j, int kk, unsigned slot, unsigned next) __attribute__((always_inline)) {
                const unsigned at = (s_lds + block_of(kk, slot, next, S_BLK, s_shift)) ^ ((kk & 1) * 64);
                to = ((lds_frag_t)(uintptr_t)at)[j * 128];
            };
            auto behind_slot = [&](unsigned slot) __attribute__((always_inline)) { return slot + STAGE == S * STAGE ? 0 : slot + STAGE; };
            auto meet = [&]() __attribute__((always_inline)) {
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wavefront's fetches from the slot have returned
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            };
            auto mul = [&](frag l, frag q, typename T::block b) __attribute__((always_inline)) {
                if constexpr (LONG_B)
                    acc[b.j][b.i] = X::go(l, q, acc[b.j][b.i]);
                else
                    acc[b.i][b.j] = X::go(q, l, acc[b.i][b.j]);
            };
            // AHEAD: fetch number `nth` of a stage into a set.
            auto fetch_nth = [&](auto nth, auto set_c, unsigned slot, unsigned next) __attribute__((always_inline)) {
                constexpr typename T::fetch f = T::fetches().nth[decltype(nth)::value];
                constexpr int set = decltype(set_c)::value;
                if constexpr (f.is_long)
                    fetch_l(lf[set][AHEAD ? f.at : 0][f.kk], f.at, f.kk, slot, next);
                else
                    fetch_s(sf[AHEAD ? set : 0][f.at][f.kk], f.at, f.kk, slot, next);
            };
            // The step on set SET: the first half of its MFMAs, the meeting, the rest with the next stage's fetches.
            // (Met at the start, a stage that arrives late holds up the MFMAs of two stages.)
            auto step_ahead = [&](auto set_c, unsigned next, unsigned after) __attribute__((always_inline)) {
                constexpr int SET = decltype(set_c)::value, MEET = NB / 2 * KK, SPAN = NB == 1 ? NM : (NM - MEET) * 3 / 4;
                static_for<NM>([&](auto mfma) __attribute__((always_inline)) {
                    constexpr int m = decltype(mfma)::value;
                    constexpr typename T::block b = T::block_at(m / KK);
                    if constexpr (m == MEET) meet();
                    mul(lf[SET][AHEAD ? b.i : 0][m % KK], sf[AHEAD ? SET : 0][b.j][m % KK], b);
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (m >= MEET) {
                        constexpr int first = T::first_at(m - MEET, NF, SPAN), last = T::first_at(m - MEET + 1, NF, SPAN);
                        static_for<last - first>([&](auto t) __attribute__((always_inline)) {
                            fetch_nth(std::integral_constant<int, first + decltype(t)::value>{}, std::integral_constant<int, 1 - SET>{}, next, after);
                        });
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
            };
            // The step in strips.  The last strip's long fragments are the last ones fetched from the slot; with four k-steps
            // half of that strip is enough to fetch behind, and the later a stage is asked for, the less often it is late.
            auto step_strips = [&](unsigned slot, unsigned next, unsigned after) __attribute__((always_inline)) {
                constexpr int LEAD = T::LEAD_B * KK, PER = 2 * FS * KK, MEET = KK > 2 ? PER / 2 : 0, SPAN = KK > 2 ? PER * 3 / 8 : 2 * KK;
                static_for<NM>([&](auto mfma) __attribute__((always_inline)) {
                    constexpr int m = decltype(mfma)::value;
                    constexpr typename T::block b = T::block_at(m / KK);
                    constexpr int strip = m < LEAD ? 0 : (m - LEAD) / PER + FL % 2, w = m < LEAD ? m : (m - LEAD) % PER;
                    constexpr int len = m < LEAD ? LEAD : PER;
                    if constexpr (strip == NS - 1 && w == MEET) meet();
                    mul(lf[strip % LSETS][AHEAD ? 0 : FL % 2 ? (b.i + 1) % 2 * (b.i > 0) : b.i % 2][m % KK], sf[0][b.j][m % KK], b);
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (strip < NS - 1) {
                        // the next strip's long fragments; in front of them, in the first strip, the last short one
                        constexpr int ns = strip == 0 ? KK : 0, n = ns + 2 * KK, span = strip == NS - 2 ? len / 2 : len * 3 / 4;
                        constexpr int first = T::first_at(w, n, span), last = T::first_at(w + 1, n, span);
                        static_for<last - first>([&](auto nth) __attribute__((always_inline)) {
                            constexpr int t = first + decltype(nth)::value, h = (t - ns) / KK, kk = t % KK;
                            if constexpr (t < ns)
                                fetch_s(sf[0][FS - 1][kk], FS - 1, kk, slot, next);
                            else
                                fetch_l(lf[(strip + 1) % LSETS][h][kk], 2 * (strip + 1) - FL % 2 + h, kk, slot, next);
                        });
                    } else {
                        // the next stage's: long fragments at once, a short one behind its last MFMA
                        static_for<(2 - FL % 2) * KK>([&](auto nth) __attribute__((always_inline)) {
                            constexpr int t = decltype(nth)::value;
                            if constexpr (w == MEET + t * SPAN / (2 * KK)) fetch_l(lf[0][t / KK][t % KK], t / KK, t % KK, next, after);
                        });
                        static_for<(FS - 1) * KK>([&](auto nth) __attribute__((always_inline)) {
                            constexpr int t = decltype(nth)::value, freed = (t / KK + 1) * 2 * KK - 1;
                            if constexpr (w == (freed > MEET ? freed : MEET) + t % KK * SPAN / (2 * KK)) fetch_s(sf[0][t / KK][t % KK], t / KK, t % KK, next, after);
                        });
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
            };
            __builtin_amdgcn_s_setprio(2);
            // MAPPED: lane e of the computing wavefronts' 256 finds where row e, or (two reorder tiles side by side) row e % TM
            // of one of them, goes.  The entry of the row map and the group sizes are asked for while the first stage is on its
            // way, and used behind the first step: they lie two round trips to memory behind the reorder table, and awaited in
            // front of the first barrier they held up the first step of every tile (whole passes, us: 2048x4096x2048 over eight ranks
            // 34.7 -> 33.3, 1152x5120x1720 with an accumulator 35.0 -> 33.9, 3456x2176x680 22.9 -> 21.3).  The barrier of the second
            // step publishes the maps; with too few steps for the loaders to wait for that, they are found in front of the first.
            const int e = wave * 64 + lane;
            const bool mapped_later = MAPPED && KT > S;
            int entry = 0, size0 = 0;
            const bool second_e = two_n ? e >= TM : e >= split_m;
            if (MAPPED) {
                const int row = two_n && e >= TM ? e - TM : e, r = second_e ? r1 : r0;
                if (e < (two_n ? 2 * TM : TM))
                    entry = p.RE[(r / rLDN << bm_shift) + (second_e && two_m ? -split_m : m0 & ((1 << bm_shift) - 1)) + row];
                if (MODE == MODE_RS && lane < p.G) size0 = p.cseg[lane];
            }
            auto write_maps = [&]() __attribute__((always_inline)) {
                int first0 = 0, count0 = 0, first1 = 0, count1 = 0;  // MODE_RS: the groups' slots
                if (MODE == MODE_RS) {
                    find_group_range(p.cseg, p.G, r0, lane, size0, &first0, &count0);
                    first1 = first0;
                    count1 = count0;
                    if (r1 != r0) find_group_range(p.cseg, p.G, r1, lane, size0, &first1, &count1);
                }
                if (e < (two_n ? 2 * TM : TM)) {
                    row_map[e] = entry;
                    if (MODE == MODE_RS)
                        rs_map[e] = rs_row(p.cseg, p.G, 1 << bm_shift, ranks, (p.M >> log_ranks) * RTN, entry, (second_e ? first1 : first0) << bm_shift,
                                           (second_e ? count1 : count0) << bm_shift);
                }
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): written when the next barrier is passed
            };
            if (MAPPED && !mapped_later) write_maps();
            if (signalling && wave == 0) {
                g0 = find_group(p.cseg, p.G, r0, lane);
                g1 = r1 != r0 ? find_group(p.cseg, p.G, r1, lane) : g0;
            }
            unsigned slot = 0;
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            // Behind the last stage, zeros never used are fetched.
            if constexpr (AHEAD) {
                static_for<NF>([&](auto t) __attribute__((always_inline)) { fetch_nth(t, std::integral_constant<int, 0>{}, 0, STAGE); });
                for (int kt = 0;;) {
                    unsigned next = behind_slot(slot);
                    step_ahead(std::integral_constant<int, 0>{}, next, behind_slot(next));
                    if (++kt == KT) break;
                    if (mapped_later && kt == 1) write_maps();
                    slot = behind_slot(next);
                    step_ahead(std::integral_constant<int, 1>{}, slot, behind_slot(slot));
                    if (++kt == KT) break;
                }
            } else {
#pragma unroll
                for (int t = 0; t < (2 - FL % 2) * KK; t++) fetch_l(lf[0][t / KK][t % KK], t / KK, t % KK, 0, STAGE);
#pragma unroll
                for (int t = 0; t < (FS - 1) * KK; t++) fetch_s(sf[0][t / KK][t % KK], t / KK, t % KK, 0, STAGE);
                for (int kt = 0; kt < KT; kt++) {
                    const unsigned next = behind_slot(slot), after = behind_slot(next);
                    step_strips(slot, next, after);
                    if (mapped_later && kt == 0) write_maps();
                    slot = next;
                }
            }
            // To the compiler these two loads may still be on their way behind the loop (it does not know that one of its steps, or the
            // call in front of it, has used them), and where it takes their registers for something else in the epilogue it waits, with
            // every piece, for the stores of the one before: 2048x4096x2048 over eight ranks 32.5 us or 35.4, by the registers it chose.
            if (MAPPED) asm volatile("" : "+v"(entry), "+v"(size0));
            __builtin_amdgcn_s_waitcnt(0xC07F);
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            // ---- epilogue: accumulators -> 16 bit -> LDS -> 16-byte pieces of output rows.  (The thread id is laundered
            // so that this addressing is computed here instead of resting in registers across the K loop.)
            int el = lane;
            asm volatile("" : "+v"(el));
            const int erow = el & 15, ek = el >> 4;  // accumulator block: row erow, columns 4*ek .. 4*ek+3
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++) {
                    fo_u32x2 v;
                    v.x = E::pack(acc[i][j][0], acc[i][j][1]);
                    v.y = E::pack(acc[i][j][2], acc[i][j][3]);
                    *reinterpret_cast<fo_u32x2 *>(stage + (wm * WTM + i * 16 + erow) * PITCH + wn * WTN + j * 16 + ek * 4) = v;
                }
            if constexpr (ACC) {
                find_bases();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_waitcnt(0xC07F);
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                auto put = [&](int, int row, int col, uint16_t *at) __attribute__((always_inline)) {
                    store16_write_through(at, piece(row, col));
                };
                if constexpr (MODE == MODE_RS)
                    each_mapped_piece(wave * 64 + lane, row_map, p.C, std::false_type{}, put);
                else
                    each_piece(wave * 64 + lane, p.C, std::false_type{}, put);
            }
        }
        if constexpr (!ACC) {
            find_bases();
            __syncthreads();
            auto put = [&](int, int row, int col, uint16_t *at) __attribute__((always_inline)) {
                store16_write_through(at, piece(row, col));
            };
            if constexpr (MODE == MODE_SCATTER)
                each_mapped_piece(tid, row_map, p.C, std::false_type{}, put);
            else
                each_piece(tid, p.C, std::false_type{}, put);
        }
        if (signalling) {
            // Whole reorder tiles only (the launcher sees to it): every wavefront's write-through stores are
            // acknowledged, the barrier collects the workgroup, then the counters move (the reference has no fence
            // here, src/overlap/gemm_with_signal.h:337-351).
            __builtin_amdgcn_s_waitcnt(0);
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            const bool first_counts = skip_m < split_m && skip_n < split_n;
            if (wave_id == NL && ((lane == 0 && first_counts) || (lane == 1 && (two_m || two_n)))) {
                const int g = lane ? g1 : g0, r = lane ? r1 : r0;
                __hip_atomic_fetch_add(p.MM + g, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (bits & TileArgs::MONITOR) {
                    int o = __hip_atomic_fetch_add(p.MM + (RTN - 1), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(p.MM + RTN + r, o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
        tile += args.stride;
        settle();
        if (tile < count) {
            __syncthreads();  // the staged tile has been read by everyone
            if (loader) begin();
        }
    }
}

}  // namespace fo_gemm_dev
