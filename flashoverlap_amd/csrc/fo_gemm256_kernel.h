// The 256x256 workgroup tile of the gfx950 MFMA GEMM (plain, signal and scatter
// epilogues; same arguments, raster and epilogue semantics as fo_gemm_tile_kernel.h,
// whose reference citations hold here too:
// src/overlap/gemm_with_signal.h:236-256, :291-361, src/overlap/gemm_scatter.cu:15-98).
//
// Four wavefronts, one per SIMD, each computing 128x128 of the tile with
// v_mfma_f32_16x16x32_{f16,bf16}: 64 accumulator blocks = all 256 accumulation
// registers of a lane, operand fragments in about 110 architectural registers.
// One wavefront per SIMD issues its instructions strictly in order, so whatever
// is not an MFMA has to leave in an MFMA's shadow: the K step is written as 128
// MFMAs with at most two other vector-memory or LDS instructions behind each
// (a fragment fetch, or the M0 update + load of an operand block), and a burst
// of such instructions anywhere shows up as idle matrix pipe.
//
// Operands travel HBM/L2 -> LDS directly (buffer_load_dwordx4 ... lds, 1 KiB per
// wavefront instruction) into two slots of 64 KiB (BK = 64: 256 rows of A and
// 256 of B, 128 bytes each, the 16-byte chunks XOR-swizzled by the choice of the
// global chunk each lane fetches, as in fo_gemm_tile_kernel.h).  The buffer
// descriptor covers the tile's rows only, and the chunks of a last, partial K
// step that lie beyond K are requested out of its range: the hardware writes
// zeros for them, nothing outside A or B is ever addressed.
//
// A K step is four strips, each two A blocks x eight B blocks x two k-steps, and
// each strip four rows of eight MFMAs.  The order inside a strip is chosen for
// energy, because large products run at this part's power limit: both k-steps of
// an accumulator block follow one another (the sum then stays in the matrix
// pipe's own path instead of going through the register file), and from one
// block to the next only one of the two operands changes.  MFMAs alone, random
// operands, at the power limit: 8.60 ns per MFMA with the k-steps 64 MFMAs apart
// and one A fragment x eight B fragments in a row, 8.14 in this order (bf16 8.05
// -> 7.74); 7.94 with four k-steps in a chain and 7.66 with eight, for which LDS
// and registers do not hold the operands.  This kernel: 8192^3 766 -> 749 us,
// 8192x4096x4096 205.5 -> 199.2, 4096x4096x512 20.7 -> 20.0, the same bits.  (With
// the two A blocks in the same order for every B block, so that A changes each
// time, 761.)
//
// Two meetings of the workgroup per K step:
//   FREE (behind row 9): every wavefront has fetched its last fragment of the
//     step's slot (B is complete by row 1, a strip's A fragments are fetched in
//     the strip before it, the last ones in row 8), so the slot may be refilled.
//     The sixteen loads of the stage two steps ahead follow, two per row in rows
//     10-12, then one per row until row 6 of the next step (two in row 13 as well:
//     8192x4096x4096 200.4 us; that row has six fragment fetches).
//   PUB (behind row 12): the other slot's loads, requested one step earlier,
//     have landed (vmcnt) in every wavefront; rows 13-15 fetch the next step's
//     first A fragments from it and the B fragments, each into the registers of the
//     block that the last strip has just finished with; the last of them follow in
//     rows 0 and 1.
// With one meeting for both, a stage's loads would have to leave within a few
// rows (the load path of a CU delivers a stage in about half a K step, and a
// wavefront that presents loads faster than they drain stalls with its MFMAs
// behind them) or land within a few rows.  The loader runs on across tile
// boundaries (the last two steps of a tile request the next tile's first two
// stages), so only the epilogue itself separates two tiles' MFMAs.
//
// Epilogue: accumulators -> 16-bit -> LDS strip of 16 rows per wavefront (behind
// the two slots) -> 16-byte stores of contiguous output-row pieces.  A tile's
// completion signal is sent from the next tile's first PUB meeting: its wait
// covers loads requested behind the tile's stores, hence the stores (vmcnt
// retires a wavefront's vector memory instructions in issue order on
// gfx9-family parts), in every wavefront, and the meeting's barrier lies between
// that wait and the counter update.
#pragma once

#include "fo_gemm_common.h"

namespace fo_gemm_dev {

// The MFMAs of this kernel: accumulator in the accumulation registers, tied to the destination
// (see fo_elem::mfma for why they are assembly); `go_load` carries a direct-to-LDS load in the
// MFMA's shadow: the M0 update in front of the MFMA, which also separates it from its use, the
// load behind it.  (Two wait states, where a scalar out of a vector lane needs five: see dma_buf16.  None of
// the K loop's comes from there, which a test checks in the built code.)
template <typename Tag> struct fo_mfma256;
#define FO_MFMA256(TAG_, OPC_)                                                                                        \
    template <> struct fo_mfma256<TAG_> {                                                                             \
        static __device__ __forceinline__ void go(fo_u32x4 a, fo_u32x4 b, fo_float4v &c) {                            \
            asm("v_mfma_f32_16x16x32_" OPC_ " %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));                            \
        }                                                                                                             \
        template <unsigned LDS_OFF>                                                                                   \
        static __device__ __forceinline__ void go_load(fo_u32x4 a, fo_u32x4 b, fo_float4v &c, unsigned lds_base,      \
                                                       fo_srd_t srd, unsigned voff, unsigned soff) {                  \
            asm volatile("s_add_u32 m0, %4, %5\n\tv_mfma_f32_16x16x32_" OPC_                                          \
                         " %0, %1, %2, %0\n\tbuffer_load_dwordx4 %3, %6, %7 offen lds"                                \
                         : "+a"(c)                                                                                    \
                         : "v"(a), "v"(b), "v"(voff), "s"(lds_base), "n"(LDS_OFF), "s"(srd), "s"(soff)                \
                         : "memory", "scc");                                                                          \
        }                                                                                                             \
    };
FO_MFMA256(fo_f16_tag, "f16")
FO_MFMA256(fo_bf16_tag, "bf16")
#undef FO_MFMA256

// Direct-to-LDS loads per wavefront in the rows behind FREE (rows 10, 11, ... wrapping into the next step).
constexpr int kLoadRows256[] = {2, 2, 2, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1};
constexpr int kLoadSpan256 = sizeof(kLoadRows256) / sizeof(int);
constexpr int loads_in_row256(int d) { return d >= 0 && d < kLoadSpan256 ? kLoadRows256[d] : 0; }
constexpr int loads_before_row256(int d) {
    int s = 0;
    for (int e = 0; e < d && e < kLoadSpan256; e++) s += kLoadRows256[e];
    return s;
}

// The LDS fetches of each row of a K step in issue order: A or B block `block`, k-step kk, from the step's slot or the next one's.
struct fetch256 {
    bool b;
    int block, kk;
    bool next;
};
struct row_fetches256 {
    int n;
    fetch256 at[6];
};
constexpr row_fetches256 fetches_of_row256(int r) {
    row_fetches256 f{};
    auto a = [&](int block, int kk, bool next = false) { f.at[f.n++] = {false, block, kk, next}; };
    auto b = [&](int block, bool next = false) {
        f.at[f.n++] = {true, block, 0, next};
        f.at[f.n++] = {true, block, 1, next};
    };
    if (r == 0) { b(5); b(6); }
    if (r == 1) { b(7); a(2, 0); a(2, 1); }
    if (r == 2) { a(3, 0); a(3, 1); }
    if (r == 4) { a(4, 0); a(4, 1); }
    if (r == 5) { a(5, 0); a(5, 1); }
    if (r == 8) { a(6, 0); a(6, 1); a(7, 0); a(7, 1); }
    if (r == 13) { a(0, 0, true); a(0, 1, true); b(0, true); a(1, 0, true); a(1, 1, true); }
    if (r == 14) { b(1, true); b(2, true); }
    if (r == 15) { b(3, true); b(4, true); }
    return f;
}

// The accumulator's values that a step requests (MODE_ACC): eight, in rows that carry no operand load, behind this step's
// last load of the next stage (row 6) and in front of FREE.  takes_before256: those in front of MFMA m of row r.
constexpr int kTakes256 = 8, kTakeAt256[kTakes256] = {7 * 8 + 1, 7 * 8 + 3, 7 * 8 + 5, 8 * 8 + 2, 8 * 8 + 6, 9 * 8 + 1, 9 * 8 + 3, 9 * 8 + 5};
constexpr int takes_before256(int r, int m) {
    int n = 0;
    while (n < kTakes256 && kTakeAt256[n] < r * 8 + m) n++;
    return n;
}

constexpr int kTakeFromSteps256 = 5;  // K steps of a tile from which on they are: four take, and the loop behind them has one at least

constexpr int kSmem256 = 2 * 65536 + 4 * 16 * (128 + 8) * 2;  // two slots + four strips of 16 padded rows

template <typename Tag, int MODE>
__global__ __launch_bounds__(256) void fo_gemm256_kernel(uint64_t A_, uint64_t B_, uint64_t K_count, uint64_t grid_m_n, uint64_t panel_bits,
                                                         uint64_t by_panel_rows, uint64_t by_last_stride, GemmArgs) {
    Front256 f;
    f.A = (const uint16_t *)(uintptr_t)A_;
    f.B = (const uint16_t *)(uintptr_t)B_;
    f.K = (int)K_count;
    f.count = (int)(K_count >> 32);
    f.grid_m = (int)grid_m_n;
    f.grid_n = (int)(grid_m_n >> 32);
    f.panel = (int)panel_bits;
    f.bits = (uint32_t)(panel_bits >> 32);
    f.by_panel.mul = (uint32_t)by_panel_rows;
    f.by_rows.mul = (uint32_t)(by_panel_rows >> 32);
    f.by_last_rows.mul = (uint32_t)by_last_stride;
    const int stride = (int)(by_last_stride >> 32);  // workgroups of the launch
    typedef fo_elem<Tag> E;
    typedef fo_mfma256<Tag> X;
    constexpr bool SUMS = MODE == MODE_SIGNAL_SUM || MODE == MODE_SCATTER_SUM;
    constexpr bool ACC = MODE == MODE_ACC || MODE == MODE_RS, COUNTS = MODE == MODE_SIGNAL || MODE == MODE_SCATTER || SUMS;
    constexpr bool MAPPED = MODE == MODE_SCATTER || MODE == MODE_RS || MODE == MODE_SCATTER_SUM;
    constexpr bool TO_RANKS = MODE == MODE_RS || MODE == MODE_SCATTER_SUM;  // sums go where a reduce-scatter takes them
    constexpr int MT = 256, BK = 64, F = 8, ROWS = 16;
    constexpr int FREE = 9;   // row behind whose MFMAs the step's slot is given up
    constexpr int PUB = 12;   // row behind whose MFMAs the next step's slot is published
    constexpr unsigned SLOT_B = 65536, BPART_B = 32768, BLOCK_B = 2048, KSTEP_X = 64, CHUNK_B = 4096;
    constexpr int PITCH = 128 + 8, CPR = 16, RPP = 4;
    constexpr unsigned STRIP_B = 2 * SLOT_B;
    constexpr int NST = 32;                                      // stores per wavefront and tile
    constexpr int YOUNG = loads_before_row256(PUB - FREE);       // loads of a step already requested at its PUB meeting
    static_assert(loads_before_row256(kLoadSpan256) == 16, "a stage is sixteen loads per wavefront");
    static_assert(FREE + kLoadSpan256 - ROWS < FREE && PUB > FREE && PUB <= 13, "load rows lie between two FREE meetings");
    // YOUNG is exact: between a FREE meeting (row 9) and the PUB meeting of the same step (row 12) rows 10-12 issue
    // loads_in_row256(0..2) loads and nothing else that counts in vmcnt; a tile's stores and the loads of rows 0-6 of
    // its successor's first step are older than those.  Further vector-memory instructions in that stretch would
    // only make the PUB wait stricter.  The wait relies on vmcnt retiring loads and stores in issue order (one
    // counter for both on this part); a part with a counter of its own for stores needs a wait on that one as well.
    static_assert(YOUNG == loads_in_row256(0) + loads_in_row256(1) + loads_in_row256(2), "loads of rows 10-12");
    static_assert(NST + 16 + YOUNG < 64, "vmcnt range: a tile's stores and a stage's loads in flight together");
    static_assert(FREE + kLoadSpan256 >= ROWS, "the rest of a stage's loads leaves in the rows of the next step");

    extern __shared__ fo_u32x4 smem[];
    const unsigned smem_lds = (unsigned)(uintptr_t)FO_LDS_PTR(smem);
    typedef const __attribute__((address_space(3))) fo_u32x4 *lds16_t;

    // A consumer wavefront may share the SIMD (it fits beside this kernel's registers); this wavefront's
    // instructions go first, the consumer's take the issue cycles that are left.
    __builtin_amdgcn_s_setprio(3);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int ntiles = f.count;
    const int KT = (f.K + BK - 1) / BK;
    const bool ktail = (f.K % BK) != 0;

    // Fragment addressing as in fo_gemm_tile_kernel.h: lane l supplies row l & 15, k-chunk l >> 4 of a 16x32 block.
    const int frow = lane & 15, fk = lane >> 4;
    const int fkey = (frow >> 1) & 7;
    const unsigned la0 = smem_lds + (unsigned)((wm * 128 + frow) * 8 + (fk ^ fkey)) * 16;
    const unsigned lb0 = smem_lds + BPART_B + (unsigned)((wn * 128 + frow) * 8 + (fk ^ fkey)) * 16;
    const unsigned wa0 = smem_lds + (unsigned)(wave * 1024);  // wave-uniform; load c of a stage: + c * CHUNK_B (lane l: + 16 l by the hardware)

    // Loader: load c < 8 of a stage brings A rows (4c + wave) * 8 + lane / 8, load c >= 8 the same rows of B;
    // LDS slot `lane` of the 1 KiB block is (row lane / 8, physical chunk lane % 8), which receives logical chunk
    // phys ^ key(row).
    const int lrow = lane >> 3;
    const int lchunk = (lane & 7) ^ (((wave * 8 + lrow) >> 1) & 7);
    const unsigned a_off = (unsigned)((wave * 8 + lrow) * f.K * 2 + lchunk * 16);
    const bool tail_out = (KT - 1) * BK + lchunk * 8 >= f.K;  // this lane's chunk of the last K step lies beyond K
    const unsigned a_off_t = tail_out ? 0x80000000u : a_off;  // beyond every descriptor's range
    // The descriptors point at the stage's first column of the tile's first row and cover exactly the
    // tile's rows from there (the host checks that this fits 31 bits).
    const unsigned a_span = (unsigned)((255 * f.K + f.K) * 2);
    // Rows of A and of B are K elements apart (GemmArgs has no other stride), so the lane offsets, the span and the
    // row-block offsets of the eight loads per operand serve both.
    unsigned soff_a[8];
#pragma unroll
    for (int c = 0; c < 8; c++) {
        soff_a[c] = __builtin_amdgcn_readfirstlane((unsigned)(c * 32 * f.K * 2));
    }

    // M and N are multiples of 128, not of 256: where half a tile is left at the end of a dimension, the tile is moved
    // back by half its size, so that all of its operand rows exist; its first half there repeats the neighbour's
    // product and is not stored (half: bit 0 along M, bit 1 along N; never in a launch that counts, see plan_launch).
    int half = f.bits >> 3;
    asm volatile("" : "+s"(half));  // in a register from here on: loaded again inside the K loop, it would turn every wait for LDS data into a wait for everything
    // Coordinates of raster position t in halves of tiles, bits 0 and 1 of *repeated: which halves another tile
    // computes (the upper rows, the left columns).
    auto locate = [&](int t, int *pm_, int *pn_, int *repeated_) {
        int qm, qn;
        fo_tile_of(f, t, &qm, &qn);
        const int rep = __builtin_amdgcn_readfirstlane(half & ((qm == f.grid_m - 1 ? 1 : 0) | (qn == f.grid_n - 1 ? 2 : 0)));
        *pm_ = __builtin_amdgcn_readfirstlane(2 * qm - (rep & 1));
        *pn_ = __builtin_amdgcn_readfirstlane(2 * qn - (rep >> 1));
        *repeated_ = rep;
    };
    int pm, pn, repeated;  // the first tile's are found once, for the loader, the slots and the tile itself
    locate(blockIdx.x, &pm, &pn, &repeated);

    // Loader state: the stage being requested (it runs two K steps ahead of the MFMAs, across tiles).
    int ld_tile = blockIdx.x, ld_kt = 0;
    unsigned a_cur = (ktail && KT == 1) ? a_off_t : a_off;  // this stage's lane offsets, A and B alike
    fo_srd_t ra, rb;
    auto point_loader = [&](int pm_, int pn_) {
        ra = fo_make_srd(f.A + (size_t)pm_ * 128 * f.K, a_span);
        rb = fo_make_srd(f.B + (size_t)pn_ * 128 * f.K, a_span);
    };
    auto set_loader_tile = [&]() {
        if (ld_tile < ntiles) {
            int pm_, pn_, rep_;
            locate(ld_tile, &pm_, &pn_, &rep_);
            point_loader(pm_, pn_);
        } else {
            ra = fo_make_srd(f.A, 0);  // behind the last tile: every load is out of range, nothing is fetched
            rb = fo_make_srd(f.B, 0);
        }
    };
    auto advance_loader = [&]() {
        ld_kt++;
        if (ld_kt == KT) {
            ld_kt = 0;
            ld_tile += stride;
            set_loader_tile();
        } else {
            // the next K step of the same tile: 128 bytes further along the rows
            const uint64_t ab = ((uint64_t)ra.y << 32 | ra.x) + BK * 2, bb = ((uint64_t)rb.y << 32 | rb.x) + BK * 2;
            ra.x = __builtin_amdgcn_readfirstlane((unsigned)ab);
            ra.y = __builtin_amdgcn_readfirstlane((unsigned)(ab >> 32));
            rb.x = __builtin_amdgcn_readfirstlane((unsigned)bb);
            rb.y = __builtin_amdgcn_readfirstlane((unsigned)(bb >> 32));
            ra.z = __builtin_amdgcn_readfirstlane(ra.z >= BK * 2 ? ra.z - BK * 2 : 0);
            rb.z = __builtin_amdgcn_readfirstlane(rb.z >= BK * 2 ? rb.z - BK * 2 : 0);
        }
        if (ktail) {
            const bool t = ld_kt == KT - 1;
            a_cur = t ? a_off_t : a_off;
        }
    };
    // load c of the loader's stage into the slot at byte offset `slot` (pipeline fill)
    auto load_chunk = [&](int c, unsigned slot) {
        if (c < 8)
            dma_buf16(ra, a_cur, soff_a[c & 7], (wa0 ^ slot) + c * CHUNK_B);
        else
            dma_buf16(rb, a_cur, soff_a[c & 7], (wa0 ^ slot) + c * CHUNK_B);
    };
    // the same riding on an MFMA (K loop)
    auto mfma_load_chunk = [&](auto chunk, fo_u32x4 x, fo_u32x4 y, fo_float4v &cc, unsigned lds_base) __attribute__((always_inline)) {
        constexpr int c = decltype(chunk)::value;
        X::template go_load<c * CHUNK_B>(x, y, cc, lds_base, c < 8 ? ra : rb, a_cur, soff_a[c & 7]);
    };

    // ---- the first stage, in front of all that its addresses do not need.  A workgroup takes one or two tiles of a product that
    // fits the chip, so what stands in front of its first load counts: the arguments in memory, the slot table and the raster's
    // divisions were 513 instructions and 21 scalar loads and waits there in the signal epilogue, these are 172 and 4 (Front256
    // arrives in registers, its divisors come from the host).  Whole passes:
    // 4096x4096x512 with its normalisation 41.1 -> 40.2 us, 4096x4096x1024 with an accumulator 52.5 -> 51.5, over eight ranks 45.8 -> 44.4.
    point_loader(pm, pn);
#pragma unroll
    for (int c = 0; c < 16; c++) load_chunk(c, 0);
    typedef const __attribute__((address_space(4))) char *args_t;
    args_t rest = (args_t)__builtin_amdgcn_kernarg_segment_ptr() + kGemmArgsAt;
    asm volatile("" : "+s"(rest));  // the other arguments are read from here on
    const __attribute__((address_space(4))) GemmArgs &p = *(const __attribute__((address_space(4))) GemmArgs *)rest;
    // Those that the first tile's group sizes and slots need, in one round trip.
    int first_BM = 0, first_BN = 0, first_TN = 0, first_G = 0;
    const int32_t *first_RA = nullptr, *first_cseg = nullptr;
    if (MODE != MODE_PLAIN) {
        first_BM = p.BM; first_BN = p.BN; first_TN = p.TN; first_RA = p.RA;
        if (COUNTS || TO_RANKS) {
            first_G = p.G; first_cseg = p.cseg;
        }
        asm volatile("" : "+s"(first_BM), "+s"(first_BN), "+s"(first_TN), "+s"(first_RA), "+s"(first_G), "+s"(first_cseg));
    }

    // ---- signalling state (signal and scatter epilogues)
    const int bm_shift = p.BM == 256 ? 8 : 7, bn_shift = p.BN == 256 ? 8 : 7;
    const int log_sub_n = 8 - bn_shift, sub_n = 1 << log_sub_n, nsub = sub_n << (8 - bm_shift);  // reorder tiles per macro tile
    typedef const __attribute__((address_space(4))) int32_t *cptr_t;
    const cptr_t RAc = (cptr_t)(uintptr_t)p.RA;
    constexpr int NPRE = kPrefixRegs / 64;
    int pre[NPRE];
#pragma unroll
    for (int q = 0; q < NPRE; q++) pre[q] = 0;
    const bool reg_search = p.G <= kPrefixRegs;
    const bool signalling = COUNTS && !p.quiet;
    const bool reorder = MODE == MODE_ACC ? p.RA != nullptr : COUNTS || MODE == MODE_RS || MODE == MODE_REORDER;
    const bool groups = signalling || TO_RANKS;  // group sizes are needed
    // The group sizes are requested between the pipeline fill's two stages and summed behind it (a round trip to memory and
    // some two dozen dependent cross-lane steps otherwise stand between the kernel's start and its first operand
    // load).  The requests are assembly: their registers are read only behind the fill's wait for loads that were
    // requested after them, and the compiler, which knows nothing of the fill's loads, would otherwise wait for
    // every one of those as well.  Lanes beyond G ask for element 0.
    int cs_raw[NPRE];
    if (groups && reg_search) {
#pragma unroll
        for (int q = 0; q < NPRE; q++) {
            const int32_t *src = first_cseg + (q * 64 + lane < first_G ? q * 64 + lane : 0);
            asm volatile("global_load_dword %0, %1, off" : "=v"(cs_raw[q]) : "v"(src) : "memory");
        }
    }
    // The first tile's storage slots, lane s the one of its reorder tile s: one load, in the same place and manner.  As scalar loads
    // they were four round trips, one behind the other (there are no scalar registers to hold them side by side), and the fill took
    // 3 us, of which the operands need 1.5.  Whole passes, us: layers 4096x4096x1024 39.7 -> 39.2, over eight ranks 44.7 -> 44.0.  Lanes beyond
    // the tile's last slot ask for that one again, without a table all of them for the first word of A.
    int slots_raw = 0;
    if (MODE != MODE_PLAIN) {
        const int q = lane < nsub ? lane : nsub - 1;
        const int at = ((pm >> (first_BM >> 8)) + (q >> log_sub_n)) * first_TN + (pn >> (first_BN >> 8)) + (q & (sub_n - 1));
        const int32_t *src = reorder ? first_RA + at : reinterpret_cast<const int32_t *>(f.A);
        asm volatile("global_load_dword %0, %1, off" : "=v"(slots_raw) : "v"(src) : "memory");
    }
    auto sum_groups = [&]() {
        if (groups && reg_search) {
            int base = 0;
#pragma unroll
            for (int q = 0; q < NPRE; q++) {
                if (q * 64 < p.G) {  // wave-uniform
                    int v = q * 64 + lane < p.G ? cs_raw[q] : 0;
#pragma unroll
                    for (int d = 1; d < 64; d <<= 1) {
                        int o = __shfl_up(v, d, 64);
                        if (lane >= d) v += o;
                    }
                    pre[q] = v + base;
                    base = __shfl(pre[q], 63, 64);
                }
            }
        }
    };
    auto group_of = [&](int r) {
        if (reg_search) {
#pragma unroll
            for (int q = 0; q < NPRE; q++) {
                unsigned long long hit = __ballot(q * 64 + lane < p.G && pre[q] > r);
                if (hit) return q * 64 + (int)__builtin_ctzll(hit);
            }
            return p.G - 1;
        }
        return find_group(p.cseg, p.G, r, lane);
    };
    // Slots of the group that holds slot r (MODE_RS).
    auto group_range = [&](int r, int *first, int *count) __attribute__((always_inline)) {
        if (reg_search) {
            const int g = group_of(r);
            int end = 0, begin = 0;
#pragma unroll
            for (int q = 0; q < NPRE; q++) {
                if (g >> 6 == q) end = __builtin_amdgcn_readlane(pre[q], g & 63);
                if (g > 0 && (g - 1) >> 6 == q) begin = __builtin_amdgcn_readlane(pre[q], (g - 1) & 63);
            }
            *first = begin;
            *count = end - begin;
        } else {
            find_group_range(p.cseg, p.G, r, lane, lane < p.G ? p.cseg[lane] : 0, first, count);
        }
    };
    // Wavefront 0 announces a macro tile's reorder tiles: lane s < nsub holds the storage slot r and the group g of
    // reorder tile s (one register each; as scalars, slots and groups of this tile and of the one whose signal is
    // still owed took twenty scalar registers through the K loop and the kernel spilled 145 of them).  Callers
    // guarantee that every wavefront's write-through stores of those tiles are acknowledged (vmcnt) and that a
    // workgroup barrier lies between that wait and this call, so the atomic itself is relaxed.
    // Reorder tiles of one group are counted with one atomic: all resident workgroups finish a tile at about the
    // same time and bump the same few counters, and atomics on one address complete one after the other, some 25 ns
    // apart (512 tiles of 256x256 in 128x128 reorder tiles, 8 groups: 7 us per launch with one atomic per tile).
    auto announce = [&](int r, int g) {
        int count = 0;      // tiles of this lane's group from this lane on
        bool first = true;  // no earlier tile of this group
#pragma unroll
        for (int q = 0; q < kMaxSub; q++) {
            const int gq = __builtin_amdgcn_readlane(g, q);
            if (q < nsub && gq == g) {
                if (q < lane) first = false;
                if (q >= lane) count++;
            }
        }
        if (lane < nsub && g >= 0) {
            if (first) __hip_atomic_fetch_add(p.MM + g, count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (p.monitor) {
                int o = __hip_atomic_fetch_add(p.MM + (p.TN - 1), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(p.MM + p.TN + r, o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    };
    // Storage slots of a further tile's reorder tiles (scalar loads).  They are requested one tile ahead, in front of the previous
    // tile's epilogue, and awaited in it: the round trip to memory then costs nothing, and no scalar load is pending at the K loop's head,
    // where it would turn every wait for LDS data into a wait for everything (scalar loads return out of order).
    int rs_next[kMaxSub] = {0, 0, 0, 0};
    auto request_slots = [&](int pm_, int pn_) {
        if (reorder) {
            const int tm_ = pm_ >> (p.BM >> 8), tn_ = pn_ >> (p.BN >> 8);  // in reorder tiles (BM, BN: 128 or 256)
#pragma unroll
            for (int s = 0; s < kMaxSub; s++)
                if (s < nsub) rs_next[s] = RAc[(tm_ + (s >> log_sub_n)) * p.TN + tn_ + (s & (sub_n - 1))];
        }
    };
    // The slots that request_slots brought, as the rest of the kernel uses them: this wavefront's own reorder tile as a
    // scalar, all of them in lanes 0 .. nsub-1 of one register.
    const int my_sub = __builtin_amdgcn_readfirstlane(((wm * 128 >> bm_shift) << log_sub_n) + (wn * 128 >> bn_shift));
    int r_mine = 0, v_rs = 0;
    auto take_slots = [&]() {
        if (reorder) {
#pragma unroll
            for (int s = 0; s < kMaxSub; s++) {
                int rr = __builtin_amdgcn_readfirstlane(rs_next[s]);
                asm volatile("" : "+s"(rr));  // the scalar loads complete here
                if (s == my_sub) r_mine = rr;
                v_rs = lane == s ? rr : v_rs;
            }
        }
    };
    int v_prev_r = 0, v_prev_g = 0;  // slots and groups (per lane) of the tile whose signal is still owed
    int owed = 0;                    // PUB meetings until that signal may be sent

    fo_float4v acc[F][F];
    fo_u32x4 af[2][2][2], bf[2][F];
    auto load_a = [&](int buf, unsigned base, int i, int kk) {
        af[buf][i % 2][kk] = *reinterpret_cast<lds16_t>(base + i * BLOCK_B);
    };
    auto load_b = [&](unsigned base, int j, int kk) {
        bf[kk][j] = *reinterpret_cast<lds16_t>(base + j * BLOCK_B);
    };

    // ---- pipeline fill: stage 0 -> slot 0 (above), stage 1 -> slot 1; the loader then stands at stage 1
    advance_loader();
#pragma unroll
    for (int c = 0; c < 16; c++) load_chunk(c, SLOT_B);
    wait_vmcnt<16>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int q = 0; q < 4; q++) load_a(0, la0 ^ (q % 2 * KSTEP_X), q / 2, q % 2);
#pragma unroll
    for (int q = 0; q < 10; q++) load_b(lb0 ^ (q % 2 * KSTEP_X), q / 2, q % 2);
    // Slots and group sizes, requested between the two stages, have arrived too (vmcnt retires in issue order).  Pinned here: to the
    // compiler they were in their registers from the request on, and nothing else keeps a use of them behind the wait.
    if (MODE != MODE_PLAIN) asm volatile("" : "+v"(slots_raw));
    if (groups && reg_search) {
#pragma unroll
        for (int q = 0; q < NPRE; q++) asm volatile("" : "+v"(cs_raw[q]));
    }
    sum_groups();

    int tile = blockIdx.x;
    unsigned slot_b = 0;  // byte offset of the slot the next K step reads
    for (;;) {
        // Later tiles: taken inside the previous tile's epilogue.  (In front of the loop, without the test, slots_raw would not live through
        // it, but the accumulating epilogue's K loop is laid out otherwise and slower: 4096x8192x8192 421.7 -> 423.5 us.)
        if (MODE != MODE_PLAIN && reorder && tile == (int)blockIdx.x) {
            v_rs = slots_raw;
            r_mine = __builtin_amdgcn_readlane(slots_raw, my_sub);
        }
        // Scatter: the row map entries of the wavefront's 128 rows, two per lane (lane l: rows l and 64 + l), are
        // requested here and rest in two registers through the K loop; the epilogue hands them to the lanes that
        // store each row.  Requested in the epilogue they cost every tile a round trip to memory with nothing to hide it.
        int32_t re_lo = 0, re_hi = 0;
        if (MAPPED) {
            const long trow = (long)(r_mine / p.rLDN) * p.BM + (wm * 128) % p.BM;
            re_lo = p.RE[trow + lane];
            re_hi = p.RE[trow + 64 + lane];
        }
#pragma unroll
        for (int i = 0; i < F; i++)
#pragma unroll
            for (int j = 0; j < F; j++)
#pragma unroll
                for (int v = 0; v < 4; v++) acc[i][j][v] = 0.f;
        if (MODE == MODE_ACC) {
            // All of them are written here: with two ways to the first MFMA the compiler would write each block's in front of
            // its own, inside the wait states that the assembly does not bring.
#pragma unroll
            for (int i = 0; i < F; i++)
#pragma unroll
                for (int j = 0; j < F; j++) asm volatile("" : "+a"(acc[i][j]));
        }
        fo_mfma_fence();

        // MODE_ACC: the accumulator's values of the wavefront's block, 32 pieces a lane: this wavefront owns the SIMD and has the
        // registers.  They are requested a quarter at a time in the tile's first four steps (a half that is not stored: with an
        // empty range), where the memory is idle, and read behind the last.  Loads return in order, so the place matters:
        // behind this step's last load of the next stage, whose wait then counts them as younger, and one K step in front of
        // the wait for the stage behind that.  Requested in the epilogue, with every CU at its end at the same time, they cost a
        // round trip and their bandwidth in front of the first store (whole passes, us, in the epilogue -> in the first steps:
        // 4096x4096x512 44.0 -> 41.6, 4096x4096x1024 55.9 -> 52.2, 4096x8192x264 85.7 -> 77.1, 3456x4352x3072 100.2 -> 97.3,
        // 8064x8064x4096 463.8 -> 455.7; 8192x8192x2048 by the serial call 276.5 -> 272.4).
        fo_u32x4 old[ACC ? NST : 1];
        // Not where rows are so long that the block's offsets leave a 31-bit range (half, bit 2).
        const bool early = MODE == MODE_ACC && KT >= kTakeFromSteps256 && !(half & 4);
        int take_row = 0, take_step = 0;
        unsigned take_lane = 0;
        __amdgpu_buffer_rsrc_t take_from;
        if (early) {
            const int ldp = reorder ? p.rLDN * p.BN : p.N;
            const long trow = !reorder ? (long)(pm + wm) * 128 : (long)(r_mine / p.rLDN) * p.BM + (wm * 128) % p.BM;
            const long tcol = !reorder ? (long)(pn + wn) * 128 : (long)(r_mine % p.rLDN) * p.BN + (wn * 128) % p.BN;
            const bool keep = !((repeated & 1) && wm == 0) && !((repeated & 2) && wn == 0);
            take_from = __builtin_amdgcn_make_buffer_rsrc((void *)(p.ACC + trow * ldp + tcol), 0, keep ? (unsigned)(127 * ldp + 128) * 2 : 0, 0x00027000);
            take_step = RPP * ldp * 2;
            take_lane = (unsigned)(lane / CPR * ldp + lane % CPR * 8) * 2;
        }
        auto take = [&](auto nth) __attribute__((always_inline)) {
            constexpr int k = decltype(nth)::value;
            old[ACC ? k : 0] = __builtin_bit_cast(fo_u32x4, __builtin_amdgcn_raw_buffer_load_b128(take_from, take_lane, take_row, 0));
            take_row += take_step;
            asm volatile("" ::: "memory");  // stays here: the step's waits count it
        };
        // One K step.  TAKES: the quarter of the accumulator's pieces that it requests (-1: none).
        auto k_step = [&](auto takes) __attribute__((always_inline)) {
            constexpr int TAKES = decltype(takes)::value;
            unsigned la_ = la0 ^ slot_b, lb_ = lb0 ^ slot_b;
            asm volatile("" : "+v"(la_), "+v"(lb_));
            // by slot (the step's, the next step's) and k-step, found here: computed at each fetch, they stand between the MFMAs
            const unsigned a_at[2][2] = {{la_, la_ ^ KSTEP_X}, {la_ ^ SLOT_B, la_ ^ SLOT_B ^ KSTEP_X}};
            const unsigned b_at[2][2] = {{lb_, lb_ ^ KSTEP_X}, {lb_ ^ SLOT_B, lb_ ^ SLOT_B ^ KSTEP_X}};
            // load targets: this step's slot, the previous step's (wave-uniform by construction; said so for the assembly's scalar operands)
            const unsigned lds_cur = __builtin_amdgcn_readfirstlane(wa0 ^ slot_b), lds_prev = lds_cur ^ SLOT_B;
            static_for<ROWS>([&](auto row) __attribute__((always_inline)) {
                constexpr int r = decltype(row)::value, strip = r / 4, next_a = (strip + 1) % 2;
                constexpr row_fetches256 fetches = fetches_of_row256(r);
                // The row's direct-to-LDS loads ride on MFMA 1 and, if there are two, MFMA 5.
                constexpr int d = r > FREE ? r - FREE - 1 : r + ROWS - FREE - 1;  // rows since the one behind FREE
                static_for<F>([&](auto mfma) __attribute__((always_inline)) {
                    constexpr int m = decltype(mfma)::value;
                    constexpr int j = r % 4 * 2 + m / 4, h = (m / 2 % 2) ^ (j % 2), i = strip * 2 + h, kk = m % 2;
                    constexpr int c = m / 4;
                    if constexpr (m % 4 == 1 && c < loads_in_row256(d))
                        mfma_load_chunk(std::integral_constant<int, loads_before_row256(d) + c>{}, bf[kk][j], af[strip % 2][h][kk], acc[i][j],
                                        r > FREE ? lds_cur : lds_prev);
                    else
                        X::go(bf[kk][j], af[strip % 2][h][kk], acc[i][j]);
                    __builtin_amdgcn_sched_barrier(0);
                    constexpr int first = m * fetches.n / F, last = (m + 1) * fetches.n / F;
                    static_for<last - first>([&](auto nth) __attribute__((always_inline)) {
                        constexpr fetch256 f = fetches.at[first + decltype(nth)::value];
                        if constexpr (f.b)
                            load_b(b_at[f.next][f.kk], f.block, f.kk);
                        else
                            load_a(next_a, a_at[f.next][f.kk], f.block, f.kk);
                    });
                    if constexpr (TAKES >= 0 && takes_before256(r, m + 1) > takes_before256(r, m))
                        take(std::integral_constant<int, TAKES * kTakes256 + takes_before256(r, m)>{});
                    __builtin_amdgcn_sched_barrier(0);
                });
                if constexpr (r == FREE) {
                    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wavefront's fetches from the step's slot have returned
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                    advance_loader();
                }
                if constexpr (r == PUB) {
                    // The stage the next step reads has landed; younger and allowed in flight: this step's YOUNG loads.
                    // In a tile's first step the wait also covers the previous tile's stores: part of the stage's
                    // loads was requested behind them (rows 0-6), and vmcnt retires in issue order.
                    // (The accumulator's values this step asked for are younger than that stage as well.)
                    wait_vmcnt<YOUNG + (TAKES >= 0 ? kTakes256 : 0)>();
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            slot_b ^= SLOT_B;
        };
        // A wavefront whose half of the tile another tile computes multiplies nothing: it brings its share of the operands and
        // meets the others.  (Large products are bound by energy; with M or N an odd multiple of 128 up to a tenth of their MFMAs
        // were such repeats.  Whole passes without an accumulator, us: 4224x7168x3584 bf16 183.7 -> 179.0, 8064x8064x4096 bf16 418 ->
        // 409, 6272x5888x2048 152.5 -> 150.2, of which an epilogue without the counters' code brings one percent.  Not in the
        // accumulating epilogues, which hold the accumulator's values through the K loop: a second way through it there spills
        // 500 registers.)
        const bool idle = (MODE == MODE_PLAIN || MODE == MODE_REORDER) && (((repeated & 1) && wm == 0) || ((repeated & 2) && wn == 0));
        if (idle) {
            constexpr int BEFORE = loads_before_row256(ROWS - FREE - 1);  // of a stage's loads, those in front of the step's end
            for (int kt = 0; kt < KT; kt++) {
#pragma unroll
                for (int c = BEFORE; c < 16; c++) load_chunk(c, slot_b ^ SLOT_B);
                __builtin_amdgcn_s_barrier();  // FREE
                asm volatile("" ::: "memory");
                advance_loader();
#pragma unroll
                for (int c = 0; c < YOUNG; c++) load_chunk(c, slot_b);
                wait_vmcnt<YOUNG>();
                __builtin_amdgcn_s_barrier();  // PUB
                asm volatile("" ::: "memory");
#pragma unroll
                for (int c = YOUNG; c < BEFORE; c++) load_chunk(c, slot_b);
                slot_b ^= SLOT_B;
            }
            // what a step's rows 13-15 fetch
#pragma unroll
            for (int q = 0; q < 4; q++) load_a(0, la0 ^ slot_b ^ (q % 2 * KSTEP_X), q / 2, q % 2);
#pragma unroll
            for (int q = 0; q < 10; q++) load_b(lb0 ^ slot_b ^ (q % 2 * KSTEP_X), q / 2, q % 2);
        } else {
        if (MODE == MODE_PLAIN || MODE == MODE_REORDER) {  // as above: all of them are written on this side of the wait states
#pragma unroll
            for (int i = 0; i < F; i++)
#pragma unroll
                for (int j = 0; j < F; j++) asm volatile("" : "+a"(acc[i][j]));
            fo_mfma_fence();
        }
        // A tile whose predecessor's signal is still owed leaves the K loop after its first step, sends the signal and
        // re-enters: that step's PUB meeting has waited for the predecessor's stores in every wavefront (part of the
        // stage's loads was requested behind them, rows 0-6, and vmcnt retires in issue order), with the meeting's
        // barrier behind the wait.  The test inside the step (one scalar compare and branch per K step, after the PUB
        // meeting) cost the large square 4 us.
        int kt = 0;
        int kt_stop = (COUNTS && owed > 0) ? 1 : KT;
        if constexpr (MODE == MODE_ACC) {
            if (early) {
                k_step(std::integral_constant<int, 0>{});
                k_step(std::integral_constant<int, 1>{});
                k_step(std::integral_constant<int, 2>{});
                k_step(std::integral_constant<int, 3>{});
                kt = 4;
            }
        }
        for (;;) {
        do {
            k_step(std::integral_constant<int, -1>{});
        } while (++kt < kt_stop);
            if (!COUNTS || owed == 0) break;
            owed = 0;
            if (wave == 0) announce(v_prev_r, v_prev_g);
            // Nothing scalar stays in flight behind this rare path: with a scalar load possibly pending, the K
            // loop's waits for LDS data would all have to be waits for everything.
            __builtin_amdgcn_s_waitcnt(0xC07F);
            if (kt >= KT) break;
            kt_stop = KT;
        }
        }

        fo_mfma_fence();
        const int next = tile + stride;
        const bool has_next = next < ntiles;
        int next_pm = 0, next_pn = 0, next_repeated = 0;
        if (has_next) {
            locate(next, &next_pm, &next_pn, &next_repeated);
            request_slots(next_pm, next_pn);
        }

        int v_done = 0;  // the slots of the tile that this epilogue stores (per lane)
        // ---- epilogue.  A wavefront's 128x128 block lies inside one reorder tile (BM and BN are multiples of
        // 128), so slot and base address are scalars.  The lane id is laundered so that this addressing is
        // recomputed per tile instead of living in registers across the K loop.
        {
            int el = lane;
            asm volatile("" : "+v"(el));
            const int erow = el & 15, ek = el >> 4;  // accumulator block: row erow, columns 4*ek .. 4*ek+3
            uint16_t *strip = reinterpret_cast<uint16_t *>(reinterpret_cast<char *>(smem) + STRIP_B) + wave * (16 * PITCH);
            const int srow = el / CPR, scol = el % CPR;
            const int ldp = reorder ? p.rLDN * p.BN : p.N;  // leading dimension of the output view
            const int row0 = (wm * 128) % p.BM, col0 = (wn * 128) % p.BN;
            const int r = r_mine;
            const int v_cur = v_rs;  // this tile's slots: the next tile's replace them inside the loop below
            const long trow = !reorder ? (long)(pm + wm) * 128 : (long)(r / p.rLDN) * p.BM + row0;
            const long tcol = !reorder ? (long)(pn + wn) * 128 : (long)(r % p.rLDN) * p.BN + col0;
            char *cbase = reinterpret_cast<char *>(p.C) + (trow * ldp + tcol) * 2;  // wave-uniform
            const unsigned lane_off = (unsigned)(srow * ldp + scol * 8) * 2;
            const bool stream_out = p.stream_out != 0;  // wave-uniform
            const bool keep = !((repeated & 1) && wm == 0) && !((repeated & 2) && wn == 0);  // wave-uniform
            // The accumulator's values are awaited together, in front of the first store: a later wait would count the
            // stores between them as well.
            char *abase = ACC || SUMS ? reinterpret_cast<char *>(p.ACC) + (trow * ldp + tcol) * 2 : nullptr;
            // TO_RANKS: the accumulator rows of the wavefront's rows, held as re_lo and re_hi are.
            int ac_lo = 0, ac_hi = 0;
            const bool sums = MODE == MODE_ACC || (MODE == MODE_RS && p.ACC) || (SUMS && r >= p.sum_from);  // wave-uniform
            // SUMS: the sums of such a tile; a reduce-scatter without an accumulator only wants its rows
            const bool adds = sums && (MODE != MODE_SCATTER_SUM || p.ACC);
            const int own_first = TO_RANKS ? p.rank * p.seg_rows : 0, own_rows = TO_RANKS && p.OWN && (sums || !SUMS) ? p.seg_rows : 0;
            auto row_of = [&](int k, int lo, int hi) __attribute__((always_inline)) {  // row k * RPP + srow of the block: its entry sits in that lane
                return __builtin_amdgcn_ds_bpermute((k * RPP % 64 + srow) * 4, k * RPP < 64 ? lo : hi);
            };
            if (MODE == MODE_RS || (MODE == MODE_SCATTER_SUM && sums)) {
                int first, count;
                group_range(r, &first, &count);
                ac_lo = rs_row(p.cseg, p.G, p.BM, p.W, p.seg_rows, re_lo, first * p.BM, count * p.BM);
                ac_hi = rs_row(p.cseg, p.G, p.BM, p.W, p.seg_rows, re_hi, first * p.BM, count * p.BM);
            }
            // SUMS, in the workgroup's last tile: the accumulator's values travel into the two slots, which nobody reads any more,
            // piece by piece in the order in which they are wanted: a wavefront's pieces lie where its operand loads went, each
            // lane's where it reads them, and no other wavefront has part in it.  (In registers, as with MODE_ACC, they would
            // leave no room on the SIMD for the consumer that runs beside the earlier waves.)
            auto piece_lds = [&](int k) __attribute__((always_inline)) { return (wa0 ^ (k / 16 * SLOT_B)) + k % 16 * CHUNK_B; };
            if (SUMS && adds && !has_next) {
                if (MAPPED) asm volatile("" : "+v"(re_lo), "+v"(re_hi), "+v"(ac_lo), "+v"(ac_hi));  // nothing else is awaited behind the loads
                unsigned rows = 0, rows_step = __builtin_amdgcn_readfirstlane(RPP * ldp * 2);
                const fo_srd_t from = fo_make_srd(TO_RANKS ? reinterpret_cast<char *>(p.ACC) : abase, 0x7fffffffu);
#pragma unroll
                for (int k = 0; k < NST; k++) {
                    if (TO_RANKS) {
                        const int to = row_of(k, ac_lo, ac_hi);
                        dma_buf16(from, to < 0 ? 0x80000000u : (unsigned)(to * ldp + (int)tcol + scol * 8) * 2, 0, piece_lds(k));
                    } else {
                        dma_buf16(from, lane_off, rows, piece_lds(k));
                        rows += rows_step;
                        asm volatile("" : "+s"(rows));  // one scalar, not one for each piece
                    }
                }
            }
            if (ACC && sums && keep && !early) {
#pragma unroll
                for (int k = 0; k < NST; k++) {
                    if (MODE == MODE_RS) {
                        const int to = row_of(k, ac_lo, ac_hi);
                        old[k] = *reinterpret_cast<const fo_u32x4 *>(p.ACC + (size_t)(to < 0 ? 0 : to) * ldp + tcol + scol * 8);
                    } else {
                        old[ACC ? k : 0] = *reinterpret_cast<const fo_u32x4 *>(abase + (size_t)(k * RPP) * ldp * 2 + lane_off);
                    }
                }
                // MODE_RS: awaited on this way.  Awaited behind the point where it meets the one without an accumulator, they were to
                // the compiler still to come on the other, and on both every piece waited, counting, for the stores in front of
                // it.  Whole calls with the normalisation, us: 4096x3328x4096 bf16 122.5 -> 103.5, 3456x4352x3072 108.2 -> 93.5,
                // 8192x8192x1024 in 32 groups 221.5 -> 207.0; without an accumulator 8192x4096x4096 in 24 240.2 -> 214.6.
                if (MODE == MODE_RS) {
#pragma unroll
                    for (int k = 0; k < NST; k++) asm volatile("" : "+v"(old[ACC ? k : 0]));
                }
            } else if (!early) {
#pragma unroll
                for (int k = 0; k < (ACC ? NST : 1); k++) old[k] = fo_u32x4{0, 0, 0, 0};
            }
#pragma unroll
            for (int i = 0; i < F; i++) {  // 16 output rows = one row of accumulator blocks
                __builtin_amdgcn_sched_barrier(0);
                int pitch = ldp;
                if (SUMS) asm volatile("" : "+s"(pitch));  // a strip's offsets are computed in the strip
#pragma unroll
                for (int j = 0; j < F; j++) {
                    fo_float4v a4 = acc[i][j];
                    asm volatile("" : "+a"(a4));  // leaves the accumulation registers here, not in one sweep in front of the epilogue
                    fo_u32x2 v;
                    v.x = E::pack(a4[0], a4[1]);
                    v.y = E::pack(a4[2], a4[3]);
                    *reinterpret_cast<fo_u32x2 *>(strip + erow * PITCH + j * 16 + ek * 4) = v;
                }
                // the strip is private to this wavefront: order its LDS writes before its reads
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_s_waitcnt(0xC07F);
                __builtin_amdgcn_wave_barrier();
                if (MODE == MODE_ACC && sums && i == 0) {
#pragma unroll
                    for (int k = 0; k < NST; k++) asm volatile("" : "+v"(old[ACC ? k : 0]));
                }
                if (SUMS && adds && !has_next) {
                    // this strip's values have landed; behind them the later strips' and the stores of the earlier ones
                    constexpr int PER = MODE == MODE_SIGNAL_SUM ? 2 * (16 / RPP) : 16 / RPP;
                    switch (i) {  // i is a constant: the loop is unrolled
                        case 0: wait_vmcnt<28>(); break;
                        case 1: wait_vmcnt<24 + PER>(); break;
                        case 2: wait_vmcnt<20 + 2 * PER>(); break;
                        case 3: wait_vmcnt<16 + 3 * PER>(); break;
                        case 4: wait_vmcnt<12 + 4 * PER>(); break;
                        case 5: wait_vmcnt<8 + 5 * PER>(); break;
                        case 6: wait_vmcnt<4 + 6 * PER>(); break;
                        default: wait_vmcnt<7 * PER>(); break;
                    }
                    asm volatile("" ::: "memory");
                }
                // SUMS: the accumulator's piece k; in another than the last tile, which a caller's own order of the slots may
                // ask for, from memory
                auto value_of = [&](int k) __attribute__((always_inline)) {
                    fo_u32x4 x;
                    if (!has_next) {
                        x = *reinterpret_cast<lds16_t>(piece_lds(k) + el * 16);
                    } else {
                        if (TO_RANKS) {
                            const int to = row_of(k, ac_lo, ac_hi);
                            x = *reinterpret_cast<const fo_u32x4 *>(p.ACC + (size_t)(to < 0 ? 0 : to) * pitch + tcol + scol * 8);
                        } else {
                            x = *reinterpret_cast<const fo_u32x4 *>(abase + (size_t)(k * RPP) * pitch * 2 + lane_off);
                        }
                        asm volatile("" : "+v"(x));  // awaited here: where the two ways meet, the other one would wait for its stores
                    }
                    return x;
                };
                if (keep)
#pragma unroll
                for (int ps = 0; ps < 16 / RPP; ps++) {
                    const int row = ps * RPP + srow;
                    fo_u32x4 v = *reinterpret_cast<const fo_u32x4 *>(strip + row * PITCH + scol * 8);
                    if (MAPPED) {
                        const int k = i * (16 / RPP) + ps;
                        const long prow = row_of(k, re_lo, re_hi);
                        uint16_t *to = p.C + (size_t)prow * pitch + tcol + scol * 8;
                        if (TO_RANKS && (ACC || sums)) {
                            const int ac = row_of(k, ac_lo, ac_hi);
                            if ((SUMS ? adds : sums) && ac >= 0)
                                store16_write_through(p.ACC + (size_t)ac * pitch + tcol + scol * 8, fo_add8<Tag>(SUMS ? value_of(k) : old[ACC ? k : 0], v));
                            if ((unsigned)(ac - own_first) < (unsigned)own_rows)
                                store16_write_through(p.OWN + (size_t)(ac - own_first) * pitch + tcol + scol * 8, v);
                            store16_write_through(to, v);
                        } else if (stream_out) {
                            store16_write_through_nt(to, v);
                        } else {
                            store16_write_through(to, v);
                        }
                    } else {
                        char *sb = cbase + (size_t)(i * 16 + ps * RPP) * pitch * 2;
                        if constexpr (MODE == MODE_ACC || MODE == MODE_SIGNAL_SUM) {
                            if (sums) {
                                char *ab = abase + (size_t)(i * 16 + ps * RPP) * pitch * 2;
                                const fo_u32x4 sum = fo_add8<Tag>(SUMS ? value_of(i * (16 / RPP) + ps) : old[ACC ? i * (16 / RPP) + ps : 0], v);
                                if (stream_out)
                                    store16_write_through_nt(ab, lane_off, sum);
                                else
                                    store16_write_through(ab, lane_off, sum);
                            }
                        }
                        if (stream_out)
                            store16_write_through_nt(sb, lane_off, v);
                        else
                            store16_write_through(sb, lane_off, v);
                    }
                    if (SUMS) __builtin_amdgcn_sched_barrier(0);  // a piece at a time: four take more registers than the kernels beside this one leave
                }
                __builtin_amdgcn_s_waitcnt(0xC07F);  // strip reads done before the next pass overwrites it
                __builtin_amdgcn_wave_barrier();
                // The next tile's slots, requested in front of this epilogue, have arrived with the pass's waits: they
                // leave their four scalar registers here.
                if (i == 0 && has_next) take_slots();
            }
            v_done = v_cur;
        }

        if (signalling) {
            // lane s: group of reorder tile s, -1 where another workgroup tile counts it.  (No launch that counts has half
            // tiles, see plan_launch; with the test gone, the code the compiler makes of this is 0.3 % slower on 8192^3.)
            int v_g = -1;
            if (wave == 0) {
#pragma unroll
                for (int s = 0; s < kMaxSub; s++) {
                    if (s < nsub && !((repeated & 1) && s < sub_n) && !((repeated & 2) && s % sub_n == 0)) {
                        const int slot = __builtin_amdgcn_readlane(v_done, s), g = group_of(slot);
                        v_g = lane == s && !(SUMS && slot >= p.sum_from) ? g : v_g;
                    }
                }
            }
            if (has_next) {
                owed = 1;  // PUB meetings until this tile's stores have been waited for in every wavefront
                v_prev_r = v_done;
                v_prev_g = v_g;
            } else {
                // Last tile: every lane waits until its own write-through stores are acknowledged, the barrier
                // collects the workgroup, then one lane bumps the counters (the reference has no fence here,
                // src/overlap/gemm_with_signal.h:337-351).
                __builtin_amdgcn_s_waitcnt(0);
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                if (wave == 0) {
                    if (owed > 0) announce(v_prev_r, v_prev_g);
                    announce(v_done, v_g);
                }
            }
        }
        if (!has_next) break;
        tile = next;
        pm = next_pm;
        pn = next_pn;
        repeated = next_repeated;
    }
    __builtin_amdgcn_s_waitcnt(0);  // nothing of this wavefront is in flight when it ends
}

}  // namespace fo_gemm_dev
