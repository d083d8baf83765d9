// What the kernels of the gfx950 MFMA GEMM share: launch arguments, the group search, counted waits, stores and
// the direct-to-LDS load.
//
//   C[M,N] = A[M,K] . B[N,K]^T   (both operands K-contiguous), fp32 accumulate.
//
// Replaces the CUTLASS kernels behind gemm_func_table / signal_func_table /
// scatter_func_table of the reference (src/gemm/gemm.cu:23-110,
// src/overlap/gemm_signal.cu:15-97, src/overlap/gemm_scatter.cu:15-98; epilogue
// semantics src/overlap/gemm_with_signal.h:236-256, :291-361).
//
// Two kernels: fo_gemm256_kernel.h (256x256 workgroup tiles, four wavefronts, persistent) and
// fo_gemm_tile_kernel.h (everything smaller).  Both use v_mfma_f32_16x16x32_{f16,bf16} over ascending K: in an
// MFMA-only loop under this part's power limit that form sustains 14 % more than 32x32x16 (a quarter of the
// accumulator registers per instruction, half of their traffic per flop), and large products are power-limited.
#pragma once

#include <cstddef>
#include <cstring>
#include <type_traits>
#include <utility>

#include "fo_common.h"

namespace fo_gemm_dev {

// f(integral_constant 0), f(1), ... f(N - 1): the body of a K step, whose every index decides which instruction stands where.
// As loops for the optimiser to unroll, the choices are made in its passes, over thousands of branches; here they are made
// before it starts (CPU seconds to compile an instantiation of the 256x256 kernel 172 -> 3, 150 of them in value numbering,
// of the smaller tiles 23 -> 14; the code is the same but for fewer address computations where a whole stage is fetched
// ahead: GEMM alone, fp16, us, 512x4096x4088 22.8 -> 21.8, 1024x4096x4088 33.0 -> 32.0, 1536x4096x4088 54.2 -> 52.3).
template <typename F, int... I>
__device__ __forceinline__ void static_for_each(std::integer_sequence<int, I...>, F &&f) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    static_for_each(std::make_integer_sequence<int, (N > 0 ? N : 0)>{}, static_cast<F &&>(f));
}

// MODE_ACC: for a call that stays on one stream.  The tile is stored as the plain epilogue does (RA null) or reordered,
// without counters, and ACC[o] = round16(ACC[o] + C[o]) is done for every element stored.
// MODE_RS: the same for a reduce-scatter (the scatter epilogue's row map, rLDN == 1): C is cut into ranges of rows, one
// per group, and each range into W chunks of consecutive rows; row i of chunk q of a range that starts at row f is added
// to row q * seg_rows + f / W + i of the accumulator (if any) and, for q == rank, stored to row f / W + i of OWN (if any).
// MODE_SIGNAL_SUM, MODE_SCATTER_SUM (256x256 kernel only): the signal and scatter epilogues where tiles from storage slot
// sum_from on are not counted but added to the accumulator as MODE_ACC and MODE_RS do.  MODE_REORDER (the same kernel): the signal
// epilogue's store, nothing counted.
enum { MODE_PLAIN = 0, MODE_SIGNAL = 1, MODE_SCATTER = 2, MODE_ACC = 3, MODE_RS = 4, MODE_SIGNAL_SUM = 5, MODE_SCATTER_SUM = 6, MODE_REORDER = 7 };

// Division by a number that the host knows: n / d for n and d below 32768, exactly (the product exceeds n / d * 2^31 by
// less than n * d).
struct fo_div {
    uint32_t mul;  // 2^31 / d rounded up
};
__host__ __device__ inline __attribute__((always_inline)) int fo_divide(int n, fo_div d) {
    return (int)((uint64_t)(uint32_t)(2 * n) * d.mul >> 32);
}
constexpr long kMaxDivide = 32767;
inline fo_div fo_divisor(long d) { return {d > 0 ? (uint32_t)(((1ULL << 31) + d - 1) / d) : 0}; }

// Position t of the raster that fo_wg_to_tile walks (xcd_remap 0 or 1), by divisors that the host prepared.
__host__ __device__ inline __attribute__((always_inline)) void fo_raster_tile(int t, int remap, int grid_m, int grid_n, int panel,
                                                                              fo_div by_panel, fo_div by_rows, fo_div by_last_rows,
                                                                              int *pm, int *pn) {
    const int nt = grid_m * grid_n, x = t & 7, rem = nt & 7;
    const int v = remap ? x * (nt >> 3) + (x < rem ? x : rem) + (t >> 3) : t;
    const int q = fo_divide(v, by_panel), first_m = q * panel, in = v - first_m * grid_n;
    const bool last = grid_m - first_m < panel;
    fo_div by;
    by.mul = last ? by_last_rows.mul : by_rows.mul;
    const int rows = last ? grid_m - first_m : panel, col = fo_divide(in, by);
    *pm = first_m + in - col * rows;
    *pn = col;
}

// A launch as the host describes it, and, behind those words that its first load needs, the 256x256 kernel's arguments.
struct alignas(64) GemmArgs {
    const uint16_t *A;
    const uint16_t *B;
    int M, N, K;           // K is also the row stride of both operands
    int grid_m, grid_n, panel, xcd_remap;  // the raster of this launch's parent tiles
    int first, sub_m, sub_n, count;        // this launch: positions from `first`, each cut into sub_m x sub_n macro tiles, `count` of them
    uint16_t *C;
    uint16_t *ACC;         // MODE_ACC, MODE_RS: the accumulator
    int BM, BN, TN, rLDN;  // reorder/signal tile, tiles along N, reshaped width in tiles
    const int32_t *RA;
    const int32_t *RE;
    const int32_t *cseg;
    int G;
    int32_t *MM;
    int monitor;
    int quiet;                             // signalling epilogues: store the tiles reordered, touch no counter
    int half;                              // 256x256 kernel: half a tile is left at the end of M (bit 0), N (bit 1); rows too long for early requests (bit 2)
    uint16_t *OWN;                         // MODE_RS: this rank's rows
    int W, rank, seg_rows;                 // MODE_RS: ranks, this rank, rows of the view per rank
    int stream_out;                        // 256x256 kernel: store the output with the non-temporal hint
    int sum_from;                          // MODE_SIGNAL_SUM, MODE_SCATTER_SUM: first storage slot that is summed

    static GemmArgs of(const GemmArgs &a, int, int) { return a; }
};
// What the 256x256 kernel's epilogue reads of it, C and on, are two 64-byte lines of its launch's 256 bytes of arguments (in front stand
// Front256's seven words, one of padding and the part up to C); eight bytes earlier they are three: 4096x4096x512 with an accumulator 40.65 -> 41.0 us.
constexpr int kGemmArgsAt = 64;
static_assert(offsetof(GemmArgs, C) == 64 && sizeof(GemmArgs) == 192, "the kernel's part begins on a line and ends with the second one");

// The smaller tiles' arguments: 112 bytes, because a launch takes the host 2.7 us with up to 112 bytes of arguments and 3.1 to
// 3.7 with 120 or more, those that the runtime adds for gridDim among them (an empty kernel in a process with torch, which
// brings its own runtime; a launch of the struct above had 208 bytes and 256 that were added).  One plain product: 3.9 -> 3.1 us of host time; whole
// passes that wait for the host: 128x4096x1024 11.8 -> 11.4 us, 128x3328x488 9.5 -> 9.0, 128x2432x320 12.6 -> 12.1.  (The launch's
// size out of the dispatch packet instead of an argument: the packet lies in host memory, 9 us more on every kernel.)
// What the kernel can derive is derived there, what only one epilogue needs shares its place, and the fields that the first
// operand load needs stand in front: they arrive in registers with the wavefront (see TileRest).
struct TileArgs {
    const uint16_t *A;
    const uint16_t *B;
    int M, N, K;            // K is also the row stride of both operands
    int grid_m, grid_n;
    int stride;             // workgroups of the launch
    fo_div by_panel, by_rows, by_last_rows;  // divisors of the raster walk: tiles of a panel, its rows, the last panel's (general: panel, first, count)
    uint32_t bits;
    uint16_t *C;
    const int32_t *RA;
    union {
        uint16_t *ACC;      // MODE_ACC, MODE_RS
        int32_t *MM;        // the epilogues that count
    };
    const int32_t *cseg;
    const int32_t *RE;
    union {
        uint16_t *OWN;      // MODE_RS, whose rLDN is 1
        int rLDN;
    };
    int G;

    // bits
    static constexpr uint32_t GENERAL = 1;  // another walk than the divisors', or numbers too large for them or for the bits below
    static constexpr uint32_t TALL = 2, WIDE = 4;    // reorder tiles of 256 rows, columns (else 128)
    static constexpr uint32_t MONITOR = 8, QUIET = 16;
    static constexpr int REMAP = 5;                  // two bits: xcd_remap
    static constexpr int SUB_M = 7, SUB_N = 9;       // two bits each, general: log2 of the tiles a position is cut into along M, N
    static constexpr int RANKS = 11, RANK = 15;      // MODE_RS: four bits, log2 of W; eight bits, rank
    static constexpr int PANEL = 23;                 // eight bits, not general: panel

    static TileArgs of(const GemmArgs &a, int workgroups, int mode) {
        const long positions = (long)a.grid_m * a.grid_n;
        const bool general = a.xcd_remap == 2 || a.sub_m * a.sub_n > 1 || a.count != positions || positions > kMaxDivide || a.panel > 255;
        TileArgs t = {};
        t.A = a.A; t.B = a.B; t.C = a.C;
        t.M = a.M; t.N = a.N; t.K = a.K;
        t.grid_m = a.grid_m; t.grid_n = a.grid_n; t.stride = workgroups;
        if (general) {
            t.by_panel.mul = (uint32_t)a.panel;
            t.by_rows.mul = (uint32_t)a.first;
            t.by_last_rows.mul = (uint32_t)a.count;
        } else {
            t.by_panel = fo_divisor((long)a.panel * a.grid_n);
            t.by_rows = fo_divisor(a.panel);
            t.by_last_rows = fo_divisor(a.panel > 0 ? a.grid_m % a.panel : 1);
        }
        t.RA = a.RA; t.RE = a.RE; t.cseg = a.cseg; t.G = a.G;
        if (mode == MODE_ACC || mode == MODE_RS)
            t.ACC = a.ACC;
        else
            t.MM = a.MM;
        if (mode == MODE_RS)
            t.OWN = a.OWN;
        else
            t.rLDN = a.rLDN;
        auto log2 = [](int n) { return (uint32_t)__builtin_ctz((unsigned)n); };  // W, sub_m and sub_n are powers of two
        t.bits = (general ? GENERAL : 0) | log2(a.sub_m) << SUB_M | log2(a.sub_n) << SUB_N | (uint32_t)a.xcd_remap << REMAP |
                 (a.BM == 256 ? TALL : 0) | (a.BN == 256 ? WIDE : 0) | (a.monitor ? MONITOR : 0) | (a.quiet ? QUIET : 0) |
                 log2(a.W) << RANKS | (uint32_t)a.rank << RANK | (general ? 0 : (uint32_t)a.panel << PANEL);
        return t;
    }
};
static_assert(sizeof(TileArgs) == 112, "a launch costs more from here on");
// The kernel takes the fields in front of C as seven words of 64 bits, which arrive in registers with the wavefront, and the rest as
// they are.  (Words, not pointers: with pointers and integers one by one, thirteen arguments, a launch was as dear as with 208 bytes.)
struct TileRest {
    uint64_t words[7];
};
static_assert(offsetof(TileArgs, C) == 56 && sizeof(TileRest) == sizeof(TileArgs) - 56, "the fields in front, and the rest");

// Tiles of a launch.
__host__ __device__ inline __attribute__((always_inline)) int fo_tile_count(const TileArgs &p) {
    return p.bits & TileArgs::GENERAL ? (int)p.by_last_rows.mul : p.grid_m * p.grid_n;
}


// Tile of unit u of a launch: what fo_unit_to_tile gives, without its divisions where the host could prepare them.  (A
// division is some thirty instructions, and in front of a kernel's first load those are fetched from memory as well.)
__host__ __device__ inline __attribute__((always_inline)) void fo_tile_of(const TileArgs &p, int u, int *pm, int *pn) {
    const int remap = p.bits >> TileArgs::REMAP & 3;
    if (__builtin_expect(p.bits & TileArgs::GENERAL, 0)) {
        int sub_m = 1 << (p.bits >> TileArgs::SUB_M & 3), sub_n = 1 << (p.bits >> TileArgs::SUB_N & 3);
        int grid_m = p.grid_m, grid_n = p.grid_n, panel = (int)p.by_panel.mul;
#ifdef __HIP_DEVICE_COMPILE__
        asm volatile("" : "+s"(sub_m), "+s"(sub_n), "+s"(grid_m), "+s"(grid_n), "+s"(panel));  // its divisions stay in here
#endif
        fo_unit_to_tile(u, (int)p.by_rows.mul, sub_m, sub_n, grid_m, grid_n, panel, remap, pm, pn);
        return;
    }
    fo_raster_tile(u, remap, p.grid_m, p.grid_n, p.bits >> TileArgs::PANEL & 255, p.by_panel, p.by_rows, p.by_last_rows, pm, pn);
}

// What the first operand load of the 256x256 kernel needs, as words of 64 bits that arrive in registers with the wavefront, low half
// first: A, B, K and count, grid_m and grid_n, panel and bits, the divisors of the raster walk.
struct Front256 {
    const uint16_t *A, *B;
    int K, count, grid_m, grid_n, panel;
    fo_div by_panel, by_rows, by_last_rows;  // tiles of a panel (waves of whole tile rows: workgroups of a wave), its rows, the last panel's
    uint32_t bits;                           // 1: numbers too large for the divisors; from bit 1: xcd_remap, two bits; from bit 3: half

    static Front256 of(const GemmArgs &a) {
        Front256 f = {};
        const bool waves = a.xcd_remap == 2;
        f.A = a.A; f.B = a.B; f.K = a.K; f.count = a.count;
        f.grid_m = a.grid_m; f.grid_n = a.grid_n; f.panel = a.panel;
        const bool general = (long)a.grid_m * a.grid_n > kMaxDivide || (!waves && a.panel <= 0);
        if (!general) {
            f.by_panel = fo_divisor(waves ? a.panel >> 12 : (long)a.panel * a.grid_n);
            f.by_rows = fo_divisor(waves ? 1 : a.panel);
            f.by_last_rows = fo_divisor(waves ? 1 : a.grid_m % a.panel);
        }
        f.bits = (general ? 1 : 0) | (uint32_t)a.xcd_remap << 1 | (uint32_t)a.half << 3;
        return f;
    }
};

// Raster position t of such a launch: what fo_wg_to_tile gives.
__host__ __device__ inline __attribute__((always_inline)) void fo_tile_of(const Front256 &f, int t, int *pm, int *pn) {
    const int remap = f.bits >> 1 & 3;
    if (__builtin_expect(f.bits & 1, 0)) {
        int grid_m = f.grid_m, grid_n = f.grid_n, panel = f.panel;
#ifdef __HIP_DEVICE_COMPILE__
        asm volatile("" : "+s"(grid_m), "+s"(grid_n), "+s"(panel));  // its divisions stay in here
#endif
        fo_wg_to_tile(t, grid_m, grid_n, panel, remap, pm, pn);
        return;
    }
    if (remap == 2) {
        fo_row_wave_tile(t, fo_divide(t, f.by_panel), f.panel, pm, pn);
        return;
    }
    fo_raster_tile(t, remap, f.grid_m, f.grid_n, f.panel, f.by_panel, f.by_rows, f.by_last_rows, pm, pn);
}

// Every operand row begins on a 128-byte line.
inline bool on_lines(const GemmArgs &a) { return (((uintptr_t)a.A | (uintptr_t)a.B | (uintptr_t)a.K * 2) & 127) == 0; }

constexpr int kMaxSub = 4;        // reorder tiles per macro tile (256x256 over 128x128)
constexpr int kPrefixRegs = 256;  // group search on prefix sums held in registers (one per 64 groups) up to this many groups

// Inclusive prefix sum over a wavefront's lanes by the vector unit's own paths (six round trips to the LDS unit otherwise).
// All lanes take part.
template <int CTRL, int ROWS> __device__ __forceinline__ int add_shifted(int v) {
    return v + __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false);
}
__device__ __forceinline__ int wave_prefix_sum(int v) {
    v = add_shifted<0x111, 0xf>(v);     // row_shr:1, 2, 4, 8: inside rows of sixteen lanes
    v = add_shifted<0x112, 0xf>(v);
    v = add_shifted<0x114, 0xf>(v);
    v = add_shifted<0x118, 0xf>(v);
    v = add_shifted<0x142, 0xa>(v);     // row_bcast:15: a row's sum to the next, rows 1 and 3
    return add_shifted<0x143, 0xc>(v);  // row_bcast:31: the first half's to rows 2 and 3
}

// Group of storage slot r: smallest g with cseg[0]+..+cseg[g] > r
// (src/overlap/gemm_with_signal.h:343-349), found by one wavefront with a
// 64-wide prefix sum per step instead of a serial scan.  All 64 lanes call it.
__device__ __forceinline__ int find_group(const int32_t *cseg, int G, int r, int lane) {
    int base = 0;
    for (int it = 0; it < G; it += 64) {
        int idx = it + lane;
        const int s = base + wave_prefix_sum(idx < G ? cseg[idx] : 0);
        unsigned long long hit = __ballot(idx < G && s > r);
        if (hit) return it + (int)__builtin_ctzll(hit);
        base = __builtin_amdgcn_readlane(s, 63);
    }
    return G - 1;  // unreachable when sum(cseg) covers every slot (validated on the host)
}

// The same, with the group's first storage slot and its slot count.  n0: this lane's group size, cseg[lane] (0 beyond G).
__device__ __forceinline__ void find_group_range(const int32_t *cseg, int G, int r, int lane, int n0, int *first, int *count) {
    int base = 0;
    *first = *count = 0;
    for (int it = 0; it < G; it += 64) {
        const int idx = it + lane, n = it == 0 ? n0 : idx < G ? cseg[idx] : 0;
        const int s = base + wave_prefix_sum(n);
        unsigned long long hit = __ballot(idx < G && s > r);
        if (hit) {
            const int at = (int)__builtin_ctzll(hit);
            *count = __builtin_amdgcn_readlane(n, at);
            *first = __builtin_amdgcn_readlane(s, at) - *count;
            return;
        }
        base = __builtin_amdgcn_readlane(s, 63);
    }
}

// MODE_RS: accumulator row of view row `row`, whose group holds the rows [first, first + count); -1 for a row that the
// map sent out of its group's range and that belongs to nobody's (the host's row maps do not).
__device__ __forceinline__ int rs_row(const int32_t *cseg, int G, int BM, int W, int seg_rows, int row, int first, int count) {
    if (row < first || row >= first + count) {
        first = 0;
        int g = 0;
        for (; g < G; g++) {
            count = cseg[g] * BM;
            if (row < first + count) break;
            first += count;
        }
        if (g == G || row < 0) return -1;
    }
    const int chunk = count / W, in = row - first, q = in / chunk;
    return q * seg_rows + first / W + (in - q * chunk);
}

// s_waitcnt vmcnt(n) only (expcnt/lgkmcnt left at their maxima); gfx9 encoding:
// vmcnt = imm[15:14]:imm[3:0], expcnt = imm[6:4], lgkmcnt = imm[11:8].
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// 16-byte global stores written as assembly so that the number of vector memory
// instructions in flight is known exactly (the main loop waits on vmcnt with
// non-zero counts; the compiler does not see these instructions in its own
// count, which can only make its waits longer, never shorter).  All of them write
// through (system-scope cache policy).  In the signalled epilogues the tile must be
// visible to other XCDs before its counter is bumped, and a tile that never becomes
// dirty in L2 needs no releasing write-back before the signal.  Elsewhere the lines
// left dirty in the L2s would be written back between this kernel and the next,
// when nothing else runs (GEMM with an accumulator, us: 1152x5120x1720 28.4 -> 26.7,
// 1024x4096x2048 20.0 -> 18.8, 512x4096x4096 21.8 -> 21.2, 1024x8192x2048 34.0 ->
// 33.4; whole passes: sequence 38.0 -> 36.1, ragged 35.1 -> 33.9).  The trailing s_nop covers
// the wait states gfx9 requires between a VMEM store of more than 8 bytes and a
// VALU write of its data registers.
__device__ __forceinline__ void store16_write_through(void *ptr, fo_u32x4 v) {
    asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 1" : : "v"(ptr), "v"(v) : "memory");
}
// saddr forms: wave-uniform base (SGPR pair) + 32-bit per-lane byte offset
__device__ __forceinline__ void store16_write_through(char *base, unsigned lane_off, fo_u32x4 v) {
    asm volatile("global_store_dwordx4 %0, %1, %2 sc0 sc1\n\ts_nop 1"
                 :
                 : "v"(lane_off), "v"(v), "s"((__attribute__((address_space(1))) char *)base)
                 : "memory");
}
// The same with the non-temporal hint, for outputs too large to be found in a cache by whoever reads them
// next (GemmArgs::stream_out): the resident workgroups finish their tiles together and store 128 KB each
// at once, and output lines that took room in the L2 would push out the operand panels the next tile's
// first K steps are about to share.  8192^3: GEMM alone 1.7 % faster, the overlapped step unchanged; on
// the 8192x4096 output (67 MB), which the consumer finds in the memory-side cache, the hint made the
// overlapped step 2 % and the serial step 8 % slower, so smaller outputs go without it.
__device__ __forceinline__ void store16_write_through_nt(void *ptr, fo_u32x4 v) {
    asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1 nt\n\ts_nop 1" : : "v"(ptr), "v"(v) : "memory");
}
__device__ __forceinline__ void store16_write_through_nt(char *base, unsigned lane_off, fo_u32x4 v) {
    asm volatile("global_store_dwordx4 %0, %1, %2 sc0 sc1 nt\n\ts_nop 1"
                 :
                 : "v"(lane_off), "v"(v), "s"((__attribute__((address_space(1))) char *)base)
                 : "memory");
}
#define FO_LDS_PTR(p) ((__attribute__((address_space(3))) void *)(p))

typedef unsigned int fo_srd_t __attribute__((ext_vector_type(4)));  // buffer descriptor

// Raw buffer of `bytes` bytes at a wave-uniform address.
__device__ __forceinline__ fo_srd_t fo_make_srd(const void *base, unsigned bytes) {
    const uint64_t b = (uint64_t)(uintptr_t)base;
    fo_srd_t r;
    r.x = __builtin_amdgcn_readfirstlane((unsigned)b);
    r.y = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32) & 0xFFFF);  // stride 0: raw buffer
    r.z = __builtin_amdgcn_readfirstlane(bytes);
    r.w = 0x00020000u;  // 32-bit data format, no swizzle
    return r;
}

// 16 bytes per lane, global -> LDS: address = descriptor base + soff + voff (out of range: zeros),
// LDS address = lds_addr + lane * 16 (through M0; the s_nop is the wait state between an M0 write and its use).
// A vector-memory instruction that reads a scalar register has to stay five wait states behind a vector instruction that
// wrote it, and the compiler, which does not look into this statement, may return a spilled scalar (v_readlane) right in
// front of it.  Where it does, dma_buf16_sum takes its place; a test looks for such pairs in the built code.
__device__ __forceinline__ void dma_buf16(fo_srd_t srd, unsigned voff, unsigned soff, unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds_addr), "v"(voff), "s"(srd), "s"(soff)
                 : "memory");
}
// The same with soff = row_off + col_off, added here: the load reads a scalar that a scalar instruction wrote, which needs
// no distance.  (As fast on the tiles that use it; five wait states instead cost 128x256 tiles 1 %.  On smaller tiles,
// which keep their offsets in scalar registers, this form is up to 4 % slower: 384x2304x4760 in 64x64 tiles, 22.3 -> 23.1.)
__device__ __forceinline__ void dma_buf16_sum(fo_srd_t srd, unsigned voff, unsigned row_off, unsigned col_off, unsigned lds_addr) {
    unsigned soff;
    asm volatile("s_mov_b32 m0, %1\n\ts_add_u32 %0, %4, %5\n\tbuffer_load_dwordx4 %2, %3, %0 offen lds"
                 : "=&s"(soff)
                 : "s"(lds_addr), "v"(voff), "s"(srd), "s"(row_off), "s"(col_off)
                 : "memory", "scc");
}

}  // namespace fo_gemm_dev
