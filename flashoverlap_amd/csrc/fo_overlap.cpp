// Host orchestration of the overlap path: the counterpart of class OverlapImpl
// (src/overlap_impl.h:12-43, src/overlap_impl.cu) behind a C handle.  Two HIP
// streams; every call only enqueues work and returns.  May be captured into a HIP graph.
#include <initializer_list>
#include <mutex>
#include <new>
#include <vector>

#include "fo_common.h"

namespace {

// Words of the workspace (device int32[kWorkspaceWords], zero between calls).
enum {
    kWsLeft = 0,    // workgroups of the one-launch consumer that have left
    kWsGaveUp = 1,  // set by any bounded wait of a call that ran out of polls
    kWsJoin = 4,    // consumer stream -> GEMM stream
    kWsFork = 5,    // GEMM stream -> consumer stream
    kWorkspaceWords = 16,
};

// Defaults of the scheduling choices below; a handle can override them
// (fo_overlap_set_schedule), they are measurements on one MI355X, not laws.
//
// Two launches per group cost a few microseconds each; beyond kFusedFromGroups
// groups the single wait+reduce launch is the faster consumer.  With few, large
// groups the per-group launches win: a kernel that starts when its group is
// complete needs no polling workgroups resident beside the GEMM.
//
// In automatic mode a GEMM shorter than kInStreamBelowFlop (about 50 us of this
// GPU) keeps the whole call on the GEMM stream: the GEMM with its reordered
// store, whose epilogue does the all-reduce consumer's work too (with the monitor on: the signalling
// GEMM, one wait that resets every counter and one consumer launch).  Fork, join and pollers beside the
// GEMM cost more than such a GEMM can hide (4096x4096x512 with 256 groups:
// 71 us overlapped, 44 us in stream).
//
// kManyCopiesFromFlop, kFewCopies: see fo_overlap_gemm_reducescatter.  They are no thresholds of a handle.
//
// kTogetherFromN, kTogetherUpToK, kTogetherAnyKUpToN: what is consumed and normalised by one kernel (rows_together below).
//
// kGemmFlopPerNs: what a GEMM is expected to sustain, for sizing the pause
// between polls only.
constexpr int kFusedFromGroups = 16;
constexpr double kInStreamBelowFlop = 6.4e10;
constexpr double kManyCopiesFromFlop = 5e11;
constexpr int kFewCopies = 16, kFewCopiesOfShort = 6;
constexpr int kTogetherFromN = 1024;
constexpr int kTogetherUpToK = 3072;
constexpr int kTogetherAnyKUpToN = 2048;
constexpr double kGemmFlopPerNs = 1.2e6;

}  // namespace

struct fo_overlap {
    hipStream_t gemm_stream = nullptr;
    hipStream_t comm_stream = nullptr;  // null: every call stays on the GEMM stream
    hipEvent_t forked = nullptr, joined = nullptr;  // used only while the GEMM stream is being captured
    int32_t *workspace = nullptr;
    bool gemm_ready = false;
    bool overlap_ready = false;
    int rank = 0, world = 1;
    void *acc = nullptr;
    int64_t acc_nelem = 0;
    int fused = -1;        // -1: choose per call (one launch when there are many groups)
    long max_polls = -1;   // bound of every device-side wait; -1: FO_WAIT_MAX_POLLS, 0: none
    int fused_from_groups = kFusedFromGroups;
    double in_stream_below_flop = kInStreamBelowFlop;
    int token = 1;         // value the fork and join words carry from one stream to the other
    // A handle-free call: its words may hold what another call left.  They are cleared first, and the consumer stream
    // must not start before that.
    bool static_words = false;
    // Link-rate model (fo_overlap_set_link_rate): bytes per second a collective over the group's bytes would
    // sustain; 0: none.  With a rate every consumer launch is followed on its stream by a kernel that holds the
    // stream for the bytes' link time, so that the schedule can be timed against a link-bound collective on
    // one GPU.
    double link_bytes_per_s = 0;
};

namespace {

// With a link rate the automatic choices go to per-wave launches on the second stream: the link time
// follows each consumer launch, and it is what the second stream is there to hide.
//
// Longer GEMMs stay on one stream too where there is nothing to overlap: `idle`, a call without a consumer and without a
// normalisation (4224x7168x3584 221 -> 215 us, 3712x8192x3456 216 -> 207) or as the reduce-scatter says, and a product of at most one round of 256x256
// tiles, whose groups all complete at its end, so that the second stream adds its launches and polls and hides
// nothing (us, two streams -> one: 2304x4096x3560 96 -> 83, 1792x4608x4520 125 -> 108, 2048x4224x6968 256 -> 167,
// 2176x5888x3312 133 -> 127, 4096x4096x4096 133 -> 125, 2048x8192x3000 128 -> 118).  `scatter`, a reduce-scatter: up to five
// sixths of a round, with launches behind the GEMM (4096x4096x2560 with four ranks 98 -> 100).  in_stream_below_flop = 0 still asks for two streams always.
//
// `ragged`, a call that could do either and whose M or N is an odd multiple of 128: a launch that counts keeps the order of
// the groups in the Algo's own tile (plan_launch), one that does not takes 256x256 tiles with half tiles at the end, and
// what that saves is more than the second stream hides (us, two streams -> one, with an accumulator and the normalisation:
// 3456x4352x3072 127 -> 93, 2432x7040x7056 271 -> 245, 8064x8064x4096 586 -> 465, 6272x8192x7168 661 -> 636; reduce-scatter,
// eight ranks: 3456x4352x3072 123 -> 95, 4224x7168x3584 205 -> 194, 6272x8192x7168 651 -> 630, 8192x8064x7168 801 -> 703).
// `fits`: the accumulator is one that every path takes; one that is not aligned is left to the one-launch consumer.
bool in_stream(const fo_overlap *h, int M, int N, int K, bool idle, bool monitor, bool ragged, bool fits, bool scatter) {
    if (h->overlap_ready && !h->comm_stream) return true;  // (a planner's handle may not have been initialised)
    if (h->fused >= 0 || h->link_bytes_per_s > 0 || h->in_stream_below_flop <= 0) return false;
    if (2.0 * M * N * K < h->in_stream_below_flop) return true;
    if (monitor || !fits) return false;  // the monitor's GEMM counts and is waited for in any case
    return idle || ragged || (long)((M + 255) / 256) * ((N + 255) / 256) * 6 <= (long)fo_main_tile_resident() * (scatter ? 5 : 6);
}

// An all-reduce that could do either, longer than all of those: whether the GEMM's epilogue, which does the sums while the tile
// is in LDS and asks for the accumulator's values during the product, costs less than the consumer beside the GEMM, which reads
// the product back and takes bandwidth and power from it, and the last wave's behind it.  Whole calls with an accumulator, us, two
// streams -> one.  Without the normalisation up to four waves: 8192x8192x1024 205 -> 195, 6144x8192x3072 bf16 308 -> 298,
// 4096x8192x8192 438 -> 431, 8192x8192x8192 bf16 811 -> 806; eight, 16384x8192x2048, 570 -> 579.  With it the second stream also
// brings the rows of each wave that is whole rows (xcd_remap 2), which one stream has to leave for the end: 6144x8192x2048 217 ->
// 227, 16384x8192x1024 366 -> 384, 8192x8192x3584 bf16 396 -> 407; not with few columns of K (8192x8192x512 161 -> 149, 16384x8192x512
// 301 -> 300, 6144x8192x768 142 -> 146), nor with two waves, of which only the first is beside the GEMM (8192x4096x1024 115 -> 104,
// 8192x4096x3072 205 -> 199, x4096 245 -> 247).  Where waves are not whole rows there is nothing to bring: 5120x8192x1024 156 -> 142,
// 6144x6144x4096 301 -> 286, 8192x7168x4096 bf16 439 -> 411, 7168x8192x8192 777 -> 767.
// `one_launch`, so many groups that one polling launch would consume them and the rows follow at the end: one stream at every
// size measured (8192x8192x3584 bf16 in 32 groups 430 -> 409, 8192x8192x8192 in 64 847 -> 828, 8192x8192x2048 in 1024 333 -> 281,
// 4096x8192x4096 in 20 261 -> 241; without the normalisation 16384x8192x1024 in 40 441 -> 375, x4096 bf16 in 100 902 -> 882).
constexpr int kRowsWaitFromK = 640, kRowsWaitTwoWavesFromK = 3584;
bool epilogue_sums(int algo, int M, int N, int K, bool norm, bool one_launch) {
    const long tiles = (long)((M + 255) / 256) * ((N + 255) / 256), wave = fo_main_tile_resident();
    if (one_launch) return true;
    if (!norm) return tiles <= 4 * wave;
    fo_raster r;
    if (fo_pick_raster(algo, M, N, &r)) return false;
    return r.xcd_remap != 2 || K < kRowsWaitFromK || (tiles <= 2 * wave && K < kRowsWaitTwoWavesFromK);
}

int fused_grid(const fo_overlap *h, int G) {  // 0: per-group launches, otherwise workgroups of the one launch
    if (h->fused < 0) return G > h->fused_from_groups && h->link_bytes_per_s <= 0 ? 256 : 0;
    if (h->fused == 1) return 256;
    return h->fused;
}

// Pause between a workgroup's polls in the one-launch consumer: 100 ns per
// workgroup keeps the GEMM's slowdown near one percent, but no more than about
// a sixtieth of the GEMM's expected duration, so that a short problem is not
// left waiting for a sleeping poller.
int fused_poll_gap_ns(int M, int N, int K, int grid) {
    const double gemm_ns = 2.0 * M * N * K / kGemmFlopPerNs;
    double gap = grid * 100.0;
    if (gap > gemm_ns / 60) gap = gemm_ns / 60;
    if (gap < 500) gap = 500;
    return (int)gap;
}

// Pieces per group for the one-launch consumer: about 32 KiB each, at most one per workgroup.
int fused_slices(int64_t total_elems, int G, int grid) {
    const int64_t per_group = total_elems / G;
    int64_t s = per_group / 16384;
    if (s < 1) s = 1;
    if (s > grid) s = grid;
    return (int)s;
}

// Groups [i, j) that complete in the same wave of the persistent GEMM (their last
// tiles fall into the same stretch of `wave` consecutive storage slots, which
// is the order the hint assigns) are waited for by one launch: they become
// ready within microseconds of each other, and a launch per group would only
// add its latency to the tail.  done = tiles of the groups before i.
int batch_end(const int32_t *cseg_host, int G, int i, long done, int wave) {
    if (wave <= 0) return i + 1;
    const long w = (done + cseg_host[i] - 1) / wave;
    int j = i + 1;
    long d = done + cseg_host[i];
    while (j < G && (d + cseg_host[j] - 1) / wave == w) d += cseg_host[j++];
    return j;
}

// Storage slots of the batches in front of the last.
long slots_before_last_batch(const int32_t *cseg_host, int G, int wave) {
    long done = 0;
    for (int i = 0; i < G;) {
        const int j = batch_end(cseg_host, G, i, done, wave);
        if (j == G) break;
        for (; i < j; i++) done += cseg_host[i];
    }
    return done;
}

// Link time of `bytes` on `stream` (nothing without a rate).
int link_time(const fo_overlap *h, int64_t bytes, fo_stream_t stream) {
    if (h->link_bytes_per_s <= 0 || bytes <= 0) return FO_OK;
    return fo_pace_with((double)bytes / h->link_bytes_per_s, stream);
}

// Asked before a call enqueues anything: the largest stretch it could ask for (all of C) must be one that
// fo_pace_with accepts, so that a refusal cannot come between the fork and the join.
int link_fits(const fo_overlap *h, int64_t bytes) {
    if (h->link_bytes_per_s <= 0) return FO_OK;
    return (double)bytes / h->link_bytes_per_s > kMaxPaceSeconds ? FO_ERR_LIMIT : FO_OK;
}

int check_segments(const int32_t *cseg_host, int G, long tiles) {
    if (!cseg_host || G <= 0) return FO_ERR_SEGMENTS;
    long sum = 0;
    for (int i = 0; i < G; i++) {
        if (cseg_host[i] <= 0) return FO_ERR_SEGMENTS;
        sum += cseg_host[i];
    }
    return sum == tiles ? FO_OK : FO_ERR_SEGMENTS;
}

// Whether `out` (elements of 16 bits) shares no memory with any of the others.  A GEMM whose epilogue also writes `out`
// writes it while other workgroups still read operands; one that is followed by a consumer does not.
struct span {
    const void *p;
    int64_t n;
};
bool apart(span out, std::initializer_list<span> others) {
    const uintptr_t a = (uintptr_t)out.p, a_end = a + out.n * 2;
    for (const span &o : others) {
        const uintptr_t b = (uintptr_t)o.p;
        if (out.p && o.p && a < b + o.n * 2 && b < a_end) return false;
    }
    return true;
}

// Whether the consumer launches take these buffers (16-byte accesses; null: none).
bool aligned(const void *C, const void *acc, const void *own = nullptr) {
    return !(((uintptr_t)C | (uintptr_t)acc | (uintptr_t)own) & 15);
}

// While the GEMM stream is being captured into a HIP graph the two streams are tied
// together with events, as in the reference (src/overlap_impl.cu:246, :260-263): the
// event wait pulls the consumer stream into the capture, and in the graph the dependency
// is an edge, not a wait at run time.
bool capturing(const fo_overlap *h) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(h->gemm_stream, &st) != hipSuccess) return false;
    return st == hipStreamCaptureStatusActive;
}

// GEMM stream -> consumer stream, right before the GEMM is enqueued.  Outside a capture it
// goes through memory (a one-lane set on the GEMM stream, a one-lane wait on the other) and
// only the one-launch consumer needs it: its workgroups poll from the moment they start,
// and polls slow down whatever shares the memory system with them, so they must not start
// while the GEMM stream is still busy with the work that precedes the GEMM (the
// reference's wait kernels may start early: a single sleeping lane disturbs nobody).
int fork(fo_overlap *h, bool captured, bool polling_consumer) {
    if (captured) {
        if (!h->forked || !h->joined) return FO_ERR_STATE;  // a handle-free call has no events to capture with
        FO_HIP_CHECK(hipEventRecord(h->forked, h->gemm_stream));
        FO_HIP_CHECK(hipStreamWaitEvent(h->comm_stream, h->forked, 0));
        return FO_OK;
    }
    if (!polling_consumer && !h->static_words) return FO_OK;
    int rc = fo_set(h->workspace + kWsFork, h->token, h->gemm_stream);
    if (rc) return rc;
    return fo_wait_with(h->token, h->workspace + kWsFork, h->max_polls, h->workspace + kWsGaveUp, h->comm_stream);
}

// consumer stream -> GEMM stream.  The reference records an event on the consumer stream
// and makes the GEMM stream wait for it (src/overlap_impl.cu:260-263); an event wait across
// queues measured about 12 us here, so outside a capture the join goes through memory: a
// one-lane kernel at the end of the consumer stream sets the workspace's join word (stream order
// makes all earlier work there complete and visible first), a one-lane wait behind the
// GEMM on the GEMM's stream consumes it.  The wait cannot start before the GEMM has ended
// and everything it waits for was enqueued before it; the GEMM stream continues about 4 us
// after the consumer's end.
int join(fo_overlap *h, bool captured) {
    if (captured) {
        FO_HIP_CHECK(hipEventRecord(h->joined, h->comm_stream));
        FO_HIP_CHECK(hipStreamWaitEvent(h->gemm_stream, h->joined, 0));
        return FO_OK;
    }
    int rc = fo_set(h->workspace + kWsJoin, h->token, h->comm_stream);
    if (rc) return rc;
    return fo_wait_with(h->token, h->workspace + kWsJoin, h->max_polls, h->workspace + kWsGaveUp, h->gemm_stream);
}

}  // namespace

extern "C" int fo_overlap_plan_batches(const int32_t *cseg_host, int G, int wave_tiles, int32_t *first) {
    if (!cseg_host || !first || G <= 0) return FO_ERR_ARG;
    for (int i = 0; i < G; i++)
        if (cseg_host[i] <= 0) return FO_ERR_SEGMENTS;
    int n = 0;
    long done = 0;
    for (int i = 0; i < G;) {
        const int j = batch_end(cseg_host, G, i, done, wave_tiles);
        first[n++] = i;
        for (int g = i; g < j; g++) done += cseg_host[g];
        i = j;
    }
    first[n] = G;
    return n;
}

extern "C" int fo_overlap_create(fo_overlap_t **out) {
    if (!out) return FO_ERR_ARG;
    *out = new (std::nothrow) fo_overlap();
    return *out ? FO_OK : FO_ERR_ARG;
}

extern "C" int fo_overlap_destroy(fo_overlap_t *h) {
    if (!h) return FO_ERR_ARG;
    // release everything even if one step fails; report the first failure
    hipError_t first = hipSuccess;
    auto note = [&](hipError_t e) {
        if (first == hipSuccess) first = e;
    };
    if (h->comm_stream) {
        note(hipStreamSynchronize(h->comm_stream));
        note(hipStreamDestroy(h->comm_stream));
    }
    if (h->forked) note(hipEventDestroy(h->forked));
    if (h->joined) note(hipEventDestroy(h->joined));
    if (h->workspace) note(hipFree(h->workspace));
    delete h;
    return (int)first;
}

extern "C" int fo_overlap_set_gemm_stream(fo_overlap_t *h, fo_stream_t gemm_stream) {
    if (!h) return FO_ERR_ARG;
    h->gemm_stream = static_cast<hipStream_t>(gemm_stream);
    h->gemm_ready = true;
    return FO_OK;
}

extern "C" int fo_overlap_init(fo_overlap_t *h) {
    if (!h) return FO_ERR_ARG;
    if (h->overlap_ready) return FO_OK;
    // Default priority on purpose (the reference asks for priority -5,
    // src/overlap_impl.cu:140): mixed-priority streams are avoided on this platform.
    FO_HIP_CHECK(hipStreamCreateWithFlags(&h->comm_stream, hipStreamNonBlocking));
    FO_HIP_CHECK(hipEventCreateWithFlags(&h->forked, hipEventDisableTiming));
    FO_HIP_CHECK(hipEventCreateWithFlags(&h->joined, hipEventDisableTiming));
    FO_HIP_CHECK(hipMalloc(&h->workspace, kWorkspaceWords * sizeof(int32_t)));
    FO_HIP_CHECK(hipMemset(h->workspace, 0, kWorkspaceWords * sizeof(int32_t)));
    h->overlap_ready = true;
    return FO_OK;
}

extern "C" int fo_overlap_set_world(fo_overlap_t *h, int rank, int world) {
    if (!h || world <= 0 || rank < 0 || rank >= world) return FO_ERR_ARG;
    h->rank = rank;
    h->world = world;
    return FO_OK;
}

extern "C" int fo_overlap_set_accumulator(fo_overlap_t *h, void *acc, int64_t nelem) {
    if (!h || nelem < 0) return FO_ERR_ARG;
    h->acc = acc;
    h->acc_nelem = acc ? nelem : 0;
    return FO_OK;
}

extern "C" int fo_overlap_set_fused_consumer(fo_overlap_t *h, int fused) {
    if (!h) return FO_ERR_ARG;
    h->fused = fused < 0 ? -1 : fused;
    return FO_OK;
}

extern "C" int fo_overlap_set_wait_limit(fo_overlap_t *h, int64_t max_polls) {
    if (!h || max_polls < -1) return FO_ERR_ARG;
    h->max_polls = (long)max_polls;
    return FO_OK;
}

extern "C" int fo_overlap_set_schedule(fo_overlap_t *h, double in_stream_below_flop, int fused_from_groups) {
    if (!h) return FO_ERR_ARG;
    h->in_stream_below_flop = in_stream_below_flop < 0 ? kInStreamBelowFlop : in_stream_below_flop;
    h->fused_from_groups = fused_from_groups < 0 ? kFusedFromGroups : fused_from_groups;
    return FO_OK;
}

extern "C" int fo_overlap_set_link_rate(fo_overlap_t *h, double gigabytes_per_second) {
    if (!h || !(gigabytes_per_second >= 0)) return FO_ERR_ARG;
    h->link_bytes_per_s = gigabytes_per_second * 1e9;
    return FO_OK;
}

extern "C" int fo_overlap_status(fo_overlap_t *h, int32_t *gave_up) {
    if (!h || !gave_up) return FO_ERR_ARG;
    *gave_up = 0;
    if (!h->overlap_ready) return FO_OK;
    FO_HIP_CHECK(hipStreamSynchronize(h->comm_stream));
    if (h->gemm_ready) FO_HIP_CHECK(hipStreamSynchronize(h->gemm_stream));
    FO_HIP_CHECK(hipMemcpy(gave_up, h->workspace + kWsGaveUp, sizeof(int32_t), hipMemcpyDeviceToHost));
    // A wait that gave up may have left the fork or join word set; both streams are idle now.
    if (*gave_up) FO_HIP_CHECK(hipMemset(h->workspace, 0, kWorkspaceWords * sizeof(int32_t)));
    return FO_OK;
}

extern "C" fo_stream_t fo_overlap_comm_stream(fo_overlap_t *h) {
    return h ? static_cast<fo_stream_t>(h->comm_stream) : nullptr;
}

extern "C" int fo_overlap_gemm(fo_overlap_t *h, int dtype, int M, int N, int K, const void *A,
                               const void *B, void *C, int algo) {
    if (!h) return FO_ERR_ARG;
    if (!h->gemm_ready) return FO_ERR_STATE;
    return fo_gemm(dtype, M, N, K, A, B, C, algo, h->gemm_stream);
}

namespace {

// The reorder+RMSNorm that follows the overlapped GEMM in the reference's layers (example/RMSNorm.py:20-34
// behind example/RowParallelLinear.py:50-66), enqueued by the overlapped call itself: a tile row of the output
// can be normalised as soon as the group that holds its last tile has been consumed, so the rows follow the
// consumer batch by batch on the consumer stream and only the last batch's rows remain behind the GEMM.
struct norm_plan {
    void *Y = nullptr;
    const void *Wt = nullptr;
    float eps = 0.f;
    const int32_t *RA_host = nullptr;
};

// Rows of tile rows [first, end) of Y, on `stream`.
int norm_tile_rows(const norm_plan &np, int dtype, const void *C, int M, int N, int BM, int BN, int rLDN,
                   const int32_t *RA, int first, int end, bool beside_gemm, fo_stream_t stream) {
    return fo_norm_rows_with(dtype, C, np.Y, np.Wt, first * BM, (end - first) * BM, M, N, BM, BN, rLDN, RA, np.eps,
                             fo_streams((int64_t)M * N * 4), beside_gemm, 0, stream);
}

// Tile rows whose tiles all lie in storage slots below `done` and that have not been normalised yet, as
// runs of consecutive tile rows [first, end); at most kMaxRuns runs per batch (a reorder table that scatters the
// rows of a wave leaves the rest to the last batch, which takes everything that is left).
// last_slot[tm] = largest slot of tile row tm; -1 once handed out.  Appends to `runs`.
constexpr int kMaxRuns = 4;
void ready_tile_rows(long *last_slot, int TM, long done, bool final_batch, std::vector<int> &runs) {
    int n = 0;
    for (int tm = 0; tm < TM;) {
        if (last_slot[tm] < 0 || last_slot[tm] >= done) {
            tm++;
            continue;
        }
        int end = tm;
        while (end < TM && last_slot[end] >= 0 && last_slot[end] < done) end++;
        if (!final_batch && n == kMaxRuns) break;
        runs.push_back(tm);
        runs.push_back(end);
        for (int t = tm; t < end; t++) last_slot[t] = -1;
        n++;
        tm = end;
    }
}

// Largest storage slot of every tile row of the reorder table; FO_ERR_ARG for an entry outside [0, TM*TN).
int last_slots(const int32_t *RA_host, int TM, int TN, std::vector<long> &last_slot) {
    last_slot.assign(TM, 0);
    for (int tm = 0; tm < TM; tm++)
        for (int tn = 0; tn < TN; tn++) {
            const long r = RA_host[(long)tm * TN + tn];
            if (r < 0 || r >= (long)TM * TN) return FO_ERR_ARG;
            if (r > last_slot[tm]) last_slot[tm] = r;
        }
    return FO_OK;
}

// Whether batches that are whole tile rows are consumed and normalised by one kernel, which reads C once for both.  `last`:
// the batch behind the GEMM, where the one kernel is the faster in any case (28 us instead of 17 + 12 and a launch on 8192
// columns; whole call, us, 4096x8192x4096 241.6 -> 236.1, 8192x2048x4096 135.2 -> 129.9).
// Beside the GEMM it depends on how long a wave of it lasts.  In a short one the consumer and the rows (61 + 30 to 55 us
// for a quarter of 8192x8192, together 71) fall behind if they follow one another; a long one has time for that, and a
// consumer of one wavefront per CU takes less from it.  Whole call, us, one after the other and together beside the GEMM, 8192
// columns: fp16, 8192 rows, K = 1536 236 and 228, 2048 273.5 and 271.9, 2560 321.6 and 314.3, 3072 370.4 and 370.1, 3328
// 378.6 and 385.0, 3584 401.2 and 409.2, 4096 442.3 and 454.4, 6144 651 and 658, 8192 815 and 830; bf16 239 and 222, 268 and 262,
// 323 and 302, 363 and 361, 367 and 372, 388 and 395, 425 and 432, 631 and 629, 778 and 789; 16384x4096 bf16 K = 2048 278 and
// 258, 3072 379.5 and 371.7, 3584 397 and 402, 8192 778 and 781.  Rows of up to 2048 elements are the faster together at
// every K (16384x2048 fp16 3584 225 and 222, 8192 427 and 422; 65536x1024 3584 462 and 445, 8192 851 and 846).
// The kernel's registers (at most 128) fit beside the 256x256 kernel that counts, and not beside 128x256 tiles that do, no
// more than the row kernel's by itself.  Those tiles are taken where 256 does not divide M or N; a batch is whole rows there
// in an order of the caller's only, much of it follows the GEMM, and the one kernel is the faster at every K (rows in row-major
// order, fp16: 8064x8192 by 128x256 tiles, K = 1600 328 and 302, 4096 564 and 547, 7168 890 and 869; by 128x128 tiles 4096 699
// and 657; 8064x4096x8192 497 and 482).
// Rows in more than one run are in an order that the GEMM does not follow: such a batch is complete late, when little is
// left of the GEMM, and a launch for each run is the faster than one consumer launch and a launch for each run's rows
// (8192x8192 fp16 in four batches of two, of four runs: K = 2048 309 and 291, 339 and 323, 3584 438 and 412, 473 and 449, 8192
// 831 and 829, 880 and 862).
// Shorter rows leave most of the workgroup's lanes idle in what was the consumer's traffic (us, by two kernels and by one, fp16
// / bf16: 131072x256x4096 480 and 523 / 498 and 544, 65536x512x2048 218 and 227 / 230 and 240.5; 32768x1024x4096 257
// and 251 / 251 and 242).
bool rows_together(int M, int N, int K, int BN, int rLDN, int runs, bool last) {
    const bool ragged = M % 256 || N % 256;
    return fo_consumes_norm_rows(M, N, BN, rLDN) && N >= kTogetherFromN &&
           (last || ragged || runs > 1 || K <= kTogetherUpToK || N <= kTogetherAnyKUpToN);
}

// Whether a batch that fills the storage slots [done, done + tiles) is exactly the tile rows `runs` it completes.
bool whole_rows(const int32_t *RA_host, int TN, const std::vector<int> &runs, long done, long tiles) {
    long rows = 0;
    for (size_t k = 0; k + 1 < runs.size(); k += 2) {
        rows += runs[k + 1] - runs[k];
        for (long t = (long)runs[k] * TN; t < (long)runs[k + 1] * TN; t++)
            if (RA_host[t] < done) return false;  // the rows' largest slot lies in the batch: asked before
    }
    return rows * TN == tiles;
}

int check_slots(const int32_t *RA_host, int T) {  // FO_ERR_ARG for an entry outside [0, T)
    uint32_t most = 0;
    for (int t = 0; t < T; t++) most = (uint32_t)RA_host[t] > most ? (uint32_t)RA_host[t] : most;
    return most < (uint32_t)T ? FO_OK : FO_ERR_ARG;
}

int norm_runs(const norm_plan &np, const std::vector<int> &runs, int dtype, const void *C, int M, int N, int BM, int BN, int rLDN,
              const int32_t *RA, bool beside_gemm, fo_stream_t stream) {
    for (size_t k = 0; k + 1 < runs.size(); k += 2) {
        int rc = norm_tile_rows(np, dtype, C, M, N, BM, BN, rLDN, RA, runs[k], runs[k + 1], beside_gemm, stream);
        if (rc) return rc;
    }
    return FO_OK;
}

// Whether the accumulator shares no memory with operands and product.
bool accumulator_apart(const fo_overlap *h, int M, int N, int K, const void *A, const void *B, const void *C) {
    const int64_t mn = (int64_t)M * N;
    return h->acc && apart({h->acc, mn}, {{A, (int64_t)M * K}, {B, (int64_t)N * K}, {C, mn}});
}

// Whether an all-reduce stays on the GEMM stream.  fits: the consumer launches take the buffers.
bool allreduce_in_stream(const fo_overlap *h, int M, int N, int K, int G, int algo, bool norm, bool monitor, bool fits, bool acc_apart) {
    const bool automatic = h->fused < 0 && h->link_bytes_per_s <= 0 && h->in_stream_below_flop > 0;
    return in_stream(h, M, N, K, !h->acc && !norm, monitor, M % 256 || N % 256, fits, false) ||
           (automatic && !monitor && fits && acc_apart && epilogue_sums(algo, M, N, K, norm, fused_grid(h, G) != 0));
}

// An all-reduce that chose two streams and launches per batch by itself: the storage slot from which on the GEMM does the sums
// itself (M * N / (BM * BN): nowhere).  Those of the last wave: nothing is left to overlap them with, and behind
// the GEMM they are a wait, a launch and a second read of the product (17 + 4 us on 4096x8192, of which the GEMM's epilogue
// takes 17).  Where the groups' ends are not the waves', the consumer also need not wait for the last wave to begin with the
// rest of its first group.  Whole calls, us, consumer -> GEMM: groups across waves, 8192x8192x2048 in one 288 -> 274, 8192x4096x4096
// in three 253 -> 242, by the pair of calls 8192x4096x2560 in one 203 -> 184; groups that end with waves, by the pair
// 4096x8192x8192 422 -> 419, 8192x8192x8192 828 -> 824.  There the call that also normalises keeps its one kernel for the last
// batch's sums and rows (4096x8192x1536 131 against 135 with sums in the GEMM).
//
// The rows that the last wave completes then follow on the GEMM stream, while the consumer's may still read the product and update
// the accumulator, and rows of earlier waves may be written while the GEMM reads its operands: only rows that share memory with
// none of these.
int allreduce_sum_from(const fo_overlap *h, int M, int N, int K, int rLDN, int BN, const int32_t *cseg_host, int G, int wave, int algo,
                       const void *A, const void *B, const void *C, const norm_plan *np, bool monitor, bool acc_apart,
                       int32_t *sum_from) {
    const int64_t mn = (int64_t)M * N;
    int32_t first = 0;
    int rc = fo_gemm_last_wave(algo, M, N, &first, sum_from);
    if (rc) return rc;
    if (h->fused >= 0 || fused_grid(h, G) || monitor || h->link_bytes_per_s > 0 || !acc_apart) return FO_OK;
    if (!fo_block_in_range((int64_t)rLDN * BN)) return FO_OK;
    if (np && !(apart({np->Y, mn}, {{A, (int64_t)M * K}, {B, (int64_t)N * K}, {C, mn}, {h->acc, mn}}) &&
                apart({h->acc, mn}, {{np->Wt, N}})))
        return FO_OK;
    if (!np || slots_before_last_batch(cseg_host, G, wave) < first) *sum_from = first;
    return FO_OK;
}

// GemmAllReduceOverlap on whatever `h` describes: a caller's handle, or the
// streams and static workspace of a handle-free call.  np: the normalisation to enqueue behind the consumer
// (null: none).
int allreduce_overlap(fo_overlap *h, int dtype, int M, int N, int K, const void *A, const void *B, void *C,
                      int32_t *MM, const int32_t *RA, int TM, int TN, int rLDN, const int32_t *cseg_host,
                      const int32_t *cseg_dev, int G, int algo, int monitor, const norm_plan *np = nullptr) {
    int32_t info[12];
    int rc = fo_algo_info(algo, info);
    if (rc) return rc;
    if (M <= 0 || N <= 0 || M % info[0] || N % info[1]) return FO_ERR_SHAPE;
    if (TM != M / info[0] || TN != N / info[1]) return FO_ERR_SHAPE;  // RA.shape must match the Algo's tile
    rc = check_segments(cseg_host, G, (long)TM * TN);
    if (rc) return rc;
    const int64_t tile_elems = (int64_t)info[0] * info[1];
    if (h->acc && h->acc_nelem < (int64_t)M * N) return FO_ERR_ARG;
    rc = link_fits(h, (int64_t)M * N * 2);
    if (rc) return rc;
    std::vector<long> last_slot;  // per tile row: its largest storage slot
    if (np) {
        if (!np->Y || !np->Wt || !np->RA_host) return FO_ERR_ARG;
        if (N % 8 || N > 16384 || (int64_t)M * N * 2 > 0xFFFFFFFFLL) return FO_ERR_SHAPE;
    }

    const bool fits = !h->acc || aligned(C, h->acc);
    const int64_t mn = (int64_t)M * N;
    const bool acc_apart = accumulator_apart(h, M, N, K, A, B, C);
    const bool same_stream = allreduce_in_stream(h, M, N, K, G, algo, np != nullptr, monitor != 0, fits, acc_apart);
    if (np) {
        // on one stream all rows follow in one launch, whatever their slots
        rc = same_stream ? check_slots(np->RA_host, TM * TN) : last_slots(np->RA_host, TM, TN, last_slot);
        if (rc) return rc;
    }
    const int fused = same_stream ? 0 : fused_grid(h, G);
    fo_stream_t cstream = same_stream ? h->gemm_stream : h->comm_stream;
    int32_t wave = 0;
    if (same_stream) {
        wave = TM * TN;  // every group in one batch
    } else if (!fused) {
        rc = fo_gemm_wave_tiles(dtype, algo, M, N, &wave);
        if (rc) return rc;
    }
    // Whatever can be refused is refused here: a refusal between the launches would leave counters standing and the
    // streams apart.
    rc = fo_gemm_signal_check(dtype, M, N, K, rLDN, cseg_dev, G, A, B, C, MM, RA, nullptr, monitor, algo);
    if (rc) return rc;
    if (!fused && !fits) return FO_ERR_SHAPE;
    int32_t sum_from = TM * TN;
    if (!same_stream) {
        rc = allreduce_sum_from(h, M, N, K, rLDN, info[1], cseg_host, G, wave, algo, A, B, C, np, monitor != 0, acc_apart, &sum_from);
        if (rc) return rc;
    }
    const bool captured = !same_stream && capturing(h);
    if (h->static_words) {
        // By a kernel, not a memset node, in case the GEMM stream is being captured.  The give-up word is left standing:
        // fo_static_status reads and clears it.
        rc = fo_fill_words(h->workspace, kWorkspaceWords + G, 0, h->gemm_stream, kWsGaveUp);
        if (rc) return rc;
    }
    if (!same_stream) {
        rc = fork(h, captured, fused != 0);
        if (rc) return rc;
    }
    // On one stream the order of the launches is all the synchronisation there is
    // to do: unless the caller wants the monitor's stamps, the GEMM then leaves
    // the counters alone (they stay zero, as the waits would have left them).
    const bool quiet = same_stream && !monitor;
    // With nothing to wait for, the GEMM's epilogue does the consumer's work on the tile it holds in LDS.
    const bool consumed = quiet && acc_apart;
    const bool sums_last = sum_from < TM * TN;  // the last wave's sums by the GEMM itself
    rc = sums_last  ? fo_gemm_signal_sums(dtype, M, N, K, rLDN, cseg_dev, G, A, B, C, MM, RA, nullptr, h->acc, sum_from, nullptr, 1, 0,
                                          algo, h->gemm_stream)
         : consumed ? fo_gemm_accumulate(dtype, M, N, K, rLDN, cseg_dev, G, A, B, C, h->acc, RA, algo, h->gemm_stream)
         : quiet  ? fo_gemm_reordered_quiet(dtype, M, N, K, rLDN, cseg_dev, G, A, B, C, RA, nullptr, algo,
                                            h->gemm_stream)
                  : fo_gemm_signal(dtype, M, N, K, rLDN, cseg_dev, G, A, B, C, MM, RA, monitor, algo,
                                h->gemm_stream);
    if (rc) return rc;  // the GEMM was refused: nothing of this call follows on either stream

    // C' and the accumulator together against the memory-side cache
    const bool stream_acc = fo_streams((int64_t)M * N * 4);
    if (fused) {
        rc = fo_wait_reduce_groups_with(dtype, C, h->acc, MM, cseg_dev, G, tile_elems, 1, 0, nullptr, 0,
                                        h->workspace, fused, fused_slices((int64_t)M * N, G, fused),
                                        fused_poll_gap_ns(M, N, K, fused), stream_acc, h->max_polls, h->comm_stream);
        if (rc) return rc;
        rc = link_time(h, (int64_t)M * N * 2, h->comm_stream);
        if (rc) return rc;
        if (np) {  // that launch ends when the last group has been consumed: every row at once
            rc = norm_tile_rows(*np, dtype, C, M, N, info[0], info[1], rLDN, RA, 0, TM, false, h->comm_stream);
            if (rc) return rc;
        }
    } else {
        int64_t off = 0;
        long done = 0;
        uint16_t *c = static_cast<uint16_t *>(C);
        uint16_t *acc = static_cast<uint16_t *>(h->acc);
        const bool consumes_rows = np && acc && !same_stream && h->link_bytes_per_s <= 0 &&
                                   apart({acc, mn}, {{C, mn}, {np->Y, mn}, {np->Wt, N}}) &&
                                   apart({np->Y, mn}, {{C, mn}});  // the accumulator takes the product, not rows written over it
        for (int i = 0; i < G;) {
            const int j = batch_end(cseg_host, G, i, done, wave);
            long tiles = 0;
            for (int g = i; g < j; g++) tiles += cseg_host[g];
            // The batch that the last wave completes: what is left to the consumer is the beginning of its first group, if
            // that began in an earlier wave.  The GEMM counts no more of it than that.
            const bool last_wave = done + tiles > sum_from;
            if (last_wave) tiles = done < sum_from ? sum_from - done : 0;
            const int64_t n = tiles * tile_elems;
            if (last_wave && !tiles) break;
            if (!quiet) {
                int32_t *gave_up = h->workspace ? h->workspace + kWsGaveUp : nullptr;
                rc = last_wave  ? fo_wait_with((int)tiles, MM + i, h->max_polls, gave_up, cstream)
                     : j - i == 1 ? fo_wait_with(cseg_host[i], MM + i, h->max_polls, gave_up, cstream)  // resets the counter
                                : fo_wait_groups_with(j - i, cseg_dev + i, MM + i, h->max_polls, gave_up, cstream);
                if (rc) return rc;
            }
            std::vector<int> runs;
            const bool behind_gemm = j == G && !last_wave;  // every batch but the last runs beside the GEMM
            if (np && !same_stream) ready_tile_rows(last_slot.data(), TM, done + tiles, behind_gemm, runs);
            const bool with_rows = consumes_rows && rows_together(M, N, K, info[1], rLDN, (int)runs.size() / 2, behind_gemm) &&
                                   whole_rows(np->RA_host, TN, runs, done, tiles);
            if (acc && !consumed && !with_rows) {  // the groups of a batch are one contiguous range
                rc = fo_consumer_reduce_with(dtype, c + off, acc + off, n, 1, 0, nullptr, 0, stream_acc, cstream,
                                             !behind_gemm && !same_stream);
                if (rc) return rc;
            }
            rc = link_time(h, n * 2, cstream);
            if (rc) return rc;
            off += n;
            done += tiles;
            if (np && same_stream) {
                rc = norm_tile_rows(*np, dtype, C, M, N, info[0], info[1], rLDN, RA, 0, TM, false, cstream);
                if (rc) return rc;
            } else if (with_rows) {
                for (size_t k = 0; k + 1 < runs.size(); k += 2) {
                    rc = fo_consume_norm_rows_with(dtype, C, acc, np->Y, np->Wt, runs[k] * info[0], (runs[k + 1] - runs[k]) * info[0], M, N,
                                                   info[0], info[1], RA, np->eps, fo_streams(mn * 4), !behind_gemm, cstream);
                    if (rc) return rc;
                }
            } else if (np) {
                rc = norm_runs(*np, runs, dtype, C, M, N, info[0], info[1], rLDN, RA, !behind_gemm, cstream);
                if (rc) return rc;
            }
            i = j;
        }
        if (sums_last && np) {  // the rows that the last wave completed: nothing but the GEMM in front of them
            std::vector<int> runs;
            ready_tile_rows(last_slot.data(), TM, (long)TM * TN, true, runs);
            rc = norm_runs(*np, runs, dtype, C, M, N, info[0], info[1], rLDN, RA, false, h->gemm_stream);
            if (rc) return rc;
        }
    }
    return same_stream ? FO_OK : join(h, captured);
}

}  // namespace

// Which tile rows fo_overlap_gemm_allreduce_norm normalises behind which batch of groups, for a caller that wants
// to know (and for tests on a machine without a GPU): the same planner the call uses.
extern "C" int fo_overlap_plan_norm_rows(const int32_t *RA_host, int TM, int TN, const int32_t *cseg_host, int G,
                                         int wave_tiles, int32_t *runs, int max_runs) {
    if (!RA_host || !runs || TM <= 0 || TN <= 0 || max_runs <= 0) return FO_ERR_ARG;
    int rc = check_segments(cseg_host, G, (long)TM * TN);
    if (rc) return rc;
    std::vector<long> last_slot;
    rc = last_slots(RA_host, TM, TN, last_slot);
    if (rc) return rc;
    int n = 0, batch = 0;
    long done = 0;
    for (int i = 0; i < G; batch++) {
        const int j = batch_end(cseg_host, G, i, done, wave_tiles);
        for (int g = i; g < j; g++) done += cseg_host[g];
        std::vector<int> ready;
        ready_tile_rows(last_slot.data(), TM, done, j == G, ready);
        for (size_t k = 0; k + 1 < ready.size(); k += 2) {
            if (n == max_runs) return FO_ERR_LIMIT;
            runs[3 * n] = batch;
            runs[3 * n + 1] = ready[k];
            runs[3 * n + 2] = ready[k + 1];
            n++;
        }
        i = j;
    }
    return n;
}

// Whether the call consumes and normalises a batch of whole tile rows by one kernel.
extern "C" int fo_overlap_plan_rows_together(int M, int N, int K, int BN, int rLDN, int runs, int last) {
    if (M <= 0 || N <= 0 || K <= 0 || BN <= 0 || rLDN <= 0 || runs <= 0) return FO_ERR_ARG;
    return rows_together(M, N, K, BN, rLDN, runs, last != 0) ? 1 : 0;
}

namespace {

// What both planners below refuse, and the Algo's tile.
int check_plan(const fo_overlap *h, int M, int N, int K, int rLDN, const int32_t *cseg_host, int G, int algo, int32_t *info) {
    if (!h || K <= 0) return FO_ERR_ARG;
    int rc = fo_algo_info(algo, info);
    if (rc) return rc;
    if (M <= 0 || N <= 0 || M % info[0] || N % info[1]) return FO_ERR_SHAPE;
    const long tiles = (long)(M / info[0]) * (N / info[1]);
    if (rLDN <= 0 || tiles % rLDN) return FO_ERR_SHAPE;
    return check_segments(cseg_host, G, tiles);
}

}  // namespace

// What the calls do with these buffers (whose addresses alone are looked at), for a caller that wants to know and for tests on a
// machine without a GPU: the functions the calls decide by.
extern "C" int fo_overlap_plan_allreduce(const fo_overlap_t *h, int M, int N, int K, const void *A, const void *B, const void *C,
                                         const void *Y, const void *Wt, int rLDN, const int32_t *cseg_host, int G, int wave_tiles,
                                         int algo, int monitor) {
    int32_t info[12], sum_from = 0;
    int rc = check_plan(h, M, N, K, rLDN, cseg_host, G, algo, info);
    if (rc) return rc;
    norm_plan np;
    np.Y = const_cast<void *>(Y);
    np.Wt = Wt;
    const bool acc_apart = accumulator_apart(h, M, N, K, A, B, C), fits = !h->acc || aligned(C, h->acc);
    const bool same_stream = allreduce_in_stream(h, M, N, K, G, algo, Y != nullptr, monitor != 0, fits, acc_apart);
    if (!fits && (same_stream || !fused_grid(h, G))) return FO_ERR_SHAPE;
    if (same_stream) return 0;
    rc = allreduce_sum_from(h, M, N, K, rLDN, info[1], cseg_host, G, wave_tiles, algo, A, B, C, Y ? &np : nullptr, monitor != 0, acc_apart, &sum_from);
    return rc ? rc : sum_from;
}

extern "C" int fo_overlap_gemm_allreduce(fo_overlap_t *h, int dtype, int M, int N, int K,
                                         const void *A, const void *B, void *C, int32_t *MM,
                                         const int32_t *RA, int TM, int TN, int rLDN,
                                         const int32_t *cseg_host, const int32_t *cseg_dev, int G,
                                         int algo, int monitor) {
    if (!h || !MM) return FO_ERR_ARG;
    if (!h->gemm_ready || !h->overlap_ready) return FO_ERR_STATE;
    return allreduce_overlap(h, dtype, M, N, K, A, B, C, MM, RA, TM, TN, rLDN, cseg_host, cseg_dev, G, algo,
                             monitor);
}

extern "C" int fo_overlap_gemm_allreduce_norm(fo_overlap_t *h, int dtype, int M, int N, int K, const void *A,
                                              const void *B, void *C, int32_t *MM, const int32_t *RA,
                                              const int32_t *RA_host, int TM, int TN, int rLDN,
                                              const int32_t *cseg_host, const int32_t *cseg_dev, int G, int algo,
                                              int monitor, void *Y, const void *Wt, float eps) {
    if (!h || !MM) return FO_ERR_ARG;
    if (!h->gemm_ready || !h->overlap_ready) return FO_ERR_STATE;
    norm_plan np;
    np.Y = Y;
    np.Wt = Wt;
    np.eps = eps;
    np.RA_host = RA_host;
    return allreduce_overlap(h, dtype, M, N, K, A, B, C, MM, RA, TM, TN, rLDN, cseg_host, cseg_dev, G, algo, monitor,
                             &np);
}

namespace {

// How a reduce-scatter is carried out.
struct scatter_route {
    bool by_epilogue;      // whole rows of the output view are each rank's, and every buffer lies apart
    bool own_in_consumer;  // the consumer also writes this rank's rows
    bool fits;             // the consumer launches take the buffers
    bool same_stream;
};

scatter_route route_scatter(const fo_overlap *h, int M, int N, int K, const void *A, const void *B, const void *C, const void *D,
                            int rLDN, int G, int BM, bool monitor) {
    scatter_route r;
    const int W = h->world;
    const int64_t seg_stride = (int64_t)M * N / W;
    // Where whole rows of the output view are this rank's, the GEMM's epilogue can do what follows it on one stream: a copy
    // per group (4-5 us each on this GPU) and the consumer.  2048x4096x2048, four groups, eight ranks, no accumulator, whole
    // pass with the normalisation: 42.0 us with copies, 37.5 so.
    const span a = {A, (int64_t)M * K}, b = {B, (int64_t)N * K}, prod = {C, (int64_t)M * N}, sum = {h->acc, (int64_t)M * N};
    r.by_epilogue = rLDN == 1 && BM % W == 0 && !(((uintptr_t)C | (uintptr_t)D | (uintptr_t)h->acc) & 15) &&
                    apart(sum, {a, b, prod}) && apart({D, seg_stride}, {a, b, prod, sum});
    // With an accumulator and W > 1 the consumer also writes this rank's chunk of
    // every group to D (ncclReduceScatter(C+acc -> D+acc/W, n/W) with one rank
    // present, src/overlap_impl.cu:312-313); otherwise a copy per group does.
    r.own_in_consumer = D && h->acc && W > 1;
    r.fits = !h->acc || aligned(C, h->acc, r.own_in_consumer ? D : nullptr);
    // The epilogue leaves nothing to overlap, and what it adds to the GEMM is less than two streams cost (whole calls with the
    // normalisation, us, two streams and one): with an accumulator where there is one round, which no consumer runs beside,
    // 4096x4096x4096 130 and 120, 4096x4096x8192 bf16 212 and 203; and where groups are so many that one polling launch would
    // consume them, 4096x8192x4096 bf16 in twenty 244 and 225, 8192x8192x3584 bf16 in 32 415 and 401, 8192x8192x8192 in 64 835
    // and 819, 16384x8192x2048 in 64 564 and 558.  Fewer groups and more rounds are left to the consumer: two rounds are the same
    // either way (8192x4096x4096 in eight 234 and 234, 4096x8192x1536 129 and 128), four are not (8192x8192x3584 bf16 387 and 401).
    // Without an accumulator all there is to overlap are copies, and many take longer than the GEMM (8192x4096x4096 in 24
    // groups 284, on one stream 215).  Up to sixteen groups stay on two streams, where their counters are waited for and reset,
    // which a caller can see, at 1 to 9 % (16384x8192x1024 285 and 273, 8192x4096x4096 in sixteen 201 and 196).
    const bool one_round = (long)((M + 255) / 256) * ((N + 255) / 256) <= (long)fo_main_tile_resident();
    const bool idle = r.by_epilogue && (h->acc ? one_round || fused_grid(h, G) != 0 : G > kFewCopies);
    // A ragged call's gain on one stream (see in_stream) is there by the epilogue (us, eight ranks, two streams' 8064x8064x7168 in
    // four groups with launches behind the GEMM 750, so 719) and with one consumer launch for all groups or a few copies behind it.
    const bool few_copies = !h->acc && G <= (2.0 * M * N * K >= kManyCopiesFromFlop ? kFewCopies : kFewCopiesOfShort);
    const bool ragged = (M % 256 || N % 256) && (r.by_epilogue || (h->acc && W > 1) || few_copies);
    r.same_stream = in_stream(h, M, N, K, idle, monitor, ragged, r.fits, true);
    return r;
}

// A reduce-scatter that chose two streams and launches per batch by itself: the storage slot from which on the GEMM does the
// rest itself (M * N / (BM * BN): nowhere).  The last batch's sums and rows, where that batch is of the last wave only (us:
// 8192x4096x4096, eight ranks 235.6 -> 230.4, 8192x8192x3584 bf16 398 -> 389, 4096x8192x2048 bf16 146.7 -> 143.3).
// Without an accumulator this rank's rows of those groups, else a copy per group behind the GEMM (8192x4096x4096 bf16 in
// sixteen groups, eight ranks, 211.8 -> 203.5; 8192x4096x2048 in four, four ranks, 124.0 -> 122.5).
int scatter_sum_from(const fo_overlap *h, const scatter_route &r, int M, int N, const void *D, const int32_t *cseg_host, int G,
                     int wave, int algo, bool monitor, int32_t *sum_from) {
    int32_t first = 0;
    int rc = fo_gemm_last_wave(algo, M, N, &first, sum_from);
    if (rc) return rc;
    if (h->fused >= 0 || fused_grid(h, G) || monitor || h->link_bytes_per_s > 0) return FO_OK;
    if (!r.by_epilogue || !(h->acc || D) || h->world <= 1) return FO_OK;
    if ((int64_t)M * N * 2 > 0x7FFFFFFFLL) return FO_OK;  // the accumulator is read through one 31-bit buffer range
    const long before = slots_before_last_batch(cseg_host, G, wave);
    if (before >= first) *sum_from = (int32_t)before;
    return FO_OK;
}

}  // namespace

extern "C" int fo_overlap_plan_reducescatter(const fo_overlap_t *h, int M, int N, int K, const void *A, const void *B,
                                             const void *C, const void *D, int rLDN, const int32_t *cseg_host, int G,
                                             int wave_tiles, int algo, int monitor) {
    int32_t info[12], sum_from = 0;
    int rc = check_plan(h, M, N, K, rLDN, cseg_host, G, algo, info);
    if (rc) return rc;
    const scatter_route r = route_scatter(h, M, N, K, A, B, C, D, rLDN, G, info[0], monitor != 0);
    if (!r.fits && (r.same_stream || !fused_grid(h, G))) return FO_ERR_SHAPE;
    if (r.same_stream) return 0;
    rc = scatter_sum_from(h, r, M, N, D, cseg_host, G, wave_tiles, algo, monitor != 0, &sum_from);
    return rc ? rc : sum_from;
}

extern "C" int fo_overlap_gemm_reducescatter(fo_overlap_t *h, int dtype, int M, int N, int K,
                                             const void *A, const void *B, void *C, void *D,
                                             int32_t *MM, const int32_t *RA, const int32_t *RE,
                                             int TM, int TN, int rLDN, const int32_t *cseg_host,
                                             const int32_t *cseg_dev, int G, int algo, int monitor) {
    if (!h || !MM || !RE) return FO_ERR_ARG;
    if (!h->gemm_ready || !h->overlap_ready) return FO_ERR_STATE;
    int32_t info[12];
    int rc = fo_algo_info(algo, info);
    if (rc) return rc;
    if (M <= 0 || N <= 0 || M % info[0] || N % info[1]) return FO_ERR_SHAPE;
    if (TM != M / info[0] || TN != N / info[1]) return FO_ERR_SHAPE;
    rc = check_segments(cseg_host, G, (long)TM * TN);
    if (rc) return rc;
    const int W = h->world;
    const int64_t tile_elems = (int64_t)info[0] * info[1];
    if (tile_elems % (8 * W) || ((int64_t)M * N) % W) return FO_ERR_SHAPE;
    const int64_t seg_stride = (int64_t)M * N / W;
    if (h->acc && h->acc_nelem < (int64_t)M * N) return FO_ERR_ARG;
    rc = link_fits(h, (int64_t)M * N * 2);
    if (rc) return rc;

    const scatter_route route = route_scatter(h, M, N, K, A, B, C, D, rLDN, G, info[0], monitor != 0);
    const bool same_stream = route.same_stream, own_in_consumer = route.own_in_consumer;
    const int fused = same_stream ? 0 : fused_grid(h, G);
    fo_stream_t cstream = same_stream ? h->gemm_stream : h->comm_stream;
    int32_t wave = 0;
    if (same_stream) {
        wave = TM * TN;  // every group in one batch
    } else if (!fused) {
        rc = fo_gemm_wave_tiles(dtype, algo, M, N, &wave);
        if (rc) return rc;
    }
    rc = fo_gemm_signal_check(dtype, M, N, K, rLDN, cseg_dev, G, A, B, C, MM, RA, RE, monitor, algo);
    if (rc) return rc;
    if (!fused && !route.fits) return FO_ERR_SHAPE;
    int32_t sum_from = TM * TN;
    if (!same_stream) {
        rc = scatter_sum_from(h, route, M, N, D, cseg_host, G, wave, algo, monitor != 0, &sum_from);
        if (rc) return rc;
    }
    const bool captured = !same_stream && capturing(h);
    if (!same_stream) {
        rc = fork(h, captured, fused != 0);
        if (rc) return rc;
    }
    const bool quiet = same_stream && !monitor;  // as in fo_overlap_gemm_allreduce
    if (quiet && route.by_epilogue) {
        rc = fo_gemm_reduce_scatter(dtype, M, N, K, cseg_dev, G, A, B, C, h->acc, D, RA, RE, W, h->rank, algo, h->gemm_stream);
        if (rc) return rc;
        return link_time(h, (int64_t)M * N * 2, h->gemm_stream);
    }
    rc = quiet ? fo_gemm_reordered_quiet(dtype, M, N, K, rLDN, cseg_dev, G, A, B, C, RA, RE, algo,
                                         h->gemm_stream)
         : sum_from < TM * TN
             ? fo_gemm_signal_sums(dtype, M, N, K, rLDN, cseg_dev, G, A, B, C, MM, RA, RE, h->acc, sum_from, D, W, h->rank, algo,
                                   h->gemm_stream)
               : fo_gemm_scatter(dtype, M, N, K, rLDN, cseg_dev, G, A, B, C, MM, RA, RE, monitor, algo,
                                 h->gemm_stream);
    if (rc) return rc;

    uint16_t *c = static_cast<uint16_t *>(C);
    uint16_t *d = static_cast<uint16_t *>(D);
    uint16_t *acc = static_cast<uint16_t *>(h->acc);
    const bool stream_acc = fo_streams((int64_t)M * N * 4);
    if (fused) {
        rc = fo_wait_reduce_groups_with(dtype, C, h->acc, MM, cseg_dev, G, tile_elems, W, seg_stride,
                                        own_in_consumer ? D : nullptr, h->rank, h->workspace, fused,
                                        fused_slices((int64_t)M * N, G, fused), fused_poll_gap_ns(M, N, K, fused),
                                        stream_acc, h->max_polls, cstream);
        if (rc) return rc;
        rc = link_time(h, (int64_t)M * N * 2, cstream);
        if (rc) return rc;
    }
    int64_t off = 0;
    long done = 0;
    for (int i = 0; i < G;) {
        if (done >= sum_from) break;
        const int j = fused ? i + 1 : batch_end(cseg_host, G, i, done, wave);
        const int64_t off_batch = off;
        if (!fused && !quiet) {
            int32_t *gave_up = h->workspace ? h->workspace + kWsGaveUp : nullptr;
            rc = j - i == 1 ? fo_wait_with(cseg_host[i], MM + i, h->max_polls, gave_up, cstream)
                            : fo_wait_groups_with(j - i, cseg_dev + i, MM + i, h->max_polls, gave_up, cstream);
            if (rc) return rc;
        }
        if (!fused && acc && W > 1 && j - i > 1) {
            // the groups of one wave in one launch; each keeps its own W chunks
            long most = 0;
            for (int g = i; g < j; g++) most = cseg_host[g] > most ? cseg_host[g] : most;
            rc = fo_consumer_reduce_groups_with(dtype, c + off, acc + off / W, cseg_dev + i, j - i, most,
                                                tile_elems, W, seg_stride, own_in_consumer ? d + off / W : nullptr,
                                                h->rank, stream_acc, cstream, j < G && !same_stream);
            if (rc) return rc;
        }
        for (int g = i; g < j; g++) {
            const int64_t n = cseg_host[g] * tile_elems;
            if (!fused && acc && !(W > 1 && j - i > 1)) {
                rc = fo_consumer_reduce_with(dtype, c + off, acc + off / W, n, W, seg_stride,
                                             own_in_consumer ? d + off / W : nullptr, h->rank, stream_acc, cstream,
                                             j < G && !same_stream);
                if (rc) return rc;
            }
            if (d && !own_in_consumer)
                FO_HIP_CHECK(hipMemcpyAsync(d + off / W, c + off + (int64_t)h->rank * (n / W),
                                            (size_t)(n / W) * 2, hipMemcpyDeviceToDevice,
                                            static_cast<hipStream_t>(cstream)));
            off += n;
            done += cseg_host[g];
        }
        if (!fused) {
            rc = link_time(h, (off - off_batch) * 2, cstream);
            if (rc) return rc;
        }
        i = j;
    }
    return same_stream ? FO_OK : join(h, captured);
}

extern "C" int fo_overlap_gemm_allreduce_serial(fo_overlap_t *h, int dtype, int M, int N, int K,
                                                const void *A, const void *B, void *C, int algo) {
    if (!h) return FO_ERR_ARG;
    if (!h->gemm_ready) return FO_ERR_STATE;
    if (h->acc && h->acc_nelem < (int64_t)M * N) return FO_ERR_ARG;
    const int64_t mn = (int64_t)M * N;
    int rc = link_fits(h, mn * 2);
    if (rc) return rc;
    if (h->acc && !aligned(C, h->acc)) return FO_ERR_SHAPE;
    const bool consumed = accumulator_apart(h, M, N, K, A, B, C);
    rc = consumed ? fo_gemm_accumulate(dtype, M, N, K, 1, nullptr, 0, A, B, C, h->acc, nullptr, algo, h->gemm_stream)
                  : fo_gemm(dtype, M, N, K, A, B, C, algo, h->gemm_stream);
    if (!rc && h->acc && !consumed) rc = fo_consumer_reduce(dtype, C, h->acc, mn, h->gemm_stream);
    if (rc) return rc;
    return link_time(h, (int64_t)M * N * 2, h->gemm_stream);
}

extern "C" int fo_overlap_seg_allreduce(fo_overlap_t *h, int dtype, void *C, int64_t MN,
                                        const int32_t *cseg_host, int G, int seg_num) {
    if (!h || !C || !cseg_host || G <= 0 || seg_num <= 0 || MN <= 0) return FO_ERR_ARG;
    if (!h->gemm_ready) return FO_ERR_STATE;
    if (MN % seg_num || G < seg_num) return FO_ERR_SHAPE;
    if (h->acc && h->acc_nelem < MN) return FO_ERR_ARG;
    const int64_t unit = MN / seg_num;
    int64_t off = 0;
    if (h->acc && !aligned(C, h->acc)) return FO_ERR_SHAPE;
    for (int s = 0; s < seg_num; s++) {  // all of them before the first is enqueued
        const int64_t n = unit * cseg_host[s];
        if (off + n > MN) return FO_ERR_SEGMENTS;
        if (h->acc && n < 0) return FO_ERR_ARG;
        if (h->acc && n % 8) return FO_ERR_SHAPE;
        const int rc = link_fits(h, n * 2);
        if (rc) return rc;
        off += n;
    }
    off = 0;
    uint16_t *c = static_cast<uint16_t *>(C);
    uint16_t *acc = static_cast<uint16_t *>(h->acc);
    for (int s = 0; s < seg_num; s++) {  // the reference iterates SegNum times over cSEG_CPU
        const int64_t n = unit * cseg_host[s];
        if (acc) {
            int rc = fo_consumer_reduce(dtype, c + off, acc + off, n, h->gemm_stream);
            if (rc) return rc;
        }
        int rc = link_time(h, n * 2, h->gemm_stream);
        if (rc) return rc;
        off += n;
    }
    return FO_OK;
}

// ---------------------------------------------------------------- handle-free call that allocates nothing
// Callers that cannot allocate (code under a harness that forbids it, serving
// loops) have no handle: a handle owns a hipMalloc'ed workspace and, in the
// reference's interface, the caller brings the counters MM in a tensor of its own.
// Here both live in this file-scope array: kWorkspaceWords flag words, then one
// counter per group.  Each device the library runs on holds its own copy until the
// process ends; its address is asked for once per device.
constexpr int kStaticMaxGroups = 4096;
static __device__ __align__(256) int32_t scratch[kWorkspaceWords + kStaticMaxGroups];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
int32_t *g_scratch_ptr[kMaxDevices];  // device address of `scratch` on each device (the array's name is not one)
int g_scratch_token[kMaxDevices];     // last fork/join token handed out on each device

int scratch_of_current_device(int32_t **ptr, int *token) {
    int dev = 0;
    FO_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return FO_ERR_STATE;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        FO_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return FO_ERR_STATE;
        g_scratch_ptr[dev] = static_cast<int32_t *>(p);
    }
    *ptr = g_scratch_ptr[dev];
    // never 0 (the words' resting value) and never the previous call's, so a word
    // that an abandoned wait left behind cannot pass for this call's
    g_scratch_token[dev] = g_scratch_token[dev] >= (1 << 30) ? 1 : g_scratch_token[dev] + 1;
    *token = g_scratch_token[dev];
    return FO_OK;
}

}  // namespace

extern "C" int fo_gemm_allreduce_overlap_static(int dtype, int M, int N, int K, const void *A, const void *B,
                                                void *C, void *acc, const int32_t *RA, int TM, int TN, int rLDN,
                                                const int32_t *cseg_host, const int32_t *cseg_dev, int G, int algo,
                                                int fused, fo_stream_t gemm_stream, fo_stream_t comm_stream) {
    if (G > kStaticMaxGroups) return FO_ERR_LIMIT;
    if (G <= 0 || !cseg_host || !cseg_dev) return FO_ERR_SEGMENTS;
    int32_t *ws = nullptr;
    int token = 0;
    int rc = scratch_of_current_device(&ws, &token);
    if (rc) return rc;
    fo_overlap ctx;
    ctx.gemm_stream = static_cast<hipStream_t>(gemm_stream);
    ctx.comm_stream = comm_stream == gemm_stream ? nullptr : static_cast<hipStream_t>(comm_stream);
    ctx.workspace = ws;
    ctx.gemm_ready = ctx.overlap_ready = true;
    ctx.acc = acc;
    ctx.acc_nelem = acc ? (int64_t)M * N : 0;
    ctx.fused = fused < 0 ? -1 : fused;
    ctx.token = token;
    ctx.static_words = true;
    if (ctx.comm_stream && capturing(&ctx)) return FO_ERR_STATE;  // two streams under capture need the handle's events
    return allreduce_overlap(&ctx, dtype, M, N, K, A, B, C, ws + kWorkspaceWords, RA, TM, TN, rLDN, cseg_host,
                             cseg_dev, G, algo, 0);
}

// Whether a bounded device-side wait of an allocation-free call gave up since the
// last query on this device.  The calls have no handle to ask; the flag word of the
// static array is sticky across calls until it is read here.
extern "C" int fo_static_status(fo_stream_t gemm_stream, fo_stream_t comm_stream, int32_t *gave_up) {
    if (!gave_up) return FO_ERR_ARG;
    *gave_up = 0;
    int32_t *ws = nullptr;
    int token = 0;
    int rc = scratch_of_current_device(&ws, &token);
    if (rc) return rc;
    FO_HIP_CHECK(hipStreamSynchronize(static_cast<hipStream_t>(gemm_stream)));
    if (comm_stream != gemm_stream) FO_HIP_CHECK(hipStreamSynchronize(static_cast<hipStream_t>(comm_stream)));
    FO_HIP_CHECK(hipMemcpy(gave_up, ws + kWsGaveUp, sizeof(int32_t), hipMemcpyDeviceToHost));
    // A wait that gave up may have left the fork or join word set; both streams are idle now.
    if (*gave_up) FO_HIP_CHECK(hipMemset(ws, 0, kWorkspaceWords * sizeof(int32_t)));
    return FO_OK;
}
