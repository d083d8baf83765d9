"""What the framework is timed on: whole passes of a row-parallel projection and the normalisation behind
it, through the entry points a user's program calls, from one decode batch to the large square.

A case names one of six ways to use the framework (`op`), the problem and the type:

  layers    OverlapRowParallelLayer (all_reduce) followed by ReorderRMSNorm: the drop-in layers of a model block
  layers_rs OverlapRowParallelLayer (reduce_scatter, W ranks) followed by ReorderRMSNorm on this rank's rows
  pair      OverlapImpl.gemm_allreduce_overlap with an accumulator (the other ranks' sum), then reorder_rmsnorm
  step      Overlap.gemm_allreduce_rmsnorm_overlap: the one call that also normalises, with an accumulator
  step_rs   Overlap.gemm_reducescatter_overlap with an accumulator for all W ranks' rows, then the
            normalisation of the first rank's rows
  serial    OverlapImpl.gemm_allreduce and rmsnorm on one stream: what a shape gets whose tuned split is a
            single group
"""
import math
import os

import numpy as np
import torch

# As the benchmark and the tests do: a lost signal ends in a flagged exit, not in a waiter that spins for good.
os.environ.setdefault("FO_WAIT_MAX_POLLS", "200000000")

import flashoverlap_amd as fo  # noqa: E402
from flashoverlap_amd import layers, layout, ops  # noqa: E402

EPS = 1e-6
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}


def _case(name, op, M, N, K, bm, bn, dtype, group_tiles, W=1):
    return {"name": name, "op": op, "M": M, "N": N, "K": K, "bm": bm, "bn": bn, "dtype": dtype,
            "group_tiles": group_tiles, "W": W}


def listed():
    return [
        # Decode: one batch of 128 tokens against an eighth of the input features; launches and latency.
        _case("decode_layers", "layers", 128, 4096, 1024, 128, 128, "f16", 16),
        # Decode of a wider model with a whole down-projection's K: the weight has to be streamed in.
        _case("decode_wide_layers", "layers", 256, 8192, 3584, 128, 128, "bf16", 64),
        # A short prompt (or a chunk of a chunked prefill).
        _case("chunk_step", "step", 512, 4096, 4096, 128, 128, "f16", 64),
        # A prompt length that 256 does not divide and a K-slice that is no multiple of a K step.
        _case("ragged_pair", "pair", 1152, 5120, 1720, 128, 128, "bf16", 120),
        # A shape whose tuned split is one group: no second stream.
        _case("single_group_serial", "serial", 1024, 8192, 2048, 128, 256, "f16", 256),
        # Sequence parallelism over eight ranks, no accumulator attached: the reduce-scatter layers.
        _case("sequence_layers_rs", "layers_rs", 2048, 4096, 2048, 128, 128, "f16", 128, 8),
        # Row-parallel K-slice with very fine wave groups (the benchmark's second workload).
        _case("k_slice_step", "step", 4096, 4096, 512, 128, 128, "f16", 4),
        # Prefill of a packed batch whose rows are no multiple of 256 and whose width is no power of two.
        _case("packed_layers", "layers", 4224, 7168, 3584, 128, 256, "bf16", 231),
        # Reduce-scatter layout, eight row-chunk segments (the benchmark's fourth workload).
        _case("segments_step_rs", "step_rs", 8192, 4096, 4096, 128, 128, "f16", 256, 8),
        # Down-projection (the benchmark's third workload).
        _case("down_projection_step", "step", 8192, 8192, 3584, 256, 128, "bf16", 512),
        # The shape of the command-line tools' defaults, by the drop-in pair of calls.
        _case("default_shape_pair", "pair", 4096, 8192, 8192, 128, 256, "f16", 512),
        # The large square of the headline benchmark.
        _case("large_square_step", "step", 8192, 8192, 8192, 128, 256, "f16", 256),
    ]


def _log(rng, lo, hi, step):
    """A multiple of `step` in [lo, hi], uniform over the logarithm."""
    x = math.exp(rng.uniform(math.log(lo), math.log(hi + step)))
    return max(lo, min(hi, int(x) // step * step))


def draw(rng):
    op = rng.choice(["layers", "layers", "layers_rs", "pair", "step", "step", "step_rs", "serial"])
    bm, bn = rng.choice([(128, 128), (128, 128), (128, 256), (256, 128)])
    M = _log(rng, bm, 8192, bm)             # one decode batch to a long packed prefill
    N = _log(rng, 1024, 8192, bn)           # output features
    K = _log(rng, 256, 8192, 8)             # this rank's slice of the input features
    tiles = (M // bm) * (N // bn)
    groups = min(tiles, rng.choice([1, 2, 3, 4, 5, 8, 16]))
    if tiles >= 256 and rng.random() < 0.15:
        group_tiles = 4                     # very fine groups
    else:
        group_tiles = -(-tiles // groups)
    W = rng.choice([2, 4, 8]) if op in ("layers_rs", "step_rs") else 1
    c = _case("", op, M, N, K, bm, bn, rng.choice(["f16", "bf16"]), group_tiles, W)
    del c["name"]
    return c


def _inputs(case, seed):
    """Activations with a few outlier features, as hidden states have them; a weight that keeps the output's scale."""
    M, N, K, td = case["M"], case["N"], case["K"], DTYPES[case["dtype"]]
    g = torch.Generator(device="cuda").manual_seed(seed)
    A = torch.randn(M, K, generator=g, device="cuda")
    cols = torch.from_numpy(np.random.default_rng(seed).permutation(K)[: max(1, K // 100)]).cuda()
    A[:, cols] *= 4
    B = torch.randn(N, K, generator=g, device="cuda") * K ** -0.5
    gamma = 1 + 0.1 * torch.randn(N, generator=g, device="cuda")
    return A.to(td), B.to(td), gamma.to(td), g


def prepare(case, seed):
    M, N, K, bm, bn, W, op = (case[k] for k in ("M", "N", "K", "bm", "bn", "W", "op"))
    td = DTYPES[case["dtype"]]
    A, B, gamma, g = _inputs(case, seed)
    TM, TN = M // bm, N // bn
    algo = fo._capi.find_algo(bm, bn, swizzle=4)
    cseg = layout.cseg_from_waves(TM * TN, case["group_tiles"])
    s = {"op": op, "A": A, "B": B, "gamma": gamma, "M": M, "N": N, "bm": bm, "bn": bn, "W": W, "algo": algo}
    if op == "serial":
        layers.load_library()
        ov = torch.classes.flashoverlap_class.OverlapImpl()
        ov.nccl_init(0, 1, torch.ops.flashoverlap_op.generate_nccl_id())
        ov.cutlass_init()
        ov.overlap_init()
        s["acc"] = torch.randn(M, N, generator=g, device="cuda").to(td)
        ov.set_accumulator(s["acc"])
        s.update(ov=ov, C=torch.empty(M, N, device="cuda", dtype=td), Y=torch.empty(M, N, device="cuda", dtype=td))
        return s
    hint = fo._capi.schedule_order(algo, M, N)
    if op in ("layers", "layers_rs"):
        layers.load_library()
        config = {"BM": bm, "BN": bn, "hint": hint, "cSeg": cseg, "Algo": algo}
        s["proj"] = layers.OverlapRowParallelLayer(0, W, K, N, M, config,
                                                   "all_reduce" if op == "layers" else "reduce_scatter",
                                                   torch.ops.flashoverlap_op.generate_nccl_id(), dtype=td)
        # Reduce-scatter: this rank keeps bm / W rows of every tile.
        s["norm"] = layers.ReorderRMSNorm(N, M // W, bm // W, bn, hint, eps=EPS, dtype=td)
        with torch.no_grad():
            s["proj"].weight.copy_(B)
            s["norm"].weight.copy_(gamma)
        return s
    s["cseg_cpu"] = torch.tensor(cseg, dtype=torch.int32)
    s["cseg_gpu"] = s["cseg_cpu"].cuda()
    s["RA"] = layout.reorder_indices(TM * TN, hint).reshape(TM, TN)
    s["RA_cpu"] = s["RA"].cpu()
    s["MM"] = torch.zeros(layout.counter_size(len(cseg), TM, TN), dtype=torch.int32, device="cuda")
    s["C"] = torch.empty(M, N, device="cuda", dtype=td)
    s["acc"] = torch.randn(M * N, generator=g, device="cuda").to(td)  # what the other ranks have summed so far
    s["Y"] = torch.empty(M // W, N, device="cuda", dtype=td)
    if op == "pair":
        layers.load_library()
        ov = torch.classes.flashoverlap_class.OverlapImpl()
        ov.nccl_init(0, 1, torch.ops.flashoverlap_op.generate_nccl_id())
        ov.cutlass_init()
        ov.overlap_init()
    else:
        ov = ops.Overlap(rank=0, world=W)
    ov.set_accumulator(s["acc"])
    s["ov"] = ov
    if op == "step_rs":
        s["RE"] = layout.generate_row_mapping(M, N, bm, bn, cseg, W)
        s["D"] = torch.empty(M // W, N, device="cuda", dtype=td)
    return s


def run(s):
    op = s["op"]
    with torch.no_grad():
        if op in ("layers", "layers_rs"):
            out = s["proj"](s["A"])
            return {"out": out, "y": s["norm"](out)}
        A, B, C, Y, ov, algo, bm, bn = (s[k] for k in ("A", "B", "C", "Y", "ov", "algo", "bm", "bn"))
        if op == "serial":
            ov.gemm_allreduce(A, B, C, algo)
            torch.ops.flashoverlap_op.rmsnorm(C, Y, s["gamma"], EPS)
            return {"out": C, "acc": s["acc"], "y": Y}
        MM, RA, cs_cpu, cs_gpu = s["MM"], s["RA"], s["cseg_cpu"], s["cseg_gpu"]
        if op == "pair":
            ov.gemm_allreduce_overlap(A, B, C, MM, RA, 1, cs_cpu, cs_gpu, algo, False)
            torch.ops.flashoverlap_op.reorder_rmsnorm_eps(C, Y, s["gamma"], bm, bn, 1, RA, EPS)
            return {"out": C, "acc": s["acc"], "y": Y, "counters": MM}
        if op == "step":
            ov.gemm_allreduce_rmsnorm_overlap(A, B, C, MM, RA, s["RA_cpu"], 1, cs_cpu, cs_gpu, algo, Y, s["gamma"],
                                              eps=EPS)
            return {"out": C, "acc": s["acc"], "y": Y, "counters": MM}
        W, D = s["W"], s["D"]
        ov.gemm_reducescatter_overlap(A, B, C, D, MM, RA, s["RE"], 1, cs_cpu, cs_gpu, algo)
        ops.reorder_rmsnorm(s["acc"].view(W, s["M"] // W, s["N"])[0], Y, s["gamma"], bm // W, bn, 1, RA, eps=EPS)
        return {"out": C, "rows": D, "acc": s["acc"], "y": Y, "counters": MM}


def work(case):
    """Operands read once, product, accumulator, this rank's rows and normalised rows written once, the accumulator
    read once."""
    M, N, K, W, op = (case[k] for k in ("M", "N", "K", "W", "op"))
    product = 2.0 * M * N
    total = 2.0 * (M * K + N * K + N) + product
    if op not in ("layers", "layers_rs"):
        total += 2 * product                      # accumulator
    if op in ("layers_rs", "step_rs"):
        total += product / W                      # this rank's rows
    total += product / W                          # normalised rows
    return {"bytes": total, "flops": 2.0 * M * N * K}


def tolerance(case):
    """Sums in 32 bits in another order, each result rounded to 16 bits up to three times."""
    if case["dtype"] == "f16":
        return {"rel": 1e-3, "max": 1e-2}
    return {"rel": 8e-3, "max": 5e-2}
