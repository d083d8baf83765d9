"""GPU tests of the layers' native call path: what it enqueues, refuses and leaves to the registered operators."""
import pytest
import torch
import torch.utils._python_dispatch  # noqa: F401

pytestmark = pytest.mark.gpu


def _projection(fo, M, N, K, comm_op="all_reduce", W=1):
    from flashoverlap_amd import layers
    algo = fo._capi.find_algo(128, 128)
    hint = fo._capi.schedule_order(algo, M, N)
    T = (M // 128) * (N // 128)
    config = {"BM": 128, "BN": 128, "Algo": algo, "hint": hint, "cSeg": [T // 2, T - T // 2]}
    return layers.OverlapRowParallelLayer(0, W, K, N, M, config, comm_op, [0] * 16), hint


class Watched:
    """An OverlapImpl whose calls through Python are noted."""

    def __init__(self, impl):
        self.impl, self.calls = impl, []

    def handle(self):
        return self.impl.handle()

    def __getattr__(self, name):
        def call(*args):
            self.calls.append(name)
            return getattr(self.impl, name)(*args)
        return call


@pytest.mark.parametrize("comm_op", ["all_reduce", "reduce_scatter"])
def test_a_refused_layer_call_is_not_made_again(fo, comm_op):
    """What the C ABI refuses is raised, not tried again by the other path: a refusal may come behind the GEMM."""
    M, N, K = 256, 512, 64
    proj, _ = _projection(fo, M, N, K, comm_op, 2)
    odd = torch.zeros(M * N + 8, device="cuda", dtype=torch.float16)[1:M * N + 1]  # off its 16-byte pieces
    proj.overlap_class.set_accumulator(odd)
    proj.overlap_class = Watched(proj.overlap_class)
    x = torch.randn(M, K, device="cuda").half()
    with torch.no_grad(), pytest.raises(RuntimeError, match=r"gemm_(allreduce|reducescatter)_overlap failed: .*code -2"):
        proj(x)
    assert proj.overlap_class.calls == []
    torch.cuda.synchronize()
    proj.overlap_class = proj.overlap_class.impl
    proj.overlap_class.clear_accumulator()
    with torch.no_grad():
        assert proj(x).shape == (M // 2 if comm_op == "reduce_scatter" else M, N)
    torch.cuda.synchronize()
    assert (proj.counter == 0).all()


class Tagged(torch.Tensor):
    """A subclass without a dispatch of its own."""


class Seen(torch.overrides.TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


class Dispatched(torch.utils._python_dispatch.TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


def test_the_norm_layer_keeps_classes_and_is_seen(fo):
    """A subclass goes through torch.empty_like and the registered operator, and so does every call that a mode or the
    profiler follows; the values are those of the native call."""
    from flashoverlap_amd import layers
    M, N = 256, 1024
    hint = fo._capi.schedule_order(fo._capi.find_algo(128, 128), M, N)
    norm = layers.ReorderRMSNorm(N, M, 128, 128, hint)
    x = torch.randn(M, N, device="cuda").half()
    with torch.no_grad():
        want = norm(x)
        tagged = norm(x.as_subclass(Tagged))
        assert type(want) is torch.Tensor and type(tagged) is Tagged
        with Seen() as seen:
            followed = norm(x)
        assert any("reorder_rmsnorm_eps" in name for name in seen.names), seen.names
        with Dispatched() as dispatched:
            seen_below = norm(x)
        assert any("empty_like" in name for name in dispatched.names)  # the composite operator itself is above such modes
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
            profiled = norm(x)
        assert any("reorder_rmsnorm_eps" in event.key for event in prof.key_averages())
    for y in (tagged.as_subclass(torch.Tensor), followed, seen_below, profiled):
        assert torch.equal(y, want)


def test_the_projection_layer_takes_a_subclass(fo):
    M, N, K = 256, 512, 64
    proj, hint = _projection(fo, M, N, K)
    proj.overlap_class = Watched(proj.overlap_class)
    x = torch.randn(M, K, device="cuda").half()
    with torch.no_grad():
        want = proj(x)
        assert proj.overlap_class.calls == []
        got = proj(x.as_subclass(Tagged))
        assert proj.overlap_class.calls == ["gemm_allreduce_overlap"]
    assert torch.equal(got.as_subclass(torch.Tensor), want)


def test_calls_without_the_extension_module(fo, monkeypatch, tmp_path):
    """The kernel library alone serves the overlapped calls and the normalisation, with the same results."""
    ops, M, N, K = fo.ops, 256, 512, 64
    algo = fo._capi.find_algo(128, 128)
    T, TN = M // 128 * (N // 128), N // 128
    A, B = torch.randn(M, K, device="cuda").half(), torch.randn(N, K, device="cuda").half()
    w = torch.rand(N, device="cuda").half()
    RA = torch.arange(T, dtype=torch.int32, device="cuda").flip(0).contiguous().reshape(M // 128, TN)
    RE = fo.layout.generate_row_mapping(M, N, 128, 128, [T // 2, T // 2], 2)
    cs = torch.tensor([T // 2, T // 2], dtype=torch.int32)

    def results():
        MM = torch.zeros(fo.layout.counter_size(2, M // 128, TN), dtype=torch.int32, device="cuda")
        C, Y, Z = (torch.empty(M, N, device="cuda", dtype=torch.float16) for _ in range(3))
        D = torch.empty(M // 2, N, device="cuda", dtype=torch.float16)
        ov = ops.Overlap(world=2)
        ov.gemm_reducescatter_overlap(A, B, C, D, MM, RA, RE, 1, cs, cs.cuda(), algo)
        ov.gemm_allreduce_overlap(A, B, C, MM, RA, 1, cs, cs.cuda(), algo)
        ov.gemm_allreduce_rmsnorm_overlap(A, B, C, MM, RA, RA.cpu(), 1, cs, cs.cuda(), algo, Y, w)
        ops.reorder_rmsnorm(C, Z, w, 128, 128, 1, RA)
        torch.cuda.synchronize()
        ov.close()
        return C, D, Y, Z, MM

    want = results()
    monkeypatch.setattr(fo._capi, "NATIVE_LIB", str(tmp_path / "_fo_native.so"))
    monkeypatch.setattr(fo._capi, "_native", None)
    assert all(torch.equal(a, b) for a, b in zip(results(), want))


def test_native_calls_decline_one_wrong_argument(fo):
    """The native calls take the right arguments (error code 0) and leave alone (None) every call with one wrong one."""
    ops, native, M, N, K = fo.ops, fo._capi.native(), 256, 512, 64
    algo = fo._capi.find_algo(128, 128)
    T, TN = M // 128 * (N // 128), N // 128
    half = lambda *s: torch.zeros(*s, device="cuda", dtype=torch.float16)
    ints = lambda *s: torch.zeros(*s, device="cuda", dtype=torch.int32)
    A, B, C, D, Y, w, acc = half(M, K), half(N, K), half(M, N), half(M // 2, N), half(M, N), half(N), half(M * N)
    MM, RA, cs = ints(TN), torch.arange(T, dtype=torch.int32, device="cuda").reshape(M // 128, TN), torch.tensor([T // 2] * 2, dtype=torch.int32)
    RE = fo.layout.generate_row_mapping(M, N, 128, 128, [T // 2] * 2, 2)
    ov = ops.Overlap(world=2)
    ov.set_accumulator(acc)
    h = ov._h.value
    off = lambda t: torch.zeros(2 * t.numel(), device=t.device, dtype=t.dtype)[::2].view(t.shape)  # every other element
    tensor = [lambda t: None, lambda t: t.cpu() if t.is_cuda else t.cuda(), lambda t: t.float(), off]
    small = lambda t: t.reshape(-1)[:-1]
    number = [lambda v: None, lambda v: float(v), lambda v: 1 << 40]
    calls = {
        "allreduce": ([h, A, B, C, MM, RA, 1, cs, cs.cuda(), algo, False, acc],
                      {0: number[:2], 1: tensor, 2: tensor, 3: tensor + [small], 4: tensor + [small], 5: tensor + [small],
                       6: number + [lambda v: 3], 7: tensor, 8: tensor, 9: number + [lambda v: -1], 11: [tensor[2], small]}),
        "allreduce_norm": ([h, A, B, C, MM, RA, RA.cpu(), 1, cs, cs.cuda(), algo, False, acc, Y, w, 1e-5],
                           {6: tensor + [small], 13: tensor + [small], 14: tensor + [small], 15: [lambda v: 1]}),
        "reducescatter": ([h, A, B, C, D, MM, RA, RE, 1, cs, cs.cuda(), algo, False, acc, 2],
                          {4: tensor + [small], 7: tensor + [small], 14: number[:2] + [lambda v: 0]}),
        "reorder_rmsnorm": ([C, Y, w, 128, 128, 1, RA, 1e-5],
                            {0: tensor, 1: tensor + [small], 2: tensor + [small], 3: number + [lambda v: 96], 4: number, 5: number,
                             6: tensor + [small], 7: [lambda v: 1]}),
    }
    for name, (right, wrong) in calls.items():
        assert getattr(native, name)(*right) == 0, name
        assert getattr(native, name)(*right, 0) is None and getattr(native, name)(*right[:-1]) is None
        for i, changes in wrong.items():
            for k, change in enumerate(changes):
                args = list(right)
                args[i] = change(args[i])
                assert getattr(native, name)(*args) is None, (name, i, k)
    torch.cuda.synchronize()
    assert (MM == 0).all() and ov.status() == 0
    ov.close()
