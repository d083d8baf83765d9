"""GPU tests of the layers' native call path: what it enqueues, refuses and leaves to the registered operators."""
import pytest
import torch

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
