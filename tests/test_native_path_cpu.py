"""The native call path leaves alone what it does not recognise: None, nothing enqueued, for the Python path to judge."""
import pytest
import torch

import flashoverlap_amd as fo

H = torch.float16
I32 = dict(dtype=torch.int32)


def _overlap_args():
    A, B, C = torch.zeros(128, 64, dtype=H), torch.zeros(128, 64, dtype=H), torch.zeros(128, 128, dtype=H)
    one = torch.ones(1, **I32)
    algo = fo._capi.find_algo(128, 128)
    return [1, A, B, C, torch.zeros(1, **I32), torch.zeros(1, 1, **I32), 1, one, one, algo, False, None]


@pytest.mark.parametrize("change", [{}, {0: 0}, {0: None}, {1: None}, {4: torch.zeros(1)}, {6: 1.0}, {6: 1 << 40}, {9: -1}, {11: 3}])
def test_allreduce_declines(change):
    args = _overlap_args()  # tensors in host memory: declined whatever else is right
    for i, v in change.items():
        args[i] = v
    assert fo._capi.native().allreduce(*args) is None
    assert fo._capi.native().allreduce(*args[:-1]) is None
    assert fo._capi.native().allreduce(*args, 0) is None


def test_norm_and_layers_decline():
    native = fo._capi.native()
    X, w, RA = torch.zeros(128, 128, dtype=H), torch.zeros(128, dtype=H), torch.zeros(1, 1, **I32)
    assert native.reorder_rmsnorm(X, X, w, 128, 128, 1, RA, 1e-5) is None
    assert native.reorder_rmsnorm(X, X, w, 128, 128, 1, RA, 1) is None
    assert native.reorder_rmsnorm_layer(X, w, 128, 128, RA, 1e-5) is None
    assert native.reorder_rmsnorm_layer(X, None, 128, 128, RA, 1e-5) is None
    one, algo = torch.ones(1, **I32), fo._capi.find_algo(128, 128)
    assert native.allreduce_layer(1, X, X, one, RA, one, one, algo) is None
    assert native.reducescatter_layer(1, X, X, one, RA, one, one, one, algo, 0) is None


def test_the_kernel_library_alone_is_enough(monkeypatch, tmp_path):
    """Without the extension module (a build without the torch parts) the Python path serves the calls: here it refuses
    tensors in host memory itself."""
    monkeypatch.setattr(fo._capi, "NATIVE_LIB", str(tmp_path / "_fo_native.so"))
    monkeypatch.setattr(fo._capi, "_native", None)
    ops = fo.ops
    X, w, RA = torch.zeros(128, 128, dtype=H), torch.zeros(128, dtype=H), torch.zeros(1, 1, **I32)
    with pytest.raises(ValueError, match="must live on the GPU"):
        ops.reorder_rmsnorm(X, X.clone(), w, 128, 128, 1, RA, stream=None)
    assert fo._capi.native().allreduce(*_overlap_args()) is None
