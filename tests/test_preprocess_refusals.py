"""What the scene processing refuses before a kernel is launched (no GPU needed: the library is a stub that records calls)."""
import pytest
import torch

from adop_amd import _capi
from adop_amd import preprocess as pp


class _Recorder:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append(name)
            return _capi.ADOP_OK

        return call


@pytest.fixture
def stub(monkeypatch):
    lib = _Recorder()
    monkeypatch.setattr(_capi, "load_library", lambda: lib)
    monkeypatch.setattr(pp, "_checked_position", lambda p: p.contiguous())
    monkeypatch.setattr(pp, "_box_and_stretch", lambda p: ((None, None), 1.0))
    monkeypatch.setattr(pp, "_stream_ptr", lambda: None)
    monkeypatch.setattr(pp, "_morton_order", lambda p, box, by_keys: lambda: torch.arange(p.shape[0]))
    monkeypatch.setattr(pp, "_knn_distance", lambda p, *a: torch.zeros(p.shape[0]))
    return lib


def test_normals_on_the_device_of_the_points_are_taken(stub):
    normal = torch.zeros(600, 1, dtype=torch.int32)
    out = pp.PreprocessPointCloud(torch.zeros(600, 4), normal)
    assert out[1].shape == normal.shape
    assert stub.calls == ["adop_shuffle_points", "adop_radius_blocks"]


@pytest.mark.parametrize("block_size", [256, 64])
@pytest.mark.parametrize("normal", [
    torch.zeros(600, dtype=torch.int32, device="meta"),     # of another device
    torch.zeros(600, 1, dtype=torch.int32, device="meta"),
    torch.zeros(1, 600, dtype=torch.int32),                 # as many numbers as points, in one row
    torch.zeros(300, 2, dtype=torch.int32),
    torch.zeros(599, 1, dtype=torch.int32),
    torch.zeros((), dtype=torch.int32),
], ids=["device", "device, column", "one row", "pairs", "short", "scalar"])
def test_normals_no_kernel_may_read_are_refused(stub, normal, block_size):
    with pytest.raises(RuntimeError, match="normal must be"):
        pp.PreprocessPointCloud(torch.zeros(600, 4), normal, block_size=block_size)
    assert stub.calls == []
