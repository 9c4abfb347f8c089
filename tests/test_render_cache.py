"""Which scratch memory and which layer buffers a pass of PointRendererCache gets (no GPU needed: the library is a stub that
records the addresses it is handed, the current stream and its capture state are set by the test)."""
import ctypes as C
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from adop_amd import _capi, render, scenes


class _Library:
    def __init__(self):
        self.calls = []  # (stream, address of the workspace, its size, address of the first depth buffer)

    def adop_workspace_size_for(self, scene, views, layers, w, h, flags):
        s = C.cast(scene, C.POINTER(_capi.Scene)).contents
        return 1024 * views * (w * h + s.num_poses + s.num_cameras * s.intrinsics_cols)

    def _record(self, buffers, workspace, size, stream):
        fb = C.cast(buffers, C.POINTER(_capi.ForwardBuffers)).contents
        self.calls.append((stream.value, workspace.value, size, fb.layers[0].depth))
        return _capi.ADOP_OK

    def adop_forward(self, scene, views, n, params, buffers, workspace, size, stats, stream):
        return self._record(buffers, workspace, size, stream)

    def adop_backward(self, scene, views, n, params, buffers, grads, workspace, size, stats, stream):
        return self._record(buffers, workspace, size, stream)


class _Ctx:
    def save_for_backward(self, *t):
        self.saved_tensors = t


@pytest.fixture
def rig(monkeypatch):
    now = SimpleNamespace(stream=1, capturing=False, lib=_Library())
    monkeypatch.setattr(_capi, "load_library", lambda: now.lib)
    monkeypatch.setattr(render, "_raw_stream", lambda: now.stream)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: now.capturing)
    now.cache = render.PointRendererCache()
    now.alive = []

    def info(w=32, h=24, poses=1, points=64):
        cloud = render.NeuralPointCloud(np.zeros((points, 4), np.float32), None, np.arange(points), "cpu")
        scene = render.NeuralScene(cloud, torch.zeros(4, points), torch.zeros(4),
                                   torch.from_numpy(np.stack([scenes.look_at_view((0, 0, -3.0))] * poses)),
                                   torch.from_numpy(scenes.pinhole_row(30, 30, 16, 12)[None]))
        return render.NeuralRenderInfo(scene=scene, images=[scenes.make_view(w, h)], params=scenes.default_params(),
                                       num_layers=2, cache=now.cache)

    def forward(info, ctx=None):
        now.alive.append(now.cache.workspace)  # (addresses are compared: none is to be used twice)
        now.alive += now.cache.layers_cuda
        render.BlendPointCloudForward(ctx, info)
        return now.lib.calls[-1]

    def backward(info, ctx):
        now.alive.append(now.cache.workspace)
        render.BlendPointCloudBackward(ctx, info, [torch.zeros(1, 4, 24 >> l, 32 >> l) for l in range(2)])
        return now.lib.calls[-1]

    now.info, now.forward, now.backward = info, forward, backward
    return now


def test_passes_of_one_size_on_one_stream_share_it(rig):
    info = rig.info()
    first = rig.forward(info, _Ctx())
    ctx = _Ctx()
    second = rig.forward(info, ctx)
    assert second[1:3] == first[1:3] and second[3] != first[3]  # (the layers of a pass with a context belong to it)
    assert rig.backward(info, ctx)[1:3] == first[1:3]
    a = rig.forward(info)
    assert rig.forward(info) == a  # without one they stay too


@pytest.mark.parametrize("other", [dict(w=40), dict(h=30), dict(poses=5), dict(points=65)], ids=str)
@pytest.mark.parametrize("with_ctx", [False, True])
def test_another_size_takes_another_one(rig, other, with_ctx):
    ctx = (lambda: _Ctx()) if with_ctx else (lambda: None)
    a, b = rig.info(), rig.info(**other)
    first, second, third = rig.forward(a, ctx()), rig.forward(b, ctx()), rig.forward(a, ctx())
    assert first[1] != second[1] != third[1]
    assert third[2] == first[2]


@pytest.mark.parametrize("with_ctx", [False, True])
def test_two_streams_share_nothing(rig, with_ctx):
    ctx = (lambda: _Ctx()) if with_ctx else (lambda: None)
    info, seen = rig.info(), []
    for rig.stream in (1, 2, 1):
        seen.append(rig.forward(info, ctx()))
    assert [c[0] for c in seen] == [1, 2, 1]
    assert seen[0][1] != seen[1][1] != seen[2][1]
    assert seen[0][3] != seen[1][3] != seen[2][3]


def test_a_backward_pass_takes_that_of_its_own_stream_and_size(rig):
    info, ctx = rig.info(), _Ctx()
    need = rig.forward(info, ctx)[2]
    rig.stream = 2
    other = rig.forward(rig.info(w=8, h=8), _Ctx())  # another, smaller pass through the cache, on another stream
    rig.stream = 1
    got = rig.backward(info, ctx)
    assert got[1] != other[1] and got[2] == need > other[2]


@pytest.mark.parametrize("with_ctx", [False, True])
def test_a_captured_pass_shares_nothing_with_others(rig, with_ctx):
    ctx = (lambda: _Ctx()) if with_ctx else (lambda: None)
    info, seen = rig.info(), []
    for rig.capturing in (False, True, True, False):
        seen.append(rig.forward(info, ctx()))
    assert len({c[1] for c in seen}) == 4
    assert len({c[3] for c in seen}) == 4
