"""One PointRendererCache through passes of changing sizes, scenes and streams, and beside a captured pass: every pass gives
what a cache of its own gives."""
import numpy as np
import pytest

from helpers import announce

pytestmark = pytest.mark.gpu


class Ctx:
    def save_for_backward(self, *t):
        self.saved_tensors = t


def _info(hs, cache, forward_path):
    import torch
    from adop_amd import render

    hs.params.forward_path = forward_path
    return render.NeuralRenderInfo(scene=render.NeuralScene.from_host(hs, "cuda"), images=list(hs.views), params=hs.params,
                                   num_layers=hs.num_layers, cache=cache, train=True,
                                   dropout_points=None if hs.dropout is None else torch.from_numpy(hs.dropout).cuda())


def _scenes(forward_path):
    from adop_amd import scenes

    small = scenes.config3(n=30_000, w=160, h=90, channels=4)
    more_poses = scenes.config3(n=30_000, w=160, h=90, channels=4)
    more_poses.poses_se3 = np.stack([more_poses.poses_se3[0]] * 70)
    large = scenes.config3(n=200_000, w=480, h=270, channels=4)
    return [small, large, more_poses]


def _pass(info, gout):
    from adop_amd import render

    ctx = Ctx()
    images, _ = render.BlendPointCloudForward(ctx, info)
    grads = render.BlendPointCloudBackward(ctx, info, gout)
    return list(ctx.depth_index), images, grads


def _same(got, want, what):
    import torch

    torch.cuda.synchronize()
    for a, b in zip(got[0], want[0]):
        assert torch.equal(a, b), what
    for a, b in zip(got[1] + got[2], want[1] + want[2]):
        assert float((a.double() - b.double()).abs().max()) <= 1e-4 * float(b.double().abs().max()) + 1e-12, what


@pytest.mark.parametrize("forward_path", [1, 2], ids=["direct", "tiles"])
def test_one_cache_for_two_streams_sizes_and_scenes(forward_path):
    import torch
    from adop_amd import render, scenes

    announce(f"one cache, 3 scenes, 2 streams in turn, forward_path={forward_path}")
    cache = render.PointRendererCache()
    hosts = _scenes(forward_path)
    infos = [_info(hs, cache, forward_path) for hs in hosts]
    gouts = [[torch.from_numpy(g).cuda() for g in scenes.upstream_grads(hs, 5)] for hs in hosts]
    want = []
    for hs, gout in zip(hosts, gouts):
        want.append(_pass(_info(hs, render.PointRendererCache(), forward_path), gout))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = []
    for k in range(24):  # nothing waits in between: passes on the two streams may run at the same time
        with torch.cuda.stream(streams[(k // 2 + k) % 2]):
            got.append((k % 3, _pass(infos[k % 3], gouts[k % 3])))
    for k, (i, g) in enumerate(got):
        _same(g, want[i], f"pass {k}, scene {i}")


@pytest.mark.parametrize("forward_path", [1, 2], ids=["direct", "tiles"])
def test_a_backward_pass_beside_a_forward_pass_on_another_stream(forward_path):
    import torch
    from adop_amd import render, scenes

    announce(f"forward on stream A, another forward on stream B, backward on A, forward_path={forward_path}")
    cache = render.PointRendererCache()
    small, large, _ = _scenes(forward_path)
    gout = [torch.from_numpy(g).cuda() for g in scenes.upstream_grads(large, 5)]
    want = _pass(_info(large, render.PointRendererCache(), forward_path), gout)
    info, other = _info(large, cache, forward_path), _info(small, cache, forward_path)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    for k in range(6):
        ctx = Ctx()
        with torch.cuda.stream(a):
            images, _ = render.BlendPointCloudForward(ctx, info)
        with torch.cuda.stream(b):  # (a smaller scene: its workspace would not do)
            render.BlendPointCloudForward(Ctx(), other)
        with torch.cuda.stream(a):
            grads = render.BlendPointCloudBackward(ctx, info, gout)
        _same((list(ctx.depth_index), images, grads), want, f"round {k}")


@pytest.mark.parametrize("forward_path", [1, 2], ids=["direct", "tiles"])
def test_a_captured_pass_beside_others_without_a_context(forward_path):
    """A forward pass without a context leaves its buffers to the next one; a captured pass between two such passes takes
    none of theirs and leaves them none of its own."""
    import torch
    from adop_amd import render

    announce(f"captured forward between forwards without a context, forward_path={forward_path}")
    cache = render.PointRendererCache()
    small, large, _ = _scenes(forward_path)
    infos = {id(hs): _info(hs, cache, forward_path) for hs in (small, large)}

    def forward(hs):
        images, _ = render.BlendPointCloudForward(None, infos[id(hs)])
        return [L.depth_index_tensor for L in cache.layers_cuda], images

    want = [t.clone() for t in forward(small)[0]]
    torch.cuda.synchronize()
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            recorded, recorded_images = forward(small)
    torch.cuda.synchronize()
    for k in range(4):
        eager, _ = forward(small)
        for t in recorded:
            t.fill_(7)
        kept = [t.clone() for t in eager]
        forward(large)  # gives the eager buffers back
        torch.cuda.empty_cache()
        graph.replay()
        torch.cuda.synchronize()
        for l, t in enumerate(recorded):
            assert torch.equal(t, want[l]), (k, l)
            assert torch.equal(kept[l], want[l]), (k, l)
