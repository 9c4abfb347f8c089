"""Clouds of more than 2^26 points through the steps that gather whole points: torch's gather of rows of 16 bytes returns wrong
rows at that size.  Expected rows come from gathers of 2^24 rows each."""
import numpy as np
import pytest

from helpers import announce
from test_torch_wrapper_gpu import _module

pytestmark = pytest.mark.gpu
N = (1 << 26) + 4096


def _rows(t, index):
    import torch

    return torch.cat([t[i] for i in index.split(1 << 24)])


@pytest.fixture(scope="module")
def cloud():
    import torch

    p = torch.rand(N, 4, generator=torch.Generator("cuda").manual_seed(5), device="cuda")
    yield p
    del p
    torch.cuda.empty_cache()


def _check_prepared(got, cloud, normal):
    import torch

    position, moved_normal, data, order = got
    assert torch.equal(torch.sort(order).values, torch.arange(N, device="cuda"))
    assert torch.equal(position[:, :3], _rows(cloud, order)[:, :3])
    assert torch.equal(position[:, 3], data[:, 3]) and bool((data[:, 3] > 0).all())
    assert torch.equal(moved_normal, _rows(normal, order))


def test_preparation_in_cpp(cloud):
    import torch

    announce(f"C++ PreprocessPointCloud, N={N}")
    normal = torch.arange(N, dtype=torch.int32, device="cuda").reshape(-1, 1)
    _check_prepared(_module().preprocess_point_cloud(cloud, normal, 1, 256, 3), cloud, normal)


def test_preparation_step_by_step(cloud):
    import torch
    from adop_amd import preprocess as pp

    announce(f"PreprocessPointCloud in single steps, normals as rows of 16 bytes, N={N}")
    normal = torch.arange(N, dtype=torch.float32, device="cuda").reshape(-1, 1).repeat(1, 4)
    _check_prepared(pp.PreprocessPointCloud(cloud, normal, rank=1, block_size=128, seed=3), cloud, normal)


def test_filters_in_cpp(cloud):
    import torch
    from adop_amd import preprocess as pp, scenes

    announce(f"C++ FilterPointCloud, N={N}")
    poses = torch.from_numpy(scenes.look_at_view((0.5, 0.5, -20.0))[None]).cuda()
    intr = torch.from_numpy(scenes.pinhole_row(300, 300, 160, 120)[None]).cuda()
    frames = [scenes.make_view(320, 240)]
    tuples = [(v.w, v.h, v.image_index, v.camera_index, v.camera_model_type, v.crop_fx, v.crop_fy, v.crop_cx, v.crop_cy,
               v.crop_s) for v in frames]
    p = cloud.clone()
    p[-1000:] = p[:1000]  # close points behind the 2^26th
    got = _module().filter_point_cloud(p, poses, intr, tuples)
    assert N - 1200 < got.shape[0] <= N - 1000 and torch.equal(got, pp.FilterPointCloud(p, poses, intr, frames))


def test_radii_of_a_host_scene(cloud):
    import torch
    from types import SimpleNamespace
    from adop_amd import preprocess as pp

    announce(f"AttachDropOutRadii, N={N}")
    hs = SimpleNamespace(position=cloud.cpu().numpy(), normal=None, params=SimpleNamespace(), meta={})
    pp.AttachDropOutRadii(hs, rank=1, seed=3)
    got = torch.from_numpy(hs.position).cuda()
    data = pp.ComputeRadius(cloud, 1, torch.Generator("cuda").manual_seed(3))
    order = pp.SortBlocksByRadius(data[:, 3])
    assert torch.equal(got[:, :3], _rows(cloud, order)[:, :3])
    assert np.array_equal(hs.position[:, 3], _rows(data, order)[:, 3].cpu().numpy())
