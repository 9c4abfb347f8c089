"""Point-cloud preprocessing of SceneData (data/SceneData.cpp:96-118) on the device: the filters for lonely and
close points, Morton order, shuffled 256-point blocks, the radius of every point from its 4th nearest neighbour,
blocks sorted by radius.

The order of the cloud and the radii decide how the rasterizer runs (coherent wavefronts, the LOD early exit), so the
steps sit next to it.  The distance search and the Morton codes are HIP kernels behind the C-ABI
(``adop_knn_distance``, ``adop_morton_codes``, ``adop_point_distance_to_camera``, ``adop_close_points``), and so are the
passes that move whole points (``adop_gather_points``, ``adop_shuffle_points``, ``adop_radius_blocks``); torch sorts and
draws the random numbers.
"""
import ctypes as C

import torch

from . import _capi
from .render import _check, _stream_ptr


def _ptr(t):
    return None if t is None else C.c_void_p(t.data_ptr())


def _checked_position(position):
    assert position.is_cuda and position.dtype == torch.float32 and position.dim() == 2 and position.shape[1] == 4
    return position.contiguous()


def _check_normal(normal, position):
    """The kernels take the address of the normals as it is: a tensor of another device, or one of fewer rows than there are
    points, is refused here."""
    if normal is not None and (normal.device != position.device or normal.dim() < 1 or normal.shape[0] < position.shape[0]):
        raise RuntimeError(f"normal must be a tensor of at least {position.shape[0]} rows on {position.device}, "
                           f"not {tuple(normal.shape)} on {normal.device}")


_RADIUS_BLOCK = 256  # the block size of adop_radius_blocks


def _box_and_stretch(position):
    """((min, max), how far the box of the cloud exceeds that of a part of it on average, on the worst axis)."""
    lib = _capi.load_library()
    box = torch.empty(int(lib.adop_bounding_box_size()) // 4, dtype=torch.float32, device=position.device)
    _check(lib.adop_bounding_box(_ptr(position), int(position.shape[0]), _ptr(box), _stream_ptr()), lib)
    host = box[:12].tolist()  # (one read: the host waits in it)
    lo, hi, part_lo, part_hi = host[:3], host[3:6], host[6:9], host[9:]
    stretch = max((b - a) / (d - c) if d > c else 1.0 for a, b, c, d in zip(lo, hi, part_lo, part_hi))
    return ((C.c_float * 3)(*lo), (C.c_float * 3)(*hi)), stretch


def _bbox(position):
    return _box_and_stretch(position)[0]


def _knn_workspace(position):
    lib = _capi.load_library()
    return torch.empty(int(lib.adop_knn_workspace_size(int(position.shape[0]))), dtype=torch.uint8, device=position.device)


def _knn_distance(position, rank, box, ws=None):
    n = int(position.shape[0])
    lib = _capi.load_library()
    out = torch.empty(n, dtype=torch.float32, device=position.device)
    ws = _knn_workspace(position) if ws is None else ws
    rc = lib.adop_knn_distance(_ptr(position), n, int(rank), *box, _ptr(out), _ptr(ws), int(ws.numel()), _stream_ptr())
    _check(rc, lib)
    return out


def _morton_codes(position, box):
    lib = _capi.load_library()
    codes = torch.empty(int(position.shape[0]), dtype=torch.int64, device=position.device)
    _check(lib.adop_morton_codes(_ptr(position), int(position.shape[0]), *box, _ptr(codes), _stream_ptr()), lib)
    return codes


# Up to the first number of points the sort of whole codes takes no longer than the shorter one and the look at its flag; above the
# second the keys do not tell the points of a surface apart any more and the ties cost more than the shorter sort saves.  By
# keys against by codes: 3 M points 0.24 to 0.27 ms (volume to surface) against 0.36, 10 M 0.57 to 0.83 against 0.99, 2^24
# 0.97 to 1.62 against 1.61, 30 M 1.8 to 3.9 against 2.8.
_KEY_SORT_FROM, _KEY_SORT_TO = 1 << 20, 1 << 24
# A far outlier leaves all other points few keys: sorted by them in vain (10 M points: 1.41 ms in place of 0.98).
_KEY_SORT_STRETCH = 4.0


def _sorts_by_keys(n, stretch):
    return _KEY_SORT_FROM <= n <= _KEY_SORT_TO and stretch <= _KEY_SORT_STRETCH


def _morton_order(position, box, by_keys):
    """Stable order of the points along the Morton curve, as a function that returns it (the host waits in it for the flag
    of adop_morton_ties: what it can do beforehand, it does before)."""
    n = int(position.shape[0])
    if not by_keys:
        order = torch.sort(_morton_codes(position, box), stable=True).indices
        return lambda: order
    lib = _capi.load_library()
    codes = torch.empty(n, dtype=torch.int64, device=position.device)
    keys = torch.empty(n, dtype=torch.int32, device=position.device)
    _check(lib.adop_morton_keys(_ptr(position), n, *box, _ptr(codes), _ptr(keys), _stream_ptr()), lib)
    keys, order = torch.sort(keys, stable=True)
    too_long = torch.empty(1, dtype=torch.int32, device=position.device)
    _check(lib.adop_morton_ties(_ptr(keys), _ptr(order), _ptr(codes), n, _ptr(too_long), _stream_ptr()), lib)
    return lambda: torch.sort(codes, stable=True).indices if int(too_long.item()) else order


def _gather_points(position, index):
    """position[index] for rows of 4 floats.  (torch's own gather of rows of 16 bytes takes ten times as long; at 2^26 rows it
    raises, and of more it returns wrong ones without an error.)"""
    lib = _capi.load_library()
    out = torch.empty(int(index.shape[0]), 4, dtype=torch.float32, device=position.device)
    _check(lib.adop_gather_points(_ptr(position), int(position.shape[0]), _ptr(index), int(index.shape[0]), _ptr(out),
                                  _stream_ptr()), lib)
    return out


def _gather_rows(rows, index, part=1 << 25):
    """rows[index] for rows of any size, in parts that torch's gather can take."""
    return rows[index] if index.shape[0] <= part else torch.cat([rows[i] for i in index.split(part)])


def KNearestNeighbourDistance(position, rank=4):
    """Distance of every point to its ``rank``-th nearest other point: ``data[i](0)`` of ComputeRadius
    (SceneData.cpp:441-463).  position: [N,4] f32 on the device."""
    position = _checked_position(position)
    return _knn_distance(position, rank, _bbox(position))


def MortonCodes(position):
    """63-bit Morton code of every point inside the cloud's bounding box (the key of ReorderMorton64)."""
    position = _checked_position(position)
    return _morton_codes(position, _bbox(position))


def _camera_distance(position, poses_se3, intrinsics, frames, knn_ws=None):
    assert position.is_cuda and position.dtype == torch.float32 and position.dim() == 2 and position.shape[1] == 4
    assert poses_se3.is_cuda and poses_se3.dtype == torch.float64 and poses_se3.shape[1] == 8
    assert intrinsics.is_cuda and intrinsics.dtype == torch.float32 and intrinsics.shape[1] == 13
    position, poses_se3, intrinsics = position.contiguous(), poses_se3.contiguous(), intrinsics.contiguous()
    lib = _capi.load_library()
    s = _capi.Scene()
    s.position, s.num_points = position.data_ptr(), int(position.shape[0])
    s.poses_se3, s.num_poses = poses_se3.data_ptr(), int(poses_se3.shape[0])
    s.intrinsics, s.num_cameras, s.intrinsics_cols = intrinsics.data_ptr(), int(intrinsics.shape[0]), 13
    views = (_capi.View * len(frames))(*frames)
    out = torch.empty(s.num_points, dtype=torch.float32, device=position.device)
    ws = torch.empty(int(lib.adop_frames_workspace_size(len(frames))), dtype=torch.uint8, device=position.device)
    if knn_ws is None:
        rc = lib.adop_point_distance_to_camera(C.byref(s), views, len(frames), _ptr(out), _ptr(ws), int(ws.numel()),
                                               _stream_ptr())
    else:
        rc = lib.adop_point_distance_to_camera_grid(C.byref(s), views, len(frames), _ptr(out), _ptr(ws), int(ws.numel()),
                                                    _ptr(knn_ws), int(knn_ws.numel()), _stream_ptr())
    _check(rc, lib)
    return out


def PointDistanceToCamera(position, poses_se3, intrinsics, frames):
    """SceneData::PointDistanceToCamera (SceneData.cpp:645-669): distance of every point to the nearest camera that
    sees it.  position [N,4] f32, poses_se3 [F,8] f64 (view transforms), intrinsics [K,13] f32 on the device;
    ``frames``: one adop view per frame (w, h, image_index, camera_index)."""
    return _camera_distance(position, poses_se3, intrinsics, frames)


def RemoveLonelyPoints(position, camera_distance, n=5, dis_th=0.02):
    """Keep mask of SceneData::RemoveLonelyPoints (SceneData.cpp:550-595): a point goes when the distance to its
    n-th nearest neighbour, relative to its camera distance, exceeds ``dis_th``."""
    d = KNearestNeighbourDistance(position, n)
    return ~(d / camera_distance > dis_th)


def _decide_close_points(position, radius, box, state, ws, rounds_per_call, resume):
    """Rounds of the close-point filter until every point is decided.  resume = 1: ``ws`` holds the search grid of these
    points and ``state`` what is decided already."""
    lib = _capi.load_library()
    undecided = torch.empty(rounds_per_call, dtype=torch.int32, device=position.device)
    while True:
        rc = lib.adop_close_points(_ptr(position), int(position.shape[0]), _ptr(radius), *box, _ptr(state), _ptr(undecided),
                                   rounds_per_call, resume, _ptr(ws), int(ws.numel()), _stream_ptr())
        _check(rc, lib)
        if int(undecided[-1].item()) == 0:
            return state == 1
        resume = 1


def RemoveClosePoints(position, camera_distance, dis_th=0.00005, rounds_per_call=8):
    """Keep mask of SceneData::RemoveClosePoints (SceneData.cpp:598-642): in index order, a point goes when a point
    kept before it lies within dis_th / camera_distance of it."""
    position = _checked_position(position)
    radius = (dis_th / camera_distance).to(torch.float32).contiguous()
    state = torch.empty(int(position.shape[0]), dtype=torch.int32, device=position.device)
    return _decide_close_points(position, radius, _bbox(position), state, _knn_workspace(position), rounds_per_call, 0)


def FilterPointCloud(position, poses_se3, intrinsics, frames, lonely=(5, 0.02), close=0.00005):
    """The two filters of a new scene in the reference's order (SceneData.cpp:98-99): RemoveLonelyPoints(5, 0.02), then
    RemoveClosePoints(0.00005) on what is left.  Returns the ids of the surviving points, ascending.

    One search grid serves both, and the distances to the cameras: a point the first filter takes is erased before the
    second one starts, and neither the distances nor the order of the others change by its staying in the grid."""
    position = _checked_position(position)
    box, ws = _bbox(position), _knn_workspace(position)
    n, dis_th = lonely
    distance = _knn_distance(position, n, box, ws)
    cam = _camera_distance(position, poses_se3, intrinsics, frames, ws)  # per point: erasing others does not change it
    state = (distance / cam > dis_th).to(torch.int32) * 2  # 2: erased
    radius = (close / cam).to(torch.float32)
    ids = _decide_close_points(position, radius, box, state, ws, 8, 1).nonzero().squeeze(1)
    if ids.numel() == 0:  # (the first point the lonely filter leaves stays, so it has left none)
        raise RuntimeError("FilterPointCloud: no point is left")
    return ids


def ReorderMorton64(position):
    """Permutation that sorts the cloud along the Morton curve (stable: equal codes keep their order)."""
    return torch.sort(MortonCodes(position), stable=True).indices


def RandomBlockShuffle(num_points, block_size=256, generator=None):
    """Permutation that shuffles whole blocks of ``block_size`` consecutive points (a last, shorter block stays
    last)."""
    nb = num_points // block_size
    dev = "cuda"
    perm = torch.randperm(nb, generator=generator, device="cpu").to(dev)
    idx = (perm[:, None] * block_size + torch.arange(block_size, device=dev)[None, :]).reshape(-1)
    tail = torch.arange(nb * block_size, num_points, device=dev)
    return torch.cat([idx, tail])


def ComputeRadius(position, rank=4, generator=None):
    """SceneData::ComputeRadius (SceneData.cpp:441-484): returns ``data`` [N,4] with data[:,0] = distance to the
    rank-th neighbour, data[:,2] = sqrt(1 / u), u ~ U(0,1), data[:,3] = data[:,0] * data[:,2] (the drop-out radius the
    rasterizer reads as position.w, NeuralPointCloudCuda.cpp:21-35)."""
    n = int(position.shape[0])
    data = torch.zeros(n, 4, dtype=torch.float32, device=position.device)
    data[:, 0] = KNearestNeighbourDistance(position, rank)
    if generator is not None and generator.device.type == "cpu":  # a host generator: draw there
        u = torch.rand(n, generator=generator, dtype=torch.float64, device="cpu").to(position.device)
    else:
        u = torch.rand(n, generator=generator, dtype=torch.float64, device=position.device)
    data[:, 2] = torch.sqrt(1.0 / u.clamp_min_(1e-300)).to(torch.float32)
    data[:, 3] = data[:, 0] * data[:, 2]
    return data


def SortBlocksByRadius(radius, block_size=256):
    """Permutation that sorts every full block of ``block_size`` points by ascending radius
    (SceneData.cpp:671-684; the last, shorter block keeps its order)."""
    n = int(radius.shape[0])
    nb = n // block_size
    head = radius[: nb * block_size].reshape(nb, block_size)
    order = torch.sort(head, dim=1, stable=True).indices + (torch.arange(nb, device=radius.device) * block_size)[:, None]
    return torch.cat([order.reshape(-1), torch.arange(nb * block_size, n, device=radius.device)])


def PreprocessPointCloud(position, normal=None, rank=4, block_size=256, seed=0):
    """The initial processing of a new scene in the reference's order (SceneData.cpp:101-104): ReorderMorton64,
    RandomBlockShuffle(256), ComputeRadius, SortBlocksByRadius(256).  Returns (position [N,4] with the drop-out radius in
    w, normal, data [N,4], order) where ``order`` maps new to original point ids."""
    gen = torch.Generator(device="cpu").manual_seed(int(seed))
    gen_dev = torch.Generator(device=position.device).manual_seed(int(seed))  # the per-point numbers are drawn on the device
    position = _checked_position(position)
    _check_normal(normal, position)
    n = int(position.shape[0])
    if block_size != _RADIUS_BLOCK or (normal is not None and (normal.dtype != torch.int32 or normal.numel() != n)):
        order = ReorderMorton64(position)
        order = order[RandomBlockShuffle(n, block_size, gen)]
        position = _gather_points(position, order)
        data = ComputeRadius(position, rank, gen_dev)
        by_radius = SortBlocksByRadius(data[:, 3], block_size)
        order = order[by_radius]
        position = _gather_points(position, by_radius)
        data = _gather_points(data, by_radius)
        position[:, 3] = data[:, 3]
        return position, (None if normal is None else _gather_rows(normal, order).contiguous()), data, order
    # The same steps in passes over whole points: one gather along both permutations, one kernel for the radii and the
    # order inside the blocks.  One bounding box serves the codes and the search: the points stay the same.
    lib = _capi.load_library()
    shape = None if normal is None else normal.shape
    normal = None if normal is None else normal.contiguous()
    box, stretch = _box_and_stretch(position)
    order = _morton_order(position, box, _sorts_by_keys(n, stretch))
    blocks = torch.randperm(n // block_size, generator=gen, device="cpu").to(position.device)
    order = order()
    shuffled, ids = torch.empty_like(position), torch.empty(n, dtype=torch.int32, device=position.device)
    shuffled_normal = None if normal is None else torch.empty_like(normal)
    _check(lib.adop_shuffle_points(_ptr(position), _ptr(normal), _ptr(order), _ptr(blocks), n, block_size, _ptr(shuffled),
                                   _ptr(shuffled_normal), _ptr(ids), _stream_ptr()), lib)
    distance = _knn_distance(shuffled, rank, box)
    uniform = torch.rand(n, generator=gen_dev, dtype=torch.float64, device=position.device)
    out, data = torch.empty_like(position), torch.empty_like(position)
    out_normal = None if normal is None else torch.empty(shape, dtype=torch.int32, device=position.device)
    _check(lib.adop_radius_blocks(_ptr(shuffled), _ptr(shuffled_normal), _ptr(ids), _ptr(distance), _ptr(uniform), n,
                                  _ptr(out), _ptr(out_normal), _ptr(data), _ptr(order), _stream_ptr()), lib)
    return out, out_normal, data, order


def AttachDropOutRadii(hs, rank=4, block_size=256, seed=0):
    """Gives a host scene (``scenes.HostScene`` in the reference's point order) what the rasterizer's LOD test reads,
    as a new scene gets it (SceneData.cpp:103-104): ``position.w`` = ComputeRadius' drop-out radius, every 256-point
    block sorted by it; switches ``drop_out_points_by_radius`` on (the reference's default, Settings.h:36-37).  The
    descriptors and the dropout mask of the synthetic scenes are independent random numbers per point and stay."""
    pos = torch.from_numpy(hs.position).cuda()
    gen = torch.Generator(device=pos.device).manual_seed(int(seed))
    data = ComputeRadius(pos, rank, gen)
    order = SortBlocksByRadius(data[:, 3], block_size)
    pos = _gather_points(pos.contiguous(), order)
    pos[:, 3] = data[order, 3]
    hs.position = pos.cpu().numpy()
    if hs.normal is not None:
        hs.normal = torch.from_numpy(hs.normal).cuda()[order].cpu().numpy()
    hs.params.drop_out_points_by_radius = 1
    hs.meta["lod_radius_test"] = True
    return hs
