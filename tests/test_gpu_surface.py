"""GPU parity of the fused surface maps (nest_surface_maps) against the same
expressions as tensor operations on the CPU."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _allmap(W, H, seed):
    """A wavy surface at depth ~3 with every kind of depth: none (alpha 0,
    depth 0), infinite and NaN."""
    g = torch.Generator().manual_seed(seed)
    y, x = torch.meshgrid(torch.arange(H).float(), torch.arange(W).float(), indexing="ij")
    a = torch.rand((14, H, W), generator=g)
    a[1] = 0.3 + 0.7 * a[1]
    a[0] = (3 + 0.3 * torch.sin(x / 7) + 0.2 * torch.cos(y / 5)) * a[1]
    a[5] = a[0] / a[1] + 0.01
    if W * H > 8:
        a[0:2, H // 2, W // 3:] = 0.0
        a[0, 0, 0], a[1, 0, 0] = 1.0, 0.0
        a[5, H - 1, W // 2] = float("nan")
        a[5, H // 3, W - 1] = float("-inf")
    return a


@pytest.mark.parametrize("W,H", [(1, 1), (2, 5), (3, 3), (64, 4), (97, 61)])
@pytest.mark.parametrize("ratio", [0.0, 0.3, 1])
def test_surface_maps_fused(W, H, ratio):
    """Depths bit for bit.  Points are within ~1e-6 of coordinates of ~3
    (binary32 products and sums in another order), their differences over two
    pixels at least ~0.03 long, so the normals within 1e-4."""
    from nest_splat.camera import look_at
    from nest_splat.renderer import surface_maps
    cam = look_at((0.4, -3.0, 1.0), (0, 0, 0), 50.0, W, H)
    a = _allmap(W, H, W + H)
    ref = surface_maps(cam, a, ratio)
    dev = a.to(DEV)
    out = surface_maps(cam, dev, ratio)
    assert set(out) == set(ref)
    for k, v in ref.items():
        o = out[k].cpu()
        assert o.shape == v.shape and out[k].stride() == v.stride(), k
        if k == "rend_normal":
            np.testing.assert_allclose(o.numpy(), v.numpy(), atol=1e-6)
        elif k == "surf_normal":
            big = (ref["surf_depth"].abs() > 1e30)  # -inf became the lowest finite: its neighbours overflow
            near = torch.nn.functional.max_pool2d(big.float(), 3, 1, 1)[0] > 0
            keep = ~near.expand_as(v)
            np.testing.assert_allclose(o[keep].numpy(), v[keep].numpy(), atol=1e-4)
        else:
            np.testing.assert_array_equal(o.numpy(), v.numpy(), err_msg=k)


@pytest.mark.parametrize("ratio", [0.0, 0.3])
def test_surface_normal_against_64_bits(ratio):
    """The normal of the back-projected depth map in 64 bits, from the same
    32-bit map, ray matrix and view matrix.  A point's coordinates come from
    terms below 4 with three 32-bit roundings (7e-7); each of the two
    differences, at least 0.04 long, errs by up to twice that, 3.6e-5 of its
    length: 7e-5 of the normal, so 1e-4."""
    from nest_splat.camera import look_at, view_ray_matrix
    from nest_splat.renderer import surface_maps
    W, H = 97, 61
    cam = look_at((0.4, -3.0, 1.0), (0, 0, 0), 50.0, W, H)
    a = _allmap(W, H, 9)
    y, x = torch.meshgrid(torch.arange(H).double(), torch.arange(W).double(), indexing="ij")
    a[1] = a[1].clamp_min(0.3)
    a[0] = ((3 + 0.3 * torch.sin(x / 7) + 0.2 * torch.cos(y / 5)) * a[1]).float()
    a[5] = a[0] / a[1] + 0.01
    d = a.double()
    depth = (1 - ratio) * d[0] / d[1] + ratio * d[5]
    rays = torch.stack([x, y, torch.ones_like(x)], -1) @ torch.from_numpy(view_ray_matrix(cam)).double()
    origin = np.linalg.inv(np.asarray(cam.world_view_transform, dtype=np.float64).T)[:3, 3]
    pts = depth[..., None] * rays + torch.from_numpy(origin)
    dy, dx = pts[2:, 1:-1] - pts[:-2, 1:-1], pts[1:-1, 2:] - pts[1:-1, :-2]
    assert dx.norm(dim=-1).min() > 0.04 and dy.norm(dim=-1).min() > 0.04 and pts.abs().max() < 4
    n = torch.zeros((H, W, 3), dtype=torch.float64)
    n[1:-1, 1:-1] = torch.nn.functional.normalize(torch.cross(dy, dx, dim=-1), dim=-1)
    out = surface_maps(cam, a.to(DEV), ratio)["surf_normal"].cpu().double()
    err = (out - (n * d[1][..., None]).permute(2, 0, 1)).abs().max().item()
    print(f"surf_normal max error {err:.1e}", flush=True)
    assert err <= 1e-4


def test_surface_maps_gradient_and_views_keep_the_general_path():
    """A map that gradients follow, and one that is not contiguous."""
    from nest_splat.camera import look_at
    from nest_splat.renderer import surface_maps
    W, H = 33, 20
    cam = look_at((0.4, -3.0, 1.0), (0, 0, 0), 50.0, W, H)
    a = _allmap(W, H, 5).to(DEV)
    g = a.clone().requires_grad_(True)
    assert surface_maps(cam, g)["rend_normal"].requires_grad
    with torch.no_grad():
        ref = surface_maps(cam, g)
    out = surface_maps(cam, a.permute(0, 2, 1).contiguous().permute(0, 2, 1))
    for k in ("surf_depth", "rend_normal"):
        np.testing.assert_allclose(out[k].cpu().numpy(), ref[k].cpu().numpy(), atol=1e-6)


def test_surface_maps_of_another_camera_size_keep_the_general_path():
    """A map that is not the camera's size does what the tensor operations do
    with it: broadcast where they broadcast, raise where they raise."""
    from nest_splat.camera import look_at
    from nest_splat.renderer import surface_maps
    cam = look_at((0.4, -3.0, 1.0), (0, 0, 0), 50.0, 1, 9)
    a = _allmap(9, 1, 3)
    ref, out = surface_maps(cam, a), surface_maps(cam, a.to(DEV))
    for k, v in ref.items():
        assert out[k].shape == v.shape, k
    np.testing.assert_array_equal(out["surf_depth"].cpu().numpy(), ref["surf_depth"].numpy())
    cam = look_at((0.4, -3.0, 1.0), (0, 0, 0), 50.0, 24, 10)
    for H, W in ((20, 12), (5, 7)):
        for dev in ("cpu", DEV):
            with pytest.raises(RuntimeError):
                surface_maps(cam, _allmap(W, H, 4).to(dev))


def test_surface_maps_have_memory_of_their_own():
    """A map that a loss saved for its backward is not touched by an in-place
    change of another map, and a map kept alone keeps no other map's memory."""
    from nest_splat.camera import look_at
    from nest_splat.renderer import surface_maps
    W, H = 33, 20
    cam = look_at((0.4, -3.0, 1.0), (0, 0, 0), 50.0, W, H)
    out = surface_maps(cam, _allmap(W, H, 6).to(DEV))
    names = ("rend_normal", "surf_normal", "surf_depth", "depth_expected", "depth_median")
    for k in names:
        assert out[k].untyped_storage().nbytes() == 4 * out[k].numel(), k
    for saved, changed in zip(names, names[1:] + names[:1]):
        w = torch.ones((), device=DEV, requires_grad=True)
        loss = (w * out[saved]).sum()
        out[changed].add_(1.0)
        loss.backward()


def test_surface_maps_of_another_device_keep_the_general_path(monkeypatch):
    """With another device current, a launch would not be this map's device's."""
    from nest_splat import renderer
    from nest_splat.camera import look_at
    W, H = 33, 20
    cam = look_at((0.4, -3.0, 1.0), (0, 0, 0), 50.0, W, H)
    a = _allmap(W, H, 7).to(DEV)
    assert renderer._plain_map(a)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: DEV.index + 1)
    assert not renderer._plain_map(a)
    monkeypatch.setattr(renderer, "_surface_maps_fused", None)
    out = renderer.surface_maps(cam, a)
    monkeypatch.undo()
    np.testing.assert_array_equal(out["surf_depth"].cpu().numpy(), renderer.surface_maps(cam, a)["surf_depth"].cpu().numpy())


def test_surface_maps_under_autocast_keep_the_general_path():
    """Autocast rounds the products of the tensor operations: types and values
    are theirs."""
    from nest_splat.camera import look_at
    from nest_splat.renderer import surface_maps
    W, H = 33, 20
    cam = look_at((0.4, -3.0, 1.0), (0, 0, 0), 50.0, W, H)
    a = _allmap(W, H, 8).to(DEV)
    for dtype in (torch.float16, torch.bfloat16):
        with torch.autocast("cuda", dtype=dtype), torch.no_grad():
            out = surface_maps(cam, a)
            general = surface_maps(cam, a.permute(0, 2, 1).contiguous().permute(0, 2, 1))
        for k, v in general.items():
            assert out[k].dtype == v.dtype, k
        assert out["rend_normal"].dtype == dtype
