"""Texture gradients of half maps: summed in f32 and rounded once
(VT_ATTR_F16_SUMS), against the oracle's f32 sums of the same terms, in
launches with four lanes per ray and with one, and past 2^32 texels."""
import numpy as np
import pytest
import torch

from oracle import core
from tests import helpers as H
from vorotracing_amd import _C, camera

pytestmark = pytest.mark.gpu


def _scene(which):
    if which == "r8":
        return H.mini_heightfield_r8(), camera.orbit_rays(5, 128, 96)
    s = H.small_random(1500, seed=5, R=8, Rs=4)
    rays = camera.pinhole_rays(48, 40, eye=(0.3, -3.2, 0.4))
    if which == "image":
        return s, rays
    return s, np.ascontiguousarray(rays.reshape(-1, 6)[:: 1920 // int(which)][:int(which)])


def _scene_args(s, dev):
    return (H.to_dev(s.points, dev), H.to_dev(s.diffuse.astype(np.float16), dev),
            H.to_dev(s.specular.astype(np.float16), dev), H.to_dev(s.density, dev), H.to_dev(s.adjacency, dev),
            H.to_dev(s.offsets, dev))


def _backward(s, rays, error, dev, scn=None, shift=0):
    """(gradients on the GPU, the half forward and upstream gradient) of a
    backward without stats; scn: another scene that holds s from cell ``shift`` on."""
    start = H.start_for(s, rays)
    rng = np.random.default_rng(1)
    fw = core.trace_fwd(s.points, s.diffuse.astype(np.float16), s.specular.astype(np.float16), s.diff_res, s.spec_res,
                        s.density, s.adjacency, s.offsets, rays, start, weight_threshold=0.001)
    g = rng.normal(size=rays.shape[:-1] + (4,)).astype(np.float16)
    e = rng.uniform(0, 1, size=rays.shape[:-1] + (1,)).astype(np.float16) if error else None
    d = lambda a: None if a is None else H.to_dev(a, dev)  # noqa: E731
    out = _C.trace_vorotracing_bwd(*(scn or _scene_args(s, dev)), d(rays), d(start + np.uint32(shift)), d(fw["rgba"]),
                                   d(g), None, None, None, d(e), 0.0, d(fw["distortion"]), None, d(fw["W_total"]),
                                   d(fw["S_total"]), d(fw["t_far"]), 0.001, 1024)
    torch.cuda.synchronize()
    return out, start, fw, g, e


def _oracle_sums(s, rays, start, fw, g, e):
    """f32 sums of the same terms, their absolute sums and counts."""
    f = lambda a: None if a is None else a.astype(np.float32)  # noqa: E731
    sums = core.trace_bwd(s.points, f(s.diffuse.astype(np.float16)), f(s.specular.astype(np.float16)), s.diff_res,
                          s.spec_res, s.density, s.adjacency, s.offsets, rays, start, f(fw["rgba"]), f(g),
                          ray_error=f(e), distortion=fw["distortion"], W_total=fw["W_total"], S_total=fw["S_total"],
                          t_far=fw["t_far"], weight_threshold=0.001)
    return sums, *H.f16_train_sums(s, rays, start, 0.001, fw, g, ray_error=e)


@pytest.mark.parametrize("which,error", [("image", False), ("image", True), ("r8", False), ("r8", True), ("1", False),
                                         ("7", False), ("23", False), ("87", False), ("87", True)])
def test_half_gradients_are_rounded_once(gpu, which, error):
    """The 1 and 7 rays leave quads to scatter that are fewer than the record's
    columns, 23 and 87 a partial wave; with an error the launch has one lane per ray."""
    s, rays = _scene(which)
    out, start, fw, g, e = _backward(s, rays, error, gpu)
    sums, A, K = _oracle_sums(s, rays, start, fw, g, e)
    H.assert_one_rounding(out[1].cpu().numpy(), sums["diffuse_grad"], A["diffuse_grad"], K["diffuse_grad"], "diffuse")
    H.assert_one_rounding(out[2].cpu().numpy(), sums["specular_grad"], A["specular_grad"], K["specular_grad"], "specular")
    H.assert_grad_close(out[0].cpu().numpy(), sums["points_grad"], "points_grad", abs_sum=A["points_grad"])
    H.assert_grad_close(out[3].cpu().numpy(), sums["density_grad"], "density_grad", abs_sum=A["density_grad"])
    if error:
        H.assert_f16_sum_close(out[5].cpu().numpy(), core.trace_bwd(
            s.points, s.diffuse.astype(np.float16), s.specular.astype(np.float16), s.diff_res, s.spec_res, s.density,
            s.adjacency, s.offsets, rays, start, fw["rgba"], g, ray_error=e, distortion=fw["distortion"],
            W_total=fw["W_total"], S_total=fw["S_total"], t_far=fw["t_far"], weight_threshold=0.001)["point_error"],
            A["point_error"], K["point_error"], "point_error")


@pytest.mark.parametrize("why", ["size", "memory"])
@pytest.mark.parametrize("which,error", [("image", False), ("image", True), ("87", False), ("7", False)])
def test_half_atomics(gpu, monkeypatch, why, which, error):
    """Past the sizes up to which the sums pay, and where they cannot be
    allocated, gradients are added with half atomics (VT_ATTR_F16): within the
    accumulation bound of the oracle's half sums."""
    s, rays = _scene(which)
    if why == "size":
        monkeypatch.setattr(_C, "SUMS_VALUES", 0)
        monkeypatch.setattr(_C, "SUMS_VALUES_PER_RAY", 0)
    else:
        empty, slots = torch.empty, 4 * s.points.shape[0]

        def no_memory(*size, **kw):
            if kw.get("dtype") == torch.float32 and isinstance(size[0], int) and size[0] > slots:
                raise torch.OutOfMemoryError("no memory for the sums")
            return empty(*size, **kw)

        monkeypatch.setattr(torch, "empty", no_memory)
    codes = []
    workspace = _C._cell_workspace
    monkeypatch.setattr(_C, "_cell_workspace", lambda *a: codes.append(workspace(*a)) or codes[-1])
    out, start, fw, g, e = _backward(s, rays, error, gpu)
    assert [c[0] for c in codes] == [1] and codes[0][1].numel() == 4 * s.points.shape[0]
    want = core.trace_bwd(s.points, s.diffuse.astype(np.float16), s.specular.astype(np.float16), s.diff_res, s.spec_res,
                          s.density, s.adjacency, s.offsets, rays, start, fw["rgba"], g, ray_error=e,
                          distortion=fw["distortion"], W_total=fw["W_total"], S_total=fw["S_total"], t_far=fw["t_far"],
                          weight_threshold=0.001)
    _, A, K = _oracle_sums(s, rays, start, fw, g, e)
    for got, key in ((out[1], "diffuse_grad"), (out[2], "specular_grad")) + (((out[5], "point_error"),) if error else ()):
        H.assert_f16_sum_close(got.cpu().numpy(), want[key], A[key], K[key], key)
    H.assert_grad_close(out[0].cpu().numpy(), want["points_grad"], "points_grad", abs_sum=A["points_grad"])


def test_more_texels_than_a_grid_has_threads(gpu, monkeypatch):
    """11.3 million cells of 8x8 and 8x8 maps are 4.3e9 texels: more than 2^32,
    which bounds a grid's threads.  The cells that the rays meet are the last."""
    monkeypatch.setattr(_C, "SUMS_VALUES", 1 << 40)
    s = H.small_random(400, seed=11, R=8, Rs=8)
    rays = camera.pinhole_rays(24, 16, eye=(0.3, -3.2, 0.4))
    pad = 11_300_000
    n, tex = pad + s.points.shape[0], 3 * 64
    assert 2 * tex * n > 1 << 32
    off = torch.zeros(n + 1, dtype=torch.int32, device=gpu)
    off[pad:] = torch.from_numpy(s.offsets.astype(np.int32)).to(gpu)
    adj = H.to_dev((s.adjacency + np.uint32(pad)).astype(np.uint32), gpu)
    pts, den = torch.zeros((n, 3), device=gpu), torch.zeros((n, 1), device=gpu)
    pts[pad:], den[pad:] = H.to_dev(s.points, gpu), H.to_dev(s.density, gpu).reshape(-1, 1)
    maps = [torch.zeros((n, tex), dtype=torch.float16, device=gpu) for _ in range(2)]
    for m, a in zip(maps, (s.diffuse, s.specular)):
        m[pad:] = H.to_dev(a.astype(np.float16), gpu)
    (pg, dg, sg, deng, _, _), start, fw, g, e = _backward(s, rays, False, gpu,
                                                          (pts, *maps, den, adj, off.view(torch.uint32)), pad)
    sums, A, K = _oracle_sums(s, rays, start, fw, g, e)
    H.assert_one_rounding(dg[pad:].cpu().numpy(), sums["diffuse_grad"], A["diffuse_grad"], K["diffuse_grad"], "diffuse")
    H.assert_one_rounding(sg[pad:].cpu().numpy(), sums["specular_grad"], A["specular_grad"], K["specular_grad"], "specular")
    H.assert_grad_close(pg[pad:].cpu().numpy(), sums["points_grad"], "points_grad", abs_sum=A["points_grad"])
    for grad in (pg, dg, sg, deng):
        assert int(torch.count_nonzero(grad[pad:])) > 0
        assert not any(bool(part.any()) for part in grad[:pad].split(1 << 20))
