"""The kernels that larger launches run, which small frames do not reach:
renders of more than SMALL_RENDER_TILES_ALONE tiles without statistics (one
lane per ray, the packed walk, the footprint tables) and training passes of
more tiles than four lanes per ray take, for every map size, entry and storage.
Renders are held against the statistics renders of the same frames, which other
tests hold against the oracle; training against small launches of the same rays."""
import numpy as np
import pytest
import torch

from tests import helpers as H
from vorotracing_amd import _C, camera, native, scene
from vorotracing_amd.infer import VoroTracingInfer
from vorotracing_amd.model import VoroTracing

pytestmark = pytest.mark.gpu

LARGE, SMALL = (301, 397), (61, 75)  # 1,900 and 80 tiles, ragged
KW = dict(weight_threshold=0.001, cell_skip_threshold=1e-3)


def _infer(gpu, maps, quantize):
    return VoroTracingInfer(VoroTracing.from_scene(scene.random_scene(1500, seed=3, R=maps[0], Rs=maps[1]), device=gpu),
                            quantize=quantize)


def _bits(x):
    return x.view(torch.int16)


def _tiles(hw):
    return native.num_tiles(1, *hw, *VoroTracingInfer.TILE)


@pytest.mark.parametrize("hw", [LARGE, SMALL])
@pytest.mark.parametrize("maps", [(4, 4), (8, 4), (4, 8), (8, 8)])
@pytest.mark.parametrize("quantize", ["fp16", "q8"])
def test_renders_of_every_layout(gpu, quantize, maps, hw):
    """Image rays, camera lanes and camera lanes with a start cell per row: the
    statistics render's bits, with the packed walk and the tables and without."""
    assert _tiles(SMALL) <= native.SMALL_RENDER_TILES < native.SMALL_RENDER_TILES_ALONE < _tiles(LARGE)
    inf = _infer(gpu, maps, quantize)
    h, w = hw
    cams = {"orbit": [camera.Camera.orbit(3, w, h)],
            "rolling": [camera.Camera.fisheye_rolling(w, h, eye=camera.orbit_eye(4))]}
    rays = native.camera_rays(cams["orbit"], gpu)[0].contiguous()
    want = inf.render(rays, stats=native.new_stats(h * w, gpu), **KW)
    want_cams = {k: inf.render_cameras(c, stats=native.new_stats(h * w, gpu), **KW) for k, c in cams.items()}
    assert inf.camera_start_points(cams["rolling"])[1] and not inf.camera_start_points(cams["orbit"])[1]
    for x in (want, *want_cams.values()):
        assert float(x[..., 3].max()) > 0.5
    for walk in (True, False):
        for quads in (True, False):
            inf.packed_walk, inf.quad_maps = walk, quads
            assert (inf.walk_layout() is not None) == walk and (inf.quad_tables() is not None) == quads
            assert torch.equal(_bits(inf.render(rays, **KW)), _bits(want)), (walk, quads)
            for k, c in cams.items():
                assert torch.equal(_bits(inf.render_cameras(c, **KW)), _bits(want_cams[k])), (walk, quads, k)


@pytest.mark.parametrize("quantize", ["fp16", "q8"])
def test_stale_caches_of_large_drop_in_renders(gpu, quantize):
    """The drop-ins' cached walk layout and tables are rebuilt after an in-place
    change of the density and of the maps: a frame whose kernel reads both."""
    inf = _infer(gpu, (8, 4), quantize)
    rays = native.camera_rays([camera.Camera.orbit(3, LARGE[1], LARGE[0])], gpu)[0].contiguous()
    sp, perm = inf.get_starting_point(rays), torch.arange(rays.numel() // 6, dtype=torch.int32, device=gpu)
    den = inf.density.clone()
    maps = inf.diffuse_fp16.clone() if quantize == "fp16" else inf.diffuse_q8.clone()

    def render():
        scn = (den, inf.point_adjacency, inf.point_adjacency_offsets, rays, sp, inf.adjacent_diff)
        if quantize == "fp16":
            return _C.trace_vorotracing_infer(inf.primal_points, maps, inf.specular_fp16, *scn, perm, 0.01, 1024, 1e-3)
        return _C.trace_vorotracing_infer_q8(inf.primal_points, maps, inf.specular_q8, *scn, inf.diff_scale,
                                             inf.diff_offset, inf.spec_scale, inf.spec_offset, 0.01, 1024, 1e-3,
                                             ray_perm_in=perm)

    saved, last = (_C.DROP_IN_WALK, _C.DROP_IN_QUADS), None
    try:
        for change in (lambda: None, lambda: den.mul_(0.5), lambda: maps.copy_(maps.flip(0))):
            change()
            _C.DROP_IN_WALK = _C.DROP_IN_QUADS = False
            plain = render()
            _C.DROP_IN_WALK = _C.DROP_IN_QUADS = True
            assert torch.equal(_bits(render()), _bits(plain))
            assert last is None or not torch.equal(_bits(last), _bits(plain))
            last = plain
    finally:
        _C.DROP_IN_WALK, _C.DROP_IN_QUADS = saved


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("flat", [True, False])
def test_training_without_contribution_or_error(gpu, flat, f16):
    """Flat batches in a lane order and images, in a launch with one lane per ray
    and in small ones with four: per-ray outputs bit for bit, gradients against
    the sums over the small ones."""
    s = scene.random_scene(1200, seed=5, R=4, Rs=8)
    m = VoroTracing.from_scene(s, device=gpu)
    dt = torch.float16 if f16 else torch.float32
    scn = (m.primal_points.detach(), m.att_diffuse.detach().to(dt), m.att_specular.detach().to(dt),
           m.activated_density().detach(), m.point_adjacency, m.point_adjacency_offsets)
    h, w, n = 121, 131, 12  # 272 tiles an image
    rays = H.to_dev(np.stack([camera.orbit_rays(k, w, h, n=n, radius=4.0) for k in range(n)]), gpu)
    if flat:
        rays = rays.reshape(-1, 6)[torch.randperm(n * h * w, generator=torch.Generator().manual_seed(4)).to(gpu)]
        rays = torch.cat([rays, rays[:20000]]).contiguous()
    tiles = (rays.shape[0] + 63) // 64 if flat else n * native.num_tiles(1, h, w, 8, 8)
    assert tiles > 3072
    start = m.get_starting_point(rays)
    cuts = [slice(0, 1), slice(777, 777 + 5041), slice(150000, 150000 + 64 * 1700)] if flat else [slice(0, 1), slice(6, 9)]
    gen = torch.Generator(device=gpu).manual_seed(1)
    up = torch.zeros(list(rays.shape[:-1]) + [4], device=gpu)
    for c in cuts:
        up[c] = torch.randn(up[c].shape, generator=gen, device=gpu)
    up = up.to(dt)

    def both(c):
        r, sp, g = rays[c].contiguous(), start[c].contiguous(), up[c].contiguous()
        out = _C.trace_vorotracing_fwd(*scn, r, sp, None, 0.001, 1024, False)
        grads = _C.trace_vorotracing_bwd(*scn, r, sp, out[0], g, None, None, None, None, 0.0, out[5], None, out[6],
                                         out[7], out[8], 0.001, 1024)
        return [x for x in out if x is not None], grads[:4]

    whole, want = both(slice(None))
    parts = [both(c) for c in cuts]
    for c, (out, _) in zip(cuts, parts):
        for a, b in zip(out, whole):
            b = b[c].contiguous()
            assert a.numel() == b.numel() and torch.equal(a.flatten().view(torch.uint8), b.flatten().view(torch.uint8))
    for i, x in enumerate(want):
        H.assert_launches_sum([p[1][i] for p in parts], x, f16 and i in (1, 2), i)
