"""Launches of few tiles run with four lanes per ray, larger ones with one
(vt_walk.h walk_step_group, the *_GROUP_TILES rules): the same rays rendered or
trained in a small launch and inside a large one give the same bits per ray,
and the same gradients up to the order of their sums.  The small launches are
held against the oracle by the other tests' frames.  test_gpu_one_lane.py has
flat batches, and half training without contribution or error."""
import numpy as np
import pytest
import torch

from tests import helpers as H
from vorotracing_amd import _C, _lib, camera, native, scene
from vorotracing_amd.infer import VoroTracingInfer
from vorotracing_amd.model import VoroTracing

pytestmark = pytest.mark.gpu

MOST = 3072  # tiles of the largest launch with four lanes per ray


def _images(gpu, n, h, w):
    """n images of one camera each (n, h, w, 6)."""
    return H.to_dev(np.stack([camera.orbit_rays(k, w, h, n=n, radius=4.0) for k in range(n)]), gpu)


def _tiles(rays):
    if rays.dim() == 2:
        return (rays.shape[0] + 63) // 64
    b = 1 if rays.dim() == 3 else rays.shape[0]
    return b * ((rays.shape[-3] + 7) // 8) * ((rays.shape[-2] + 7) // 8)


@pytest.mark.parametrize("h,w", [(121, 131), (8, 9), (64, 64)])
@pytest.mark.parametrize("quantize", ["fp16", "q8"])
def test_render_small_and_large_launch(gpu, quantize, h, w):
    m = VoroTracing.from_scene(scene.random_scene(1500, seed=3, R=8, Rs=4), device=gpu)
    inf = VoroTracingInfer(m, quantize=quantize)
    n = MOST // _tiles(_images(gpu, 1, h, w)[0]) + 1
    rays = _images(gpu, n, h, w)
    assert _tiles(rays) > MOST >= _tiles(rays[0])
    kw = dict(weight_threshold=0.001, cell_skip_threshold=1e-3)
    whole = inf.render(rays, **kw)
    for k in (0, n // 2, n - 1):
        assert torch.equal(inf.render(rays[k].contiguous(), **kw), whole[k])
    flat = rays[:, ::3, ::2].reshape(-1, 6).contiguous()
    flat = flat.repeat(-(-(64 * MOST + 1) // flat.shape[0]), 1)
    start = inf.bvh.start_cells(inf.primal_points, flat)
    whole = inf.render(flat, start_point=start, **kw)
    for count in (1, 63, 65, 1001):
        assert torch.equal(inf.render(flat[:count].contiguous(), start_point=start[:count].contiguous(), **kw),
                           whole[:count])


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("h,w", [(121, 131), (9, 8)])
def test_training_small_and_large_launch(gpu, f16, h, w):
    """Every per-ray output of the forward bit for bit (depth quantiles and
    statistics of the distortion among them); contribution and gradients of the
    large launch against the sums over the small ones."""
    s = scene.random_scene(1200, seed=5, R=4, Rs=8)
    m = VoroTracing.from_scene(s, device=gpu)
    dt = torch.float16 if f16 else torch.float32
    scn = (m.primal_points.detach(), m.att_diffuse.detach().to(dt), m.att_specular.detach().to(dt),
           m.activated_density().detach(), m.point_adjacency, m.point_adjacency_offsets)
    n = MOST // _tiles(_images(gpu, 1, h, w)[0]) + 1
    rays = _images(gpu, n, h, w)
    assert _tiles(rays) > MOST
    g = torch.Generator(device=gpu).manual_seed(1)
    start = m.get_starting_point(rays)
    lead = list(rays.shape[:-1])
    q = torch.tensor([0.7, 0.3], device=gpu).expand(lead + [2]).contiguous()
    # upstream gradients for a few of the images: the others add nothing
    some = sorted({0, n // 2, n - 1})
    up = torch.zeros(lead + [4], device=gpu)
    gd = torch.zeros(lead + [1], device=gpu)
    gq = torch.zeros(lead + [2], device=gpu)
    for k in some:
        up[k] = torch.randn(up[k].shape, generator=g, device=gpu)
        gd[k] = 0.01 * torch.rand(gd[k].shape, generator=g, device=gpu)
        gq[k] = 0.1 * torch.randn(gq[k].shape, generator=g, device=gpu)
    up = up.to(dt)

    def both(sel):
        r, sp, qs = rays[sel].contiguous(), start[sel].contiguous(), q[sel].contiguous()
        out = _C.trace_vorotracing_fwd(*scn, r, sp, qs, 0.001, 1024, True)
        rgba, depth, idx, _, _, dist, wt, st, tf = out
        err = torch.ones(list(r.shape[:-1]) + [1], dtype=dt, device=gpu) * 0.5
        grads = _C.trace_vorotracing_bwd(*scn, r, sp, rgba, up[sel].contiguous(), qs, idx, gq[sel].contiguous(), err, 0.0,
                                         dist, gd[sel].contiguous(), wt, st, tf, 0.001, 1024)
        return out, grads

    whole, wgrads = both(slice(None))
    parts = {k: both(k) for k in some}
    for k, (out, _) in parts.items():
        for name, a, b in zip(("rgba", "depth", "depth_idx", None, "n", "distortion", "W", "S", "t_far"), out, whole):
            if name:
                assert torch.equal(a.view(torch.int16 if a.dtype == torch.float16 else torch.int32),
                                   b[k].view(torch.int16 if a.dtype == torch.float16 else torch.int32)), (k, name)
    # (with a contribution and an error, half launches run one lane per ray whatever their size)
    for i in range(4):
        H.assert_launches_sum([p[1][i] for p in parts.values()], wgrads[i], f16 and i in (1, 2), i)


def test_contribution_and_point_error(gpu):
    """The lane that adds to the shared outputs adds once per ray: against a large launch of the same rays repeated."""
    m = VoroTracing.from_scene(scene.random_scene(600, seed=9, R=4), device=gpu)
    scn = (m.primal_points.detach(), m.att_diffuse.detach(), m.att_specular.detach(),
           m.activated_density().detach(), m.point_adjacency, m.point_adjacency_offsets)
    ray = _images(gpu, 1, 64, 72)
    times = MOST // _tiles(ray[0]) + 1
    sums = []
    for rays in (ray[0], ray.repeat(times, 1, 1, 1)):
        rays = rays.contiguous()
        start = m.get_starting_point(rays)
        out = _C.trace_vorotracing_fwd(*scn, rays, start, None, 0.001, 1024, True)
        err = torch.ones(list(rays.shape[:-1]) + [1], device=gpu)
        grads = _C.trace_vorotracing_bwd(*scn, rays, start, out[0], torch.zeros_like(out[0]), None, None, None, err, 0.0,
                                         out[5], None, out[6], out[7], out[8], 0.001, 1024)
        sums.append((out[3].double(), grads[5].double()))
    for a, b in zip(sums[0], sums[1]):
        assert float((times * a - b).norm()) <= 1e-5 * float(b.norm())
        assert float(a.sum()) > 0


@pytest.mark.parametrize("h,w", [(64, 72), (9, 8)])
def test_forward_ignores_an_order_without_splits(gpu, monkeypatch, h, w):
    """vt_trace_fwd: "with a split count of 0 the order is ignored"; its other
    words are then unset memory, here past the last tile."""
    m = VoroTracing.from_scene(scene.random_scene(600, seed=9, R=4), device=gpu)
    scn = (m.primal_points.detach(), m.att_diffuse.detach(), m.att_specular.detach(),
           m.activated_density().detach(), m.point_adjacency, m.point_adjacency_offsets)
    rays = _images(gpu, 1, h, w)[0].contiguous()
    start = m.get_starting_point(rays)
    tiles = _tiles(rays)
    order = torch.full((tiles + 1,), 0x7fffffff, dtype=torch.int32, device=gpu)
    order[tiles] = 0
    cost = torch.zeros(tiles, dtype=torch.int32, device=gpu)

    class Unset:
        def __init__(self, o):
            self.o = o

        def launch_args(self, *args, **kw):
            cost.zero_()
            return self.o, cost.data_ptr()

    got = []
    for o in (None, order.data_ptr()):
        monkeypatch.setattr(_C, "_train_schedule", lambda *args, o=o: (Unset(o), None))
        out = _C.trace_vorotracing_fwd(*scn, rays, start, None, 0.001, 1024, False)
        got.append([x.view(torch.int32).clone() for x in out if x is not None] + [cost.clone()])
    assert all(torch.equal(a, b) for a, b in zip(*got))
    assert int(cost.min()) > 0


@pytest.mark.parametrize("tiles", [1, 255, 257, 2000])
@pytest.mark.parametrize("split_waves", [0, 4096])
def test_order_says_how_even_the_load_is(gpu, tiles, split_waves):
    """VT_TILE_ORDER_LOAD: bits 31 and 30 of the word after the order, for costs
    around both limits; order and split count as without it."""
    ws = torch.empty(int(_lib.load().vt_tile_order_workspace_size(tiles)), dtype=torch.uint8, device=gpu)
    rng = np.random.default_rng(tiles)
    for longest in (1000, 1220, 1240, 1420, 1450, 2000):
        cost = rng.integers(500, 900, size=tiles)
        # the last tile costs the others' sum over (longest - 1): sum / max = longest, near enough
        cost[-1] = max(cost[:-1].sum() // (longest - 1), 1) if tiles > 1 else 700
        total, most = int(cost.sum()), int(cost.max())
        c = torch.from_numpy(cost.astype(np.int32)).to(gpu)
        got = []
        for flag in (0, 1 << 31):
            order = torch.empty(tiles + 1, dtype=torch.int32, device=gpu)
            _lib.call("vt_tile_order", c.data_ptr(), tiles, split_waves | flag, order.data_ptr(), ws.data_ptr(),
                      torch.cuda.current_stream(gpu).cuda_stream)
            got.append(order.cpu().numpy().view(np.uint32).astype(np.int64))
        assert np.array_equal(got[0][:tiles], got[1][:tiles])
        assert got[1][tiles] == got[0][tiles] | (most * 1228 > total) << 31 | (most * 1434 > total) << 30


@pytest.mark.parametrize("flat", [False, True])
@pytest.mark.parametrize("even", [False, True])
def test_backward_chosen_by_the_load(gpu, even, flat):
    """Between the lines the costs of the forward choose the kernel that runs:
    launches as long as their longest tile (four lanes) and launches of tiles
    all alike (one lane) have the gradients of the launch without an order."""
    m = VoroTracing.from_scene(scene.random_scene(600, seed=9, R=4), device=gpu)
    scn = (m.primal_points.detach(), m.att_diffuse.detach(), m.att_specular.detach(),
           m.activated_density().detach(), m.point_adjacency, m.point_adjacency_offsets)
    image = _images(gpu, 1, 64, 72)[0]
    if even:
        image = image[24:32, 32:40].repeat(8, 9, 1).contiguous()
    rays = image.repeat(31, 1, 1, 1).contiguous()
    if not even:
        rays[8:, ..., 3:] *= -1.0  # away from the scene: a few steps
    tiles = _tiles(rays)
    assert 1920 < tiles <= 3072
    perm = None
    if flat:  # the lane order that makes the same tiles of 64 rays
        n = torch.arange(rays.numel() // 6, device=gpu).reshape(31, 8, 8, 9, 8)
        perm = n.permute(0, 1, 3, 2, 4).reshape(-1).to(torch.int32).contiguous()
        rays = rays.reshape(-1, 6)
    start = m.get_starting_point(rays)
    g = torch.randn(list(rays.shape[:-1]) + [4], generator=torch.Generator(device=gpu).manual_seed(2), device=gpu)
    got, saved = [], _C.TRAIN_TILE_ORDER
    try:
        for order in (False, True):
            _C.TRAIN_TILE_ORDER = order
            _C._TRAIN_SCHEDULES.clear()
            out = _C.trace_vorotracing_fwd(*scn, rays, start, None, 0.001, 1024, False, ray_perm=perm)
            got.append(_C.trace_vorotracing_bwd(*scn, rays, start, out[0], g, None, None, None, None, 0.0, out[5], None,
                                                out[6], out[7], out[8], 0.001, 1024, ray_perm=perm)[:4])
        sch = next(iter(_C._TRAIN_SCHEDULES.values()))
        word = int(sch.order.view(torch.int32)[tiles].item())
        cost = sch.cost.view(torch.int32).long()
    finally:
        _C.TRAIN_TILE_ORDER = saved
        _C._TRAIN_SCHEDULES.clear()
    long = int(cost.max()) * (1434 if flat else 1228) > int(cost.sum())
    assert long == (not even) and bool(word & (1 << (30 if flat else 31))) == long
    for a, b in zip(*got):
        assert float((a.double() - b.double()).norm()) <= 1e-5 * float(a.double().norm()) and float(a.abs().sum()) > 0


def _ragged_scene(gpu, which):
    """Cells with lists of 0 to 300 random neighbours (around 24, the faces that
    four lanes search at once), sites snapped so that exit distances tie, or of
    such sizes that face records and quotients leave their range."""
    rng = np.random.default_rng(len(which))
    n = 600
    nf = rng.choice([0, 1, 3, 4, 5, 23, 24, 25, 26, 47, 48, 49, 71, 300], size=n, p=[.02] + [.07] * 2 + [.08] * 10 + [.04])
    off = np.concatenate([[0], np.cumsum(nf)]).astype(np.uint32)
    adj = np.concatenate([rng.integers(0, n, off[-1]), np.zeros(32, np.int64)]).astype(np.uint32)
    pts = rng.uniform(-1, 1, size=(n, 3))
    if which == "ties":
        pts = np.round(pts * 2) / 2
    elif which == "large":
        pts *= 10.0 ** rng.uniform(0, 30, size=(n, 1))
    elif which == "small":
        pts *= 10.0 ** rng.uniform(-40, 0, size=(n, 1))
    elif which == "not finite":
        pts[rng.integers(0, n, 40), rng.integers(0, 3, 40)] = rng.choice([np.nan, np.inf, -np.inf], 40)
    rays = rng.normal(size=(40, 48, 6))
    if which == "ties":
        rays = np.round(rays)
    with np.errstate(over="ignore"):
        a = dict(points=pts.astype(np.float32), adjacency=adj, offsets=off, rays=rays.astype(np.float32),
                 diffuse=rng.normal(size=(n, 64)).astype(np.float16), specular=rng.normal(size=(n, 64)).astype(np.float16),
                 density=np.exp(rng.normal(-3, 1, size=n)).astype(np.float32),
                 start=rng.integers(0, n, size=(40, 48)).astype(np.uint32))
    return {k: H.to_dev(v, gpu) for k, v in a.items()}


def _same_bits(a, b):
    """Equal bit for bit, any NaN as another."""
    if a.is_floating_point():
        return bool(((a == b) & (torch.signbit(a) == torch.signbit(b)) | a.isnan() & b.isnan()).all())
    return torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("which", ["plain", "ties", "large", "small", "not finite"])
def test_ragged_lists_and_hard_quotients(gpu, which):
    """Renders and training forwards of few tiles, four lanes per ray, against
    the same calls with statistics, one lane per ray."""
    s = _ragged_scene(gpu, which)
    adj_diff = native.prefetch(s["points"], s["adjacency"], s["offsets"])
    for shape, tiled in (((40, 48), (8, 8)), ((1920,), None)):
        rays, start = s["rays"].reshape(*shape, 6), s["start"].reshape(shape)
        got = [native.infer_f16(s["points"], s["diffuse"], s["specular"], s["density"], s["adjacency"], s["offsets"],
                                adj_diff, rays, start, weight_threshold=1e-4, max_intersections=60, stats=st, tiled=tiled)
               for st in (None, native.new_stats(1920, gpu))]
        assert _same_bits(*got) and bool((got[0][..., 3] > 0.1).any())
        maps = [s[k].float()[:, :48].contiguous() for k in ("diffuse", "specular")]
        q = torch.tensor([0.7, 0.3], device=gpu).expand(*shape, 2).contiguous()
        out = [_C.trace_vorotracing_fwd(s["points"], *maps, s["density"].reshape(-1, 1), s["adjacency"], s["offsets"], rays,
                                        start, q, 1e-4, 60, False, stats=st) for st in (None, native.new_stats(1920, gpu))]
        for a, b in zip(*out):
            assert a is None and b is None or _same_bits(a, b)
