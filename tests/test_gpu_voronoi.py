"""GPU Voronoi adjacency (vt_voronoi_build) against the host Delaunay
(scipy/qhull): for sites in general position, each cell's neighbour set must
equal qhull's; lists come out ascending, the CSR tail holds the padding."""
import numpy as np
import pytest
import torch

from tests import helpers as H
from vorotracing_amd import ops, scene

pytestmark = pytest.mark.gpu


def _qhull_sets(points):
    adj, off = scene.delaunay_csr(points, pad=0)
    return [np.sort(adj[off[i]:off[i + 1]]) for i in range(points.shape[0])], off


def _check(points, gpu):
    adj, off, status = ops.build_voronoi_adjacency(H.to_dev(points, gpu))
    torch.cuda.synchronize()
    adj, off = adj.cpu().numpy(), off.cpu().numpy()
    want, woff = _qhull_sets(points)
    assert off.shape == (points.shape[0] + 1,)
    assert adj.shape[0] == off[-1] + 32 and not adj[off[-1]:].any()
    bad = [i for i in range(points.shape[0]) if not np.array_equal(adj[off[i]:off[i + 1]], want[i])]
    assert not bad, f"{len(bad)} cells differ from qhull, first {bad[:5]}"
    assert off[-1] == woff[-1]
    assert all(np.all(np.diff(adj[off[i]:off[i + 1]].astype(np.int64)) > 0) for i in range(points.shape[0]))


@pytest.mark.parametrize("n,seed", [(500, 0), (3000, 1)])
def test_random_cube(gpu, n, seed):
    pts = np.random.default_rng(seed).uniform(-2, 2, size=(n, 3)).astype(np.float32)
    _check(pts, gpu)


def test_c1_sites(gpu):
    _check(H.c1_scene().points, gpu)


def test_mini_heightfield_sites(gpu):
    """Config-3 distribution at test size: a thin dense surface layer plus a sparse background."""
    _check(H.mini_heightfield().points, gpu)


def test_heightfield_131k(gpu):
    """C3's site distribution at 131,072 sites: dense surface cells whose lists exceed the
    64-entry slots, background cells next to the surface and the convex-hull cells of the cube."""
    pts = scene._heightfield_sites(np.random.default_rng(3), 131072, 0.8, 4.0, 0.01).astype(np.float32)
    _check(pts, gpu)


def test_ellipsoid_surface(gpu):
    """Every site on a convex surface is a convex-hull site, so every cell is unbounded.  An
    ellipsoid (unlike a sphere) keeps 5 sites off a common sphere: general position."""
    d = np.random.default_rng(5).normal(size=(3000, 3))
    pts = (d / np.linalg.norm(d, axis=1, keepdims=True) * np.array([1.0, 0.7, 0.5])).astype(np.float32)
    _check(pts, gpu)


def test_model_scene_renders_the_same(gpu):
    """A scene whose adjacency comes from the GPU builder renders like the qhull one (same sets,
    ascending order; the walk's choice depends on the order only through exact ties)."""
    from vorotracing_amd import camera
    from vorotracing_amd.model import VoroTracing

    s = H.small_random(800, seed=9)
    rays = H.to_dev(camera.pinhole_rays(48, 32, eye=(0.3, -3.5, 0.5)), gpu)
    m1 = VoroTracing.from_scene(s, device=gpu)
    adj, off, _ = ops.build_voronoi_adjacency(m1.primal_points)
    s_sorted = scene.Scene(s.name, s.points, s.density_raw, s.diffuse, s.specular,
                           adj.cpu().numpy(), off.cpu().numpy(), s.diff_res, s.spec_res, dict(s.params))
    m2 = VoroTracing.from_scene(s_sorted, device=gpu)
    a = m1(rays, weight_threshold=0.001)[0]
    b = m2(rays, weight_threshold=0.001)[0]
    torch.cuda.synchronize()
    assert torch.equal(a, b)


@pytest.mark.parametrize("guess", ["previous", "shuffled", "junk"])
def test_warm_start_equals_cold(gpu, guess):
    """A warm-started build (initial_guesses, cuda/__init__.py:16-37) gives
    the cold build's CSR and qhull's sets, whatever the guesses: the
    adjacency before the sites moved (the training refresh), lists of other
    sites, or ids out of range."""
    rng = np.random.default_rng(17)
    pts0 = scene._heightfield_sites(rng, 40000, 0.8, 4.0, 0.01).astype(np.float32)
    adj0, off0, _ = ops.build_voronoi_adjacency(H.to_dev(pts0, gpu))
    pts = (pts0 + rng.normal(0.0, 2e-3, size=pts0.shape)).astype(np.float32)  # the sites moved
    g_adj, g_off = adj0, off0
    if guess == "shuffled":
        o64 = off0.to(torch.int64)
        g_off = (o64[-1] - o64.flip(0)).to(torch.uint32).contiguous()  # other cells' list lengths and entries
    elif guess == "junk":
        g_adj = torch.full_like(adj0, 0xFFFFFFF0)
        g_adj[::3] = torch.arange(0, g_adj[::3].numel(), device=gpu, dtype=torch.int64).to(torch.uint32)
    pd = H.to_dev(pts, gpu)
    cold = ops.build_voronoi_adjacency(pd)
    warm = ops.build_voronoi_adjacency(pd, initial_guesses=g_adj, initial_guesses_offsets=g_off)
    torch.cuda.synchronize()
    assert torch.equal(warm[1], cold[1]) and torch.equal(warm[0], cold[0])
    if guess == "previous":
        _check(pts, gpu)


def test_model_refresh_warm_start(gpu):
    """VoroTracing.update_triangulation seeds the build with the current
    adjacency; the refreshed CSR equals a cold build's."""
    from vorotracing_amd.model import VoroTracing

    s = H.small_random(3000, seed=21)
    m = VoroTracing.from_scene(s, device=gpu)
    with torch.no_grad():
        m.primal_points.add_(torch.randn_like(m.primal_points) * 1e-3)
    m.update_triangulation()
    adj, off, _ = ops.build_voronoi_adjacency(m.primal_points)
    torch.cuda.synchronize()
    assert torch.equal(m.point_adjacency, adj) and torch.equal(m.point_adjacency_offsets, off)


@pytest.mark.parametrize("n", [2, 3, 4, 5, 7, 8, 9, 63, 64, 65, 66, 511, 512, 513, 32767, 32769, 65535, 65537])
def test_site_counts_at_tree_edges(gpu, n):
    """Site counts around the builder's groups (8 sites per leaf box, 64 boxes
    per box above, 64 seeds per cell) and around the count from which its
    sort takes all Morton bits.  Up to 4 sites in general position are all
    neighbours of each other."""
    pts = np.random.default_rng(100 + n).uniform(-1, 1, size=(n, 3)).astype(np.float32)
    if n >= 5:
        _check(pts, gpu)
        return
    adj, off, _ = ops.build_voronoi_adjacency(H.to_dev(pts, gpu))
    adj, off = adj.cpu().numpy(), off.cpu().numpy()
    for i in range(n):
        assert np.array_equal(adj[off[i]:off[i + 1]], [j for j in range(n) if j != i])


@pytest.mark.parametrize("faces", [30, 40, 64, 65, 120, 230])
def test_cell_with_many_faces(gpu, faces):
    """A site inside a sphere of others has them all as neighbours: cells of one
    vertex per lane, of two and of eight, and lists longer than a slot."""
    d = np.random.default_rng(faces).normal(size=(faces, 3))
    shell = d / np.linalg.norm(d, axis=1, keepdims=True) * np.array([1.0, 0.97, 0.94])
    pts = np.concatenate([[[0.01, -0.02, 0.015]], shell]).astype(np.float32)
    _check(pts, gpu)


@pytest.mark.parametrize("e", [-125, -100, -70, -40, -20, 30, 44, 60, 64, 90, 125])
def test_any_unit(gpu, e):
    """Sites times 2^e have the neighbours that they have at 1, lists of more
    than a wave's vertices among them (squares of such coordinates leave f32),
    in a cold build and from the neighbours at 1."""
    pts = np.unique(np.round(H.mini_heightfield().points[::4] * 2.0 ** 20) / 2.0 ** 20, axis=0).astype(np.float32)
    ref = ops.build_voronoi_adjacency(H.to_dev(pts, gpu))
    far = np.ldexp(pts, e).astype(np.float32)
    assert np.array_equal(np.ldexp(far.astype(np.float64), -e), pts), "a coordinate lost bits"
    guesses = dict(initial_guesses=ref[0], initial_guesses_offsets=ref[1])
    for kw in ({}, guesses):
        got = ops.build_voronoi_adjacency(H.to_dev(far, gpu), **kw)
        assert torch.equal(got[1], ref[1]) and torch.equal(got[0], ref[0])


@pytest.mark.parametrize("n", [9, 200, 6000])
def test_coplanar_sites_on_a_tilted_plane(gpu, n):
    """Exactly coplanar sites (z = x / 2 + y / 4 on a dyadic grid): every cell is
    an open column, whose neighbours are those of the plane's own Delaunay
    triangulation; with a volume of sites above, of the whole set's."""
    from scipy.spatial import Delaunay

    rng = np.random.default_rng(n)
    xy = np.unique(np.round(rng.uniform(-1, 1, size=(n, 2)) * 2 ** 16) / 2 ** 16, axis=0)
    pts = np.concatenate([xy, 0.5 * xy[:, :1] + 0.25 * xy[:, 1:]], axis=1)
    e = np.array([1.0, 0.0, 0.5]) / np.sqrt(1.25)
    f = np.array([0.0, 1.0, 0.25]) - 0.1 * np.array([1.0, 0.0, 0.5])
    flat = np.stack([pts @ e, pts @ f / np.linalg.norm(f)], axis=1)
    ptr, idx = Delaunay(flat).vertex_neighbor_vertices
    adj, off, _ = ops.build_voronoi_adjacency(H.to_dev(pts.astype(np.float32), gpu))
    adj, off = adj.cpu().numpy(), off.cpu().numpy()
    for i in range(len(pts)):
        assert np.array_equal(adj[off[i]:off[i + 1]], np.sort(idx[ptr[i]:ptr[i + 1]])), i
    up = rng.uniform(-1, 1, size=(n, 3))
    up[:, 2] = 0.5 * up[:, 0] + 0.25 * up[:, 1] + 0.02 + 2 * np.abs(up[:, 2])
    _check(np.concatenate([pts, up]).astype(np.float32), gpu)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("n,hub,seed", [(7, False, 4), (50, False, 4), (200, False, 4), (240, True, 11), (240, True, 15),
                                        (100, True, 0)])
def test_coplanar_sites_on_a_circle(gpu, n, hub, seed, axis):
    """Sites on a circle, in f32 and so not quite: their cells are columns that
    all meet within 1e-7 of its centre, with faces down to 1e-10 wide there; with
    a site at the centre (hub), a column that some of the others cut by less
    than 1e-7.  Neighbours of the plane's own Delaunay triangulation."""
    from scipy.spatial import Delaunay

    a = np.random.default_rng(seed).uniform(0, 2 * np.pi, n)
    flat = np.concatenate([np.zeros((int(hub), 2)), np.stack([np.cos(a), np.sin(a)], axis=1)]).astype(np.float32)
    flat = np.unique(flat, axis=0)
    ptr, idx = Delaunay(flat.astype(np.float64)).vertex_neighbor_vertices
    adj, off, _ = ops.build_voronoi_adjacency(H.to_dev(np.ascontiguousarray(np.insert(flat, axis, 0.0, axis=1)), gpu))
    adj, off = adj.cpu().numpy(), off.cpu().numpy()
    for i in range(len(flat)):
        assert np.array_equal(adj[off[i]:off[i + 1]], np.sort(idx[ptr[i]:ptr[i + 1]])), i


@pytest.mark.parametrize("tilt", [False, True])
@pytest.mark.parametrize("w,h", [(2, 2), (5, 40), (30, 31)])
def test_coplanar_grid(gpu, w, h, tilt):
    """A grid in a plane (tilted: of rectangles, in z = x): four sites on every
    circle, whose diagonal columns touch in a line and are no neighbours, in a
    cold build and from guesses that hold them."""
    i, j = (x.ravel() for x in np.meshgrid(np.arange(w), np.arange(h), indexing="ij"))
    pts = np.stack([i, j, i if tilt else 0 * i], axis=1).astype(np.float32)
    near = np.maximum(abs(i[:, None] - i), abs(j[:, None] - j)) == 1
    side = near & (abs(i[:, None] - i) + abs(j[:, None] - j) == 1)
    want = [np.nonzero(x)[0] for x in side]
    guess = [np.nonzero(x)[0] for x in near]
    guesses = dict(initial_guesses=H.to_dev(np.concatenate(guess).astype(np.uint32), gpu),
                   initial_guesses_offsets=H.to_dev(np.cumsum([0] + [len(g) for g in guess]).astype(np.uint32), gpu))
    for kw in ({}, guesses):
        adj, off, _ = ops.build_voronoi_adjacency(H.to_dev(pts, gpu), **kw)
        adj, off = adj.cpu().numpy(), off.cpu().numpy()
        for c in range(len(pts)):
            assert np.array_equal(adj[off[c]:off[c + 1]], want[c]), c


@pytest.mark.parametrize("n,sparse,depth,seed", [(10000, 20, 1e-2, 3), (3000, 30, 1e-2, 3), (10000, 10, 1e-3, 1),
                                                 (10000, 25, 1e-3, 1)])
def test_sparse_sites_about_a_dense_shell(gpu, n, sparse, depth, seed):
    """Cells that see more of a dense surface, before their other neighbours
    close them, than 512 vertices hold, and end with at most 255 neighbours."""
    rng = np.random.default_rng(seed)
    p = rng.normal(size=(n, 3))
    p *= (1 - depth * rng.uniform(0, 1, (n, 1))) / np.linalg.norm(p, axis=1, keepdims=True)
    m = n // sparse
    up = rng.normal(size=(m, 3))
    up *= (1.02 + rng.exponential(1.0, (m, 1))) / np.linalg.norm(up, axis=1, keepdims=True)
    _check(np.concatenate([p, up]).astype(np.float32), gpu)


@pytest.mark.parametrize("scale", [1e-6, 1.0, 1e6])
def test_clusters_of_very_different_density(gpu, scale):
    """Clusters a thousandth of the scene wide beside sparse sites (a Morton
    grid coarser than a cluster, reaches that differ a thousandfold)."""
    rng = np.random.default_rng(8)
    sparse = rng.uniform(-1, 1, size=(3000, 3))
    dense = [c + 1e-3 * rng.normal(size=(700, 3)) for c in rng.uniform(-1, 1, size=(3, 3))]
    _check((scale * np.concatenate([sparse, *dense])).astype(np.float32), gpu)


def test_sites_on_common_spheres(gpu):
    """Sites on a 1/64 grid (no two alike): many fives on common spheres, whose
    Delaunay neighbours are not unique.  The build succeeds and gives the
    neighbours that share a face of some area: those that qhull finds however
    the sites are moved by less than matters."""
    pts = np.unique(np.round(np.random.default_rng(0).uniform(-1, 1, size=(3000, 3)) * 64) / 64, axis=0)
    adj, off, _ = ops.build_voronoi_adjacency(H.to_dev(pts.astype(np.float32), gpu))
    adj, off = adj.cpu().numpy().astype(np.int64), off.cpu().numpy().astype(np.int64)
    n = pts.shape[0]

    def pairs(a, o):
        return set(zip(np.repeat(np.arange(n), np.diff(o.astype(np.int64))).tolist(), a[:o[-1]].tolist()))

    sure = None
    for seed in range(24):
        got = pairs(*scene.delaunay_csr(pts + 1e-9 * np.random.default_rng(seed).normal(size=pts.shape), pad=0))
        sure = got if sure is None else sure & got
    assert pairs(adj, off) == sure


def test_lattice(gpu):
    """A cubic lattice: the neighbours along the axes, none across edges or corners."""
    g = np.stack(np.meshgrid(*[np.arange(10)] * 3, indexing="ij"), -1).reshape(-1, 3)
    adj, off, _ = ops.build_voronoi_adjacency(H.to_dev(g.astype(np.float32), gpu))
    adj, off = adj.cpu().numpy(), off.cpu().numpy()
    for i in range(len(g)):
        assert np.array_equal(adj[off[i]:off[i + 1]], np.flatnonzero(np.abs(g - g[i]).sum(1) == 1))
