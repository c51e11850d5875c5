// vt_voronoi.hip -- Voronoi neighbours (the Delaunay adjacency CSR) of a site
// set, built on the GPU.  Replaces the adjacency step of
// vorotracing.cuda.build_voronoi_adjacency (cuda/__init__.py:16-46, which
// calls Paragram; the synthetic scenes of this build use host qhull).
//
// One wave per cell, clipped in double precision in site-local coordinates:
//   * it starts as a box around all sites (6 planes), 10^6 times their
//     extent, so that the faces between convex-hull sites (unbounded in the
//     Delaunay sense) keep a part inside it;
//   * a site q cuts the cell by its bisector plane d.x <= |d|^2/2 (d = q - p,
//     exact in double for f32 inputs) when some vertex lies strictly outside;
//   * every site within 2R of the cell's own (R: largest vertex distance) is
//     offered to it, or ruled out together with its neighbours by a bounding
//     box that no cutting site can lie in;
//   * the neighbours are the sites whose planes keep a face, ascending.
// The cell is kept as the triangulation of its dual (Ray, Sokolov, Lefebvre,
// Levy, "Meshless Voronoi on the GPU", 2018): a vertex is a triangle of three
// plane ids; a cut removes the vertices strictly outside the plane and closes
// the hole with triangles (u, v, new plane) along the boundary edges (u, v).
//
// The cell lives in the wave's registers: lane l holds vertices l, l + 64, ...
// (position and plane ids), so that a plane is tested against all vertices by
// one dot product and one ballot, and a cut costs a few LDS exchanges: each
// triangle knows the triangles across its three edges (VorLds::nb), a removed
// vertex finds the boundary edges among its own three by testing bits of the
// removed set, the new triangles go to free lanes and meet along the boundary
// through two per-plane tables.  First pass: 64 vertices per cell (one per
// lane); cells with more run again with 128, then with 512 and 1,024.
//
// Sites are sorted along a Morton curve and kept in a tree of bounding boxes
// that is 64 children wide, one child per lane: 8 sites per box at the bottom.
// A tree follows the sites' density, where a uniform grid left some cells with
// dozens of sites and most with none.  A cell is first cut by nearby sites (64
// around it on the curve, nearest first, then those of a small ball; or the
// caller's guesses), which usually leaves it near its final shape, and then
// offered what the tree still holds within its reach.
//
// What bounds it: instruction issue.  The first pass runs 9,900 VALU and 5,400
// scalar instructions per cell (22 cuts of about 200, 33 box tests of 80, 11
// batches of sites of 150), 10.4 G VALU instructions in 20.6 ms at 5 waves per
// SIMD: one in flight in 90 % of the SIMDs' quad-cycles (SQ_ACTIVE_INST_VALU),
// though an f32 one alone takes half of a quad-cycle (41 % of that peak).  The
// later passes are bound by their longest cells.  1M heightfield sites: 131 ms
// with the cell in LDS and a uniform grid, 33 ms so; 262k torus sites after a
// move, from their old adjacency: 38.9 and 6.5 ms.
#include "vt_internal.h"
#include "vt_prims.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace vt {

constexpr uint32_t VOR_NONE = 0xffffffffu;
constexpr int VOR_BLOCK = 64; // one wave

// Neighbour lists: LIST_K entries per site; longer lists in slots of BIG_K.
constexpr int LIST_K = 64;
constexpr int BIG_K = 255;
// Vertices per lane of the passes, each of which takes the cells that overflow
// the one before (plane slots: 64 per vertex slot; a cell of T vertices has T /
// 2 + 2 faces, so the slots never run out first).  1M heightfield sites queue
// 10,423 cells for the second pass and 938 for the third.  A pass ends with its
// longest cell, 3 to 4 ms there whatever the vertices per lane: a pass of 4
// between the second and the third cost 3 ms more in all.  The fourth runs only
// when the host finds cells queued for it: those beside a far denser surface,
// of which a cell sees more, before its other neighbours close it, than it
// keeps (255 neighbours at most): one of 10,500 sites in and about a thin shell.
constexpr int NV_SMALL = 1, NV_MID = 2, NV_LARGE = 8, NV_HUGE = 16;

// The site tree: level 0 has boxes of VOR_LEAF consecutive sorted sites,
// level k + 1 boxes of 64 boxes of level k; the walk starts at level `top`,
// the first with at most 64.
constexpr uint32_t VOR_LEAF = 8;
constexpr int VOR_LEVELS = 4; // 8 * 64^4 sites and more: 2^27
struct VorBox;
struct VorTree {
    const float4 *sites;               // sorted (x, y, z, original index)
    const float4 *boxes;               // (lo, -), (hi, -) per box, level after level
    uint32_t count[VOR_LEVELS];
    int top;
    const VorBox *box;
};

// The builder works on the sites scaled by 2^-k, k the exponent of their
// largest extent (exact, and Voronoi neighbours do not depend on scale): the
// f32 squares and lengths that rule sites out then neither overflow nor
// underflow, whatever unit the sites are in.  Unscaled squares left the builder
// with wrong lists from extents of 2^44 on and at 2^-70.
struct VorBox {
    double lo[3], hi[3]; // what every cell starts as (scaled)
    double diag2;        // squared diagonal of the sites' own box
    int k;
};

// No scale for one place or sites that are not finite.  Extents below 1e-6
// count as 1e-6, down to 2^-40 of that.
__device__ __forceinline__ void scaled_box(const float *bbox, VorBox &b)
{
    double ext = 0.0;
    for (int a = 0; a < 3; ++a)
        ext = fmax(ext, (double)bbox[3 + a] - (double)bbox[a]);
    b.k = ext > 0.0 && ext < 1e39 ? min(max(ilogb(ext), -126), 126) : 0;
    double most = fmin(ldexp(1e-6, -b.k), 0x1p40);
    b.diag2 = 0.0;
    for (int a = 0; a < 3; ++a) {
        b.lo[a] = ldexp((double)bbox[a], -b.k);
        b.hi[a] = ldexp((double)bbox[3 + a], -b.k);
        b.diag2 = fma(b.hi[a] - b.lo[a], b.hi[a] - b.lo[a], b.diag2);
        most = fmax(most, b.hi[a] - b.lo[a]);
    }
    for (int a = 0; a < 3; ++a) {
        b.lo[a] -= 1e6 * most;
        b.hi[a] += 1e6 * most;
    }
}
__device__ __forceinline__ float4 scaled_site(const float *points, uint32_t i, int k)
{
    const float *p = points + 3 * (size_t)i;
    return make_float4(ldexpf(p[0], -k), ldexpf(p[1], -k), ldexpf(p[2], -k), __uint_as_float(i));
}

// Boxes before a level's first (level wave-uniform: scalar selects).
__host__ __device__ __forceinline__ uint32_t level_begin(const VorTree &t, int level)
{
    uint32_t b = level > 0 ? t.count[0] : 0u;
    b += level > 1 ? t.count[1] : 0u;
    return b + (level > 2 ? t.count[2] : 0u);
}
__device__ __forceinline__ uint32_t level_count(const VorTree &t, int level)
{
    return level == 0 ? t.count[0] : level == 1 ? t.count[1] : level == 2 ? t.count[2] : t.count[3];
}

enum { VOR_OK = 0, VOR_FULL = 1, VOR_DEGENERATE = 2 };
// which table overflowed (bits of the fails[F_REASON] word)
enum { FULL_PLANES = 1, FULL_VERTICES = 4, FULL_LISTS = 8 };

// Passes after the first, and their queues
constexpr int RETRIES = 3;
template <int NV> constexpr int QUEUE_OF = NV == NV_MID ? 0 : NV == NV_LARGE ? 1 : 2;

// fails[] words: failures, the cells queued for each further pass and those
// passes' work counters, big-list slots
enum {
    F_FULL = 0,
    F_DEGENERATE = 1,
    F_BIG = 2,
    F_FIRST_BAD = 3,
    F_REASON = 4,
    F_RETRY = 5,
    F_NEXT = F_RETRY + RETRIES,
    F_WORDS = F_NEXT + RETRIES
};

struct d3 {
    double x, y, z;
};
__device__ __forceinline__ d3 cross_d(double4 a, double4 b)
{
    return d3{fma(a.y, b.z, -(a.z * b.y)), fma(a.z, b.x, -(a.x * b.z)), fma(a.x, b.y, -(a.y * b.x))};
}
__device__ __forceinline__ double dot_d(d3 a, d3 b) { return fma(a.x, b.x, fma(a.y, b.y, a.z * b.z)); }

// intersection of three planes n.x <= w
__device__ __forceinline__ d3 plane_vertex(double4 a, double4 b, double4 c)
{
    const d3 bc = cross_d(b, c), ca = cross_d(c, a), ab = cross_d(a, b);
    const double s = 1.0 / fma(a.x, bc.x, fma(a.y, bc.y, a.z * bc.z));
    return d3{fma(a.w, bc.x, fma(b.w, ca.x, c.w * ab.x)) * s, fma(a.w, bc.y, fma(b.w, ca.y, c.w * ab.y)) * s,
              fma(a.w, bc.z, fma(b.w, ca.z, c.w * ab.z)) * s};
}

// LDS of one wave.
template <int NV> struct VorLds {
    static constexpr int T = 64 * NV; // vertices, and plane slots
    double4 P[T];
    uint32_t nid[T];          // site of a plane (VOR_NONE: box plane, unused slot)
    uint32_t by_u[T], by_v[T]; // new triangle (tag) whose boundary edge starts / ends at a plane
    // triangles across the edges (a, b), (b, c), (c, a) of (a, b, c)
    typename std::conditional<NV == 1, uchar4, ushort4>::type nb[T];
    uint32_t edge[T];         // boundary edges of a cut
    uint32_t hits[128];       // leaf boxes to look into
    uint32_t used[T / 32];
    uint8_t gone[T];          // (several vertices per lane) removed by the current cut
};

__device__ __forceinline__ void lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ uint32_t rank_in(uint64_t m)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
__device__ __forceinline__ float readlane_f(float x, int l)
{
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(x), l));
}
__device__ __forceinline__ double readlane_d(double x, int l)
{
    const uint64_t b = (uint64_t)__double_as_longlong(x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
// One DPP step within rows of 16 lanes.
template <int CTRL> __device__ __forceinline__ uint32_t dpp_u(uint32_t x)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, true);
}
// Largest / smallest value of the wave (all lanes active): a butterfly within
// each row of 16 lanes (quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_ror 4,
// row_ror 8), then the four row results.
__device__ __forceinline__ float wave_max_f(float x)
{
    x = fmaxf(x, __uint_as_float(dpp_u<0xb1>(__float_as_uint(x))));
    x = fmaxf(x, __uint_as_float(dpp_u<0x4e>(__float_as_uint(x))));
    x = fmaxf(x, __uint_as_float(dpp_u<0x124>(__float_as_uint(x))));
    x = fmaxf(x, __uint_as_float(dpp_u<0x128>(__float_as_uint(x))));
    return fmaxf(fmaxf(readlane_f(x, 0), readlane_f(x, 16)), fmaxf(readlane_f(x, 32), readlane_f(x, 48)));
}
__device__ __forceinline__ uint32_t wave_min_u(uint32_t x)
{
    x = min(x, dpp_u<0xb1>(x));
    x = min(x, dpp_u<0x4e>(x));
    x = min(x, dpp_u<0x124>(x));
    x = min(x, dpp_u<0x128>(x));
    const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)x, 0), b = (uint32_t)__builtin_amdgcn_readlane((int)x, 16);
    const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)x, 32), d = (uint32_t)__builtin_amdgcn_readlane((int)x, 48);
    return min(min(a, b), min(c, d));
}
// Ascending bitonic sort of one value per lane.
__device__ __forceinline__ uint32_t wave_sort_u(uint32_t x, int lane)
{
#pragma unroll 1
    for (int k = 2; k <= 64; k <<= 1)
#pragma unroll 1
        for (int j = k >> 1; j > 0; j >>= 1) {
            const uint32_t y = (uint32_t)__shfl_xor((int)x, j);
            const bool low = ((lane & j) == 0) == ((lane & k) == 0);
            x = low ? min(x, y) : max(x, y);
        }
    return x;
}

// The cell of one site: vertices in registers, wave-uniform scalars beside.
template <int NV> struct VorCell {
    d3 v[NV];
    float fx[NV], fy[NV], fz[NV], fl[NV]; // the vertices in f32, and their lengths
    uint32_t tri[NV];      // plane ids, 10 bits each
    uint64_t alive[NV];    // slots in use (vertex 64 k + l: bit l of alive[k])
    uint64_t freep[NV];    // plane slots that no vertex used when last counted
    uint32_t gen;          // cuts of this wave so far (tags of by_u / by_v)
    int full;              // FULL_* bits of a capacity failure
    // after radii():
    float r2;              // squared radius of all vertices, rounded up
    float bmin[3], bmax[3]; // bounding box of the near vertices and the origin, rounded outward
    uint64_t farv[NV];     // vertices beyond far
    float far;
};

// Bounds of the tests that rule sites out are evaluated in f32 and widened by
// SLACK, far above their rounding (a few 2^-24 of the summed magnitudes).
constexpr float SLACK = 1e-5f;

template <int NV> __device__ __forceinline__ void cell_radii(VorCell<NV> &c, int lane)
{
    float r = 0.0f, mn[3] = {0.0f, 0.0f, 0.0f}, mx[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        c.farv[k] = 0;
        if (NV > 1 && !c.alive[k])
            continue;
        const bool on = (c.alive[k] >> lane) & 1u;
        const bool far = on && !(c.fl[k] <= c.far);
        c.farv[k] = __ballot(far);
        if (on)
            r = fmaxf(r, c.fl[k]);
        if (on && !far) {
            const float x[3] = {c.fx[k], c.fy[k], c.fz[k]};
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                mn[a] = fminf(mn[a], x[a]);
                mx[a] = fmaxf(mx[a], x[a]);
            }
        }
    }
    r = wave_max_f(r);
    c.r2 = r * r * (1.0f + SLACK);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        c.bmin[a] = -wave_max_f(-mn[a]) * (1.0f + SLACK);
        c.bmax[a] = wave_max_f(mx[a]) * (1.0f + SLACK);
    }
}

template <int NV> __device__ __forceinline__ void set_f32(VorCell<NV> &c, int k)
{
    c.fx[k] = (float)c.v[k].x, c.fy[k] = (float)c.v[k].y, c.fz[k] = (float)c.v[k].z;
    c.fl[k] = sqrtf(fmaf(c.fx[k], c.fx[k], fmaf(c.fy[k], c.fy[k], c.fz[k] * c.fz[k])));
}

// What a lane's site is offered with in f32: its offset x, SLACK |x| and
// |x|^2 / 2 less its slack.
struct VorOffer {
    float x, y, z, slack, w;
};
// Can the site of lane l cut some vertex?  (f32, never missing one: x.v is off
// by less than SLACK |x| |v|.  Most offers miss, for a third of the
// instructions of the test in double.)
template <int NV> __device__ __forceinline__ bool may_cut(const VorCell<NV> &c, const VorOffer &o, int l)
{
    const float x = readlane_f(o.x, l), y = readlane_f(o.y, l), z = readlane_f(o.z, l);
    const float slack = readlane_f(o.slack, l), w = readlane_f(o.w, l);
    uint64_t any = 0;
#pragma unroll
    for (int k = 0; k < NV; ++k)
        if (NV == 1 || c.alive[k]) // (vertices take the lowest free slots)
            any |= __ballot(!(fmaf(x, c.fx[k], fmaf(y, c.fy[k], fmaf(z, c.fz[k], slack * c.fl[k]))) < w)) & c.alive[k];
    return any != 0;
}

// Marks the planes that some vertex uses in s.used.
template <int NV> __device__ __forceinline__ void cell_mark_used(VorLds<NV> &s, const VorCell<NV> &c, int lane)
{
    for (int w = lane; w < VorLds<NV>::T / 32; w += 64)
        s.used[w] = 0;
    lds_sync();
#pragma unroll
    for (int k = 0; k < NV; ++k)
        if ((c.alive[k] >> lane) & 1u) {
            const uint32_t t = c.tri[k], a = t & 1023u, b = (t >> 10) & 1023u, d = t >> 20;
            atomicOr(&s.used[a >> 5], 1u << (a & 31));
            atomicOr(&s.used[b >> 5], 1u << (b & 31));
            atomicOr(&s.used[d >> 5], 1u << (d & 31));
        }
    lds_sync();
}

// A plane slot (wave-uniform), or -1: the next of those free when last
// counted, else the planes that the vertices use are counted again.
template <int NV> __device__ __forceinline__ int cell_plane_slot(VorLds<NV> &s, VorCell<NV> &c, int lane)
{
#pragma unroll 1
    for (int round = 0; round < 2; ++round) {
#pragma unroll
        for (int k = 0; k < NV; ++k)
            if (c.freep[k]) {
                const int l = (int)__builtin_ctzll(c.freep[k]);
                c.freep[k] &= c.freep[k] - 1;
                return 64 * k + l;
            }
        if (round)
            break;
        cell_mark_used(s, c, lane);
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)s.used[2 * k]);
            const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)s.used[2 * k + 1]);
            c.freep[k] = ~(((uint64_t)hi << 32) | lo);
        }
        c.freep[0] &= ~0x3full; // the box planes stay
    }
    return -1;
}

// The site of a cell, and the squared distances [lo2, hi2) of the sites that
// are offered to it.
struct VorReach {
    float px, py, pz;
    float lo2, hi2; // of offset2(); hi2 infinite: no bound
};
// Squared length of an f32 offset between sites: what the bands compare, the
// same for a site wherever it is met.
__device__ __forceinline__ float offset2(float x, float y, float z) { return fmaf(x, x, fmaf(y, y, z * z)); }

// The hole that the removed vertices `out` leave is closed with a triangle (u,
// v, q) along every boundary edge (u, v): the edges of removed vertices
// towards a kept one, each triangle in a free slot (those of the removed ones
// among them), which keeps the removed side's orientation.  A cut of a convex
// cell removes a disc, so the boundary is one cycle: every plane on it starts
// exactly one edge and ends exactly one, and the triangles of neighbouring
// edges find each other by the plane between them.
__device__ __forceinline__ int hole_fits(uint32_t cnt, uint32_t room, int &full)
{
    if (cnt > room) {
        full |= FULL_VERTICES;
        return VOR_FULL;
    }
    return cnt < 3 ? VOR_DEGENERATE : VOR_OK;
}

// Triangle (u, v, q) of slot me, whose edge (u, v) has `keep` on its other
// side, after every new triangle has entered by_u and by_v.  Returns whether
// it fails (not one cycle, or a vertex of nearly parallel planes).
template <int NV>
__device__ __forceinline__ bool new_vertex(const VorLds<NV> &s, VorCell<NV> &c, int k, uint32_t me, uint32_t u,
                                           uint32_t v, double4 pq, int q, uint32_t &next, uint32_t &prev)
{
    const uint32_t tag = c.gen << 10 | me;
    next = s.by_u[v];
    prev = s.by_v[u];
    bool bad = s.by_u[u] != tag || s.by_v[v] != tag || next >> 10 != c.gen || prev >> 10 != c.gen;
    const d3 x = plane_vertex(s.P[u], s.P[v], pq);
    bad = bad || !(dot_d(x, x) < 1e300);
    c.v[k] = x;
    set_f32(c, k);
    c.tri[k] = u | v << 10 | (uint32_t)q << 20;
    next &= 1023u;
    prev &= 1023u;
    return bad;
}

// One vertex per lane: the links of a triangle are the bytes of a word, and
// the lanes of all new triangles run together.
template <int NV>
__device__ __forceinline__ int close_hole_1(VorLds<NV> &s, VorCell<NV> &c, const uint64_t *out, double4 pq, int q,
                                            uint32_t site, int lane)
{
    uint32_t *nb = reinterpret_cast<uint32_t *>(s.nb);
    uint8_t *nb8 = reinterpret_cast<uint8_t *>(s.nb);
    const uint64_t gone = out[0];
    const uint32_t to = nb[lane], t = c.tri[0];
    const bool o = (gone >> lane) & 1u;
    const uint32_t n0 = to & 63u, n1 = (to >> 8) & 63u, n2 = (to >> 16) & 63u;
    const bool b0 = o && !((gone >> n0) & 1u), b1 = o && !((gone >> n1) & 1u), b2 = o && !((gone >> n2) & 1u);
    const uint64_t m0 = __ballot(b0), m1 = __ballot(b1), m2 = __ballot(b2);
    const uint32_t c0 = (uint32_t)__popcll(m0), c1 = c0 + (uint32_t)__popcll(m1), cnt = c1 + (uint32_t)__popcll(m2);
    const uint64_t f = ~c.alive[0] | gone;
    const int fits = hole_fits(cnt, (uint32_t)__popcll(f), c.full);
    if (fits != VOR_OK)
        return fits;
    // edge: u | v << 10 | kept << 20 | removed << 26
    const uint32_t me26 = (uint32_t)lane << 26;
    if (b0)
        s.edge[rank_in(m0)] = (t & 0xfffffu) | n0 << 20 | me26;
    if (b1)
        s.edge[c0 + rank_in(m1)] = t >> 10 | n1 << 20 | me26;
    if (b2)
        s.edge[c1 + rank_in(m2)] = t >> 20 | (t & 1023u) << 10 | n2 << 20 | me26;
    c.gen = (c.gen + 1u) & 0x3fffffu;
    if (lane == 0) {
        s.P[q] = pq;
        s.nid[q] = site;
    }
    lds_sync();
    const uint32_t j = rank_in(f);
    const bool mine = ((f >> lane) & 1u) && j < cnt;
    bool bad = false;
    if (mine) {
        const uint32_t e = s.edge[j], u = e & 1023u, v = (e >> 10) & 1023u, kept = (e >> 20) & 63u, was = e >> 26;
        const uint32_t tag = c.gen << 10 | (uint32_t)lane;
        s.by_u[u] = tag;
        s.by_v[v] = tag;
        // the kept triangle's link across the edge, read by every lane before any is written
        const uint32_t back = nb[kept];
        const uint32_t at = (back & 255u) == was ? 0u : ((back >> 8) & 255u) == was ? 1u : 2u;
        lds_sync();
        nb8[4u * kept + at] = (uint8_t)lane;
        uint32_t next, prev;
        bad = new_vertex(s, c, 0, (uint32_t)lane, u, v, pq, q, next, prev);
        nb[lane] = kept | next << 8 | prev << 16;
    }
    c.alive[0] = (c.alive[0] & ~gone) | __ballot(mine);
    lds_sync();
    return __ballot(bad) ? VOR_DEGENERATE : VOR_OK;
}

// Several vertices per lane.
template <int NV>
__device__ __forceinline__ int close_hole(VorLds<NV> &s, VorCell<NV> &c, const uint64_t *out, double4 pq, int q,
                                          uint32_t site, int lane)
{
    constexpr uint32_t T = VorLds<NV>::T;
    uint32_t cnt = 0, room = 0;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        room += (uint32_t)__popcll(~c.alive[k] | out[k]);
        if (!out[k])
            continue;
        const uint32_t me = 64u * k + (uint32_t)lane;
        const bool o = (out[k] >> lane) & 1u;
        const ushort4 n = s.nb[me];
        const uint32_t t = c.tri[k], id[3] = {t & 1023u, (t >> 10) & 1023u, t >> 20};
        const uint32_t to[3] = {n.x & (T - 1), n.y & (T - 1), n.z & (T - 1)};
#pragma unroll
        for (int e = 0; e < 3; ++e) {
            const bool b = o && !s.gone[to[e]];
            const uint64_t m = __ballot(b);
            const uint32_t at = cnt + rank_in(m);
            if (b && at < T) {
                // edge: u | v << 10 | kept << 20 | the kept triangle's link back << 30
                const ushort4 back = s.nb[to[e]];
                const uint32_t link = back.x == me ? 0u : back.y == me ? 1u : 2u;
                s.edge[at] = id[e] | id[(e + 1) % 3] << 10 | to[e] << 20 | link << 30;
            }
            cnt += (uint32_t)__popcll(m);
        }
    }
    const int fits = hole_fits(cnt, room, c.full);
    if (fits != VOR_OK)
        return fits;
    c.gen = (c.gen + 1u) & 0x3fffffu;
    if (lane == 0) {
        s.P[q] = pq;
        s.nid[q] = site;
    }
    lds_sync();
    uint64_t fresh[NV];
    uint32_t edge[NV], base = 0;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        fresh[k] = 0;
        if (base >= cnt)
            continue;
        const uint64_t f = ~c.alive[k] | out[k];
        const uint32_t j = base + rank_in(f);
        const bool mine = ((f >> lane) & 1u) && j < cnt;
        base += (uint32_t)__popcll(f);
        fresh[k] = __ballot(mine);
        if (mine) {
            const uint32_t me = 64u * k + (uint32_t)lane, e = s.edge[j], kept = (e >> 20) & 1023u;
            edge[k] = e;
            s.by_u[e & 1023u] = c.gen << 10 | me;
            s.by_v[(e >> 10) & 1023u] = c.gen << 10 | me;
            reinterpret_cast<uint16_t *>(&s.nb[kept])[e >> 30] = (uint16_t)me;
        }
    }
    lds_sync();
    bool bad = false;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        if (fresh[k] && ((fresh[k] >> lane) & 1u)) {
            const uint32_t me = 64u * k + (uint32_t)lane, e = edge[k];
            uint32_t next, prev;
            bad = new_vertex(s, c, k, me, e & 1023u, (e >> 10) & 1023u, pq, q, next, prev) || bad;
            s.nb[me] = make_ushort4((uint16_t)((e >> 20) & 1023u), (uint16_t)next, (uint16_t)prev, 0);
        }
        c.alive[k] = (c.alive[k] & ~out[k]) | fresh[k];
    }
    lds_sync();
    return __ballot(bad) ? VOR_DEGENERATE : VOR_OK;
}

// The box plane of a vertex that lies on one of them (else 6), and where the
// line that ends there meets the plane through the site alongside it.  A vertex
// 10^6 extents away has 6 digits fewer than that place, and the cells of
// coplanar sites are columns as wide there as at the site.
template <int NV> __device__ __forceinline__ uint32_t wall_of(const VorLds<NV> &s, uint32_t tri, d3 &at)
{
    const uint32_t a = tri & 1023u, b = (tri >> 10) & 1023u, d = tri >> 20, low = min(a, min(b, d));
    if (low >= 6u || max(min(a, b), min(max(a, b), d)) < 6u)
        return 6;
    double4 w[3] = {s.P[a], s.P[b], s.P[d]};
    (low == a ? w[0] : low == b ? w[1] : w[2]).w = 0.0;
    at = plane_vertex(w[0], w[1], w[2]);
    return low;
}

// Cut by the bisector of `site` at q (wave-uniform; the cell's own site at p):
// every lane tests its vertices, and the cell changes only when some lie
// outside.  Sites on common spheres make vertices of one place, which rounding
// may part to both sides of a plane through it, so that what a cut removes is
// no disc.  The last passes, which take such cells too, therefore leave the
// vertices within ON_PLANE |x| |v| of a plane (the rounding of x.v and of v, 500
// times) on it; a second site at the place of a neighbour still fails.  For a
// vertex on a box plane that is 10^-7 of an extent, the depth to which one of
// 240 coplanar sites on a circle cuts the cell of a site within: where it is so
// near the plane, its line decides at the site.
constexpr double ON_PLANE = 1e-13;
template <int NV, bool WARM>
__device__ __forceinline__ int cell_cut(VorLds<NV> &s, VorCell<NV> &c, const VorReach &p, float qx, float qy, float qz,
                                        uint32_t site, int lane)
{
    const double dx = (double)qx - (double)p.px, dy = (double)qy - (double)p.py, dz = (double)qz - (double)p.pz;
    const double w = 0.5 * fma(dx, dx, fma(dy, dy, dz * dz));
    uint64_t out[NV];
    uint64_t any = 0, kept = 0, clear = 0, on_plane = 0;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        out[k] = 0;
        if (NV > 1 && !c.alive[k])
            continue;
        const double xv = fma(dx, c.v[k].x, fma(dy, c.v[k].y, dz * c.v[k].z));
        const bool o = xv > w;
        if (NV >= NV_LARGE) {
            // (above) only what is outside by more than rounding is removed
            const uint64_t cut = __ballot(o) & c.alive[k];
            any |= cut;
            out[k] = __ballot(xv - w > ON_PLANE * sqrt(2.0 * w) * (double)c.fl[k]) & c.alive[k];
            on_plane |= cut & ~out[k];
            s.gone[64 * k + lane] = (out[k] >> lane) & 1u;
            kept |= c.alive[k] & ~out[k];
            clear |= out[k];
            continue;
        }
        out[k] = __ballot(o) & c.alive[k];
        if (NV > 1)
            s.gone[64 * k + lane] = (out[k] >> lane) & 1u;
        any |= out[k];
        kept |= c.alive[k] & ~out[k];
    }
    if (!any)
        return VOR_OK;
    if (NV >= NV_LARGE) {
        if (on_plane) {
            kept = 0;
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                if (!c.alive[k])
                    continue;
                bool o = ((c.alive[k] & ~out[k]) >> lane & 1u) && fma(dx, c.v[k].x, fma(dy, c.v[k].y, dz * c.v[k].z)) > w;
                d3 at;
                o = o && wall_of(s, c.tri[k], at) < 6u &&
                    fma(dx, at.x, fma(dy, at.y, dz * at.z)) - w > ON_PLANE * sqrt(2.0 * w * dot_d(at, at));
                out[k] |= __ballot(o);
                s.gone[64 * k + lane] = (out[k] >> lane) & 1u;
                kept |= c.alive[k] & ~out[k];
                clear |= out[k];
            }
        }
        bool twin = false;
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const double4 p = s.P[64 * k + lane];
            twin = twin || (s.nid[64 * k + lane] != VOR_NONE && p.x == dx && p.y == dy && p.z == dz);
        }
        if (__ballot(twin))
            return VOR_DEGENERATE;
        if (!clear)
            return VOR_OK;
    }
    if (WARM) {
        // A guess is offered again when the walk meets its site.  Its plane is
        // already a face; a vertex on it may round to "outside", and the same
        // plane again would make a vertex of parallel planes.
        bool dup = false;
#pragma unroll
        for (int k = 0; k < NV; ++k)
            dup = dup || s.nid[64 * k + lane] == site;
        if (__ballot(dup))
            return VOR_OK;
    }
    if (!kept)
        return VOR_DEGENERATE; // the site's own half-space always keeps the site
    const int q = cell_plane_slot(s, c, lane);
    if (q < 0) {
        c.full |= FULL_PLANES;
        return VOR_FULL;
    }
    const double4 pq = make_double4(dx, dy, dz, w);
    if constexpr (NV == 1)
        return close_hole_1(s, c, out, pq, q, site, lane);
    else
        return close_hole(s, c, out, pq, q, site, lane);
}

// One child box per lane: can a site in it, at a squared distance in [lo2,
// hi2), cut the cell?  It must come within 2R, and within the ball of some
// vertex v: a cut needs x.v > |x|^2 / 2 for a point x of the box.  Near
// vertices are bounded through their bounding box, far ones (of unbounded or
// stretched cells) one by one.  A NaN keeps the box.
template <int NV>
__device__ __forceinline__ uint64_t boxes_in_reach(const VorTree &t, const VorCell<NV> &c, const VorReach &r, int level,
                                                   uint32_t base, int lane)
{
    const uint32_t i = base + (uint32_t)lane;
    bool in = false, may = false;
    float l[3] = {0.0f, 0.0f, 0.0f}, h[3] = {0.0f, 0.0f, 0.0f}, need = 0.0f;
    // (box and site are f32: an offset is off by one rounding, 2^-24 of itself)
    if (i < level_count(t, level)) {
        const float4 *box = t.boxes + 2 * (size_t)(level_begin(t, level) + i);
        const float4 a = box[0], b = box[1];
        l[0] = a.x - r.px, l[1] = a.y - r.py, l[2] = a.z - r.pz;
        h[0] = b.x - r.px, h[1] = b.y - r.py, h[2] = b.z - r.pz;
        float mind2 = 0.0f, maxd2 = 0.0f, sb = 0.0f;
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            const float near = fmaxf(fmaxf(l[x], -h[x]), 0.0f), far = fmaxf(-l[x], h[x]);
            mind2 = fmaf(near, near, mind2);
            maxd2 = fmaf(far, far, maxd2);
            sb += fmaxf(l[x] * c.bmin[x], h[x] * c.bmax[x]);
        }
        in = !(mind2 * (1.0f - SLACK) > fminf(r.hi2, 4.0f * c.r2)) && !(maxd2 * (1.0f + SLACK) < r.lo2);
        need = 0.5f * mind2 * (1.0f - SLACK);
        may = !(sb * (1.0f + SLACK) < need);
    }
    if (NV > 1 && level == 0 && __popcll(__ballot(in && may)) >= 4) {
        // Cells of many faces lie beside far denser sites, and the bounding box
        // of their vertices reaches thousands of those: does the box meet the
        // ball of some near vertex (the sites closer to it than this cell's)?
        bool meets = false;
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            uint64_t m = c.alive[k] & ~c.farv[k];
            while (m) {
                const int v = (int)__builtin_ctzll(m);
                m &= m - 1;
                const float vx = readlane_f(c.fx[k], v), vy = readlane_f(c.fy[k], v), vz = readlane_f(c.fz[k], v);
                const float len = readlane_f(c.fl[k], v);
                const float x = vx - fminf(fmaxf(vx, l[0]), h[0]), y = vy - fminf(fmaxf(vy, l[1]), h[1]),
                            z = vz - fminf(fmaxf(vz, l[2]), h[2]);
                meets = meets || !(fmaf(x, x, fmaf(y, y, z * z)) > len * len * (1.0f + SLACK));
            }
        }
        may = may && meets;
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        uint64_t m = c.farv[k];
        if (!m || !__ballot(in && !may))
            continue;
        while (m) {
            const int v = (int)__builtin_ctzll(m);
            m &= m - 1;
            const float vx = readlane_f(c.fx[k], v), vy = readlane_f(c.fy[k], v), vz = readlane_f(c.fz[k], v);
            const float a = l[0] * vx, b = h[0] * vx, d = l[1] * vy, e = h[1] * vy, f = l[2] * vz, g = h[2] * vz;
            const float most = fmaxf(a, b) + fmaxf(d, e) + fmaxf(f, g);
            const float size = fmaxf(fabsf(a), fabsf(b)) + fmaxf(fabsf(d), fabsf(e)) + fmaxf(fabsf(f), fabsf(g));
            may = may || !(fmaf(size, SLACK, most) < need);
        }
    }
    return __ballot(in && may);
}

// From this many sites of a batch on, they are tested together, one per lane,
// against one vertex after another (one vertex per lane: the far ones, several:
// all of them) instead of offering each.
constexpr int MANY = 8;

// Sites of the leaf boxes s.hits[first, first + 8), one per lane: those that
// may cut the cell are offered to it, nearest first where asked (the nearer
// planes of the first ball make many farther ones miss).  Sorted positions [skip, skip + 64) have been
// offered before (skip VOR_NONE: none have).
template <int NV, bool WARM>
__device__ __forceinline__ int offer_sites(VorLds<NV> &s, VorCell<NV> &c, const VorTree &t, const VorReach &r,
                                           uint32_t first, uint32_t nhits, uint32_t at, uint32_t skip, uint32_t n,
                                           int lane)
{
    const uint32_t hit = first + (uint32_t)lane / VOR_LEAF;
    const bool nearest_first = r.lo2 == 0.0f;
    bool cand = false;
    float4 p = make_float4(r.px, r.py, r.pz, 0.0f);
    if (hit < nhits) {
        const uint32_t k = s.hits[hit] * VOR_LEAF + (uint32_t)lane % VOR_LEAF;
        cand = k < n && k != at && (skip == VOR_NONE || k - skip >= 64u);
        if (cand)
            p = t.sites[k];
    }
    const float fx = p.x - r.px, fy = p.y - r.py, fz = p.z - r.pz, d2f = offset2(fx, fy, fz);
    // (a site on top of the cell's own has no bisector)
    cand = cand && (fx != 0.0f || fy != 0.0f || fz != 0.0f) && d2f >= r.lo2 && !(d2f >= r.hi2 && r.hi2 < INFINITY) &&
           !(d2f > 4.0f * c.r2);
    const float w = 0.5f * d2f * (1.0f - SLACK);
    const float sb = fmaxf(fx * c.bmin[0], fx * c.bmax[0]) + fmaxf(fy * c.bmin[1], fy * c.bmax[1]) +
                     fmaxf(fz * c.bmin[2], fz * c.bmax[2]);
    bool far_cut = false;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        uint64_t m = c.farv[k];
        if (!m)
            continue;
        while (m) {
            const int v = (int)__builtin_ctzll(m);
            m &= m - 1;
            const float a = fx * readlane_f(c.fx[k], v), b = fy * readlane_f(c.fy[k], v), e = fz * readlane_f(c.fz[k], v);
            far_cut = far_cut || !(fmaf(fabsf(a) + fabsf(b) + fabsf(e), SLACK, a + b + e) < w);
        }
    }
    const VorOffer mine{fx, fy, fz, SLACK * sqrtf(d2f), w};
    const bool near_cut = !(sb * (1.0f + SLACK) < w);
    if (NV == NV_SMALL && __popcll(__ballot(cand && far_cut && !near_cut)) >= MANY) {
        // SLACK of a vertex 10^6 extents away passes every site within 10^-5 rad
        // of its tangent plane: all of them, where sites on a plane leave the
        // cell open.  cell_cut's own test then, one site per lane (coplanar
        // sites on a tilted plane, 50,000: 198 -> 36 ms, 100,000: 806 -> 135).
        // For every batch it cost the 1M heightfield build 5 %, in the larger
        // passes 2 % where a noisy plane lies below a volume.
        const double x = (double)p.x - (double)r.px, y = (double)p.y - (double)r.py, z = (double)p.z - (double)r.pz;
        const double wd = 0.5 * fma(x, x, fma(y, y, z * z));
        far_cut = false;
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            uint64_t a = c.farv[k];
            while (a) {
                const int v = (int)__builtin_ctzll(a);
                a &= a - 1;
                const double vx = readlane_d(c.v[k].x, v), vy = readlane_d(c.v[k].y, v), vz = readlane_d(c.v[k].z, v);
                far_cut = far_cut || fma(x, vx, fma(y, vy, z * vz)) > wd;
            }
        }
    }
    uint64_t m = __ballot(cand && (far_cut || near_cut));
    if (NV > 1 && __popcll(m) >= MANY) {
        // (a cell of many faces: the box of its vertices lets too many pass)
        float most = 0.0f;
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            uint64_t a = c.alive[k] & ~c.farv[k];
            while (a) {
                const int v = (int)__builtin_ctzll(a);
                a &= a - 1;
                const float vx = readlane_f(c.fx[k], v), vy = readlane_f(c.fy[k], v), vz = readlane_f(c.fz[k], v);
                most = fmaxf(most, fmaf(fx, vx, fmaf(fy, vy, fz * vz)));
            }
        }
        m &= __ballot(far_cut || !(most + mine.slack * fminf(sqrtf(c.r2), c.far) < w));
    }
    while (m) {
        int l = (int)__builtin_ctzll(m);
        if (nearest_first && (m & (m - 1))) {
            const bool rem = (m >> lane) & 1u;
            l = (int)(wave_min_u(rem ? (__float_as_uint(d2f) & ~63u) | (uint32_t)lane : VOR_NONE) & 63u);
        }
        m &= ~(1ull << l);
        if (!may_cut(c, mine, l))
            continue;
        const int status = cell_cut<NV, WARM>(s, c, r, readlane_f(p.x, l), readlane_f(p.y, l), readlane_f(p.z, l),
                                              __float_as_uint(readlane_f(p.w, l)), lane);
        if (status != VOR_OK)
            return status;
    }
    return VOR_OK;
}

// Offers the cell every site of the tree, in the band of r, that may cut it.
template <int NV, bool WARM>
__device__ __forceinline__ int offer_tree(VorLds<NV> &s, VorCell<NV> &c, const VorTree &t, const VorReach &r,
                                          uint32_t at, uint32_t skip, uint32_t n, int lane)
{
    uint32_t nhits = 0;
    // sites of whole groups of 8 leaf boxes, or of all that are left
    auto flush = [&](bool all) {
        uint32_t k = 0;
        while (k + 8u <= nhits || (all && k < nhits)) {
            const uint32_t gen = c.gen;
            const int status = offer_sites<NV, WARM>(s, c, t, r, k, nhits, at, skip, n, lane);
            if (status != VOR_OK)
                return status;
            if (gen != c.gen)
                cell_radii(c, lane);
            k += 8u;
        }
        if (k && k < nhits) {
            const uint32_t x = s.hits[k + ((uint32_t)lane & 7u)]; // below 8 are left
            lds_sync();
            if (lane < 8)
                s.hits[lane] = x;
            lds_sync();
        }
        nhits = k < nhits ? nhits - k : 0u;
        return (int)VOR_OK;
    };
    uint64_t m3 = t.top >= 3 ? boxes_in_reach<NV>(t, c, r, 3, 0, lane) : 1ull;
    while (m3) {
        const uint32_t b3 = (uint32_t)__builtin_ctzll(m3);
        m3 &= m3 - 1;
        uint64_t m2 = t.top >= 2 ? boxes_in_reach<NV>(t, c, r, 2, 64u * b3, lane) : 1ull;
        while (m2) {
            const uint32_t b2 = 64u * b3 + (uint32_t)__builtin_ctzll(m2);
            m2 &= m2 - 1;
            uint64_t m1 = boxes_in_reach<NV>(t, c, r, 1, 64u * b2, lane);
            while (m1) {
                const uint32_t b1 = 64u * b2 + (uint32_t)__builtin_ctzll(m1);
                m1 &= m1 - 1;
                const uint64_t m0 = boxes_in_reach<NV>(t, c, r, 0, 64u * b1, lane);
                if ((m0 >> lane) & 1u)
                    s.hits[nhits + rank_in(m0)] = 64u * b1 + (uint32_t)lane;
                nhits += (uint32_t)__popcll(m0); // at most 7 + 64
                lds_sync();
                if (nhits >= 8u) {
                    const int status = flush(false);
                    if (status != VOR_OK)
                        return status;
                }
            }
        }
    }
    return flush(true);
}

// The box planes 0..5 (+x, -x, +y, -y, +z, -z) and its 8 corners.  Corner
// (sx, sy, sz) is the triangle of planes (X, Y, Z), ordered X, Y, Z when an
// even number of them are "-" planes and X, Z, Y otherwise, so that every
// edge of the closed triangulation appears once in each direction.  Across
// the edge of two planes lies the corner on the other plane of the third axis.
template <int NV>
__device__ __forceinline__ void cell_begin(VorLds<NV> &s, VorCell<NV> &c, const VorTree &t, const VorReach &r, int lane)
{
    const double p[3] = {(double)r.px, (double)r.py, (double)r.pz};
    double lo[3], hi[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        lo[a] = t.box->lo[a] - p[a];
        hi[a] = t.box->hi[a] - p[a];
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        s.nid[64 * k + lane] = VOR_NONE;
        c.alive[k] = k == 0 ? 0xffull : 0ull;
        c.freep[k] = k == 0 ? ~0x3full : ~0ull;
        c.farv[k] = 0ull;
        c.v[k] = d3{0.0, 0.0, 0.0};
        c.fx[k] = c.fy[k] = c.fz[k] = c.fl[k] = 0.0f;
        c.tri[k] = 0;
    }
    if (lane < 6) {
        const int a = lane >> 1;
        const bool minus = lane & 1;
        s.P[lane] = make_double4(a == 0 ? (minus ? -1.0 : 1.0) : 0.0, a == 1 ? (minus ? -1.0 : 1.0) : 0.0,
                                 a == 2 ? (minus ? -1.0 : 1.0) : 0.0,
                                 minus ? -(a == 0 ? lo[0] : a == 1 ? lo[1] : lo[2])
                                       : (a == 0 ? hi[0] : a == 1 ? hi[1] : hi[2]));
    }
    if (lane < 8) {
        const int sx = (lane >> 2) & 1, sy = (lane >> 1) & 1, sz = lane & 1;
        const uint32_t X = (uint32_t)sx, Y = (uint32_t)(2 + sy), Z = (uint32_t)(4 + sz);
        const bool even = ((sx + sy + sz) & 1) == 0;
        c.v[0] = d3{sx ? lo[0] : hi[0], sy ? lo[1] : hi[1], sz ? lo[2] : hi[2]};
        set_f32(c, 0);
        c.tri[0] = even ? X | Y << 10 | Z << 20 : X | Z << 10 | Y << 20;
        s.nb[lane].x = even ? lane ^ 1 : lane ^ 2;
        s.nb[lane].y = lane ^ 4;
        s.nb[lane].z = even ? lane ^ 2 : lane ^ 1;
    }
    c.full = 0;
    lds_sync();
}

// Sites on common spheres leave faces of no area, which planes offered in one
// order keep and in another do not: those whose vertices lie in one or two
// places lose their mark in s.used, so that the neighbours do not depend on the
// order.  Only a cell with two linked vertices in one place can have any
// (SAME_PLACE |v| apart, some dozen roundings: in general position there are none).
//
// At a vertex on a box plane that is 10^-8 of an extent.  Two of them are in one
// place if their lines also pass the site in one (wall_of), by the measure of
// that place (by the far one alone, 7 of the 97 pairs of neighbours among 50
// sites on a circle, rounded to f32, were lost).
constexpr double SAME_PLACE = 1e-14;
__device__ __forceinline__ bool same_place(d3 a, d3 b, float len)
{
    return fmax(fmax(fabs(a.x - b.x), fabs(a.y - b.y)), fabs(a.z - b.z)) <= SAME_PLACE * (double)len;
}
__device__ __forceinline__ d3 readlane_d3(d3 x, int l)
{
    return d3{readlane_d(x.x, l), readlane_d(x.y, l), readlane_d(x.z, l)};
}
template <int NV> __device__ __forceinline__ void cell_drop_flat(VorLds<NV> &s, const VorCell<NV> &c, int lane)
{
    // wall_of every vertex (at: itself where there is none)
    d3 at[NV];
    uint32_t wall[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        at[k] = c.v[k];
        wall[k] = 6;
        if (!c.farv[k]) // (no vertex on a box plane)
            continue;
        if ((c.alive[k] >> lane) & 1u)
            wall[k] = wall_of(s, c.tri[k], at[k]);
    }
    // the planes are no longer needed: vertex positions take their place
    lds_sync();
#pragma unroll
    for (int k = 0; k < NV; ++k)
        s.P[64 * k + lane] = make_double4(c.v[k].x, c.v[k].y, c.v[k].z, 0.0);
    lds_sync();
    auto place_of = [&](uint32_t v) { return d3{s.P[v].x, s.P[v].y, s.P[v].z}; };
    bool close = false;
#pragma unroll
    for (int k = 0; k < NV; ++k)
        if ((c.alive[k] >> lane) & 1u) {
            const auto n = s.nb[64 * k + lane];
            const d3 v = c.v[k];
            close = close || same_place(place_of(n.x), v, c.fl[k]) || same_place(place_of(n.y), v, c.fl[k]) ||
                    same_place(place_of(n.z), v, c.fl[k]);
        }
    if (!__ballot(close))
        return;
    for (uint32_t q = 6; q < (uint32_t)VorLds<NV>::T; ++q) {
        if (!(((uint32_t)__builtin_amdgcn_readfirstlane((int)s.used[q >> 5]) >> (q & 31u)) & 1u))
            continue;
        uint64_t on[NV];
        uint32_t first = 0, second = 0;
        d3 first_at{0.0, 0.0, 0.0}, second_at{0.0, 0.0, 0.0};
        uint32_t first_wall = 6, second_wall = 6;
#pragma unroll
        for (int k = NV - 1; k >= 0; --k) {
            const uint32_t t = c.tri[k];
            on[k] = __ballot((t & 1023u) == q || ((t >> 10) & 1023u) == q || t >> 20 == q) & c.alive[k];
            if (on[k]) {
                const int l = (int)__builtin_ctzll(on[k]);
                first = 64u * k + (uint32_t)l;
                first_at = readlane_d3(at[k], l);
                first_wall = (uint32_t)__builtin_amdgcn_readlane((int)wall[k], l);
            }
        }
        bool flat = true;
        for (int place = 0; place < 2 && flat; ++place) {
            // the vertices of the face that are elsewhere
            const d3 p = place_of(place ? second : first), p_at = place ? second_at : first_at;
            const uint32_t p_wall = place ? second_wall : first_wall;
            uint64_t any = 0;
#pragma unroll
            for (int k = NV - 1; k >= 0; --k) {
                const d3 x = at[k];
                const float len = wall[k] == 6u ? c.fl[k] : (float)sqrt(fma(x.x, x.x, fma(x.y, x.y, x.z * x.z)));
                const bool same = wall[k] == p_wall && same_place(p, c.v[k], c.fl[k]) && same_place(p_at, x, len);
                on[k] &= __ballot(!same);
                any |= on[k];
                if (on[k]) {
                    const int l = (int)__builtin_ctzll(on[k]);
                    second = 64u * k + (uint32_t)l;
                    second_at = readlane_d3(x, l);
                    second_wall = (uint32_t)__builtin_amdgcn_readlane((int)wall[k], l);
                }
            }
            if (!any)
                break;
            flat = place == 0;
        }
        if (flat && lane == 0)
            s.used[q >> 5] &= ~(1u << (q & 31u));
        lds_sync();
    }
}

// A cold cell is offered its sites ball by ball: first those no farther than
// this many of the curve's 64, then balls of GROW2 times the squared radius,
// and all that can still cut it once its reach is within 4 times the last
// ball.  Near sites of every side first leave a bounded cell early; far ones
// on one side make long slivers, whose vertices lose their digits.  The third
// pass goes in smaller steps.  FAR_TIMES: distance, in radii of the first
// ball, beyond which a vertex counts as far.
template <int NV> constexpr int BALL_SITES = NV < NV_LARGE ? 16 : 6;
template <int NV> constexpr float GROW2 = NV < NV_LARGE ? 4.0f : 2.0f;
constexpr float FAR_TIMES = 4.0f;

// Voronoi cell of the site at sorted position `at`; its neighbours go to
// ids[0..m) (unordered; LDS).  Guesses: gadj[gb, ge), at most 64.
template <int NV, bool WARM>
__device__ __forceinline__ int voronoi_cell(VorLds<NV> &s, VorCell<NV> &c, const VorTree &t, uint32_t at,
                                            const float *__restrict__ points, uint32_t n, bool warm, uint32_t gb,
                                            uint32_t ge, const uint32_t *__restrict__ gadj, int lane, uint32_t *ids,
                                            int *m_out)
{
    const float4 own = t.sites[at];
    const uint32_t self = __float_as_uint(own.w);
    VorReach r{own.x, own.y, own.z, 0.0f, 0.0f};
    *m_out = 0;
    cell_begin(s, c, t, r, lane);
    const float diag2 = (float)t.box->diag2; // no two sites are farther apart
    // seeds, one per lane: the guesses, or the 64 sites around it on the curve
    uint32_t first = at < 32u ? 0u : at - 32u;
    if (first + 64u > n)
        first = n > 64u ? n - 64u : 0u;
    bool ok = false;
    float4 p = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    uint32_t site = 0;
    float near2 = 0.0f; // warm: how far the nearest sites on the curve are
    if (WARM && warm) {
        const uint32_t k = at + (uint32_t)lane - 6u;
        if (lane < 13 && k < n) { // (k wraps past the first sites)
            const float4 q = t.sites[k];
            near2 = offset2(q.x - own.x, q.y - own.y, q.z - own.z);
        }
        near2 = wave_max_f(near2);
        if (gb + (uint32_t)lane < ge) {
            site = gadj[gb + lane];
            ok = site < n && site != self;
            if (ok)
                p = scaled_site(points, site, t.box->k);
        }
    } else if (first + (uint32_t)lane < n) {
        p = t.sites[first + lane];
        site = __float_as_uint(p.w);
        ok = first + (uint32_t)lane != at;
    }
    const float dx = p.x - own.x, dy = p.y - own.y, dz = p.z - own.z, d2 = offset2(dx, dy, dz);
    ok = ok && (dx != 0.0f || dy != 0.0f || dz != 0.0f);
    const uint32_t key = wave_sort_u(ok ? (__float_as_uint(d2) & ~63u) | (uint32_t)lane : VOR_NONE, lane);
    const int found = (int)__popcll(__ballot(ok));
    float ball2 = 0.0f;
    if (found)
        ball2 = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)key, min(found, BALL_SITES<NV>) - 1) | 63u);
    const bool cold = !(WARM && warm);
    const uint64_t take = __ballot(ok && (!cold || d2 < ball2));
    const VorOffer mine{dx, dy, dz, SLACK * sqrtf(d2), 0.5f * d2 * (1.0f - SLACK)};
    int left = NV == NV_SMALL ? (int)__popcll(take) : 0; // (one copy of the cut's code in the larger passes)
    for (int i = 0; left > 0; ++i) { // sorted: those to take are the first, but for the bits cut off
        const int l = (int)((uint32_t)__builtin_amdgcn_readlane((int)key, i) & 63u);
        if (!((take >> l) & 1u))
            continue;
        --left;
        if (!may_cut(c, mine, l))
            continue;
        const int status = cell_cut<NV, WARM>(s, c, r, readlane_f(p.x, l), readlane_f(p.y, l), readlane_f(p.z, l),
                                              (uint32_t)__builtin_amdgcn_readlane((int)site, l), lane);
        if (status != VOR_OK)
            return status;
    }
    c.far = FAR_TIMES * sqrtf(ball2);
    cell_radii(c, lane);
    // cold: the rest of the first ball (the curve's sites in it have been
    // offered), and so on; warm: all within reach at once (the guesses come
    // again), when the guesses have left the cell no larger than its
    // neighbourhood
    r.hi2 = cold ? ball2 : 4.0f * c.r2 <= 64.0f * near2 ? INFINITY : near2;
    for (;;) {
        const int status = offer_tree<NV, WARM>(s, c, t, r, at, NV == NV_SMALL && cold && r.lo2 == 0.0f ? first : VOR_NONE, n, lane);
        if (status != VOR_OK)
            return status;
        const float reach2 = 4.0f * c.r2;
        if (!(r.hi2 < INFINITY) || reach2 * (1.0f + SLACK) < r.hi2)
            break;
        r.lo2 = r.hi2;
        r.hi2 = reach2 <= 16.0f * r.hi2 || !(r.hi2 > 0.0f) || r.hi2 > diag2 ? INFINITY : r.hi2 * GROW2<NV>;
    }
    cell_mark_used(s, c, lane);
    cell_drop_flat(s, c, lane);
    int m = 0;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const uint32_t q = 64u * k + (uint32_t)lane, id = s.nid[q];
        const bool u = ((s.used[q >> 5] >> (q & 31u)) & 1u) && id != VOR_NONE;
        const uint64_t b = __ballot(u);
        if (u)
            ids[m + (int)rank_in(b)] = id;
        m += (int)__popcll(b);
    }
    lds_sync();
    *m_out = m;
    return VOR_OK;
}

struct VorLists {
    uint32_t *lists, *big_lists, *big_slot, *counts;
    uint32_t big_cap;
    uint32_t *retry[RETRIES], *fails; // cells queued for the further passes
};

// One cell and its list.  A list longer than LIST_K goes to a slot of
// big_lists (big_slot[i]), shorter lists to the cell's slot of lists.  A cell
// that overflows the small tables, or fails a cut, is queued in retry[].
template <int NV, bool WARM>
__device__ __forceinline__ void cell_and_list(VorLds<NV> &s, VorCell<NV> &c, const VorTree &t, uint32_t at,
                                              const float *points, uint32_t n, const VorLists &o, const uint32_t *gofs,
                                              const uint32_t *gadj, uint32_t gcount, int lane)
{
    const uint32_t i = __float_as_uint(t.sites[at].w);
    // Guesses seed the first pass only, and only cells with at most 64 of
    // them: a cell that overflows runs again cold, so guesses never cause a
    // capacity failure.  A range that runs backwards or past the gcount
    // guesses is not read (the cell builds cold).
    bool warm = false;
    uint32_t gb = 0, ge = 0;
    if (WARM) {
        gb = gofs[i], ge = gofs[i + 1];
        warm = gb < ge && ge <= gcount && ge - gb <= 64u;
    }
    uint32_t *ids = reinterpret_cast<uint32_t *>(s.edge); // free between cuts
    int m;
    int status = voronoi_cell<NV, WARM>(s, c, t, at, points, n, warm, gb, ge, gadj, lane, ids, &m);
    uint32_t *dst = o.lists + (size_t)i * LIST_K;
    if (status == VOR_OK && m > LIST_K) {
        uint32_t slot = 0;
        if (lane == 0)
            slot = atomicAdd(o.fails + F_BIG, 1u);
        slot = (uint32_t)__builtin_amdgcn_readfirstlane((int)slot);
        if (slot < o.big_cap && m <= BIG_K) {
            dst = o.big_lists + (size_t)slot * BIG_K;
            if (lane == 0)
                o.big_slot[i] = slot;
        } else {
            status = VOR_FULL;
            c.full |= FULL_LISTS;
        }
    }
    if (status == VOR_OK) {
        // ascending by rank (the ids are distinct)
        for (int a = lane; a < m; a += 64) {
            const uint32_t v = ids[a];
            int rank = 0;
            for (int b = 0; b < m; ++b)
                rank += ids[b] < v;
            dst[rank] = v;
        }
    } else {
        m = 0;
        if (lane == 0) {
            if (NV != NV_HUGE && (NV != NV_LARGE || status == VOR_FULL) && !(c.full & FULL_LISTS)) {
                constexpr int next = NV == NV_SMALL ? QUEUE_OF<NV_MID> : NV == NV_MID ? QUEUE_OF<NV_LARGE> : QUEUE_OF<NV_HUGE>;
                o.retry[next][atomicAdd(o.fails + F_RETRY + next, 1u)] = at; // at most n entries
            } else {
                atomicAdd(o.fails + (status == VOR_FULL ? F_FULL : F_DEGENERATE), 1u);
                atomicMin(o.fails + F_FIRST_BAD, i);
                atomicOr(o.fails + F_REASON, (uint32_t)c.full);
            }
        }
    }
    if (lane == 0)
        o.counts[i] = (uint32_t)m;
    lds_sync();
}

template <int NV> __device__ __forceinline__ void lds_begin(VorLds<NV> &s, VorCell<NV> &c, int lane)
{
#pragma unroll
    for (int k = 0; k < NV; ++k)
        s.by_u[64 * k + lane] = s.by_v[64 * k + lane] = 0u; // no tag has generation 0
    c.gen = 0;
    lds_sync();
}

// First pass: block b takes the cells of sorted positions [per b, per b + per),
// whose reads share the same boxes and sites.  5 waves per SIMD (96 VGPRs, 136
// bytes spilled) ran 2 to 5 % faster than 4 (128 VGPRs) or 6.
template <bool WARM>
__global__ __launch_bounds__(VOR_BLOCK) __attribute__((amdgpu_waves_per_eu(5))) void voronoi_cells_kernel(
    const float *__restrict__ points, VorTree t, uint32_t n, uint32_t per, VorLists o,
    const uint32_t *__restrict__ gofs, const uint32_t *__restrict__ gadj, uint32_t gcount)
{
    __shared__ VorLds<NV_SMALL> s;
    VorCell<NV_SMALL> c;
    const int lane = (int)threadIdx.x;
    lds_begin(s, c, lane);
    const uint32_t b = blockIdx.x * per, e = min(b + per, n);
    for (uint32_t at = b; at < e; ++at)
        cell_and_list<NV_SMALL, WARM>(s, c, t, at, points, n, o, gofs, gadj, gcount, lane);
}

// The further passes: the queued cells, taken from a work counter.
template <int NV>
__global__ __launch_bounds__(VOR_BLOCK) void voronoi_retry_kernel(const float *__restrict__ points, VorTree t,
                                                                  uint32_t n, VorLists o)
{
    __shared__ VorLds<NV> s;
    VorCell<NV> c;
    const int lane = (int)threadIdx.x;
    constexpr int queue = QUEUE_OF<NV>;
    const uint32_t count = o.fails[F_RETRY + queue];
    lds_begin(s, c, lane);
    for (;;) {
        uint32_t k = 0;
        if (lane == 0)
            k = atomicAdd(o.fails + F_NEXT + queue, 1u);
        k = (uint32_t)__builtin_amdgcn_readfirstlane((int)k);
        if (k >= count)
            break;
        cell_and_list<NV, false>(s, c, t, o.retry[queue][k], points, n, o, nullptr, nullptr, 0u, lane);
    }
}

// ---------------------------------------------------------------------------
// the site tree

__device__ __forceinline__ uint32_t spread10(uint32_t x)
{
    x = (x | x << 16) & 0x030000ffu;
    x = (x | x << 8) & 0x0300f00fu;
    x = (x | x << 4) & 0x030c30c3u;
    return (x | x << 2) & 0x09249249u;
}

// Morton codes on a cubic grid of 2^20 steps per axis over the largest
// extent: the upper 10 bits of each axis in hi, the lower 10 in lo.
__global__ void voronoi_keys_kernel(const float *__restrict__ points, uint32_t n, const float *__restrict__ bbox,
                                    const VorBox *__restrict__ box, uint32_t *__restrict__ hi,
                                    uint32_t *__restrict__ lo, uint32_t *__restrict__ vals)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    const int k = box->k;
    const float4 p = scaled_site(points, i, k);
    float ext = 1e-30f, at[3] = {p.x, p.y, p.z};
    for (int a = 0; a < 3; ++a) {
        const float lo = ldexpf(bbox[a], -k);
        ext = fmaxf(ext, ldexpf(bbox[3 + a], -k) - lo);
        at[a] -= lo;
    }
    uint32_t h = 0, l = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float x = at[a] / ext * 1048575.0f;
        const uint32_t q = (uint32_t)fminf(fmaxf(x, 0.0f), 1048575.0f);
        h |= spread10(q >> 10) << (2 - a);
        l |= spread10(q & 1023u) << (2 - a);
    }
    hi[i] = h;
    if (lo)
        lo[i] = l;
    vals[i] = i;
}

// keys[k] = src[vals[k]]
__global__ void voronoi_take_kernel(const uint32_t *__restrict__ src, const uint32_t *__restrict__ vals, uint32_t n,
                                    uint32_t *__restrict__ keys)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n)
        keys[k] = src[vals[k]];
}

// Sorted sites and the leaf boxes (a box per VOR_LEAF lanes).
__global__ __launch_bounds__(256) void voronoi_sites_kernel(const float *__restrict__ points,
                                                            const uint32_t *__restrict__ vals, uint32_t n,
                                                            const VorBox *__restrict__ box,
                                                            float4 *__restrict__ sites, float4 *__restrict__ boxes)
{
    const uint32_t k = blockIdx.x * 256u + threadIdx.x;
    const float inf = __builtin_huge_valf();
    float lo[3] = {inf, inf, inf}, hi[3] = {-inf, -inf, -inf};
    if (k < n) {
        const float4 p = scaled_site(points, vals[k], box->k);
        sites[k] = p;
        lo[0] = hi[0] = p.x;
        lo[1] = hi[1] = p.y;
        lo[2] = hi[2] = p.z;
    }
#pragma unroll
    for (int o = 1; o < (int)VOR_LEAF; o <<= 1)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            lo[a] = fminf(lo[a], __shfl_xor(lo[a], o));
            hi[a] = fmaxf(hi[a], __shfl_xor(hi[a], o));
        }
    if (k < n && k % VOR_LEAF == 0) {
        boxes[2 * (size_t)(k / VOR_LEAF)] = make_float4(lo[0], lo[1], lo[2], 0.0f);
        boxes[2 * (size_t)(k / VOR_LEAF) + 1] = make_float4(hi[0], hi[1], hi[2], 0.0f);
    }
}

// A level's boxes from the 64 boxes below each (one wave per box).
__global__ __launch_bounds__(64) void voronoi_level_kernel(const float4 *__restrict__ below, uint32_t count,
                                                           float4 *__restrict__ boxes)
{
    const uint32_t k = blockIdx.x * 64u + threadIdx.x;
    const float inf = __builtin_huge_valf();
    float lo[3] = {inf, inf, inf}, hi[3] = {-inf, -inf, -inf};
    if (k < count) {
        const float4 a = below[2 * (size_t)k], b = below[2 * (size_t)k + 1];
        lo[0] = a.x, lo[1] = a.y, lo[2] = a.z;
        hi[0] = b.x, hi[1] = b.y, hi[2] = b.z;
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        lo[a] = -wave_max_f(-lo[a]);
        hi[a] = wave_max_f(hi[a]);
    }
    if (threadIdx.x == 0) {
        boxes[2 * (size_t)blockIdx.x] = make_float4(lo[0], lo[1], lo[2], 0.0f);
        boxes[2 * (size_t)blockIdx.x + 1] = make_float4(hi[0], hi[1], hi[2], 0.0f);
    }
}

// Lists into the CSR, 16 lanes per cell.
constexpr uint32_t COPY_LANES = 16;
__global__ void voronoi_copy_kernel(uint32_t n, const uint32_t *__restrict__ offsets,
                                    const uint32_t *__restrict__ lists, const uint32_t *__restrict__ big_lists,
                                    const uint32_t *__restrict__ big_slot, uint32_t *__restrict__ adjacency)
{
    const uint32_t i = (blockIdx.x * blockDim.x + threadIdx.x) / COPY_LANES;
    if (i >= n)
        return;
    const uint32_t b = offsets[i], m = offsets[i + 1] - b;
    const uint32_t *src = lists + (size_t)i * LIST_K;
    if (m > LIST_K)
        src = big_lists + (size_t)big_slot[i] * BIG_K;
    for (uint32_t k = threadIdx.x % COPY_LANES; k < m; k += COPY_LANES)
        adjacency[b + k] = src[k];
}

__global__ void voronoi_begin_kernel(uint32_t *fails, uint32_t *last_count, const float *bbox, VorBox *box)
{
    if (threadIdx.x == F_WORDS + 1)
        scaled_box(bbox, *box);
    if (threadIdx.x < F_WORDS)
        fails[threadIdx.x] = threadIdx.x == F_FIRST_BAD ? VOR_NONE : 0u;
    if (threadIdx.x == F_WORDS)
        *last_count = 0u; // the scan runs over n + 1 counts
}

// workspace layout (u32 words)
struct VorWs {
    uint32_t *lists, *counts, *keys, *keys_lo, *vals, *sort_ws, *scan_ws, *fails, *bbox_ws, *retry[RETRIES - 1], *big_lists,
        *big_slot, *sites, *boxes;
    float *bbox;
    VorBox *box;
    uint32_t count[VOR_LEVELS];
};

// cells with more than LIST_K neighbours
static uint32_t big_cap_for(uint32_t n) { return std::max<uint32_t>(256, n / 64); }
// Sites above which the Morton codes take all 60 bits (8 sort passes): with
// fewer, 1024 steps per axis part most sites.
constexpr uint32_t FINE_KEYS_MIN = 1u << 16;

static size_t ws_words(uint32_t n, VorWs *w, uint32_t *base)
{
    size_t off = 0;
    uint32_t *dummy;
    auto take = [&](uint32_t **p, size_t words) {
        *(w ? p : &dummy) = base + off;
        off += (words + 63) & ~(size_t)63;
    };
    VorWs local{};
    VorWs &x = w ? *w : local;
    take(&x.lists, (size_t)n * LIST_K);
    take(&x.counts, (size_t)n + 1);
    take(&x.keys, n);
    take(&x.keys_lo, 2 * (size_t)n);
    take(&x.vals, n);
    take(&x.sort_ws, radix_sort_workspace_words(n));
    take(&x.scan_ws, scan_workspace_words(n + 1));
    take(&x.fails, F_WORDS);
    take(&x.bbox_ws, 6);
    uint32_t *bb;
    take(&bb, 6);
    x.bbox = reinterpret_cast<float *>(bb);
    take(&bb, sizeof(VorBox) / 4); // (each of these starts at a multiple of 256 bytes)
    x.box = reinterpret_cast<VorBox *>(bb);
    for (uint32_t *&queue : x.retry)
        take(&queue, n);
    take(&x.big_lists, (size_t)big_cap_for(n) * BIG_K);
    take(&x.big_slot, n);
    take(&x.sites, 4 * (size_t)n);
    uint32_t count = (n + VOR_LEAF - 1) / VOR_LEAF, boxes = 0;
    for (int l = 0; l < VOR_LEVELS; ++l) {
        x.count[l] = count;
        boxes += count;
        count = (count + 63) / 64;
    }
    take(&x.boxes, 8 * (size_t)boxes);
    return off;
}

} // namespace vt

using namespace vt;

extern "C" size_t vt_voronoi_workspace_size(uint32_t num_points)
{
    return ws_words(num_points, nullptr, nullptr) * sizeof(uint32_t);
}

extern "C" int vt_voronoi_build(const float *points, uint32_t num_points, uint32_t *offsets,
                                uint32_t *num_adjacency, void *workspace, vt_stream_t stream)
{
    return vt_voronoi_build_warm(points, num_points, nullptr, nullptr, 0, offsets, num_adjacency, workspace, stream);
}

extern "C" int vt_voronoi_build_warm(const float *points, uint32_t num_points, const uint32_t *guess_offsets,
                                     const uint32_t *guess_adjacency, uint32_t num_guesses, uint32_t *offsets,
                                     uint32_t *num_adjacency,
                                     void *workspace, vt_stream_t stream)
{
    clear_error();
    VT_REQUIRE(points && offsets && num_adjacency && workspace, "null pointer argument");
    VT_REQUIRE(!guess_offsets == !guess_adjacency, "guess offsets and adjacency are given together or not at all");
    VT_REQUIRE(num_points >= 2, "at least 2 sites are needed, got %u", num_points);
    VT_REQUIRE(num_points <= (1u << 26), "too many sites (%u)", num_points);
    hipStream_t s = as_stream(stream);
    VorWs w{};
    ws_words(num_points, &w, reinterpret_cast<uint32_t *>(workspace));
    const uint32_t n = num_points;
    int rc = bbox3(points, n, w.bbox, w.bbox_ws, s);
    if (rc)
        return rc;
    // sites along a Morton curve, and the boxes over them
    voronoi_begin_kernel<<<1, 64, 0, s>>>(w.fails, w.counts + n, w.bbox, w.box);
    VT_LAUNCH_CHECK("voronoi_begin_kernel");
    const uint32_t nblocks = (n + 255) / 256;
    const bool fine = n >= FINE_KEYS_MIN;
    uint32_t *lo = w.keys_lo + n;
    voronoi_keys_kernel<<<nblocks, 256, 0, s>>>(points, n, w.bbox, w.box, fine ? w.keys_lo : w.keys,
                                                fine ? w.keys : nullptr, w.vals);
    VT_LAUNCH_CHECK("voronoi_keys_kernel");
    rc = radix_sort_pairs(w.keys, w.vals, n, 30, w.sort_ws, s);
    if (rc)
        return rc;
    if (fine) { // by the lower bits first, then (stable) by the upper
        voronoi_take_kernel<<<nblocks, 256, 0, s>>>(w.keys_lo, w.vals, n, lo);
        VT_LAUNCH_CHECK("voronoi_take_kernel");
        rc = radix_sort_pairs(lo, w.vals, n, 30, w.sort_ws, s);
        if (rc)
            return rc;
    }
    VorTree t{};
    t.sites = reinterpret_cast<const float4 *>(w.sites);
    t.box = w.box;
    float4 *boxes = reinterpret_cast<float4 *>(w.boxes);
    t.boxes = boxes;
    voronoi_sites_kernel<<<nblocks, 256, 0, s>>>(points, w.vals, n, w.box, reinterpret_cast<float4 *>(w.sites),
                                                 boxes);
    VT_LAUNCH_CHECK("voronoi_sites_kernel");
    std::copy(w.count, w.count + VOR_LEVELS, t.count);
    for (t.top = 0; t.top == 0 || w.count[t.top] > 64;) {
        const float4 *below = boxes + 2 * (size_t)level_begin(t, t.top);
        const uint32_t nbelow = w.count[t.top++];
        voronoi_level_kernel<<<w.count[t.top], 64, 0, s>>>(below, nbelow, boxes + 2 * (size_t)level_begin(t, t.top));
        VT_LAUNCH_CHECK("voronoi_level_kernel");
    }
    // (the third pass queues for the fourth where the second's queue was)
    VorLists o{w.lists, w.big_lists, w.big_slot, w.counts, big_cap_for(n), {w.retry[0], w.retry[1], w.retry[0]}, w.fails};
    const uint32_t per = std::min<uint32_t>(8, std::max<uint32_t>(1, n / 32768));
    const uint32_t blocks = (n + per - 1) / per;
    // cold builds run an instantiation without any of the warm-start code
    if (guess_offsets)
        voronoi_cells_kernel<true><<<blocks, VOR_BLOCK, 0, s>>>(points, t, n, per, o, guess_offsets, guess_adjacency,
                                                                num_guesses);
    else
        voronoi_cells_kernel<false><<<blocks, VOR_BLOCK, 0, s>>>(points, t, n, per, o, nullptr, nullptr, 0u);
    VT_LAUNCH_CHECK("voronoi_cells_kernel");
    // the retry passes run cold (guesses never cause a capacity failure)
    voronoi_retry_kernel<NV_MID><<<std::min<uint32_t>(n, 2048), VOR_BLOCK, 0, s>>>(points, t, n, o);
    VT_LAUNCH_CHECK("voronoi_retry_kernel (second pass)");
    voronoi_retry_kernel<NV_LARGE><<<std::min<uint32_t>(n, 1024), VOR_BLOCK, 0, s>>>(points, t, n, o);
    VT_LAUNCH_CHECK("voronoi_retry_kernel (third pass)");
    uint32_t tail[1 + F_WORDS];
    for (int huge = 0; huge < 2; ++huge) {
        rc = exclusive_scan_u32(w.counts, offsets, n + 1, w.scan_ws, s);
        if (rc)
            return rc;
        VT_HIP_CHECK(hipMemcpyAsync(tail, offsets + n, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
        VT_HIP_CHECK(hipMemcpyAsync(tail + 1, w.fails, F_WORDS * sizeof(uint32_t), hipMemcpyDeviceToHost, s));
        VT_HIP_CHECK(hipStreamSynchronize(s));
        const uint32_t queued = tail[1 + F_RETRY + QUEUE_OF<NV_HUGE>];
        if (huge || !queued || tail[1 + F_FULL] || tail[1 + F_DEGENERATE])
            break;
        voronoi_retry_kernel<NV_HUGE><<<std::min<uint32_t>(queued, 512), VOR_BLOCK, 0, s>>>(points, t, n, o);
        VT_LAUNCH_CHECK("voronoi_retry_kernel (fourth pass)");
    }
    if (tail[1 + F_FULL] || tail[1 + F_DEGENERATE]) {
        set_error("Voronoi build failed for %u cells over capacity (%d planes, %d vertices, %u lists longer than %d) "
                  "and %u degenerate cuts; first failing site %u; full tables (1 planes, 4 vertices, 8 "
                  "lists): %u",
                  tail[1 + F_FULL], VorLds<NV_HUGE>::T, VorLds<NV_HUGE>::T, big_cap_for(n), LIST_K,
                  tail[1 + F_DEGENERATE], tail[1 + F_FIRST_BAD], tail[1 + F_REASON]);
        return VT_ERR_INVALID;
    }
    *num_adjacency = tail[0];
    return VT_OK;
}

extern "C" int vt_voronoi_adjacency(uint32_t num_points, const uint32_t *offsets, uint32_t *adjacency,
                                    const void *workspace, vt_stream_t stream)
{
    clear_error();
    VT_REQUIRE(offsets && adjacency && workspace, "null pointer argument");
    hipStream_t s = as_stream(stream);
    VorWs w{};
    ws_words(num_points, &w, reinterpret_cast<uint32_t *>(const_cast<void *>(workspace)));
    const uint32_t per = 256 / COPY_LANES;
    voronoi_copy_kernel<<<(num_points + per - 1) / per, 256, 0, s>>>(num_points, offsets, w.lists, w.big_lists,
                                                                     w.big_slot, adjacency);
    VT_LAUNCH_CHECK("voronoi_copy_kernel");
    return VT_OK;
}
