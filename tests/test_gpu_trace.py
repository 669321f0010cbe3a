"""GPU ray queries on closed meshes: watertightness at shared edges and vertices.

The reference's ray queries come from Embree (src/embreeaccelerator.cxx:87-304), whose
triangle test is watertight; the device test is the watertight test of Woop, Benthin and
Wald (2013).  Its guarantee: a ray that crosses a closed mesh is accepted by at least one
triangle, also when it passes exactly through an edge or a vertex shared by several
triangles.  It holds only if the 2-D edge functions are evaluated antisymmetrically, i.e.
without fused multiply-adds, so rays are aimed at the exact float32 vertices and at points
on the shared edges, from several interior origins, and every one of them must hit.
"""
import numpy as np
import pytest

from naivetrace_amd import abi, configs
from naivetrace_amd.renderer import GpuRenderer
from naivetrace_amd.scene import Scene, flat

pytestmark = pytest.mark.gpu


def _closed_scene(vertices, tris):
    s = Scene()
    m = s.add_material(shader=s.add_shader(abi.SHADER_DIFFUSE, reflectance=flat(0.5)))
    s.add_mesh(vertices, tris, m)
    c = vertices.mean(axis=0)
    s.set_camera(c, c + np.array([0.0, 0.0, -1.0]), [0.0, 1.0, 0.0], 60.0)
    s.width, s.height = 8, 8
    return s


def _edge_rays(vertices, tris, origins):
    """Rays from each origin through every vertex and through points on every edge (float32)."""
    v = vertices.astype(np.float32)
    e = np.concatenate([tris[:, [0, 1]], tris[:, [1, 2]], tris[:, [2, 0]]])
    e = np.unique(np.sort(e, axis=1), axis=0)
    targets = [v]
    for s in (0.5, 0.25, 1.0 / 3.0, 0.9):
        a, b = v[e[:, 0]], v[e[:, 1]]
        targets.append((a + np.float32(s) * (b - a)).astype(np.float32))
    targets = np.concatenate(targets)
    org, d = [], []
    for o in origins:
        o = np.asarray(o, dtype=np.float32)
        dd = targets.astype(np.float64) - o
        dd /= np.linalg.norm(dd, axis=1, keepdims=True)
        org.append(np.broadcast_to(o, dd.shape))
        d.append(dd)
    return np.concatenate(org).astype(np.float32), np.concatenate(d).astype(np.float32)


def _check_no_leak(vertices, tris, origins):
    s = _closed_scene(vertices, tris)
    org, d = _edge_rays(vertices, tris, origins)
    tmax = np.full(len(org), 1e30, np.float32)
    with GpuRenderer(s, abi.default_params(8, 8)) as r:
        t, prim, _, _ = r.trace_closest(org, d, tmax)
        tb, pb, _, _ = r.trace_closest(org, d, tmax, bruteforce=True)
        occ = r.trace_occluded(org, d, tmax)
    print(f"{len(org)} rays: BVH misses {np.sum(prim < 0)}, brute-force misses {np.sum(pb < 0)}, "
          f"any-hit misses {np.sum(occ == 0)}", flush=True)
    assert np.all(prim >= 0)
    assert np.all(pb >= 0)
    assert np.all(occ == 1)
    assert np.all(np.isfinite(t)) and np.all(t > 0)


@pytest.mark.parametrize("freq", [3, 12])
def test_icosphere_edges_and_vertices_hit(gpu_lib, freq):
    v, f = configs.icosphere(freq)
    # Off-origin, non-power-of-two scale so that coordinates carry full mantissas.
    v = (v * 3.7 + np.array([10.3, -2.1, 5.9])).astype(np.float32)
    origins = [v.mean(axis=0), v.mean(axis=0) + [0.9, -0.4, 1.3], v.mean(axis=0) + [-2.1, 1.7, 0.2]]
    _check_no_leak(v, f, origins)


def test_cube_edges_and_vertices_hit(gpu_lib):
    """A unit cube split along face diagonals, seen from points inside it."""
    v = np.array([[0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 1, 0], [0, 0, 1], [1, 0, 1], [1, 1, 1], [0, 1, 1]],
                 dtype=np.float32) * np.float32(1.3) + np.float32(0.37)
    f = np.array([[0, 3, 2], [0, 2, 1], [4, 5, 6], [4, 6, 7], [0, 1, 5], [0, 5, 4],
                  [3, 7, 6], [3, 6, 2], [0, 4, 7], [0, 7, 3], [1, 2, 6], [1, 6, 5]], dtype=np.uint32)
    rng = np.random.default_rng(7)
    origins = [v.mean(axis=0)] + list(v.min(axis=0) + rng.uniform(0.1, 1.2, (6, 3)))
    _check_no_leak(v, f, origins)


def test_full_scale_bvh_matches_bruteforce(gpu_lib):
    """The benchmark's 1,008,288-triangle scene (512 x 512 heightfield + 200 icospheres of
    frequency 11): closest hits and any-hit answers of the BVH traversal equal a brute-force loop
    over every triangle on the device, for camera rays and for random rays above the terrain.
    Equal distances on different triangles are ties on shared edges and vertices."""
    s = configs.terrain_instances(64, 36)
    assert s.num_triangles == 1008288
    rng = np.random.default_rng(11)
    n = 1024
    # Camera rays: from the camera towards random points of the view.
    cam = np.array([0.0, 30.0, 70.0])
    look = np.array([0.0, 5.0, 0.0]) - cam
    look /= np.linalg.norm(look)
    right = np.cross(look, [0.0, 1.0, 0.0])
    right /= np.linalg.norm(right)
    up = np.cross(right, look)
    a = np.tan(np.radians(30.0))
    u, v = rng.uniform(-a, a, n), rng.uniform(-a * 36 / 64, a * 36 / 64, n)
    d_cam = look[None] + u[:, None] * right[None] + v[:, None] * up[None]
    d_cam /= np.linalg.norm(d_cam, axis=1, keepdims=True)
    # Random rays above the terrain, random directions (many graze the icospheres and the ground).
    o_rnd = np.column_stack([rng.uniform(-45, 45, n), rng.uniform(2, 20, n), rng.uniform(-45, 45, n)])
    d_rnd = rng.normal(size=(n, 3))
    d_rnd /= np.linalg.norm(d_rnd, axis=1, keepdims=True)
    org = np.concatenate([np.broadcast_to(cam, (n, 3)), o_rnd]).astype(np.float32)
    d = np.concatenate([d_cam, d_rnd]).astype(np.float32)
    inf = np.full(len(org), 1e30, np.float32)
    with GpuRenderer(s, abi.default_params(64, 36)) as r:
        print("full-scale BVH: tracing", len(org), "rays", flush=True)
        t, prim, _, _ = r.trace_closest(org, d, inf)
        tb, pb, _, _ = r.trace_closest(org, d, inf, bruteforce=True)
        print("full-scale BVH: brute force done", flush=True)
        occ = r.trace_occluded(org, d, inf)
        hit = pb >= 0
        # Shorter segments: occluded exactly when the brute-force hit lies inside.
        occ_half = r.trace_occluded(org, d, np.where(hit, tb * 0.5, 1e30).astype(np.float32))
        occ_past = r.trace_occluded(org, d, np.where(hit, tb * 1.001, 1e30).astype(np.float32))
    print(f"full-scale BVH: hit rate {hit.mean():.3f}, differing prims {np.sum(prim != pb)}", flush=True)
    assert hit.mean() > 0.5
    assert np.array_equal(prim >= 0, hit)
    assert np.array_equal(t[hit], tb[hit])
    assert np.mean(prim != pb) < 0.01
    assert np.array_equal(occ == 1, hit)
    assert np.all(occ_half[hit] == 0)
    assert np.all(occ_past[hit] == 1)


@pytest.mark.parametrize("count", [1, 63, 1024, 1025, 1 << 17, (1 << 17) + 1, 4 * (1 << 17) + 3])
def test_query_chunks(count):
    """Queries of one slot and of several, whole and partly filled, against the same rays asked for
    in other portions (each ray's answer is its own: equal bits) and against brute force."""
    from concurrent.futures import ThreadPoolExecutor
    rng = np.random.default_rng(count)
    pool = 5000
    org = rng.uniform(-0.3, 0.3, (pool, 3)).astype(np.float32)
    d = rng.normal(size=(pool, 3))
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    tmax = np.where(rng.random(pool) < 0.3, 0.4, 1e30).astype(np.float32)
    pick = rng.integers(0, pool, count)
    with GpuRenderer(configs.cornell_box(8, 8), abi.default_params(8, 8)) as r:
        portions = [slice(k, k + 700) for k in range(0, pool, 700)]
        parts = [r.trace_closest(org[p], d[p], tmax[p]) for p in portions]
        want = [np.concatenate([p[k] for p in parts]) for k in range(4)]
        want_occ = np.concatenate([r.trace_occluded(org[p], d[p], tmax[p]) for p in portions])
        brute = r.trace_closest(org, d, tmax, bruteforce=True)
        assert np.array_equal(want[0], brute[0])
        ask = lambda _: (r.trace_closest(org[pick], d[pick], tmax[pick]), r.trace_occluded(org[pick], d[pick], tmax[pick]))
        got, occ = ask(0)
        assert all(np.array_equal(g, w[pick]) for g, w in zip(got, want))
        assert np.array_equal(occ, want_occ[pick])
    if count == (1 << 17) + 1:  # handles of several threads, each with slots of its own
        def one(_):
            with GpuRenderer(configs.cornell_box(8, 8), abi.default_params(8, 8)) as q:
                return q.trace_closest(org[pick], d[pick], tmax[pick])
        with ThreadPoolExecutor(3) as ex:
            for g in ex.map(one, range(3)):
                assert all(np.array_equal(a, w[pick]) for a, w in zip(g, want))
