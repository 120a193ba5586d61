"""GPU tests of the forms that small builds and clusters take: the one-workgroup radix sort around its
sizes (radix.hip, k_rs_small), and the SAH clusters (bvh_build.hip, k_sah_clusters) for geometry whose
splits tie, chain or have no finite cost."""
import numpy as np
import pytest

import luisacompute_amd as lc
from luisacompute_amd import DeviceRadixSort as DRS
from luisacompute_amd import host
from oracle import binding as ob
from parity import compare_any, compare_closest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", (1, 2, 64, 1023, 1024, 1025, 2048, 2049, 4096, 4097, 8191, 8192, 8193))
@pytest.mark.parametrize("begin,end", ((0, 32), (0, 30), (7, 8), (3, 20)))
@pytest.mark.parametrize("values", (True, False), ids=("pairs", "identity"))
def test_small_sorts_are_stable(device, stream, n, begin, end, values):
    rng = np.random.default_rng(n + begin)
    keys = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    keys[rng.random(n) < 0.5] &= np.uint32(0xF0F0)  # many equal digits
    vals = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    kin, vin = host.upload(device, stream, keys), host.upload(device, stream, vals)
    count = host.upload(device, stream, np.array([0, n // 2], np.uint32))
    temp = device.create_buffer(1, DRS.temp_storage_size(n))
    for used, kw in ((n, {}), (n // 2, dict(count_buffer=count, count_index=1))):
        print(f"[sort] n {n} bits [{begin}, {end}) used {used}", flush=True)
        kout, vout = (host.upload(device, stream, np.full(n + 4, 0xA5A5A5A5, np.uint32)) for _ in range(2))
        DRS.sort_pairs(stream, temp, kin, kout, vin if values else None, vout, n, begin, end, **kw)
        got_k, got_v = np.zeros(n + 4, np.uint32), np.zeros(n + 4, np.uint32)
        stream << kout.copy_to(got_k) << vout.copy_to(got_v) << lc.synchronize()
        digit = (keys[:used].astype(np.uint64) >> begin) & ((1 << (end - begin)) - 1)
        order = np.argsort(digit, kind="stable")
        np.testing.assert_array_equal(got_k[:used], keys[:used][order])
        np.testing.assert_array_equal(got_v[:used], vals[:used][order] if values else order.astype(np.uint32))
        assert (got_k[used:] == 0xA5A5A5A5).all() and (got_v[used:] == 0xA5A5A5A5).all()


def _triangles(kind, n, rng):
    v = np.zeros((n, 3, 4), np.float32)
    if kind == "same":  # equal boxes and centroids: every split costs the same
        v[:, :, :3] = [[-1, -1, 0.25], [1, -1, 0.25], [0, 1, 0.25]]
    elif kind == "chain":  # sizes in geometric progression: the cheapest split takes one off the end
        size = np.float32(1.3) ** -np.arange(n, dtype=np.float32).clip(0, 60)
        v[:, :, :3] = np.array([[-1, -1, 0], [1, -1, 0], [0, 1, 0]], np.float32) * size[:, None, None]
        v[:, :, 2] = np.linspace(-1, 1, n, dtype=np.float32)[:, None]
    elif kind == "row":  # centroids along one axis only
        v[:, :, :3] = rng.normal(0, 0.02, (n, 3, 3))
        v[:, :, 0] += np.linspace(-2, 2, n, dtype=np.float32)[:, None]
    else:  # a box area beyond the largest float: no split has a finite cost
        v[:, :, :3] = rng.normal(0, 0.3, (n, 3, 3))
        v[0, :, :3] = [[-3e19, -3e19, 2], [3e19, -3e19, 2], [0, 3e19, 2]]
    return v.reshape(-1, 4), np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)


@pytest.mark.parametrize("kind", ("same", "chain", "row", "huge"))
@pytest.mark.parametrize("n", (3, 63, 64, 65, 1000, 3000))
def test_sah_clusters_of_hard_geometry(device, stream, kind, n):
    print(f"[sah] {kind} {n}", flush=True)
    verts, tris = _triangles(kind, n, np.random.default_rng(n))
    mesh = host.mesh_from_arrays(device, stream, verts, tris)
    accel = device.create_accel()
    accel.emplace_back(mesh)
    stream << accel.build()
    errs = mesh.validate(stream)
    assert not any(errs.values()), errs
    assert mesh.stats().leaf_primitive_count == n
    rays = lc.rays_orbit_to_ball(2000, orbit=4.0)
    scene, f = ob.single_mesh_scene(verts, tris), lc.rays_as_floats(rays)
    compare_closest(host.trace_closest(device, stream, accel, rays), scene.trace_closest2(f), rays)
    compare_any(host.trace_any(device, stream, accel, rays), scene.trace_any(f))


@pytest.mark.parametrize("n,extent", ((64, 0.125), (64, 0.5), (1000, 0.25)))
def test_sah_clusters_far_from_the_origin(device, stream, n, extent):
    """The same geometry near the origin and at a coordinate of 10,000, its vertices multiples of 2^-9,
    so that positions, centroids and extents are exact in both places: the trees are equally good (rays
    visit as many nodes and test as many triangles) however close the centroids lie for their size."""
    rng = np.random.default_rng(n)
    grid = int(extent * 512)
    at = rng.integers(0, grid, (n, 1, 3)) + rng.integers(-2, 3, (n, 3, 3))
    rays = np.zeros(20000, lc.RAY_DTYPE)
    origin = rng.integers(-grid, 2 * grid, (len(rays), 3))
    target = rng.uniform(0, extent, (len(rays), 3))
    rays["direction"] = (target - origin / 512.0).astype(np.float32)
    rays["t_min"], rays["t_max"] = 0.0, 1e30
    work = []
    for offset in (0, 10000):
        v = np.zeros((3 * n, 4), np.float32)
        v[:, :3] = (at / 512.0 + offset).reshape(-1, 3)
        mesh = host.mesh_from_arrays(device, stream, v, np.arange(3 * n, dtype=np.uint32).reshape(-1, 3))
        accel = device.create_accel()
        accel.emplace_back(mesh)
        stream << accel.build()
        rays["origin"] = (origin / 512.0 + offset).astype(np.float32)
        work.append(accel.trace_count(stream, host.upload(device, stream, rays), len(rays)))
        print(f"[far] {n} triangles over {extent} at {offset}: nodes and triangles {work[-1]}", flush=True)
        errs = mesh.validate(stream)
        assert not any(errs.values()), errs
    near, far = np.array(work, np.float64)
    assert (far <= 1.02 * near).all(), work
