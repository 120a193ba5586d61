"""GPU tests of traversal stacks deeper than their part in LDS, whose spill areas no ordinary tree of
eight children per node reaches in launches of eight lanes per ray (24 entries in LDS). The tree is a
chain: binary nodes over groups of triangles whose Morton codes are the powers of two, every box reaching
all of the others, so that a ray that takes the chain first leaves one entry per level behind it."""
import numpy as np
import pytest

import luisacompute_amd as lc
from luisacompute_amd import host
from oracle import binding as ob
from parity import compare_any, compare_closest, compare_query

pytestmark = pytest.mark.gpu
LEVELS = 30  # bits of a Morton code
PER_CODE = 8  # more than a leaf holds: every group is an inner node, which takes a stack entry
AXIS = np.array([1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0], np.float32)
SWAP = np.array([0, 1, 0, 0, 0, 0, 1, 0, 1, 0, 0, 0], np.float32)


def _chain(rng):
    """Thin triangles centred on the cells 2^k of each axis, and one at the far corner that fixes the
    scale; each reaches 3,000 in every direction, so its box holds all the cells."""
    cells = [np.eye(3)[k % 3] * 2.0 ** (k // 3) for k in range(LEVELS)] + [np.zeros(3)]
    centres = np.repeat(np.array(cells) + 0.25, PER_CODE, axis=0)
    centres = np.concatenate([centres, [[1023.75] * 3]])
    reach = rng.choice([-3000.0, 3000.0], (len(centres), 3))
    # doubled centroids are the sums of a box's corners: the third vertex lies inside the box
    v = np.zeros((len(centres), 3, 4), np.float32)
    v[:, 0, :3], v[:, 1, :3] = centres - reach, centres + reach
    v[:, 2, :3] = centres + reach * rng.uniform(0.9, 0.99, (len(centres), 3))
    return v.reshape(-1, 4), np.arange(3 * len(centres), dtype=np.uint32).reshape(-1, 3)


def _rays(n, rng):
    r = np.zeros(n, lc.RAY_DTYPE)
    r["direction"] = rng.normal(size=(n, 3))
    r["origin"] = rng.uniform(0, 900, (n, 3)) - 2000.0 * np.sign(r["direction"])
    r["t_min"], r["t_max"] = 0.0, 1e30
    return r


@pytest.fixture(scope="module", params=(1, 2, 9))
def scene(device, stream, request):
    verts, tris = _chain(np.random.default_rng(3))
    width = device.build_width()
    try:
        device.set_build_width(2)
        mesh = host.mesh_from_arrays(device, stream, verts, tris, option=lc.AccelOption(lc.AccelOption.FAST_BUILD, 1, 0))
        accel, sc, om = device.create_accel(lc.AccelOption(lc.AccelOption.FAST_BUILD, 1, 0)), ob.Scene(), ob.Mesh(verts, tris)
        for k in range(request.param):
            a = (AXIS, SWAP)[k % 2].copy()
            a[3::4] += k
            accel.emplace_back(mesh, a, opaque=k % 2 == 0)
            sc.add(om, a, opaque=k % 2 == 0)
        stream << accel.build()
        stream.synchronize()
    finally:
        device.set_build_width(width)
    assert mesh.stats().depth >= LEVELS
    assert not any(mesh.validate(stream).values())
    accel._keep = mesh
    return accel, sc.commit()


# eight lanes per ray with 1, 2, 4 and 8 rays per wave; one ray per lane; slots claimed by the waves
@pytest.mark.parametrize("n", (7, 2000, 4001, 30000, 70001, 420001))
def test_stacks_beyond_lds(device, stream, scene, n):
    print(f"[deep] {n} rays", flush=True)
    accel, sc = scene
    some = _rays(1999, np.random.default_rng(5))
    rays = np.resize(some, n)
    k = min(n, len(some))
    f = lc.rays_as_floats(some[:k])
    closest, any_hit = host.trace_closest(device, stream, accel, rays), host.trace_any(device, stream, accel, rays)
    compare_closest(closest[:k], sc.trace_closest2(f), some[:k])
    compare_any(any_hit[:k], sc.trace_any(f))
    policy = dict(surface=lc.QUERY_SURFACE_CUTOUT, cutout=0.9, procedural=lc.QUERY_PROCEDURAL_SPHERE)
    query = host.query(device, stream, accel, rays, **policy)
    compare_query(query[:k], sc.query(f, **policy), sc, f, **policy)
    rb, hb = host.upload(device, stream, rays), device.create_buffer(24, n)
    stream.synchronize()
    rc = lc.lib().lc_hip_accel_trace_closest_noalloc(device.handle, stream.handle, accel.handle, rb.handle, 0, hb.handle,
                                                     0, n, 0xFF)
    assert rc == 0, lc.lib().lc_hip_last_error()
    noalloc = np.zeros(n, lc.HIT_DTYPE)
    stream << hb.copy_to(noalloc) << lc.synchronize()
    for got in (closest, noalloc, query):
        bits = got.view(np.uint32).reshape(n, -1)
        np.testing.assert_array_equal(bits, np.resize(bits[:k], bits.shape))
    np.testing.assert_array_equal(noalloc.view(np.uint32), closest.view(np.uint32))
    np.testing.assert_array_equal(any_hit, np.resize(any_hit[:k], n))
    nodes, _ = accel.trace_count(stream, rb, n)
    assert nodes > 2 * LEVELS * n  # rays visit the whole chain


# queues counted on the device: eight lanes per ray in a launch sized for one ray per lane
@pytest.mark.parametrize("count", (1, 999, 20000, 51200, 98304, 200000))
def test_stacks_beyond_lds_of_counted_queues(device, stream, scene, count):
    print(f"[deep] counted {count} rays", flush=True)
    accel, _ = scene
    rays = np.resize(_rays(1999, np.random.default_rng(6)), 420001)
    rb, cb = host.upload(device, stream, rays), host.upload(device, stream, np.array([count], np.uint32))
    hb, ab = device.create_buffer(24, len(rays)), device.create_buffer(1, len(rays))
    accel.trace_closest_indirect(stream, rb, hb, cb)
    accel.trace_any_indirect(stream, rb, ab, cb)
    hits, occluded = np.zeros(len(rays), lc.HIT_DTYPE), np.zeros(len(rays), np.uint8)
    stream << hb.copy_to(hits) << ab.copy_to(occluded) << lc.synchronize()
    np.testing.assert_array_equal(hits[:count].view(np.uint32),
                                  host.trace_closest(device, stream, accel, rays[:count]).view(np.uint32))
    np.testing.assert_array_equal(occluded[:count], host.trace_any(device, stream, accel, rays[:count]))
