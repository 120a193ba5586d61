"""GPU tests of the triangle queue that a wave's lanes share (wave_walker.h) at the sizes where it
can go wrong: more triangles per step than the queue holds, leaves of one and of three triangles,
last steps that fill only part of a wave, hits at equal distances and at zero, and instances that
are left, skipped or masked while pairs are queued. Everything is compared with the oracle bit for
bit (hits do not depend on the order in which triangles are tested). The rays are traced as they are,
a launch with eight lanes per ray (oct_walker.h), and repeated past the size at which waves take one
ray per lane and share a queue."""
import numpy as np
import pytest

import luisacompute_amd as lc
from luisacompute_amd import host
from oracle import binding as ob
from parity import compare_any, compare_closest, random_rigid

pytestmark = pytest.mark.gpu
FAST_BUILD = (lc.AccelOption.FAST_BUILD, 1, 0)
FAST_TRACE = (lc.AccelOption.FAST_TRACE, 1, 0)


def _stack(layers, copies=1):
    """`layers` triangles across the z axis, all met by every ray along it; `copies` of each."""
    v = np.zeros((layers, 3, 4), np.float32)
    v[:, :, :2] = [[-8, -8], [8, -8], [0, 12]]
    v[:, :, 2] = (np.arange(layers, dtype=np.float32) // 2)[:, None]
    v = np.repeat(v, copies, axis=0)
    return v.reshape(-1, 4), np.arange(3 * layers * copies, dtype=np.uint32).reshape(-1, 3)


def _rays(n, rng, z=-1.0, t_min=0.0):
    r = np.zeros(n, lc.RAY_DTYPE)
    r["origin"][:, :2] = rng.uniform(-2, 2, (n, 2))
    r["origin"][:, 2] = z
    r["direction"] = [0, 0, 1]
    r["t_min"], r["t_max"] = t_min, 1e30
    return r


def _one_lane_per_ray(device, stream, accel, rays, mask=0xFF):
    """The rays repeated past 65,536: hits of the first round, each later round the same."""
    reps = 70000 // len(rays) + 1
    many = np.tile(rays, reps)
    closest, any_hit = host.trace_closest(device, stream, accel, many, mask), host.trace_any(device, stream, accel, many, mask)
    closest, any_hit = closest.reshape(reps, -1), np.asarray(any_hit).reshape(reps, -1)
    assert (closest.view(np.uint32) == closest[:1].view(np.uint32)).all() and (any_hit == any_hit[:1]).all()
    return closest[0], any_hit[0]


def _check(device, stream, accel, scene, rays, ties_exact=True):
    g = host.trace_closest(device, stream, accel, rays)
    f = lc.rays_as_floats(rays)
    ref = scene.trace_closest2(f)
    compare_closest(g, ref, rays)
    if ties_exact:  # equal distances: the smaller (instance, primitive), as in the oracle
        np.testing.assert_array_equal(g["prim"], ref["prim"])
        np.testing.assert_array_equal(g["inst"], ref["inst"])
    any_hit = host.trace_any(device, stream, accel, rays)
    compare_any(any_hit, scene.trace_any(f))
    closest2, any2 = _one_lane_per_ray(device, stream, accel, rays)
    np.testing.assert_array_equal(closest2.view(np.uint32), g.view(np.uint32))
    np.testing.assert_array_equal(any2, any_hit)
    return g


@pytest.mark.parametrize("option", (FAST_BUILD, FAST_TRACE), ids=("three_per_leaf", "one_per_leaf"))
@pytest.mark.parametrize("layers,n", ((1, 1), (3, 63), (24, 64), (24, 65), (600, 127), (600, 4097)))
def test_more_triangles_than_the_queue_holds(device, stream, option, layers, n):
    """Every ray meets every triangle: a node's leaf slots bring up to 24 per lane at once."""
    v, t = _stack(layers)
    accel = host.single_mesh_accel(device, stream, v, t, option=lc.AccelOption(*option))
    scene = ob.Scene().add(ob.Mesh(v, t)).commit()
    rays = _rays(n, np.random.default_rng(layers + n))
    g = _check(device, stream, accel, scene, rays)
    assert (g["prim"] == 0).all()
    rays["t_min"] = 1.5 + (layers // 4)  # the nearest hits lie inside the stack
    _check(device, stream, accel, scene, rays)


def test_equal_distances_and_zero(device, stream):
    """Three copies of each triangle (the smallest primitive wins), and rays that start on one: a
    hit at t = 0 keeps the sign of its zero."""
    v, t = _stack(40, copies=3)
    accel = host.single_mesh_accel(device, stream, v, t, option=lc.AccelOption(*FAST_BUILD))
    scene = ob.Scene().add(ob.Mesh(v, t)).commit()
    for z, d in ((0.0, 1.0), (0.0, -1.0), (3.0, 1.0), (3.0, -1.0), (-5.0, 1.0)):
        rays = _rays(500, np.random.default_rng(7), z=z)
        rays["direction"][:, 2] = d
        g = _check(device, stream, accel, scene, rays)
        ref = scene.trace_closest2(lc.rays_as_floats(rays))
        hit = ref["prim"] != 0xFFFFFFFF
        np.testing.assert_array_equal(g["committed_ray_t"][hit].view(np.uint32), ref["t"][hit].view(np.uint32))


@pytest.mark.parametrize("count", (2, 9, 300))
@pytest.mark.parametrize("mask", (0xFF, 0x01, 0x80))
def test_instances_left_skipped_and_masked(device, stream, count, mask):
    """Overlapping instances, some masked away and some procedural (skipped by plain traces): lanes
    leave an instance only once its queued triangles are tested, and skip to the TLAS or to the next
    instance of the same leaf."""
    rng = np.random.default_rng(count + mask)
    v, t = _stack(60)
    v2, t2 = lc.icosphere(3)
    gm = [host.mesh_from_arrays(device, stream, v, t, option=lc.AccelOption(*FAST_BUILD)),
          host.mesh_from_arrays(device, stream, v2, t2)]
    om = [ob.Mesh(v, t), ob.Mesh(v2, t2)]
    box = host.procedural_from_aabbs(device, stream, np.array([[-9, -9, -9, 9, 9, 9]], np.float32))
    accel, scene = device.create_accel(lc.AccelOption(*FAST_BUILD)), ob.Scene()
    keep = gm + [box]
    for i in range(count):
        a, m = random_rigid(rng, lo=-6.0, hi=6.0), int(rng.choice([0x01, 0x80, 0x81, 0x00]))
        if i % 7 == 3:  # procedural: an oracle instance that no ray sees
            accel.emplace_back(box, a, 0xFF)
            scene.add(om[0], a, 0x00)
        else:
            accel.emplace_back(gm[i % 2], a, m)
            scene.add(om[i % 2], a, m)
    stream << accel.build()
    accel._keep = keep
    scene.commit()
    rays = lc.rays_box_sphere(5001, initseq=91 + count, lo=-20.0, hi=20.0)
    f = lc.rays_as_floats(rays)
    closest, any_hit = host.trace_closest(device, stream, accel, rays, mask), host.trace_any(device, stream, accel, rays, mask)
    compare_closest(closest, scene.trace_closest2(f, mask), rays)
    compare_any(any_hit, scene.trace_any(f, mask))
    closest2, any2 = _one_lane_per_ray(device, stream, accel, rays, mask)
    np.testing.assert_array_equal(closest2.view(np.uint32), closest.view(np.uint32))
    np.testing.assert_array_equal(any2, any_hit)
