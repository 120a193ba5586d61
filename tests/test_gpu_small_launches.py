"""GPU tests of how a trace launch hands out its rays (trace_grid, k_trace, k_trace_oct): launches
that give every ray eight lanes, with 1 to 8 rays per wave, or one lane, with 64 rays per wave,
against larger ones whose waves claim queue slots, around the sizes where the form changes, in queue
order and sorted. Every size gives the hits of the large launch, ray by ray, and writes nothing past
its last ray."""
import numpy as np
import pytest

import luisacompute_amd as lc
from luisacompute_amd import host
from oracle import binding as ob
from parity import compare_any, compare_closest

pytestmark = pytest.mark.gpu
N = 420000  # more rays than lanes are resident (256 CUs x 24 waves x 64)
SIZES = (1, 3, 4, 5, 63, 64, 65, 1023, 1025, 2049, 4095, 4096, 4097, 8191, 8193, 65535, 65536, 65537, 262143, 262144, 262145, 393216, 393217, N)


@pytest.fixture(scope="module", params=("one", "two"))
def scene(device, stream, request):
    """One instance, or two of overlapping geometry (a two-level accel whose queues are sorted)."""
    verts, tris = lc.soup(30000, initseq=71, extent=20.0, sigma=0.3)
    affines = [np.array([1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0], np.float32)]
    if request.param == "two":
        affines.append(np.array([0, -1, 0, 20, 1, 0, 0, 0, 0, 0, 1, 0], np.float32))
    mesh = host.mesh_from_arrays(device, stream, verts, tris)
    accel, om = device.create_accel(), ob.Mesh(verts, tris)
    sc = ob.Scene()
    for a in affines:
        accel.emplace_back(mesh, a)
        sc.add(om, a)
    stream << accel.build()
    accel._keep = mesh
    sc.commit()
    rays = lc.rays_box_sphere(N, initseq=72, lo=0.0, hi=20.0)
    rb = host.upload(device, stream, rays)
    f = lc.rays_as_floats(rays[:20000])
    closest, any_hit = host.trace_closest(device, stream, accel, rays), host.trace_any(device, stream, accel, rays)
    compare_closest(closest[:20000], sc.trace_closest2(f), rays[:20000])
    compare_any(any_hit[:20000], sc.trace_any(f))
    return accel, rb, closest, any_hit


@pytest.mark.parametrize("block,sort", ((64, False), (64, True), (256, False)))
def test_every_size_gives_the_same_hits(device, stream, scene, block, sort):
    accel, rb, closest, any_hit = scene
    saved = {k: (device.trace_config(k), device.ray_sort(k)) for k in ("closest", "any")}
    hb, ab = device.create_buffer(24, N + 16), device.create_buffer(1, N + 16)
    count = device.create_buffer(4, 1)
    try:
        for k, (c, _) in saved.items():
            device.set_trace_config(k, block, c["lds_stack"], c["steps"], c["blocks_per_cu"])
            device.set_ray_sort(k, sort)
        for n in SIZES:
            print(f"[launch] block {block} sort {sort} rays {n}", flush=True)
            blank = np.full(N + 16, 0xA5, np.uint8)
            hits, occluded = np.full((N + 16) * 24, 0xA5, np.uint8).view(lc.HIT_DTYPE), blank.copy()
            stream << hb.copy_from(hits) << ab.copy_from(occluded)
            accel.trace_closest(stream, rb, hb, n)
            accel.trace_any(stream, rb, ab, n)
            stream << hb.copy_to(hits) << ab.copy_to(occluded) << lc.synchronize()
            np.testing.assert_array_equal(hits[:n].view(np.uint32), closest[:n].view(np.uint32))
            np.testing.assert_array_equal(occluded[:n], any_hit[:n])
            assert (hits[n:].view(np.uint8) == 0xA5).all() and (occluded[n:] == 0xA5).all()
        # the length read on the device: fewer rays than the launch has lanes for
        for capacity, n in ((4096, 0), (4096, 77), (65537, 1000), (N, 0), (N, 3), (N, 5000), (N, 40961),
                            (N, 51200), (N, 51201), (N, 61441), (N, 81921), (N, 98304), (N, 98305)):
            print(f"[launch] block {block} sort {sort} capacity {capacity} rays {n}", flush=True)
            hits = np.full((N + 16) * 24, 0xA5, np.uint8).view(lc.HIT_DTYPE)
            stream << hb.copy_from(hits) << count.copy_from(np.array([n], np.uint32))
            accel.trace_closest_indirect(stream, rb, hb, count, capacity=capacity)
            stream << hb.copy_to(hits) << lc.synchronize()
            occluded = blank.copy()
            stream << ab.copy_from(occluded)
            accel.trace_any_indirect(stream, rb, ab, count, capacity=capacity)
            stream << ab.copy_to(occluded) << lc.synchronize()
            np.testing.assert_array_equal(hits[:n].view(np.uint32), closest[:n].view(np.uint32))
            assert (hits[n:].view(np.uint8) == 0xA5).all()
            np.testing.assert_array_equal(occluded[:n], any_hit[:n])
            assert (occluded[n:] == 0xA5).all()
    finally:
        for k, (c, srt) in saved.items():
            device.set_trace_config(k, c["block"], c["lds_stack"], c["steps"], c["blocks_per_cu"])
            device.set_ray_sort(k, srt)
