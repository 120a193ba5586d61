"""GPU tests of nearest-commit queries (query.hip, k_query_nearest) around the sizes at which a launch
changes its form, over one instance (triangles or boxes, no TLAS) and several, against the oracle: few
queries per wave, one for each lane, and (from 327,681 on) waves that claim them and refill their lanes,
in queue order and (from 262,144 on) sorted."""
import numpy as np
import pytest

import luisacompute_amd as lc
from luisacompute_amd import host
from oracle import binding as ob
from parity import compare_query, random_boxes, random_rigid

pytestmark = pytest.mark.gpu
POLICY = dict(surface=lc.QUERY_SURFACE_CUTOUT, cutout=0.7, procedural=lc.QUERY_PROCEDURAL_SPHERE)


def _scene(device, stream, kind):
    rng = np.random.default_rng(5)
    v, t = lc.soup(4000, initseq=11, extent=2.0, sigma=0.3)
    boxes = random_boxes(rng, 500, -1.0, 2.0, 0.1, 0.9)
    gm = host.mesh_from_arrays(device, stream, v, t, option=lc.AccelOption(lc.AccelOption.FAST_BUILD, 1, 0))
    gp = host.procedural_from_aabbs(device, stream, boxes)
    om, op = ob.Mesh(v, t), ob.Procedural(boxes)
    accel, sc = device.create_accel(), ob.Scene()
    layout = {"triangles": [(gm, om, False)], "boxes": [(gp, op, True)],
              "both": [(gm, om, False), (gp, op, True), (gm, om, True), (gp, op, False)] * 8}[kind]
    for i, (g, o, opaque) in enumerate(layout):
        a = random_rigid(rng, -1, 1, 0.5, 1.5)
        m = 0xFF if kind != "both" else (0x01, 0x02, 0x03, 0xFF, 0x00)[i % 5]
        accel.emplace_back(g, a, visibility_mask=m, opaque=opaque)
        sc.add(o, a, m, opaque=opaque)
    stream << accel.build()
    accel._keep = (gm, gp)
    return accel, sc.commit()


@pytest.mark.parametrize("kind", ("triangles", "boxes", "both"))
@pytest.mark.parametrize("n", (1, 3, 63, 64, 65, 4096, 4097, 65537))
def test_query_sizes(device, stream, kind, n):
    print(f"[query] {kind} {n}", flush=True)
    accel, sc = _scene(device, stream, kind)
    rays = lc.rays_as_floats(lc.rays_box_sphere(n, initseq=77, lo=-2.0, hi=3.0))
    for mask in (0xFF, 0x02):
        g = host.query(device, stream, accel, rays, mask, **POLICY)
        compare_query(g, sc.query(rays, mask, **POLICY), sc, rays, mask=mask, **POLICY)


@pytest.fixture(scope="module", params=("triangles", "both"))
def large(device, stream, request):
    """The scene, queries and their answers from launches of at most 50,000, in which each query has a
    lane and no lane a second one."""
    accel, sc = _scene(device, stream, request.param)
    saved = device.ray_sort("closest")
    rays = lc.rays_as_floats(lc.rays_box_sphere(420001, initseq=78, lo=-2.0, hi=3.0))
    device.set_ray_sort("closest", False)
    want = np.concatenate([host.query(device, stream, accel, rays[k:k + 50000], 0xFF, **POLICY)
                           for k in range(0, len(rays), 50000)])
    some = np.random.default_rng(79).choice(len(rays), 5000, replace=False)
    compare_query(want[some], sc.query(rays[some], 0xFF, **POLICY), sc, rays[some], **POLICY)
    if request.param == "both":  # the instances overlap enough to be sorted (262,144 rays have a lane each)
        rb, steps = host.upload(device, stream, host.as_rays(rays[:262144])), []
        for on in (False, True):
            device.set_ray_sort("closest", on)
            steps.append(accel.trace_steps(stream, rb, 262144).wave_steps)
        assert steps[0] != steps[1]
    device.set_ray_sort("closest", saved)
    return accel, rays, want


@pytest.mark.parametrize("sort", (False, True))
@pytest.mark.parametrize("n", (262143, 262144, 327680, 327681, 393217, 420001))
def test_large_queries(device, stream, large, n, sort):
    print(f"[query] {n} sort {sort}", flush=True)
    accel, rays, want = large
    saved, policy = device.ray_sort("closest"), device.trace_steps("closest")
    try:
        device.set_ray_sort("closest", sort)
        for tq, refill in ((3, 48), (1, 63), (4, 0)):
            device.set_trace_steps("closest", tq, refill)
            got = host.query(device, stream, accel, rays[:n], 0xFF, **POLICY)
            np.testing.assert_array_equal(got.view(np.uint32), want[:n].view(np.uint32))
    finally:
        device.set_ray_sort("closest", saved)
        device.set_trace_steps("closest", *policy)
