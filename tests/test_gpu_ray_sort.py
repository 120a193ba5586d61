"""GPU tests of when a trace sorts its rays and of the sorted queue itself, at sizes that are sorted
(262,144 rays and more). That a launch sorts shows in its counting run: the waves take other rays
together, so they take other numbers of steps for the same visits and tests."""
import numpy as np
import pytest

import luisacompute_amd as lc
from luisacompute_amd import host
from oracle import binding as ob
from parity import compare_any, compare_closest

pytestmark = pytest.mark.gpu
N = 300001  # sorted, and every ray has a lane from the start: the counting run repeats exactly


@pytest.fixture
def sorting(device):
    """Sets ray sorting of both trace kinds; the test's end puts back what was set."""
    saved = {k: device.ray_sort(k) for k in ("closest", "any")}
    yield lambda on: [device.set_ray_sort(k, on) for k in saved]
    for k, v in saved.items():
        device.set_ray_sort(k, v)


def _sorts(stream, accel, rb, n, sorting, any_hit=False):
    steps = []
    for on in (False, True, False):
        sorting(on)
        st = accel.trace_steps(stream, rb, n, any_hit=any_hit)
        steps.append((st.wave_steps, st.nodes_visited))
    assert steps[0] == steps[2]
    return steps[0] != steps[1]


def _scene(device, stream, kind):
    verts, tris = lc.soup(20000, initseq=71, extent=20.0, sigma=0.4)
    if kind == "flat":
        verts[:, 2] = 5.0
    mesh = host.mesh_from_arrays(device, stream, verts, tris)
    at = {"one": [(0, 0, 0)], "overlapping": [(0, 0, 0), (1, 0, 0)], "flat": [(0, 0, 0), (1, 0, 0)],
          "distant": [(0, 0, 0), (1, 0, 0), (900, 900, 900)],
          "distant ones": [(0, 0, 0), (1, 0, 0)] + [(900 + 30 * k, -900, 900) for k in range(12)],
          "groups": [(150 * (k % 3) + j, 150 * (k // 3), 0) for k in range(9) for j in range(3)],
          "side by side": [(25 * (k % 3), 25 * (k // 3), 0) for k in range(9)]}[kind]
    accel, sc, om = device.create_accel(), ob.Scene(), ob.Mesh(verts, tris)
    for x, y, z in at:
        s = 0.05 if x >= 900 else 1.0
        a = np.array([s, 0, 0, x, 0, s, 0, y, 0, 0, s, z], np.float32)
        accel.emplace_back(mesh, a)
        sc.add(om, a)
    stream << accel.build()
    accel._keep = mesh
    return accel, sc.commit()


@pytest.mark.parametrize("kind,n,sorts", (
    ("one", N, True), ("one", 262144, True), ("one", 262143, False), ("overlapping", N, True), ("overlapping", 262143, False),
    ("flat", N, True), ("distant", N, True), ("distant ones", N, True), ("side by side", N, False), ("groups", N, False)))
def test_which_launches_sort(device, stream, sorting, kind, n, sorts):
    print(f"[sort] {kind} {n}", flush=True)
    accel, sc = _scene(device, stream, kind)
    rays = lc.rays_box_sphere(n, initseq=72, lo=-5.0, hi=25.0)
    rb = host.upload(device, stream, rays)
    for any_hit in (False, True):
        assert _sorts(stream, accel, rb, n, sorting, any_hit) == sorts
    got = []
    for on in (False, True):
        sorting(on)
        got.append((host.trace_closest(device, stream, accel, rays), host.trace_any(device, stream, accel, rays)))
    np.testing.assert_array_equal(got[0][0].view(np.uint32), got[1][0].view(np.uint32))
    np.testing.assert_array_equal(got[0][1], got[1][1])
    some = np.random.default_rng(n).choice(n, 3000, replace=False)
    f = lc.rays_as_floats(rays[some])
    compare_closest(got[1][0][some], sc.trace_closest2(f), rays[some])
    compare_any(got[1][1][some], sc.trace_any(f))


@pytest.mark.parametrize("kind", ("one", "overlapping"))
@pytest.mark.parametrize("any_hit", (False, True), ids=("closest", "any"))
def test_captured_sorts_follow_the_count(device, sorting, kind, any_hit):
    """A graph of a sorted trace of a queue counted on the device replays with other counts, eager work
    between the replays: each sorts and traces the first rays, as many as are counted then."""
    s = device.create_stream()
    accel, _ = _scene(device, s, kind)
    rays = lc.rays_box_sphere(N, initseq=74, lo=-5.0, hi=25.0)
    rb, cb = host.upload(device, s, rays), device.create_buffer(4, 1)
    size = 1 if any_hit else 24
    out = device.create_buffer(size, N)

    def read():
        got = np.zeros(N * size, np.uint8)
        s << out.copy_to(got) << lc.synchronize()
        return got.reshape(N, size)

    def trace():
        (accel.trace_any_indirect if any_hit else accel.trace_closest_indirect)(s, rb, out, cb)

    sorting(False)
    s << cb.copy_from(np.array([N], np.uint32))
    trace()
    want = read()
    sorting(True)
    assert _sorts(s, accel, rb, N, lambda on: sorting(on), any_hit)
    sorting(True)
    trace()  # eager first: the stream then holds the sort's working memory, without which a capture does not sort
    np.testing.assert_array_equal(read(), want)
    with s.capture() as cap:
        trace()
    sorting(False)  # the graph keeps what it recorded
    for count in (N, 0, 1, 4096, 65537, 262144, N - 1, N + 5, 77):
        print(f"[captured sort] {kind} any {any_hit} count {count}", flush=True)
        s << cb.copy_from(np.array([count], np.uint32)) << out.copy_from(np.full(N * size, 0xA5, np.uint8))
        cap.graph.launch(s)
        got = read()
        np.testing.assert_array_equal(got[:count], want[:count])
        assert (got[count:] == 0xA5).all()
        host.trace_closest(device, s, accel, rays[:1000])
