"""GPU tests of the traversal step policy (when queued triangles go first, early refill, refill
interval), of how waves claim their rays, and of the counting run's lane accounting: every policy gives
the same hits bit for bit, and the accounting is consistent with itself and with the plain counting run.
One workgroup per CU has fewer lanes than there are rays, so waves claim queue slots and refill."""
import numpy as np
import pytest

import luisacompute_amd as lc
from luisacompute_amd import host
from oracle import binding as ob
from parity import compare_any, compare_closest

pytestmark = pytest.mark.gpu
KINDS = ("closest", "any")


@pytest.fixture(scope="module", params=("one", "two"))
def soup(device, stream, request):
    """One instance, or three (two levels), one of them seen by no ray."""
    verts, tris = lc.soup(200000, initseq=61, extent=20.0, sigma=0.3)
    rays = lc.rays_box_sphere(1 << 17, initseq=62, lo=0.0, hi=20.0)
    mesh, om = host.mesh_from_arrays(device, stream, verts, tris), ob.Mesh(verts, tris)
    accel, sc = device.create_accel(), ob.Scene()
    at = [(np.array([1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0], np.float32), 0xFF)]
    if request.param == "two":
        at += [(np.array([0, -1, 0, 20, 1, 0, 0, 0, 0, 0, 1, 0], np.float32), 0xFF),
               (np.array([1, 0, 0, 5, 0, 1, 0, 5, 0, 0, 1, 5], np.float32), 0)]
    for a, mask in at:
        accel.emplace_back(mesh, a, mask)
        sc.add(om, a, mask)
    stream << accel.build()
    accel._keep = mesh
    return accel, rays, host.upload(device, stream, rays), sc.commit()


@pytest.fixture
def policy(device):
    """set(blocks_per_cu, steps, tri_quarters, refill_below, chunk, segments) for both trace kinds; what
    was set before comes back at the end of the test."""
    saved = {k: (device.trace_config(k), device.trace_steps(k), device.fetch(k)) for k in KINDS}

    def put(blocks_per_cu, steps, tri_quarters, refill_below, chunk, segments):
        for k in KINDS:
            c = saved[k][0]
            device.set_trace_config(k, c["block"], c["lds_stack"], steps, blocks_per_cu)
            device.set_trace_steps(k, tri_quarters, refill_below)
            device.set_fetch(k, chunk, segments)

    yield put
    for k, (c, st, fetch) in saved.items():
        device.set_trace_config(k, c["block"], c["lds_stack"], c["steps"], c["blocks_per_cu"])
        device.set_trace_steps(k, *st)
        device.set_fetch(k, *fetch)


def test_step_policies_give_the_same_hits(device, stream, soup, policy):
    accel, rays, rb, scene = soup
    want = host.trace_closest(device, stream, accel, rays)
    want_any = host.trace_any(device, stream, accel, rays)
    f = lc.rays_as_floats(rays[:20000])
    assert compare_closest(want[:20000], scene.trace_closest2(f), rays[:20000])["hits"] > 100
    compare_any(want_any[:20000], scene.trace_any(f))
    for bpc in (0, 1):  # a lane for every ray; slots claimed and lanes refilled
        for tq, refill, steps in ((1, 0, 16), (1, 32, 32), (2, 48, 8), (3, 0, 4), (4, 63, 1)):
            for chunk, segments in ((0, 1), (0, 8), (64, 1), (64, 8), (256, 8)):
                print(f"[policy] blocks_per_cu={bpc} tri_quarters={tq} refill_below={refill} steps={steps} "
                      f"chunk={chunk} segments={segments}", flush=True)
                policy(bpc, steps, tq, refill, chunk, segments)
                got = host.trace_closest(device, stream, accel, rays)
                np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
                np.testing.assert_array_equal(host.trace_any(device, stream, accel, rays), want_any)
    with pytest.raises(lc.LCError):
        device.set_trace_steps("closest", 0, 0)
    with pytest.raises(lc.LCError):
        device.set_trace_steps("closest", 2, 65)


def test_lane_accounting(device, stream, soup, policy):
    """Node visits and triangle tests equal the plain counting run's; each is at most one per live
    lane-iteration; live lane-iterations fit in the waves' lane slots; refills happen where waves claim
    their rays, and more of them with early refill than without."""
    accel, rays, rb, _ = soup
    n = len(rays)
    rounds, live = [], []
    for bpc, refill in ((0, 48), (1, 0), (1, 48)):
        policy(bpc, 32, 3, refill, 64, 8)
        nodes, tris = accel.trace_count(stream, rb, n)
        st = accel.trace_steps(stream, rb, n)
        print(f"[lanes] nodes {st.nodes_visited} tris {st.triangles_tested} live {st.live_lane_steps} "
              f"waves {st.wave_steps} refills {st.refill_rounds}", flush=True)
        if bpc == 0:
            assert (st.nodes_visited, st.triangles_tested) == (nodes, tris)
        else:  # a little of the work depends on which rays happen to share a wave (when a hit culls)
            assert abs(st.nodes_visited - nodes) <= 0.02 * nodes and abs(st.triangles_tested - tris) <= 0.02 * tris
        assert nodes > n and tris > 0
        assert st.nodes_visited + st.triangles_tested <= st.live_lane_steps <= 64 * st.wave_steps
        assert st.refill_rounds > 0 and st.wave_steps >= st.refill_rounds
        rounds.append(st.refill_rounds)
        live.append(st.live_lane_steps / (64 * st.wave_steps))
        sa = accel.trace_steps(stream, rb, n, any_hit=True)
        assert sa.nodes_visited + sa.triangles_tested <= sa.live_lane_steps <= 64 * sa.wave_steps
    assert rounds[2] > rounds[1]
    assert live[2] > live[0] + 0.1  # lanes whose ray ended take another
