"""GPU tests of captured launches of any size on a stream that ran a larger one: their stacks fit the
working memory that the larger launch left (a capture cannot allocate), whichever form each takes."""
import numpy as np
import pytest

import luisacompute_amd as lc
from luisacompute_amd import host

pytestmark = pytest.mark.gpu
N = 420000  # more rays than lanes are resident
MISS = np.uint32(0xFFFFFFFF)


@pytest.fixture(scope="module", params=("one", "two"))
def scene(device, stream, request):
    verts, tris = lc.soup(60000, initseq=71, extent=20.0, sigma=0.3)
    mesh = host.mesh_from_arrays(device, stream, verts, tris)
    accel = device.create_accel()
    accel.emplace_back(mesh)
    if request.param == "two":
        accel.emplace_back(mesh, np.array([0, -1, 0, 20, 1, 0, 0, 0, 0, 0, 1, 0], np.float32), opaque=False)
    stream << accel.build()
    accel._keep = mesh
    rays = host.upload(device, stream, lc.rays_box_sphere(N, initseq=72, lo=0.0, hi=20.0))
    stream.synchronize()
    return accel, rays


def _trace(kind, accel, stream, rays, out, n):
    if kind == "any":
        accel.trace_any(stream, rays, out, n)
    elif kind == "closest":
        accel.trace_closest(stream, rays, out, n)
    else:
        accel.query(stream, rays, out, n, surface=lc.QUERY_SURFACE_CUTOUT, cutout=0.8)


# launches of 1,024 and 4,096 rays take as many waves as any of their form (few rays each), those of
# 65,536 more waves than are resident at one ray per lane
@pytest.mark.parametrize("kind", ("closest", "any", "query"))
@pytest.mark.parametrize("warm,captured", ((N, 65536), (N, 1024), (65537, 65536), (1025, 1024), (8193, 4096), (4097, 4096),
                                           (65, 64), (2, 1), (393217, 393216), (327681, 327680)))
def test_smaller_captures_fit(device, scene, kind, warm, captured):
    accel, rays = scene
    s = device.create_stream()
    out = device.create_buffer(1 if kind == "any" else 24, N)
    words = (captured + 3) // 4 if kind == "any" else 6 * captured

    def read():
        got = np.zeros(out.count if kind == "any" else 6 * out.count, np.uint8 if kind == "any" else np.uint32)
        s << out.copy_to(got) << lc.synchronize()
        return got[:captured] if kind == "any" else got[:6 * captured]

    print(f"[capture] {kind} {captured} after {warm} ({words} words)", flush=True)
    _trace(kind, accel, s, rays, out, warm)  # the stream's working memory is that of this launch
    want = read()
    with s.capture() as cap:
        _trace(kind, accel, s, rays, out, captured)
    for _ in range(3):
        s << out.copy_from(np.full(out.count * (1 if kind == "any" else 24), 0xA5, np.uint8))
        cap.graph.launch(s)
        np.testing.assert_array_equal(read(), want)
