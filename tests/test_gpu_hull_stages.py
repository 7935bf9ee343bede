"""Hull builds where the device code changes hands: a call over few clouds and
one over many (other launches), clouds at the sizes and face counts where one
working set ends and the next begins, and the states saved in between, against
the C oracle.  The oracle's face counts show that each hand-over happens: a
list that ends with more faces than a working set holds has outgrown it."""
import ctypes
import time

import numpy as np
import pytest

import oracle
import ogjk
from test_gpu_hull_dense import build, ellipsoid, torch_cuda  # noqa: F401

pytestmark = pytest.mark.gpu

# Faces that the working sets hold: 16 lanes, a wave, the wave of a call over few
# clouds, a wave with more room, a block with planes, a block with vertex ids.
ROOM = [96, 160, 512, 880, 3584, 14336]
FEW_CLOUDS, FEW_POINTS, BLOCK_POINTS = 256, 32, 1024


def inside(n, seed, scale=1.0):
    """A cube's corners and n - 8 points in it: a hull of 12 faces or so."""
    rng = np.random.default_rng([n, seed])
    p = rng.uniform(-0.9, 0.9, (n, 3))
    p[rng.permutation(n)[:8]] = [[x, y, z] for x in (-1, 1) for y in (-1, 1) for z in (-1, 1)]
    return (p * scale).astype(np.float32)


def sphere(n, seed):
    u = np.random.default_rng([n, seed]).normal(size=(n, 3))
    return (u / np.linalg.norm(u, axis=1, keepdims=True)).astype(np.float32)


GROUPS = {
    # small clouds past their 16 lanes' faces, and within
    "few points": [ellipsoid(32, 46, 0.03), ellipsoid(32, 0, 1.0), sphere(32, 1), sphere(33, 2)],
    # 2 n - 4 faces around a wave's, an alone wave's and the larger wave's room
    "edges": [sphere(n, 3) for n in (80, 81, 82, 83, 255, 256, 257, 258, 259, 441, 442, 443, 444)],
    "sizes": [sphere(n, 4) for n in (511, 512, 513, 1023, 1024, 1025, 1200)],
    # face lists that blow up: bits and hash set, planes and ids, past both
    "dense": [ellipsoid(*c) for c in ((256, 0, 0.12), (512, 39, 0.2), (436, 6, 0.2), (800, 1, 0.35),
                                      (800, 9, 0.35), (600, 24, 0.5), (256, 20, 0.12),
                                      (200, 10, 0.06))],
    "inside": [inside(n, 5) for n in (8, 33, 64, 127, 500, 1025, 5000, 70000)],
}


@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("group", GROUPS)
def test_stages(torch_cuda, group, many):  # noqa: F811
    clouds = list(GROUPS[group])
    caps = [17000 if len(c) < 2000 else 4096 for c in clouds]
    if many:  # small clouds between them
        rng = np.random.default_rng(9)
        for k in range(FEW_CLOUDS + 40):
            c = sphere(int(rng.integers(3, 60)), 100 + k)
            at = int(rng.integers(0, len(clouds) + 1))
            clouds.insert(at, c)
            caps.insert(at, 4 * len(c) + 16)
    assert (len(clouds) > FEW_CLOUDS) == many
    refs = [oracle.build_hull(p, cap=c) for p, c in zip(clouds, caps)]
    lists, marks = build(torch_cuda, clouds, caps)
    for p, ref, got, left in zip(clouds, refs, lists, marks):
        assert ref is not None
        assert np.array_equal(got, ref), len(p)
        # the upper part of the workspace is written over global memory alone
        wave = ROOM[3] if many else ROOM[2]
        if len(p) > 65536:
            assert not left
        elif len(p) > BLOCK_POINTS:
            assert left == (len(ref) <= wave), (len(p), len(ref))
        elif len(ref) <= ROOM[5]:
            assert left, (len(p), len(ref))
    faces = [len(r) for r in refs]
    if group == "few points":
        assert any(len(p) <= FEW_POINTS and f > ROOM[0] for p, f in zip(clouds, faces))
    if group == "edges":
        for r in (ROOM[1], ROOM[2], ROOM[3]):
            assert r in faces and any(r < f <= r + 4 for f in faces), r
    if group == "dense":
        for r in ROOM[3:]:
            assert any(f > r for f in faces), r
        # past the planes' room on both sides of the edge set's change
        assert any(f > ROOM[4] and len(p) <= 512 for p, f in zip(clouds, faces))
        assert any(f > ROOM[4] and len(p) > 512 for p, f in zip(clouds, faces))


def test_capacities_between_stages(torch_cuda):  # noqa: F811
    """Clouds whose capacity ends just under, at and over their face count, in
    each working set: the overflow flag is the oracle's."""
    shapes = [sphere(60, 6), sphere(200, 6), sphere(400, 6), sphere(700, 6), ellipsoid(512, 39, 0.2),
              ellipsoid(800, 9, 0.35)]
    clouds, caps = [], []
    for p in shapes:
        f = len(oracle.build_hull(p, cap=17000))
        for c in (f - 1, f, f + 1, f + 100):
            clouds.append(p)
            caps.append(c)
    for fill in (0, FEW_CLOUDS):
        cs, cp = clouds + [sphere(20, 7)] * fill, caps + [96] * fill
        lists, _ = build(torch_cuda, cs, cp)
        for p, c, got in zip(cs, cp, lists):
            ref = oracle.build_hull(p, cap=c)
            if ref is None:
                assert isinstance(got, int) and got == -1, (len(p), c)
            else:
                assert np.array_equal(got, ref), (len(p), c)


def _device_args(torch, clouds, caps):
    cnt = torch.tensor([len(c) for c in clouds], dtype=torch.int32, device="cuda")
    off = torch.cumsum(cnt.long(), 0) - cnt
    fo = torch.zeros(len(clouds) + 1, dtype=torch.int64, device="cuda")
    fo[1:] = torch.cumsum(torch.tensor(caps, device="cuda"), 0)
    total = int(sum(caps))
    pts = torch.from_numpy(np.concatenate(clouds)).cuda()
    faces = torch.empty((total, 3), dtype=torch.int32, device="cuda")
    nf = torch.empty(len(clouds), dtype=torch.int32, device="cuda")
    ws = torch.empty(12 * total, dtype=torch.uint8, device="cuda")
    args = [pts.data_ptr(), off.data_ptr(), cnt.data_ptr(), len(clouds), fo.data_ptr(), total,
            faces.data_ptr(), nf.data_ptr(), ws.data_ptr(), ws.numel()]
    return args, nf, (pts, off, cnt, fo, faces, ws)


@pytest.mark.parametrize("n", [1, 3, 256])
def test_few_clouds_are_one_launch(torch_cuda, n):  # noqa: F811
    """A build of few clouds is short: each launch of it counts (14 of 55 us
    for one cloud of 8 points built by six)."""
    torch = torch_cuda
    args, nf, keep = _device_args(torch, [sphere(8, k) for k in range(n)], [48] * n)
    hip = ctypes.CDLL(next(line.split()[-1] for line in open("/proc/self/maps")
                           if "libamdhip64" in line))
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph, nodes = ctypes.c_void_p(), ctypes.c_size_t()
    assert hip.hipStreamBeginCapture(ctypes.c_void_p(stream.cuda_stream), 2) == 0  # relaxed
    st = ogjk.lib().ogjk_build_hulls(*args, ctypes.c_void_p(stream.cuda_stream))
    assert hip.hipStreamEndCapture(ctypes.c_void_p(stream.cuda_stream), ctypes.byref(graph)) == 0
    assert st == 0
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(nodes)) == 0
    assert hip.hipGraphDestroy(graph) == 0
    assert nodes.value == 1


def _seconds(torch, clouds, cap):
    args, nf, keep = _device_args(torch, clouds, [cap] * len(clouds))
    best = 1e9
    for _ in range(6):
        torch.cuda.synchronize()
        t = time.perf_counter()
        for _ in range(5):
            assert ogjk.lib().ogjk_build_hulls(*args, None) == 0
        torch.cuda.synchronize()
        best = min(best, time.perf_counter() - t)
    return best, nf


@pytest.mark.parametrize("points", [400, 1024])
def test_many_inner_point_clouds_run_side_by_side(torch_cuda, points):  # noqa: F811
    """3,000 clouds with most points inside take little longer than one: a
    wave each (1.3 times here; 12 times with a block of 16 waves per cloud)."""
    torch = torch_cuda
    shapes = [inside(points, k) for k in range(100)]
    one, nf1 = _seconds(torch, shapes[:1], 4 * points + 16)
    many, nf = _seconds(torch, shapes * 30, 4 * points + 16)
    print(f"\n[{points} points] one cloud {one / 5 * 1e6:.0f} us, 3,000 {many / 5 * 1e6:.0f} us",
          flush=True)
    assert (nf1 > 0).all() and (nf > 0).all()
    assert many < 4 * one


def test_large_clouds_run_side_by_side(torch_cuda):  # noqa: F811
    """300 clouds past the LDS working sets take no longer than 100: a wave
    each, all in flight (1.4 times with the waves of one block to a cloud)."""
    torch = torch_cuda
    shapes = [sphere(1100, k) for k in range(100)]
    few, _ = _seconds(torch, shapes, 4 * 1100 + 16)
    more, _ = _seconds(torch, shapes * 3, 4 * 1100 + 16)
    print(f"\n100 clouds {few / 5 * 1e3:.1f} ms, 300 {more / 5 * 1e3:.1f} ms", flush=True)
    assert more < 1.2 * few
