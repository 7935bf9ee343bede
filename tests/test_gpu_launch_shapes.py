"""Every launch shape as configured, over few pairs (ogjk_set_exact_lanes keeps
launches over few pairs from widening): results equal the oracle's bit for bit,
and the kernels launched are the ones named."""
import ctypes

import numpy as np
import pytest

import oracle
import ogjk
from ogjk import gen
from parity_utils import compare_f32, compare_f64, oracle_run

pytestmark = pytest.mark.gpu

LANES = [(8, 16), (16, 16), (8, 32), (16, 32), (32, 32), (32, 64), (64, 32), (64, 64)]


@pytest.fixture(scope="module")
def torch_cuda():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.fixture
def exact():
    """Sets a shape exactly; the default shape afterwards."""
    def use(lanes, fused=0, buckets=None, waves=None):
        if buckets is None:
            ogjk.set_config(*lanes, fused)
        else:
            ogjk.set_buckets(*buckets)
        if waves is not None:
            ogjk.set_block_waves(*waves)
        ogjk.set_exact_lanes()
    yield use
    ogjk.set_config(8, 32, 0)


def check(torch, out, ref, mode=oracle.GJK_EPA):
    torch.cuda.synchronize()
    simp = ogjk.simplices_from_device(out["simplices"])
    res = compare_f64(out["f64"].cpu().numpy(), simp, ref, mode)
    assert res["exact"] == res["n"], res


@pytest.fixture(scope="module")
def uneven(torch_cuda):
    b = gen.make(gen.ELLIPSOID, 1500, seed=81, box=1.3, nmin=4, nmax=900)
    ref = oracle_run(oracle.GJK_EPA, b)
    assert (ref.distances < 0).mean() > 0.1
    return b, ref, ogjk.DeviceScene(b, f64="both")


@pytest.mark.parametrize("lanes", LANES)
def test_whole_bodies(torch_cuda, uneven, exact, lanes):
    b, ref, sc = uneven
    sc.drop_clusters()
    exact(lanes)
    check(torch_cuda, sc.collide(oracle.GJK_EPA, b.n_pairs, f64_record=True), ref)


@pytest.mark.parametrize("lanes", LANES)
@pytest.mark.parametrize("cmin", [64, 400])
def test_clustered_bodies(torch_cuda, uneven, exact, lanes, cmin):
    b, ref, sc = uneven
    sc.build_clusters(cmin)
    exact(lanes)
    try:
        check(torch_cuda, sc.collide(oracle.GJK_EPA, b.n_pairs, f64_record=True), ref)
    finally:
        sc.drop_clusters()


def test_clustered_bodies_many_pairs_in_flight(torch_cuda, exact):
    """More waves than the chip has SIMDs, four pairs to a wave: large bodies at
    16 lanes, again and again, against the bodies swept whole."""
    torch = torch_cuda
    b = gen.make(gen.NOISY_SPHERE, 6000, seed=82, nverts=2500, box=1.5)
    sc = ogjk.DeviceScene(b)
    exact((64, 64))
    ref = sc.collide(oracle.GJK_EPA, b.n_pairs, f64_record=True)
    torch.cuda.synchronize()
    sc.build_clusters(1024)
    for lanes in [(16, 32), (8, 16), (16, 64)] * 3:
        exact(lanes)
        out = sc.collide(oracle.GJK_EPA, b.n_pairs, f64_record=True)
        torch.cuda.synchronize()
        assert torch.equal(out["f64"].view(torch.int64)[:, :22], ref["f64"].view(torch.int64)[:, :22])
        assert torch.equal(out["simplices"], ref["simplices"]), lanes


@pytest.fixture(scope="module")
def posed(torch_cuda):
    b = gen.make(gen.ELLIPSOID, 500, seed=83, box=0.0, nmin=8, nmax=300)
    pairs, poses = gen.posed_requests(len(b.cnt), 1, seed=84, kmin=1500, kmax=1500, tbox=1.5)[0]
    pool, off, cnt, pa, pb = oracle.posed_pool(b.coords, b.off, b.cnt, pairs, poses)
    ref = oracle.run(oracle.GJK_EPA, pool, off, cnt, pa, pb, bits=64, nthreads=8)
    assert (ref.distances < 0).mean() > 0.1
    dev = [torch_cuda.from_numpy(a).cuda() for a in (pairs, poses)]
    return ogjk.DeviceScene(b), dev, ref


@pytest.mark.parametrize("lanes", LANES)
@pytest.mark.parametrize("fused", [0, 1])
def test_posed_bodies(torch_cuda, posed, exact, lanes, fused):
    sc, (pairs, poses), ref = posed
    exact(lanes, fused)
    check(torch_cuda, sc.collide_posed(oracle.GJK_EPA, pairs, poses, f64_record=True), ref)


@pytest.mark.parametrize("epa", [16, 32, 64])
def test_fused_and_plain(torch_cuda, uneven, exact, epa):
    b, ref, sc = uneven
    sc.drop_clusters()
    exact((8, epa), fused=1)
    for plain in (False, True, "aos"):
        check(torch_cuda, sc.collide(oracle.GJK_EPA, b.n_pairs, f64_record=True, plain_f64=plain), ref)


def test_epa_alone(torch_cuda, uneven, exact):
    """EPA from a first call's simplices: the same bits whatever the lanes, and
    within the FP32 interface's rounding of the oracle's one call."""
    torch = torch_cuda
    b, ref, sc = uneven
    sc.drop_clusters()
    exact((8, 32))
    first = sc.collide(oracle.GJK, b.n_pairs)
    got = []
    for epa in (16, 32, 64):
        exact((8, epa))
        out = {k: v.clone() if v is not None else None for k, v in first.items()}
        sc.collide(oracle.EPA, b.n_pairs, out=out)
        torch.cuda.synchronize()
        got.append([out[k].cpu().numpy().view(np.uint32) for k in ("simplices", "distances", "normals")])
    for g in got[1:]:
        assert all(np.array_equal(x, y) for x, y in zip(g, got[0]))
    simp = np.ascontiguousarray(got[0][0]).view(ogjk.SIMPLEX_DTYPE).reshape(-1)
    r = compare_f32(simp, got[0][1].view(np.float32), got[0][2].view(np.float32), ref, oracle.GJK_EPA)
    assert r["max_dist_rel"] <= 1e-5, r


@pytest.mark.parametrize("cmin", [None, 256])
@pytest.mark.parametrize("buckets,waves", [
    (([64], [8, 64], [32, 64]), ([2, 1], [1, 2])),
    (([32, 256], [8, 16, 32], [16, 32, 64]), ([4, 2, 1], [2, 4, 1])),
    (([96], [16, 64], [16, 64]), ([1, 4], [4, 4]))])
def test_buckets(torch_cuda, uneven, exact, buckets, waves, cmin):
    b, ref, sc = uneven
    sc.drop_clusters()
    if cmin is not None:
        sc.build_clusters(cmin)
    exact(None, buckets=buckets, waves=waves)
    try:
        check(torch_cuda, sc.collide(oracle.GJK_EPA, b.n_pairs, f64_record=True), ref)
    finally:
        sc.drop_clusters()


class _KernelNode(ctypes.Structure):
    _fields_ = [("block", ctypes.c_uint32 * 3), ("extra", ctypes.c_void_p),
                ("func", ctypes.c_void_p), ("grid", ctypes.c_uint32 * 3),
                ("params", ctypes.c_void_p), ("shared", ctypes.c_uint32)]


def _launches(torch, call):
    """(blocks, threads) of the kernels that call(stream) launches, captured."""
    hip = ctypes.CDLL(next(line.split()[-1] for line in open("/proc/self/maps")
                           if "libamdhip64" in line))
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph, n = ctypes.c_void_p(), ctypes.c_size_t()
    assert hip.hipStreamBeginCapture(ctypes.c_void_p(stream.cuda_stream), 2) == 0  # relaxed
    call(stream.cuda_stream)
    assert hip.hipStreamEndCapture(ctypes.c_void_p(stream.cuda_stream), ctypes.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(graph, nodes, ctypes.byref(n)) == 0
    got = []
    for k in range(n.value):
        p = _KernelNode()
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(nodes[k]), ctypes.byref(p)) == 0
        got.append((p.grid[0], p.block[0]))
    assert hip.hipGraphDestroy(graph) == 0
    return got


@pytest.mark.parametrize("clustered", [False, True])
def test_exact_lanes_are_launched(torch_cuda, exact, clustered):
    """1,024 pairs: 8 GJK lanes take 128 one-wave blocks (1,024 if widened) and 64
    lanes one wave per pair, not two; widening comes back with the next shape."""
    torch = torch_cuda
    n = 1024
    b = gen.make(gen.SPHERE, n, seed=85, nverts=600 if clustered else 64, box=1.3)
    sc = ogjk.DeviceScene(b)
    if clustered:
        sc.build_clusters(512)
    out = sc.outputs(n)
    ws = torch.empty(int(ogjk.lib().ogjk_workspace_bytes(n)), dtype=torch.uint8, device="cuda")

    def call(stream):
        assert ogjk.lib().ogjk_collide_scene_ws(
            oracle.GJK, ctypes.byref(sc.scene), None, n, out["simplices"].data_ptr(),
            out["distances"].data_ptr(), out["normals"].data_ptr(), None, ws.data_ptr(), ws.numel(),
            ctypes.c_void_p(stream)) == 0

    exact((8, 32))
    assert _launches(torch, call) == [(n * 8 // 64, 64)]
    exact((64, 64))
    assert _launches(torch, call) == [(n, 64)]
    ogjk.set_config(8, 32, 0)
    assert _launches(torch, call) == [(n, 128 if clustered else 64)]
    exact(None, buckets=([], [16], [32]), waves=([2], [1]))
    assert _launches(torch, call) == [(n * 16 // 128, 128)]
    ogjk.set_buckets([], [16], [32])
    assert _launches(torch, call) == [(n, 128 if clustered else 64)]
