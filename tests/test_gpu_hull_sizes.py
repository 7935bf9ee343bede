"""Hull builds at the sizes where the device code changes hands (half a wave,
a wave, a block, the larger block, the general kernel) and where a working set
outgrows its LDS and the cloud passes to the next, against the C oracle: face
lists, order and overflow flags are equal, and so are the moments' bits."""
import numpy as np
import pytest

import oracle
import ogjk

pytestmark = pytest.mark.gpu

SIZES = [3, 4, 5, 31, 32, 33, 34, 127, 128, 129, 130, 511, 512, 513, 1023, 1024, 1025]


@pytest.fixture(scope="module")
def torch_cuda():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def cloud(kind, n, rng):
    u = rng.normal(size=(n, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    if kind == "ball":  # many points inside: insertions that see no face
        p = u * rng.uniform(0, 1, (n, 1)) ** (1 / 3)
    elif kind == "ellipsoid":  # an elongated surface: face lists past 4 n + 16
        p = u * np.array([0.3, 1.1, 2.0])
    elif kind == "lattice":  # repeated and coplanar points
        p = rng.integers(-2, 3, (n, 3)) * 0.25
    else:
        p = u
    return p.astype(np.float32)


@pytest.mark.parametrize("caps", ["fit", "4n", "huge"])
@pytest.mark.parametrize("kind", ["sphere", "ball", "ellipsoid", "lattice"])
def test_sizes(torch_cuda, kind, caps):
    torch = torch_cuda
    rng = np.random.default_rng(7)
    clouds = [cloud(kind, n, rng) for n in SIZES for _ in range(1 if n > 200 else 3)]
    order = rng.permutation(len(clouds))
    clouds = [clouds[i] for i in order]
    # fit: just what a simple hull needs (2 n - 4), so dense ones overflow; huge: the
    # working sets, not the capacity, are what a cloud outgrows
    cap = [{"fit": max(2 * len(c) - 4, 0), "4n": 4 * len(c) + 16, "huge": 40 * len(c) + 64}[caps]
           for c in clouds]
    cnt = np.array([len(c) for c in clouds], np.int32)
    off = np.concatenate([[0], np.cumsum(cnt)[:-1]]).astype(np.int64)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    pts, off, cnt = dev(np.concatenate(clouds)), dev(off), dev(cnt)
    faces, face_off, nfaces = ogjk.build_hulls(pts, off, cnt, dev(np.array(cap, np.int64)))
    mo, com, k = ogjk.hull_moments(pts, off, faces, face_off, nfaces)
    torch.cuda.synchronize()
    f, fo, nf = faces.cpu().numpy(), face_off.cpu().numpy(), nfaces.cpu().numpy()
    mo, com, k = mo.cpu().numpy(), com.cpu().numpy(), k.cpu().numpy()
    over = 0
    for i, p in enumerate(clouds):
        ref = oracle.build_hull(p, cap=cap[i])
        if ref is None:
            assert nf[i] == -1, (i, len(p))
            over += 1
            continue
        assert nf[i] == len(ref), (i, len(p))
        assert np.array_equal(f[fo[i]:fo[i] + nf[i]], ref), (i, len(p))
        m = oracle.hull_moments(p, ref)
        assert np.array_equal(mo[i].view(np.uint64), m.view(np.uint64)), (i, len(p))
        assert np.array_equal(com[i].view(np.uint32), oracle.hull_com(m).view(np.uint32)), i
        assert np.array_equal(k[i].view(np.uint32), oracle.hull_inertia_k(m).view(np.uint32)), i
    print(f"\n[{kind} {caps}] {len(clouds)} clouds, {over} past their capacity", flush=True)
