"""Hull builds of dense surface clouds, whose face lists grow to many times the
usual 2 n - 4 within their last insertions (volumes near the 1e-7 visibility
threshold): face lists against the C oracle, and which of the device's working
sets a cloud used.  Only the one-wave kernel over global memory writes the two
upper thirds of a cloud's workspace, so a mark left there shows that a cloud
did without it."""
import numpy as np
import pytest

import oracle
import ogjk

pytestmark = pytest.mark.gpu

MARK = -77


@pytest.fixture(scope="module")
def torch_cuda():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def ellipsoid(n, seed, scale):
    """n points on a rotated ellipsoid of axes up to 2 * scale."""
    rng = np.random.default_rng([n, seed])
    u = rng.normal(size=(n, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    m = np.linalg.qr(rng.normal(size=(3, 3)))[0] * rng.uniform(0.3, 2.0, (1, 3))
    return ((u @ m.T).astype(np.float32) * np.float32(scale)).astype(np.float32)


def build(torch, clouds, caps):
    """Face lists of the clouds, and per cloud whether its marks are left."""
    cnt = np.array([len(c) for c in clouds], np.int32)
    off = np.concatenate([[0], np.cumsum(cnt)[:-1]]).astype(np.int64)
    fo = np.concatenate([[0], np.cumsum(caps)]).astype(np.int64)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    pts, d_off, d_cnt, d_fo = dev(np.concatenate(clouds)), dev(off), dev(cnt), dev(fo)
    total = int(fo[-1])
    faces = torch.empty((total, 3), dtype=torch.int32, device="cuda")
    nf = torch.empty(len(clouds), dtype=torch.int32, device="cuda")
    ws = torch.full((3 * total,), MARK, dtype=torch.int32, device="cuda")
    st = ogjk.lib().ogjk_build_hulls(pts.data_ptr(), d_off.data_ptr(), d_cnt.data_ptr(),
                                     len(clouds), d_fo.data_ptr(), total, faces.data_ptr(),
                                     nf.data_ptr(), ws.data_ptr(), 12 * total, None)
    assert st == 0
    torch.cuda.synchronize()
    f, nf, ws = faces.cpu().numpy(), nf.cpu().numpy(), ws.cpu().numpy()
    lists = [f[fo[i]:fo[i] + nf[i]] if nf[i] >= 0 else int(nf[i]) for i in range(len(clouds))]
    marks = [bool((ws[3 * fo[i] + caps[i]:3 * fo[i + 1]] == MARK).all())
             for i in range(len(clouds))]
    return lists, marks


# Face counts of 5,397 to 8,357.  At an insertion of each, more than 256 of the
# visible faces lie in the sixteenth of the face list that one wave of a
# 1,024-thread block looks at.
DENSE = [(309, 24, 0.12), (512, 39, 0.2), (309, 31, 0.2), (436, 6, 0.2), (256, 33, 0.12),
         (160, 3, 0.06), (200, 26, 0.06)]


def test_dense_clouds_stay_in_lds(torch_cuda):
    """No cloud of up to 512 points whose faces fit the block's working set may
    end in the one-wave kernel (tens of milliseconds for a cloud)."""
    clouds = [ellipsoid(*c) for c in DENSE]
    lists, marks = build(torch_cuda, clouds, [9000] * len(clouds))
    for c, p, got, left in zip(DENSE, clouds, lists, marks):
        ref = oracle.build_hull(p, cap=9000)
        assert len(ref) > 5000, c
        assert np.array_equal(got, ref), c
        assert left, c
    # the same past a capacity that they exceed
    lists, marks = build(torch_cuda, clouds, [5200] * len(clouds))
    for c, p, got, left in zip(DENSE, clouds, lists, marks):
        assert got == -1 and oracle.build_hull(p, cap=5200) is None, c
        assert left, c
