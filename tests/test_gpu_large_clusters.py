"""Clustered bodies of more than 128 superclusters (131,072 vertices), whose
supercluster bounds past the 128th are formed again instead of kept, with one
and with two waves per pair and with many vertices in a query's window, against
the FP64 oracle, bit for bit."""
import numpy as np
import pytest

import oracle
import ogjk
from ogjk import gen
from parity_utils import compare_f64, oracle_run

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def bodies(n, seed, ties):
    """Two overlapping or separate noisy spheres of n vertices; ties: rounded to
    a lattice, so that hundreds of vertices share their extreme values."""
    rng = np.random.default_rng([n, seed])
    out = []
    for k in range(2):
        u = rng.normal(size=(n, 3))
        u /= np.linalg.norm(u, axis=1, keepdims=True)
        u *= 1.0 + 0.01 * rng.normal(size=(n, 1))
        if ties:
            u = np.round(u * 24) / 24
        out.append((u + k * rng.uniform(-1.9, 1.9, 3)).astype(np.float32))
    return out


@pytest.mark.parametrize("n", [131_040, 131_071, 131_072, 131_073, 135_169, 200_000])
@pytest.mark.parametrize("ties", [False, True])
def test_many_superclusters(torch_cuda, n, ties):
    torch = torch_cuda
    pairs = [bodies(n, s, ties) for s in range(6)]
    pairs.append([bodies(n, 7, ties)[0], bodies(5000, 8, ties)[1]])  # one large body of the two
    b = gen.from_bodies([p[0] for p in pairs], [p[1] for p in pairs])
    ref = oracle_run(oracle.GJK_EPA, b)
    assert (ref.distances < 0).any()
    sc = ogjk.DeviceScene(b)
    sc.build_clusters(1024)
    try:
        for exact in (False, True):  # two waves per pair, one
            ogjk.set_config(64, 64, 0)
            ogjk.set_exact_lanes(exact)
            out = sc.collide(oracle.GJK_EPA, b.n_pairs, f64_record=True)
            torch.cuda.synchronize()
            res = compare_f64(out["f64"].cpu().numpy(),
                              ogjk.simplices_from_device(out["simplices"]), ref, oracle.GJK_EPA)
            assert res["exact"] == res["n"], (exact, res)
    finally:
        ogjk.set_config(8, 32, 0)
