"""Support sweeps and EPA face storage at the sizes where they can go wrong, on
the GPU against the FP64 oracle, bit for bit: bodies whose vertex count is at,
below and above a group's width and a multiple of its four-vertex batches, for
every launch shape; clustered bodies whose counts straddle a cluster, a wave of
cluster bounds and a supercluster; and polytopes that use face slots past a
group's width."""
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


def _join(batches):
    coords, off, cnt, at = [], [], [], 0
    for b in batches:
        coords.append(np.asarray(b.coords).reshape(-1, 3))
        off.append(np.asarray(b.off) + at)
        cnt.append(b.cnt)
        at += len(coords[-1])
    cnt = np.concatenate(cnt).astype(np.int32)
    n = len(cnt) // 2
    return gen.Batch(np.concatenate(coords), np.concatenate(off).astype(np.int64), cnt,
                     np.arange(0, 2 * n, 2, dtype=np.int32), np.arange(1, 2 * n, 2, dtype=np.int32))


def _exact(torch, b, shape, cluster_min=None):
    # launches over few pairs use wider groups than configured, or two waves to a
    # clustered pair: as it is, and repeated until the configured ones run
    ref = oracle_run(oracle.GJK_EPA, b)
    once = np.stack([b.pa, b.pb], 1).astype(np.int32)
    for reps in (1, 1 + 8192 // b.n_pairs):
        pairs = torch.from_numpy(np.ascontiguousarray(np.tile(once, (reps, 1)))).cuda()
        ogjk.set_config(*shape, 0)
        try:
            sc = ogjk.DeviceScene(b)
            if cluster_min is not None:
                sc.build_clusters(cluster_min)
            out = sc.collide(oracle.GJK_EPA, len(pairs), pairs=pairs, f64_record=True)
            torch.cuda.synchronize()
        finally:
            ogjk.set_config(8, 32, 0)
        rec = out["f64"].cpu().numpy()
        simp = ogjk.simplices_from_device(out["simplices"])
        for k in range(reps):
            at = slice(k * b.n_pairs, (k + 1) * b.n_pairs)
            res = compare_f64(rec[at], simp[at], ref, oracle.GJK_EPA)
            assert res["exact"] == res["n"], (reps, k, res)
    assert (ref.distances < 0).any()


@pytest.mark.parametrize("shape", [(8, 16), (16, 32), (32, 64), (64, 64)])
def test_sweep_batch_edges(torch_cuda, shape):
    sizes = sorted({max(4, m * w + d) for w in (4, 8, 16, 32, 64) for m in (1, 2, 4, 5)
                    for d in (-1, 0, 1)})
    b = _join([gen.make(gen.SPHERE, 12, seed=100 + n, nverts=n, box=1.2) for n in sizes])
    _exact(torch_cuda, b, shape)


@pytest.mark.parametrize("sizes,cmin", [((31, 32, 33, 63, 65, 2047, 2048, 2049, 4095, 4096), 1),
                                        ((33, 4096, 4097, 4128, 5121, 9217), 1)])
def test_cluster_edges(torch_cuda, sizes, cmin):
    b = _join([gen.make(gen.NOISY_SPHERE, 6, seed=200 + n, nverts=n, box=1.2) for n in sizes])
    _exact(torch_cuda, b, (64, 64), cmin)


@pytest.mark.parametrize("lanes", [16, 32, 64])
def test_many_faces(torch_cuda, lanes):
    b = gen.make(gen.ELLIPSOID, 400, seed=300, box=0.4, nmin=200, nmax=400)
    st = oracle.run(oracle.GJK_EPA, b.coords, b.off, b.cnt, b.pa, b.pb, bits=64, nthreads=8,
                    stats=True).stats
    assert (st["epa_iters"] > 34).any()  # two more faces an iteration: slots past 64
    _exact(torch_cuda, b, (16, lanes))
