"""Training-side featurisation: descriptors of arbitrary site clouds with per-site type weights
(nepx_cloud_descriptor, the NEP / pts_to_nep surface of 05/NEP.py and 05/Processors.py) against the
FP64 oracle.  Tolerance: 1e-5 relative, row-wise max-norm."""
import os

import numpy as np
import pytest
import torch

from oracle import nep_oracle as O

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(__file__), "golden")


def _clouds(rng, P, nd, spread):
    """Random clouds: two bodies of nd/2 points each, the second displaced by up to `spread`."""
    half = nd // 2
    a = rng.normal(0, 0.5, (P, half, 3))
    b = rng.normal(0, 0.5, (P, half, 3)) + rng.uniform(0.5, spread, (P, 1, 1)) * rng.normal(0, 1, (P, 1, 3))
    return np.concatenate([a, b], axis=1).astype(np.float32)


def _rowwise(G, G64):
    return (np.abs(G - G64).max(axis=1) / np.abs(G64).max(axis=1)).max()


@pytest.mark.parametrize("hyp,nd", [((11, 6, 4), 16), ((10, 8, 4), 12), ((17, 6, 6), 24), ((10, 10, 10), 6)])
def test_cloud_descriptor_matches_oracle(gpu, hyp, nd):
    from nepx import ops
    rng = np.random.default_rng(7)
    X = _clouds(rng, 500, nd, 2.0)
    w = rng.uniform(0.5, 2.0, nd).astype(np.float32)
    r_nep = float(np.ceil(np.linalg.norm(X - X.mean(1, keepdims=True), axis=-1).max() * 100) / 100) + 0.5
    G = ops.cloud_descriptor(torch.from_numpy(X).to(gpu), *hyp, r_nep, weights=w).cpu().numpy()
    G64 = O.descriptor(X.astype(np.float64), r_nep, *hyp, weights=w.astype(np.float64))
    e = _rowwise(G, G64)
    G1 = ops.cloud_descriptor(torch.from_numpy(X).to(gpu), *hyp, r_nep).cpu().numpy()
    e1 = _rowwise(G1, O.descriptor(X.astype(np.float64), r_nep, *hyp))
    print(f"clouds {hyp} nd={nd}: weighted {e:.2e} unweighted {e1:.2e}")
    assert e < 1e-5 and e1 < 1e-5


def test_nep_class_on_reference_clouds(gpu):
    """The reference's own cube_v2 pair clouds (01/datadir sample) through NEP.get_g_fast / pts_to_nep."""
    from nepx.NEP import NEP, calculate_cutoff, pts_to_nep
    X = np.load(os.path.join(GOLD, "x12pts_cube_v2_sample.npz"))["clouds"].astype(np.float32)
    rc = calculate_cutoff(X)
    c = X - X.mean(1, keepdims=True)
    assert rc == np.ceil(np.linalg.norm(c, axis=-1).max() * 100) / 100
    nep = NEP(X)
    nep.set_hypers([10, 8, 4, rc])
    nep.set_npts(X.shape[1] // 2)
    nep.set_device(0)
    nep.set_pts_types({"pts_types": list(range(X.shape[1]))})      # types 1..12 -> sqrt weights
    G = nep.get_g_fast()
    w = np.sqrt(np.arange(X.shape[1]) + 1.0)
    assert np.abs(nep.types - w).max() < 1e-6
    e = _rowwise(G, O.descriptor(X.astype(np.float64), rc, 10, 8, 4, weights=w))
    g_plain = nep.get_g()
    e0 = _rowwise(g_plain, O.descriptor(X.astype(np.float64), rc, 10, 8, 4))
    G2, rc2 = pts_to_nep(X, {"nep_hyper": [10, 8, 4, 100], "pts_types": list(range(X.shape[1]))}, 0, None)
    print(f"reference clouds: typed {e:.2e} plain {e0:.2e}")
    assert e < 1e-5 and e0 < 1e-5 and rc2 == rc and np.array_equal(G2, G)


def test_cloud_descriptor_rejects_missing_hypers(gpu):
    from nepx.NEP import NEP
    nep = NEP(np.zeros((4, 6, 3), np.float32) + np.arange(18, dtype=np.float32).reshape(1, 6, 3))
    nep.set_hypers([9, 9, 9, 5.0])
    with pytest.raises(NotImplementedError):
        nep.get_g_fast()


@pytest.mark.parametrize("hyp", [(11, 6, 4), (10, 8, 4), (17, 6, 6), (10, 10, 10)])
@pytest.mark.parametrize("nd,P", [(2, 1), (3, 15), (4, 16), (5, 17), (31, 33), (64, 40), (65, 40), (130, 19), (6, 70001)])
def test_cloud_descriptor_tile_edges(gpu, hyp, nd, P):
    """Four lanes per cloud, 16 clouds per tile: site counts off the quad and on both sides of the staging
    limit (64), ragged last tiles, and more tiles than blocks, weighted, against the FP64 oracle."""
    from nepx import ops
    rng = np.random.default_rng(100 * nd + P)
    X = rng.normal(0, 1.0, (P, nd, 3)).astype(np.float32)
    w = rng.uniform(0.5, 2.0, nd).astype(np.float32)
    G = ops.cloud_descriptor(torch.from_numpy(X).to(gpu), *hyp, 6.0, weights=w).cpu().numpy()
    pick = np.unique(np.concatenate([np.arange(min(P, 40)), np.arange(max(0, P - 40), P)]))
    G64 = O.descriptor(X[pick].astype(np.float64), 6.0, *hyp, weights=w.astype(np.float64))
    assert np.all(np.isfinite(G)) and _rowwise(G[pick], G64) < 1e-5


def test_cloud_descriptor_into_an_unaligned_row_block(gpu):
    """Rows are stored 16 bytes at a time only where the output allows it: the same values 4 bytes off."""
    import nepx  # noqa: F401
    from nepx import _lib
    rng = np.random.default_rng(3)
    P, nd, hyp = 50, 12, (10, 8, 4)
    X = torch.from_numpy(rng.normal(0, 1.0, (P, nd, 3)).astype(np.float32)).to(gpu)
    D, out = 47, []
    for shift in (0, 1):
        buf = torch.full((P * D + 4,), float("nan"), device=gpu)
        G = buf[shift:shift + P * D]
        _lib.check(_lib.lib.nepx_cloud_descriptor(_lib.ptr(X), P, nd, None, *hyp, 6.0, G.data_ptr(),
                                                  _lib.stream_handle()), "nepx_cloud_descriptor")
        torch.cuda.synchronize()
        assert torch.isnan(buf[:shift]).all() and torch.isnan(buf[shift + P * D:]).all()
        out.append(G.clone())
    assert torch.equal(out[0], out[1]) and torch.isfinite(out[0]).all()


@pytest.mark.parametrize("n", [0, 1, 2000, 5578, 17334, 40001])
def test_featurised_rows_equal_the_device_rows(gpu, n):
    """get_g_fast copies its rows to the host plainly up to 1 MB and through two 8 MB stages beyond
    (17,331 rows of 121 floats a stage): the same bits as the descriptors on the GPU, in several
    chunks as well."""
    from nepx import ops
    from nepx.NEP import NEP
    X = np.random.default_rng(n).normal(0, 1.0, (n, 6, 3)).astype(np.float32)
    nep = NEP(X)
    nep.set_hypers([10, 10, 10, 6.0])
    want = ops.cloud_descriptor(torch.from_numpy(X).to(gpu), 10, 10, 10, 6.0).cpu().numpy()
    for chunk in (1 << 20, 19000):
        nep.chunk = chunk
        G = nep.get_g_fast()
        assert G.dtype == np.float32 and G.shape == (n, 121) and np.array_equal(G, want)


@pytest.mark.parametrize("hyp,scale", [((11, 6, 4), 1e18), ((11, 6, 4), 1e19), ((10, 8, 4), 1e18), ((17, 6, 6), 1e16),
                                       ((17, 6, 6), 1e17), ((10, 10, 10), 1e13), ((10, 10, 10), 1e14),
                                       ((10, 10, 10), 1e15)])
def test_cloud_descriptor_overflow_stays_in_its_entry(gpu, hyp, scale):
    """Site weights so large that the squared sums of the high l leave FP32's range: those entries are
    infinite, none is NaN, and the entries of the lower l are those of the FP64 oracle.  The largest square of
    an entry is at most the entry over its smallest K_lm^2 = 2 / (2l)!."""
    from math import factorial
    from nepx import ops
    rng = np.random.default_rng(3)
    nrad, nang, lmax = hyp
    X = rng.normal(0, 1.0, (40, 12, 3)).astype(np.float32)
    w = (scale * rng.uniform(0.5, 2.0, 12)).astype(np.float32)
    G = ops.cloud_descriptor(torch.from_numpy(X).to(gpu), *hyp, 6.0, weights=w).cpu().numpy()
    G64 = O.descriptor(X.astype(np.float64), 6.0, *hyp, weights=w.astype(np.float64))
    k2min = np.array([2.0 / factorial(2 * l) for l in range(1, lmax + 1)])
    safe = np.concatenate([np.ones((40, nrad + 1), bool),
                           (G64[:, nrad + 1:].reshape(40, nang + 1, lmax) / k2min < 1e38).reshape(40, -1)], 1)
    assert not np.isnan(G).any() and np.isinf(G).any() and safe.any(axis=0).sum() > nrad + 1
    assert np.isfinite(G[safe]).all()
    assert np.abs(G[safe] - G64[safe]).max() <= 1e-5 * np.abs(G64[safe]).max()


@pytest.mark.parametrize("hyp", [(11, 6, 4), (10, 8, 4), (17, 6, 6), (10, 10, 10)])
@pytest.mark.parametrize("nd", [2, 3, 4, 5, 6, 7])
def test_many_clouds_of_few_sites(gpu, hyp, nd):
    """1, 2, 5 and 6 sites with seven-wide rows, from 320 clouds a CU on: one lane per cloud, blocks of 256 (four
    lanes: 64 or 256).  Counts on both sides of the line against the FP64 oracle, in a row block that is
    4 bytes off."""
    import nepx
    from graph_util import kernel_launches
    from nepx import _lib
    line = 320 * torch.cuda.get_device_properties(gpu).multi_processor_count
    D = nepx.n_descriptor(*hyp)
    g = torch.Generator(device=gpu).manual_seed(nd)
    X = torch.randn((line + 70, nd, 3), generator=g, device=gpu)
    w = torch.from_numpy(np.random.default_rng(nd).uniform(0.5, 2.0, nd).astype(np.float32)).to(gpu)
    buf = torch.empty((line + 70) * D + 8, device=gpu)
    blocks = []
    for P in (line - 1, line, line + 70):
        def run(stream=None):
            _lib.check(_lib.lib.nepx_cloud_descriptor(_lib.ptr(X), P, nd, _lib.ptr(w), *hyp, 6.0,
                                                      buf.data_ptr() + 4, _lib.stream_handle(stream)),
                       "nepx_cloud_descriptor")
        buf.fill_(float("nan"))
        run()
        G = buf[1:1 + P * D].view(P, D)
        assert torch.isnan(buf[0]) and torch.isnan(buf[1 + P * D:]).all() and torch.isfinite(G).all()
        pick = torch.cat([torch.arange(30), torch.arange(P - 90, P)])
        G64 = O.descriptor(X[pick].cpu().numpy().astype(np.float64), 6.0, *hyp, weights=w.cpu().numpy().astype(np.float64))
        assert _rowwise(G[pick].cpu().numpy(), G64) < 1e-5
        blocks.append(kernel_launches(run)[0][1][0])
    four = 256 if hyp[2] == 10 else 64
    assert blocks == [four] + [256 if hyp[1] == 6 and nd in (2, 5, 6) else four] * 2
