"""The boxes of tree nodes are put together from the boxes of aligned runs of items: hit sets and
values against the oracle at item counts around the runs' sizes (16, 256, 4096, 65536), with boxes of
very different sizes, items at one point, and leaves of one item and of many. A box that misses one of
its items would lose that item's hits."""
import numpy as np
import pytest

from smallupbp_amd import native, scenes

from gpu_helpers import REL_TOL, gpu_context, oracle_photons, print_case, rel_err


@pytest.mark.gpu
@pytest.mark.parametrize("leaf", [1, 8])
@pytest.mark.parametrize("n", [2, 3, 15, 16, 17, 33, 255, 256, 257, 4095, 4097, 65537])
def test_hits_at_the_edges_of_the_runs(n, leaf):
    print_case("lbvh", n=n, leaf=leaf)
    rng = scenes.rng_for(n + leaf)
    media = scenes.make_media([((0.1, 0.1, 0.1), (0.5, 0.5, 0.5), 0.0, 0.8)])
    ph = scenes.make_photons(rng, n, radius=0.03)
    ph.position[n // 2: n // 2 + n // 4] = ph.position[0]
    ph.radius = (0.3 * n ** (-1.0 / 3.0) * rng.uniform(0.02, 1.0, n) ** 2).astype(np.float32)
    nq = 300
    o = np.full((nq, 3), 0.5, np.float32)
    o[nq // 2:] = rng.uniform(0, 1, (nq - nq // 2, 3)).astype(np.float32)
    d = scenes._isotropic_dirs(rng, nq)
    seg = scenes.segment_values(media, np.zeros(nq, np.int32), np.zeros(nq), np.full(nq, 2.0))
    w = scenes.Workload("lbvh", media, ph, None,
                        scenes.Queries(o, d, np.arange(nq + 1, dtype=np.int64), seg, scenes.LONG_BEAM))
    ref, rsig, _ = oracle_photons(w, accel=0)
    ctx = gpu_context(media)
    bre = native.EmbreeBre(ctx)
    bre.build(ph, leaf_size=leaf)
    qv = native.QueryBatchView.to_device(w.queries)
    assert np.array_equal(native.hit_signatures(ctx, bre, None, qv)[0], rsig)
    assert np.max(rel_err(bre.evalBre(qv).cpu().numpy(), ref)) <= REL_TOL
