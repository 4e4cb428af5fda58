"""upbp_eval_stats: candidates are the items tested against a lane's ray. 64 rays without a common origin that
each meet one cluster of 8 photons and nothing else test 512 pairs, not every cluster with every ray; rays
with a common origin test a cluster with the whole wave."""
import numpy as np
import pytest

from smallupbp_amd import native, scenes

from gpu_helpers import gpu_context, print_case

pytestmark = pytest.mark.gpu


def test_pairs_are_counted_not_waves():
    print_case("candidates")
    rng = scenes.rng_for(51)
    media = scenes.make_media([((0.1, 0.2, 0.1), (0.5, 0.4, 0.6), 0.3, 0.8), ((0, 0, 0), (0, 0, 0), 0.0, 1.0)])
    cells = (np.stack(np.meshgrid(*[np.arange(4)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5) / 4
    ph = scenes.make_photons(rng, 512, radius=0.01)
    ph.position[:] = np.repeat(cells, 8, axis=0) + 0.001 * rng.uniform(-1, 1, (512, 3))
    d = scenes._isotropic_dirs(rng, 64).astype(np.float32)
    o = (cells - 0.05 * d).astype(np.float32)
    seg = scenes.segment_values(media, np.zeros(64, np.int32), np.zeros(64), np.full(64, 0.1))
    q = scenes.Queries(o, d, np.arange(65, dtype=np.int64), seg, scenes.LONG_BEAM)
    ctx = gpu_context(media)
    bre = native.EmbreeBre(ctx)
    bre.build(ph, leaf_size=8)
    st = {}
    native.eval_batch(ctx, bre, None, native.QueryBatchView.to_device(q, order=1), stats=st)
    assert st["photon_hits"] == 512 and st["photon_candidates"] == 512
    q.origin[:] = o[0]
    q.direction[:] = d[0]
    native.eval_batch(ctx, bre, None, native.QueryBatchView.to_device(q, order=1), stats=st)
    assert st["photon_hits"] == 512 and st["photon_candidates"] == 512  # 64 rays on the one cluster
    bre.destroy()
