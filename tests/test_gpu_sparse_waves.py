"""Waves whose rays have no common origin queue ray-item pairs and test them 64 at a time, unless many of
their lanes meet a leaf (traverse.hip: queue_pairs, kSparseLanes = 16). Hit sets and values against the
oracle with bundles of rays that lie close together (runs of 1 to 64 lanes meet the same leaves), with
leaves of 1, 8 and 64 items, next to waves that do share an origin, and for SHORT queries."""
import numpy as np
import pytest

from smallupbp_amd import native, scenes

from gpu_helpers import REL_TOL, gpu_context, print_case, rel_err
from oracle import pyoracle as po


@pytest.mark.gpu
@pytest.mark.parametrize("bundle,leaf,short", [(1, 8, False), (15, 8, False), (16, 1, False), (17, 64, False),
                                               (64, 8, True), (40, 64, True)])
def test_waves_without_a_common_origin(bundle, leaf, short):
    print_case("sparse", bundle=bundle, leaf=leaf, short=short)
    rng = scenes.rng_for(bundle * 100 + leaf)
    n = 64 * 12 + 5
    media = scenes.make_media([((0.1, 0.2, 0.1), (0.5, 0.4, 0.6), 0.3, 0.8), ((0, 0, 0), (0, 0, 0), 0.0, 1.0)])
    ph = scenes.make_photons(rng, 3000, radius=0.04)
    bm = scenes.make_beams(rng, 1500, media, None, 0, 0.01, short_fraction=0.5, short_mean=0.1)
    o = rng.uniform(0, 1, (n, 3)).astype(np.float32)
    d = scenes._isotropic_dirs(rng, n)
    for s in range(0, n, bundle):  # a bundle starts near one point, in nearly one direction
        k = len(o[s:s + bundle])
        o[s:s + bundle] = o[s] + 0.002 * rng.uniform(-1, 1, (k, 3))
        d[s:s + bundle] = scenes._unit(d[s] + 0.01 * rng.uniform(-1, 1, (k, 3)))
    o[128:300] = o[128]  # waves in the middle that share an origin
    off, seg = scenes.ray_segments(media, o, d, (0, 0, 0), (1, 1, 1), 0, 1)
    w = scenes.Workload("sparse", media, ph, bm,
                        scenes.Queries(o, d, off, seg, scenes.SHORT_BEAM if short else scenes.LONG_BEAM))
    ref_p, rsig_p, _ = po.bre_eval(po.OraclePhotons(ph), media, w.queries, accel=0, signatures=True)
    ref_b, rsig_b, _ = po.beams_eval(po.OracleBeams(bm, grid_res=0), media, w.queries, accel=0, signatures=True)
    ctx = gpu_context(media)
    bre = native.EmbreeBre(ctx)
    bre.build(ph, leaf_size=leaf)
    beams = native.PhotonBeamsEvaluator(ctx)
    beams.build(bm, leaf_size=leaf)
    for order in (0, 1):  # sorted and as given
        qv = native.QueryBatchView.to_device(w.queries, order=order)
        sig_p, sig_b = native.hit_signatures(ctx, bre, beams, qv)
        assert np.array_equal(sig_p, rsig_p)
        assert np.array_equal(sig_b, rsig_b)
        out_p, out_b = native.eval_batch(ctx, bre, beams, qv)
        assert np.max(rel_err(out_p.cpu().numpy(), ref_p)) <= REL_TOL
        assert np.max(rel_err(out_b.cpu().numpy(), ref_b)) <= REL_TOL
