"""The wave queues in LDS, which some lanes fill and others empty (hashgrid.hip: vm_drain; traverse.hip:
drain_pairs, drain_photons, drain_beams), at their fullest: every lane finds every item, so that each step
queues 64 entries on top of up to 63 and the rings wrap again and again, with counts that leave none, one
or 63 entries for the end. Against the oracle."""
import numpy as np
import pytest

from smallupbp_amd import native, scenes

from gpu_helpers import REL_TOL, gpu_context, print_case, rel_err
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make,n_queries,n_paths", [(scenes.pp3d_scene, 64, 16), (scenes.pp3d_scene, 65, 21),
                                                    (scenes.pp3d_scene, 191, 40), (scenes.surf_scene, 64, 16),
                                                    (scenes.surf_scene, 129, 33)])
def test_merging_where_every_vertex_is_a_hit(make, n_queries, n_paths):
    print_case("full_ring", scene=make.__name__, q=n_queries, paths=n_paths)
    sc = make(n_paths=n_paths, n_queries=n_queries, radius=3.0, cell_count=1, seed=91)
    og = po.OracleHashGrid(sc)
    ref, ref_sig, cnt = po.vm_eval(og, sc, precision=64)
    # one bucket, walked for each of the eight cells: all that is tested is found (by the queries inside the
    # vertices' box, the others test nothing)
    assert cnt[0] == cnt[1] and cnt[0] % (8 * og.count()) == 0 and cnt[0] > 2 * og.count() * n_queries
    ctx = gpu_context(sc.media)
    grid = native.HashGrid(ctx)
    grid.build(sc.positions, sc.mis.light_vertices, sc.radius, sc.cell_count, sc.technique)
    assert np.array_equal(grid.eval(sc.queries, sc.mis, signatures=True), ref_sig)
    assert rel_err(grid.eval(sc.queries, sc.mis), ref).max() <= REL_TOL
    grid.destroy()


@pytest.mark.parametrize("n_queries,n_items", [(64, 64), (65, 65), (128, 190)])
def test_pairs_of_waves_without_a_common_origin(n_queries, n_items):
    """Bundles of 16 rays, the most that queue their pairs, through one spot where all items lie."""
    print_case("full_pairs", q=n_queries, n=n_items)
    rng = scenes.rng_for(92)
    media = scenes.make_media([((0.1, 0.2, 0.1), (0.5, 0.4, 0.6), 0.3, 0.8), ((0, 0, 0), (0, 0, 0), 0.0, 1.0)])
    ph = scenes.make_photons(rng, n_items, radius=0.05)
    ph.position[:] = 0.5 + 0.002 * (ph.position - 0.5)
    bm = scenes.make_beams(rng, n_items, media, None, 0, 0.05, short_fraction=0.5, short_mean=0.1)
    bm.origin[:] = 0.5 + 0.002 * (bm.origin - 0.5)
    bm.length[:] = 0.3
    o = rng.uniform(0.1, 0.9, (n_queries, 3)).astype(np.float32)
    aim = scenes._unit(0.5 + 0.01 * rng.uniform(-1, 1, (n_queries, 3)) - o)
    near = np.arange(n_queries) % 64 < 16
    d = np.where(near[:, None], aim, scenes._unit(o - 0.5)).astype(np.float32)  # the others look away
    off, seg = scenes.ray_segments(media, o, d, (0, 0, 0), (1, 1, 1), 0, 1)
    q = scenes.Queries(o, d, off, seg, scenes.LONG_BEAM)
    ref_p, rsig_p, _ = po.bre_eval(po.OraclePhotons(ph), media, q, accel=0, signatures=True)
    ref_b, rsig_b, _ = po.beams_eval(po.OracleBeams(bm, grid_res=0), media, q, accel=0, signatures=True)
    assert rsig_p[near, 0].min() > 0.9 * n_items
    ctx = gpu_context(media)
    bre = native.EmbreeBre(ctx)
    bre.build(ph)
    beams = native.PhotonBeamsEvaluator(ctx)
    beams.build(bm)
    qv = native.QueryBatchView.to_device(q, order=1)
    sig_p, sig_b = native.hit_signatures(ctx, bre, beams, qv)
    assert np.array_equal(sig_p, rsig_p) and np.array_equal(sig_b, rsig_b)
    out_p, out_b = native.eval_batch(ctx, bre, beams, qv)
    assert np.max(rel_err(out_p.cpu().numpy(), ref_p)) <= REL_TOL
    assert np.max(rel_err(out_b.cpu().numpy(), ref_b)) <= REL_TOL
    bre.destroy()
    beams.destroy()
