"""Beam evaluations of 512 to 32768 tiles split each tile by what it is estimated to cost (traverse.hip:
k_tile_cost, k_plan_parts, k_plan_tasks). Against the oracle where the plan can go wrong: the fewest
tiles and a ragged last one, beams that all leave one point (a few tiles carry most of the cost and get
the most parts), and batches in which some or all waves have no common origin. A second evaluation and
the allocation-free one have to give the same bits, also where the plan takes the most scratch memory."""
import numpy as np
import pytest
import torch

from smallupbp_amd import native, scenes

from gpu_helpers import REL_TOL, gpu_context, print_case, rel_err
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def scene(n_queries, n_items, clustered, other, seed=9):
    """other: the share of runs of 256 queries whose rays start anywhere"""
    rng = scenes.rng_for(seed)
    media = scenes.make_media([((0.1, 0.2, 0.1), (0.5, 0.4, 0.6), 0.3, 0.8), ((0, 0, 0), (0, 0, 0), 0.0, 1.0)])
    bm = scenes.make_beams(rng, n_items, media, None, 0, 0.005, short_fraction=0.5, short_mean=0.1)
    if clustered:
        bm.origin[:] = 0.5 + 0.01 * (bm.origin - 0.5)
        bm.length[:] = np.minimum(bm.length, 0.3)
    o, d = scenes.random_camera_rays(rng, n_queries)
    if other:
        runs = np.repeat(rng.uniform(size=(n_queries + 255) // 256) < other, 256)[:n_queries]
        o[runs] = rng.uniform(0, 1, (int(runs.sum()), 3)).astype(np.float32)
        d[runs] = scenes._isotropic_dirs(rng, int(runs.sum()))
    off, seg = scenes.ray_segments(media, o, d, (0, 0, 0), (1, 1, 1), 0, 1)
    return scenes.Workload("plan", media, None, bm, scenes.Queries(o, d, off, seg, scenes.LONG_BEAM))


@pytest.mark.parametrize("n_queries,n_items,clustered,other", [
    (32_705, 16_384, False, 0.0), (32_768, 20_000, True, 0.0), (33_333, 16_384, True, 0.3),
    (32_705, 16_384, False, 1.0)])
def test_planned_tiles_match_the_oracle(n_queries, n_items, clustered, other):
    print_case("tile_plan", q=n_queries, n=n_items, clustered=clustered, other=other)
    w = scene(n_queries, n_items, clustered, other)
    ref, rsig, _ = po.beams_eval(po.OracleBeams(w.beams, grid_res=0), w.media, w.queries, accel=0, signatures=True)
    ctx = gpu_context(w.media)
    bm = native.PhotonBeamsEvaluator(ctx)
    bm.build(w.beams)
    qv = native.QueryBatchView.to_device(w.queries)
    assert np.array_equal(native.hit_signatures(ctx, None, bm, qv)[1], rsig)
    out = native.eval_batch(ctx, None, bm, qv)[1]
    assert np.max(rel_err(out.cpu().numpy(), ref)) <= REL_TOL
    assert torch.equal(out, native.eval_batch(ctx, None, bm, qv)[1])
    # the estimate is linear in the beams' flux: sum over queries w . out = sum over beams gradient . flux
    wq = torch.rand((n_queries, 3), generator=torch.Generator().manual_seed(1)).cuda()
    g = torch.zeros((n_items, 3), device="cuda")
    native.adjoint(ctx, None, bm, qv, None, wq, None, None, None, g)
    a = float((wq.double() * out.double()).sum())
    b = float((g.double() * torch.from_numpy(w.beams.throughput).cuda().double()).sum())
    assert abs(a - b) <= 1e-3 * abs(a)
    bm.destroy()


@pytest.mark.parametrize("n_queries", [32_768, 524_288, 1_048_576, 2_097_152])
def test_noalloc_plans_give_the_same_bits(n_queries):
    print_case("tile_plan_noalloc", q=n_queries)
    w = scene(n_queries, 16_384, False, 0.0)
    ctx = gpu_context(w.media)
    bm = native.PhotonBeamsEvaluator(ctx)
    bm.build(w.beams)
    qv = native.QueryBatchView.to_device(w.queries)
    out = native.eval_batch(ctx, None, bm, qv)[1]
    got = torch.full_like(out, -1.0)
    native.eval_batch_noalloc(ctx, None, bm, qv, None, got)
    torch.cuda.synchronize()
    assert torch.equal(out, got)
    bm.destroy()
