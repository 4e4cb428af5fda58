"""Evaluations in the caller's order recorded into a graph by the caller, as the context's first call: they
allocate nothing, and the graph stays valid when a later, larger call makes the context grow its buffers.
Sizes that an eager call splits over waves (700 queries) and plans (33000). Replayed several times with
eager calls in between, each replay against the oracle."""
import numpy as np
import pytest
import torch

from smallupbp_amd import _abi, native, scenes

from gpu_helpers import REL_TOL, gpu_context, print_case, rel_err
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def scene(n_queries, n_items, seed=13):
    rng = scenes.rng_for(seed)
    media = scenes.make_media([((0.1, 0.2, 0.1), (0.5, 0.4, 0.6), 0.3, 0.8), ((0, 0, 0), (0, 0, 0), 0.0, 1.0)])
    ph = scenes.make_photons(rng, n_items, radius=0.02)
    bm = scenes.make_beams(rng, n_items, media, None, 0, 0.005, short_fraction=0.5, short_mean=0.1)
    o, d = scenes.random_camera_rays(rng, n_queries)
    off, seg = scenes.ray_segments(media, o, d, (0, 0, 0), (1, 1, 1), 0, 1)
    return scenes.Workload("capture", media, ph, bm, scenes.Queries(o, d, off, seg, scenes.LONG_BEAM))


@pytest.mark.parametrize("n_queries", [700, 33_000])
def test_captured_evaluation_outlives_larger_calls(n_queries):
    print_case("capture", q=n_queries)
    w, big = scene(n_queries, 16_384), scene(100_000, 16_384, seed=14)
    ref_p, _, _ = po.bre_eval(po.OraclePhotons(w.photons), w.media, w.queries, accel=1)
    ref_b, _, _ = po.beams_eval(po.OracleBeams(w.beams, grid_res=0), w.media, w.queries, accel=0)
    ctx = gpu_context(w.media)
    bre = native.EmbreeBre(ctx)
    bre.build(w.photons)
    bm = native.PhotonBeamsEvaluator(ctx)
    bm.build(w.beams)
    qv = native.QueryBatchView.to_device(w.queries, order=_abi.ORDER_AS_GIVEN)
    bv = native.QueryBatchView.to_device(big.queries, order=_abi.ORDER_AS_GIVEN)
    p, b = (torch.zeros((n_queries, 3), device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ctx.set_stream(torch.cuda.current_stream().cuda_stream)
        ctx.set_sync(False)
        native.eval_batch(ctx, bre, bm, qv, p, b)
    ctx.set_stream(None)
    ctx.set_sync(True)
    for _ in range(3):
        p.fill_(-1.0)
        b.fill_(-1.0)
        graph.replay()
        torch.cuda.synchronize()
        assert np.max(rel_err(p.cpu().numpy(), ref_p)) <= REL_TOL
        assert np.max(rel_err(b.cpu().numpy(), ref_b)) <= REL_TOL
        native.eval_batch(ctx, bre, bm, bv)
        ep, eb = native.eval_batch(ctx, bre, bm, qv)
        assert np.max(rel_err(ep.cpu().numpy(), ref_p)) <= REL_TOL
        assert np.max(rel_err(eb.cpu().numpy(), ref_b)) <= REL_TOL
    bre.destroy()
    bm.destroy()
