"""Device memory that calls keep: a batched plan holds the partial sums of split tiles only where some
instance is large enough to be split."""
import numpy as np
import pytest
import torch

from smallupbp_amd import native, scenes

from gpu_helpers import gpu_context, print_case

pytestmark = pytest.mark.gpu


def free_bytes():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


@pytest.mark.parametrize("n_photons,n_beams,split", [(4_000, 300, False), (20_000, 300, True)])
def test_batched_plans_hold_rows_only_where_tiles_can_be_split(n_photons, n_beams, split):
    print_case("plan_memory", photons=n_photons, beams=n_beams)
    w = scenes.bre_beams(320, 205, n_photons, n_beams, seed=23)  # 1025 tiles: planned
    ctx = gpu_context(w.media)
    bre = native.EmbreeBre(ctx)
    bre.build(w.photons)
    bm = native.PhotonBeamsEvaluator(ctx)
    bm.build(w.beams)
    assert bm.pieces < 16_384
    qv = native.QueryBatchView.to_device(w.queries)
    want = native.eval_batch(ctx, bre, bm, qv)
    p, b = (torch.full((qv.count, 3), -1.0, device="cuda") for _ in range(2))
    before = free_bytes()
    plan = native.BatchPlan(ctx, [(bre, bm, qv, 0, p, b)])
    held = before - free_bytes()
    # a row estimator's 24576 rows of 768 bytes are 18.9 MB; the rest of this plan is less than 8 MB
    assert held < (8 << 20) + (18_874_368 if split else 0)
    for graph in (False, True, True):
        p.fill_(-1.0)
        b.fill_(-1.0)
        plan.run(use_graph=graph)
        torch.cuda.synchronize()
        assert torch.equal(b, want[1])
        assert torch.allclose(p, want[0], rtol=1e-5, atol=0.0)  # the call's tiles are split too: another order
    plan.destroy()
    bre.destroy()
    bm.destroy()


@pytest.mark.parametrize("n_media", [2, 1024, 1025, 65_537, 300_000])
def test_adjoint_memory_is_bounded_for_large_media_tables(n_media):
    """The medium gradients are spread over up to 64 rows: fewer for large tables, one from 65536 media on. The
    gradients of the two media that the rays meet are those of a table of two, the others' are zero."""
    print_case("media_rows", media=n_media)
    w = scenes.adjoint_scene(64, 48, 5_000, 500)
    want = None
    for m in (len(w.media), n_media):
        media = np.resize(w.media, max(m, len(w.media)))
        ctx = gpu_context(media)
        bre = native.EmbreeBre(ctx)
        bre.build(w.photons)
        bm = native.PhotonBeamsEvaluator(ctx)
        bm.build(w.beams)
        qv = native.QueryBatchView.to_device(w.queries)
        native.eval_batch(ctx, bre, bm, qv)
        wp, wb = (torch.ones((qv.count, 3), device="cuda") for _ in range(2))
        gs, ga = (torch.zeros((len(media), 3), device="cuda") for _ in range(2))
        pp, pb = torch.zeros((w.photons.count, 3), device="cuda"), torch.zeros((w.beams.count, 3), device="cuda")
        before = free_bytes()
        native.adjoint(ctx, bre, bm, qv, wp, wb, gs, ga, pp, pb)
        # rows of 24 bytes per medium: 64 rows up to 1024 media, at most 1.6 MB, or one; the rest is small
        assert before - free_bytes() < (8 << 20) + 24 * len(media)
        hs, ha = np.zeros((len(media), 3), np.float32), np.zeros((len(media), 3), np.float32)
        native.adjoint(ctx, bre, bm, native.QueryBatchView.host(w.queries), wp.cpu().numpy(), wb.cpu().numpy(), hs, ha)
        got = [gs.cpu().numpy(), ga.cpu().numpy(), hs, ha]
        n = len(w.media)
        if want is None:
            want = got
        for g, ref in zip(got, want):
            # the same terms added in another order: a few thousand float atomics per entry
            assert np.allclose(g[:n], ref[:n], rtol=1e-3, atol=1e-4 * np.abs(ref).max())
            assert not g[n:].any()
        bre.destroy()
        bm.destroy()
