"""Evaluations of one context that return before their work has ended, on two streams in turn. Each has the
results of a call that is waited for: the second one starts in the context's buffers (the sums of a split,
the tile plan, and for sorted batches the query keys) only when the first has left them."""
import pytest
import torch

from smallupbp_amd import _abi, native, scenes

from gpu_helpers import gpu_context, print_case

pytestmark = pytest.mark.gpu


def queries(media, n, seed):
    rng = scenes.rng_for(seed)
    o, d = scenes.random_camera_rays(rng, n)
    off, seg = scenes.ray_segments(media, o, d, (0, 0, 0), (1, 1, 1), 0, 1)
    return scenes.Queries(o, d, off, seg, scenes.LONG_BEAM)


@pytest.mark.parametrize("order", [_abi.ORDER_AS_GIVEN, _abi.ORDER_SORTED])
def test_two_streams_share_a_context(order):
    print_case("streams", order=order)
    media = scenes.make_media([((0.1, 0.2, 0.1), (0.5, 0.4, 0.6), 0.3, 0.8), ((0, 0, 0), (0, 0, 0), 0.0, 1.0)])
    rng = scenes.rng_for(31)
    ctx = gpu_context(media)
    bre = native.EmbreeBre(ctx)
    bre.build(scenes.make_photons(rng, 40_000, radius=0.02))
    bm = native.PhotonBeamsEvaluator(ctx)
    bm.build(scenes.make_beams(rng, 40_000, media, None, 0, 0.005, short_fraction=0.5, short_mean=0.1))
    # planned, split, split: the largest first, so that the context's buffers have their size
    views = [native.QueryBatchView.to_device(queries(media, n, 40 + n), order=order) for n in (60_000, 700, 5_000)]
    want = [native.eval_batch(ctx, bre, bm, v) for v in views]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = [[(torch.full((v.count, 3), -1.0, device="cuda"), torch.full((v.count, 3), -1.0, device="cuda"))
            for v in views] for _ in range(4)]
    torch.cuda.synchronize()
    ctx.set_sync(False)
    k = 0
    for outs in got:
        for v, (p, b) in zip(views, outs):
            ctx.set_stream(streams[k % 2].cuda_stream)
            native.eval_batch(ctx, bre, bm, v, p, b)
            k += 1
    torch.cuda.synchronize()
    ctx.set_stream(None)
    ctx.set_sync(True)
    for outs in got:
        for (p, b), (wp, wb) in zip(outs, want):
            assert torch.equal(p, wp)
            assert torch.equal(b, wb)
    bre.destroy()
    bm.destroy()
