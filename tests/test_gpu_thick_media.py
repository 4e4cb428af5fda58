"""SHORT beams in grey media. A SHORT length's transmittance is divided by that of the channel with the
smallest coefficient, so in a grey medium it is exactly 1, and SHORT queries on photons or SHORT beams
give the same bits whatever the medium absorbs (traverse.hip: transmittance). Camera rays and rays without
a common origin, small structures and ones large enough to be split, one call and a batched plan."""
import numpy as np
import pytest
import torch

from smallupbp_amd import native, scenes

from gpu_helpers import gpu_context, print_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_queries,n_items,camera", [(700, 2_000, True), (700, 2_000, False), (900, 17_000, True),
                                                      (900, 17_000, False), (33_000, 17_000, True)])
def test_short_beams_do_not_depend_on_absorption(n_queries, n_items, camera):
    print_case("thick", q=n_queries, n=n_items, camera=camera)
    outs = []
    for absorption in (0.0, 20.0, 79.5):
        rng = scenes.rng_for(21)
        media = scenes.make_media([((absorption,) * 3, (0.5,) * 3, 0.3, 0.8), ((0, 0, 0), (0, 0, 0), 0.0, 1.0)])
        ph = scenes.make_photons(rng, n_items, radius=0.03)
        bm = scenes.make_beams(rng, n_items, media, None, 0, 0.01, short_fraction=1.0, short_mean=0.1)
        if camera:
            o, d = scenes.random_camera_rays(rng, n_queries)
        else:
            o = rng.uniform(0, 1, (n_queries, 3)).astype(np.float32)
            d = scenes._isotropic_dirs(rng, n_queries).astype(np.float32)
        off, seg = scenes.ray_segments(media, o, d, (0, 0, 0), (1, 1, 1), 0, 1)
        q = scenes.Queries(o, d, off, seg, scenes.SHORT_BEAM)
        ctx = gpu_context(media)
        bre = native.EmbreeBre(ctx)
        bre.build(ph)
        beams = native.PhotonBeamsEvaluator(ctx)
        beams.build(bm)
        qv = native.QueryBatchView.to_device(q)
        got = list(native.eval_batch(ctx, bre, beams, qv))
        bp, bb = torch.zeros_like(got[0]), torch.zeros_like(got[1])
        plan = native.BatchPlan(ctx, [(bre, beams, qv, 0, bp, bb)])
        plan.run(use_graph=False)
        torch.cuda.synchronize()
        outs.append([x.cpu() for x in got + [bp, bb]])
        plan.destroy()
        bre.destroy()
        beams.destroy()
    assert all(bool(x.any()) for x in outs[0])
    for other in outs[1:]:
        for a, b in zip(outs[0], other):
            assert torch.equal(a, b)
