"""Batched plans of 1024 tiles or more start the dearest tiles first and split the dear tiles of instances
with 16384 items or more (traverse.hip: k_tile_cost_batched). Every instance against its own evaluation,
eager and replayed: the same bits where nothing is split, to the rounding of the sums where tiles are; with
instances whose tiles are no multiple of the four that share an estimate, without photons, without beams,
with rays of no common origin, and with one ray."""
import numpy as np
import pytest
import torch

from smallupbp_amd import native, scenes

from gpu_helpers import gpu_context, print_case, rel_err


def scene(n_queries, n_photons, n_beams, spread, seed):
    rng = scenes.rng_for(seed)
    media = scenes.make_media([((0.1, 0.2, 0.1), (0.5, 0.4, 0.6), 0.3, 0.8), ((0, 0, 0), (0, 0, 0), 0.0, 1.0)])
    ph = scenes.make_photons(rng, n_photons, radius=0.02) if n_photons else None
    bm = scenes.make_beams(rng, n_beams, media, None, 0, 0.005, short_fraction=0.5, short_mean=0.1) if n_beams else None
    o, d = scenes.random_camera_rays(rng, n_queries)
    if spread:
        o = rng.uniform(0, 1, (n_queries, 3)).astype(np.float32)
        d = scenes._isotropic_dirs(rng, n_queries)
    off, seg = scenes.ray_segments(media, o, d, (0, 0, 0), (1, 1, 1), 0, 1)
    return scenes.Workload("batch", media, ph, bm, scenes.Queries(o, d, off, seg, scenes.LONG_BEAM))


@pytest.mark.gpu
@pytest.mark.parametrize("first", [20_000, 65_000])
def test_planned_batch_equals_per_instance_eval(first):
    print_case("batched_plan", first=first)
    shapes = [(first, 20_000, 18_000, False), (777, 5_000, 0, False), (30_001, 0, 6_000, False), (1, 400, 300, False),
              (5_000, 17_000, 2_000, True), (15_000, 3_000, 20_000, False)]
    ws = [scene(*s, seed=31 + i) for i, s in enumerate(shapes)]
    ctx = gpu_context(np.concatenate([w.media for w in ws]))
    inst, refs, outs = [], [], []
    for i, w in enumerate(ws):
        one = gpu_context(w.media)
        got = []
        for c in (ctx, one):
            bre = bm = None
            if w.photons is not None:
                bre = native.EmbreeBre(c)
                bre.build(w.photons)
            if w.beams is not None:
                bm = native.PhotonBeamsEvaluator(c)
                bm.build(w.beams)
            got.append((bre, bm, native.QueryBatchView.to_device(w.queries)))
        out = [torch.full((w.queries.count, 3), -1.0, device="cuda") if x is not None else None for x in got[0][:2]]
        inst.append((*got[0], 2 * i, *out))
        outs.append(out)
        refs.append(native.eval_batch(one, *got[1]))
    plan = native.BatchPlan(ctx, inst)
    for use_graph in (False, True, True):
        for out in outs:
            for x in out:
                if x is not None:
                    x.fill_(-1.0)
        torch.cuda.synchronize()
        plan.run(use_graph=use_graph)
        torch.cuda.synchronize()
        for s, (bre, bm, *_), out, ref in zip(shapes, inst, outs, refs):
            for x, r, items in zip(out, ref, (s[1], bm.pieces if bm else 0)):
                if x is None:
                    continue
                # an evaluation of rays without a common origin adds up in another order than a plan
                if items < 16_384 and not s[3]:
                    assert torch.equal(x, r)
                else:
                    assert np.max(rel_err(x.cpu().numpy(), r.cpu().numpy())) <= 2e-5
    plan.destroy()
