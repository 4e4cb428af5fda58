"""Beams of few pieces are gathered in one launch, whatever origins the rays have (traverse.hip:
kSparseFrom = 1024 pieces). Against the oracle on both sides of the line, rays with and without a common
origin in one batch, values and hit sets in both query orders."""
import numpy as np
import pytest
import torch

from smallupbp_amd import native, scenes

from gpu_helpers import REL_TOL, check_beam_ties, gpu_context, print_case, rel_err
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_beams", [1, 1023, 1024, 1025])
def test_few_pieces(n_beams):
    print_case("few_pieces", beams=n_beams)
    rng = scenes.rng_for(61)
    media = scenes.make_media([((0.1, 0.2, 0.1), (0.5, 0.4, 0.6), 0.3, 0.8), ((0, 0, 0), (0, 0, 0), 0.0, 1.0)])
    bm = scenes.make_beams(rng, n_beams, media, None, 0, 0.03, short_fraction=0.5, short_mean=0.1)
    bm.length[:] = np.minimum(bm.length, 0.2)  # one piece each
    o, d = scenes.random_camera_rays(rng, 64 * 9 + 1)
    o[200:500] = rng.uniform(0, 1, (300, 3))
    d[200:500] = scenes._isotropic_dirs(rng, 300)
    off, seg = scenes.ray_segments(media, o, d, (0, 0, 0), (1, 1, 1), 0, 1)
    q = scenes.Queries(o, d, off, seg, scenes.LONG_BEAM)
    ref, rsig, _ = po.beams_eval(po.OracleBeams(bm, grid_res=0), media, q, accel=0, signatures=True)
    ctx = gpu_context(media)
    beams = native.PhotonBeamsEvaluator(ctx)
    beams.build(bm)
    assert beams.pieces == n_beams
    for order in (0, 1):
        qv = native.QueryBatchView.to_device(q, order=order)
        out = torch.full((q.count, 3), -1.0, device="cuda")
        native.eval_batch(ctx, None, beams, qv, None, out)
        sig = native.hit_signatures(ctx, None, beams, qv)[1]
        check_beam_ties(q, bm, sig, rsig)
        same = np.all(sig == rsig, axis=1)
        assert np.max(rel_err(out.cpu().numpy()[same], ref[same])) <= REL_TOL
    beams.destroy()
