"""Batches in which some rays meet no scattering medium or have no segment at all, next to rays that do.
Which launch evaluates a tile of 64 rays, and which rows a tile plan gives it (traverse.hip:
common_origin), depends on all of its evaluated rays: here tiles whose scattering rays share an origin,
are a single one or none while the other rays start elsewhere. Sizes on both sides of every line of the
dispatch: uniform splits, plans with and without a uniform split next to them, no split. The outputs are
filled with -1 before; values and hit sets against the oracle, in both query orders."""
import numpy as np
import pytest
import torch

from smallupbp_amd import native, scenes

from gpu_helpers import REL_TOL, check_beam_ties, gpu_context, print_case, rel_err
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu
EYE = (0.5, 0.5, -2.0)


def scene(n_queries, n_items, gathering, camera, seed=11):
    """Tiles of seven kinds in turn (as given order). gathering: of how many tiles' rays any can gather
    something; the other tiles only miss. camera: every tile starts as camera rays."""
    rng = scenes.rng_for(seed)
    media = scenes.make_media([((0.1, 0.2, 0.1), (0.5, 0.4, 0.6), 0.3, 0.8), ((0, 0, 0), (0, 0, 0), 0.0, 1.0)])
    bm = scenes.make_beams(rng, n_items, media, None, 0, 0.01, short_fraction=0.5, short_mean=0.1)
    n = n_queries
    tile, lane = np.arange(n) // 64, np.arange(n) % 64
    kind = rng.permutation((n + 63) // 64)[tile] % 7
    far = np.where(np.arange(n) // 64 < gathering, False, True)
    kind[far] = np.where(kind[far] % 2 == 0, 1, 6)
    o, d = scenes.random_camera_rays(rng, n, EYE)
    away = rng.uniform(2.0, 3.0, (n, 3)).astype(np.float32)  # outside, leaving: they meet nothing
    out = scenes._unit(rng.uniform(0.1, 1.0, (n, 3))).astype(np.float32)
    inside = rng.uniform(0, 1, (n, 3)).astype(np.float32)
    iso = scenes._isotropic_dirs(rng, n).astype(np.float32)
    # 0: camera rays; 1: all start elsewhere and miss; 2: one gathers; 3, 4: half are camera rays, the others
    # miss (3) or have no segment (4); 5: all start inside; 6: none has a segment
    miss = (kind == 1) | ((kind == 2) & (lane != 17)) | ((kind == 3) & (lane % 2 == 1))
    none = ((kind == 4) & (lane % 2 == 0)) | (kind == 6)
    if camera:  # a frame padded with rays that miss or end at once
        miss &= rng.uniform(size=n) < 0.5
        none |= (kind == 1) & ~miss
    else:
        o[kind == 5], d[kind == 5] = inside[kind == 5], iso[kind == 5]
    gone = miss | none
    o[gone], d[gone] = away[gone], out[gone]
    off, seg = scenes.ray_segments(media, o, d, (0, 0, 0), (1, 1, 1), 0, 1)
    counts = np.diff(off)
    keep = np.repeat(~none, counts)
    counts[none] = 0
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    return scenes.Workload("classes", media, None, bm, scenes.Queries(o, d, off, seg[keep], scenes.LONG_BEAM)), gone


@pytest.mark.parametrize("n_queries,gathering,camera", [
    (5_000, 78, False), (40_005, 600, False), (40_005, 600, True), (524_289, 700, False), (600_000, 900, False),
    (600_000, 900, True), (2_100_000, 600, False)])
def test_tiles_of_every_class_are_written(n_queries, gathering, camera):
    print_case("tile_classes", q=n_queries, gathering=gathering, camera=camera)
    w, gone = scene(n_queries, 16_384, gathering, camera)
    ref, rsig, _ = po.beams_eval(po.OracleBeams(w.beams, grid_res=0), w.media, w.queries, accel=0, signatures=True)
    assert not ref[gone].any() and np.count_nonzero(ref.any(axis=1)) > gathering
    ctx = gpu_context(w.media)
    bm = native.PhotonBeamsEvaluator(ctx)
    bm.build(w.beams)
    for order in (0, 1):  # sorted and as given
        qv = native.QueryBatchView.to_device(w.queries, order=order)
        out = torch.full((n_queries, 3), -1.0, device="cuda")
        native.eval_batch(ctx, None, bm, qv, None, out)
        sig = native.hit_signatures(ctx, None, bm, qv)[1]
        check_beam_ties(w.queries, w.beams, sig, rsig)
        same = np.all(sig == rsig, axis=1)
        assert np.max(rel_err(out.cpu().numpy()[same], ref[same])) <= REL_TOL
        if order == 1 or n_queries <= 1 << 21:
            got = torch.full_like(out, -1.0)
            native.eval_batch_noalloc(ctx, None, bm, qv, None, got)
            torch.cuda.synchronize()
            assert torch.equal(out, got)
    bm.destroy()


@pytest.mark.parametrize("n_queries,gathering", [(5_000, 78), (40_005, 600), (600_000, 900)])
def test_rays_that_gather_nothing_do_not_matter_to_the_others(n_queries, gathering):
    """Where a tile's other rays start, if they meet no medium, changes nothing: camera rays padded with them
    keep the launch, the order and so the bits that they have when all start at the camera."""
    print_case("tile_padding", q=n_queries, gathering=gathering)
    w, gone = scene(n_queries, 16_384, gathering, True)
    ctx = gpu_context(w.media)
    bm = native.PhotonBeamsEvaluator(ctx)
    bm.build(w.beams)
    res = []
    for elsewhere in (True, False):
        if not elsewhere:
            w.queries.origin[gone] = EYE
        qv = native.QueryBatchView.to_device(w.queries, order=1)
        out = torch.full((n_queries, 3), -1.0, device="cuda")
        native.eval_batch(ctx, None, bm, qv, None, out)
        res.append((out, native.hit_signatures(ctx, None, bm, qv)[1]))
    assert np.array_equal(res[0][1], res[1][1])
    assert torch.equal(res[0][0], res[1][0])
    bm.destroy()
