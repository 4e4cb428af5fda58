"""Small batches split a tile's items over several waves (traverse.hip: ItemPart, split_parts). Hit sets
and values against the oracle where the split's arithmetic can go wrong: query counts around a tile of
64, item counts around the 256 per part and around the blocks of 64, items that all lie close together
in leaf order (one tile meets them all), and leaves of 1, 8 and 64 items, whose runs straddle blocks."""
import numpy as np
import pytest

from smallupbp_amd import native, scenes

from gpu_helpers import REL_TOL, gpu_context, print_case, rel_err
from oracle import pyoracle as po


def scene(n_queries, n_items, clustered, seed=5):
    rng = scenes.rng_for(seed)
    media = scenes.make_media([((0.1, 0.2, 0.1), (0.5, 0.4, 0.6), 0.3, 0.8), ((0, 0, 0), (0, 0, 0), 0.0, 1.0)])
    ph = scenes.make_photons(rng, n_items, radius=0.03)
    bm = scenes.make_beams(rng, n_items, media, None, 0, 0.01, short_fraction=0.5, short_mean=0.1)
    if clustered:  # around one point
        ph.position[:] = 0.5 + 0.02 * (ph.position - 0.5)
        bm.origin[:] = 0.5 + 0.02 * (bm.origin - 0.5)
        bm.length[:] = np.minimum(bm.length, 0.1)
    o, d = scenes.random_camera_rays(rng, n_queries)
    if clustered:
        d = scenes._unit(0.5 + 0.02 * (rng.uniform(size=(n_queries, 3)) - 0.5) - o)
    off, seg = scenes.ray_segments(media, o, d, (0, 0, 0), (1, 1, 1), 0, 1)
    return scenes.Workload("split", media, ph, bm, scenes.Queries(o, d, off, seg, scenes.LONG_BEAM))


@pytest.mark.gpu
@pytest.mark.parametrize("clustered", [False, True])
@pytest.mark.parametrize("n_queries,n_items,leaf", [(1, 16_383, 8), (63, 16_384, 64), (64, 16_385, 1),
                                                    (65, 16_900, 8), (200, 20_000, 64), (700, 20_000, 8)])
def test_split_tiles_match_the_oracle(n_queries, n_items, leaf, clustered):
    print_case("split", q=n_queries, n=n_items, leaf=leaf, clustered=clustered)
    w = scene(n_queries, n_items, clustered)
    ref_p, rsig_p, _ = po.bre_eval(po.OraclePhotons(w.photons), w.media, w.queries, accel=1, signatures=True)
    ref_b, rsig_b, _ = po.beams_eval(po.OracleBeams(w.beams, grid_res=0), w.media, w.queries, accel=0,
                                     signatures=True)
    ctx = gpu_context(w.media)
    bre = native.EmbreeBre(ctx)
    bre.build(w.photons, leaf_size=leaf)
    bm = native.PhotonBeamsEvaluator(ctx)
    bm.build(w.beams, leaf_size=leaf)
    qv = native.QueryBatchView.to_device(w.queries)
    sig_p, sig_b = native.hit_signatures(ctx, bre, bm, qv)
    assert np.array_equal(sig_p, rsig_p)
    assert np.array_equal(sig_b, rsig_b)
    for b, m in ((bre, bm), (bre, None), (None, bm)):
        out_p, out_b = native.eval_batch(ctx, b, m, qv)
        if b is not None:
            assert np.max(rel_err(out_p.cpu().numpy(), ref_p)) <= REL_TOL
        if m is not None:
            assert np.max(rel_err(out_b.cpu().numpy(), ref_b)) <= REL_TOL
    bre.destroy()
    bm.destroy()


def test_item_parts_cover_every_item_once(tmp_path):
    """ItemPart's own source on the host: over all parts, every item of a range is taken exactly once, and
    a part that takes none of a range's items may still meet it, but never the other way round."""
    import os
    import subprocess

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    src = open(os.path.join(root, "smallupbp_amd", "csrc", "traverse.hip")).read()
    body = src[src.index("struct ItemPart {"):]
    body = body[:body.index("\n};") + 3]
    code = """
#include <cstdint>
#include <cstdio>
#define __device__
#define __forceinline__ inline
%s
int main() {
    for (uint32_t parts = 1; parts <= 64; parts *= 2)
        for (uint32_t shift = 6; shift <= 8; ++shift)
            for (uint32_t s = 0; s < 5u << shift; s += 7)
                for (uint32_t n = 1; n <= 64; n += 1) {
                    uint64_t seen = 0;
                    for (uint32_t p = 0; p < parts; ++p) {
                        const ItemPart part = {p, parts - 1u, shift};
                        const uint64_t m = part.items(s, n);
                        if (m & seen) return 1;
                        if (m && !part.meets(s, n)) return 2;
                        for (uint32_t j = 0; j < n; ++j)
                            if (((m >> j) & 1) != ((((s + j) >> shift) & (parts - 1)) == p)) return 3;
                        seen |= m;
                    }
                    if (seen != (n >= 64 ? ~0ull : (1ull << n) - 1)) return 4;
                    for (uint32_t big = 100; big < 100000; big *= 3)
                        for (uint32_t p = 0; p < parts; ++p) {
                            bool any = false;
                            for (uint32_t b = s >> shift; b <= (s + big - 1) >> shift; ++b) any |= (b & (parts - 1)) == p;
                            if (any != ItemPart{p, parts - 1u, shift}.meets(s, big)) return 5;
                        }
                    if (n > 3 && n < 60) n += 5;
                }
    return 0;
}
""" % body
    exe = str(tmp_path / "parts")
    (tmp_path / "parts.cpp").write_text(code)
    subprocess.check_call(["g++", "-std=c++17", "-O2", str(tmp_path / "parts.cpp"), "-o", exe])
    assert subprocess.call([exe]) == 0
