"""The autotuners leave the waves per workgroup alone where the launches choose their own."""
import os
import re

import pytest

from smallupbp_amd import autotune, scenes

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_the_rule_is_the_librarys():
    src = open(os.path.join(ROOT, "smallupbp_amd", "csrc", "upbp_internal.hpp")).read()

    def constant(name):
        return int(re.search(r"\b%s = (\d+)" % name, src).group(1))

    assert autotune.SPLIT_FROM == constant("kSplitFrom")
    assert autotune.PHOTON_SPLIT_TILES == constant("kSplitWavesLight") // 2
    assert autotune.BEAM_SPLIT_TILES == constant("kPlanMostTiles")
    # beams: uniform splits end where plans begin or later, so no size in between is left whole
    assert constant("kSplitWaves") // 2 >= constant("kPlanTiles") - 1
    # one more part has to leave each kSplitItems items
    assert constant("kSplitItems") * 2 <= constant("kSplitFrom")
    for est, most in (("photons", 2048), ("beams", 32768)):
        assert autotune.takes_waves(est, 16383, 64)
        assert not autotune.takes_waves(est, 16384, 64 * most)
        assert autotune.takes_waves(est, 16384, 64 * most + 1)


@pytest.mark.gpu
def test_autotune_keeps_the_tuning_of_split_launches():
    from gpu_helpers import gpu_context, print_case
    from smallupbp_amd import native

    print_case("autotune")
    w = scenes.bre_beams(240, 150, 20_000, 20_000, seed=17)  # 563 tiles: beams planned, photons split
    ctx = gpu_context(w.media)
    bre = native.EmbreeBre(ctx)
    bre.build(w.photons)
    bm = native.PhotonBeamsEvaluator(ctx)
    bm.build(w.beams)
    qv = native.QueryBatchView.to_device(w.queries)
    ctx.set_tuning(3)
    (waves, _), ms = native.autotune(ctx, bre, bm, qv)
    assert waves == 3 and ctx.get_tuning()[0] == 3 and ms > 0
    small = scenes.bre_beams(240, 150, 10_000, 100, seed=18)  # fewer than 16384 items: whole tiles
    bre2 = native.EmbreeBre(ctx)
    bre2.build(small.photons)
    (waves, _), ms = native.autotune(ctx, bre2, None, qv)
    assert waves in (1, 2, 4) and ctx.get_tuning()[0] == waves and ms > 0
    for h in (bre, bre2, bm):
        h.destroy()


@pytest.mark.gpu
def test_tune_sweeps_only_what_the_launch_takes():
    from gpu_helpers import print_case

    print_case("tune")
    w = scenes.bre_beams(64, 36, 17_000, 1_000, seed=19)
    e = autotune.tune(w, reps=1, path=None, log=lambda *a: None)
    assert {c["waves_per_block"] for c in e["all"]["photons"]} == {4}  # split: the context's own setting
    for c in e["all"]["beams"]:
        assert c["pieces"] < autotune.SPLIT_FROM or c["waves_per_block"] == 4
    assert e["best"]["photons"] and e["best"]["beams"]
