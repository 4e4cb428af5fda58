"""The wave frustum check of a beam's first and last piece, on pairs where only the rounding of the
reference's t2 makes a hit: beams nearly perpendicular to a camera ray whose closest point to it lies
beyond one of the beam's ends. A wave whose segments start behind the eye has no frustum and tests
every piece of the leaves it visits, so both runs must find the same hits: with leaves of 64 items
the leaves a wave visits are the same in both (dist_min -1e-3 adds nothing to hit: nothing lies
behind the eye). Hit signatures are exact, so they must be equal."""
import numpy as np
import pytest

from smallupbp_amd import native, scenes

from gpu_helpers import gpu_context, print_case

W = H = 32


def _tile_rays():
    o, d = scenes.pinhole_rays(W, H)
    y, x = np.divmod(np.arange(W * H), W)
    idx = np.argsort(((y // 8) * (W // 8) + x // 8) * 64 + (y % 8) * 8 + x % 8)
    return np.ascontiguousarray(o[idx]), np.ascontiguousarray(d[idx])


def end_tie_scene(reach, seed=17, n=20_000, radius=0.003):
    """Beams across a ray (|q| below 1e-6) whose closest point to it lies up to `reach` radii before
    the beam's start or beyond its end."""
    rng = scenes.rng_for(seed)
    media = scenes.make_media([((0.1, 0.1, 0.1), (0.5, 0.5, 0.5), 0.0, 0.8)])
    o, d = _tile_rays()
    j = rng.integers(0, len(o), n)
    d64 = d[j].astype(np.float64)
    a = rng.normal(size=(n, 3))
    b = np.cross(a, d64)
    b /= np.linalg.norm(b, axis=1, keepdims=True)  # across the ray
    b32 = b.astype(np.float32)
    u = np.cross(b, d64)
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    length = rng.uniform(0.02, 0.3, n)
    beyond = rng.uniform(0.0, reach, n) * radius
    s = np.where(rng.uniform(size=n) < 0.5, -beyond, length + beyond)  # foot of the closest point
    p = o[j] + d64 * rng.uniform(2.2, 2.8, n)[:, None] + u * (rng.uniform(0.0, 0.95, n) * radius)[:, None]
    org = p - b * s[:, None]
    beams = scenes.Beams(org.astype(np.float32), b32, length.astype(np.float32),
                         rng.uniform(0, 1e-4, (n, 3)).astype(np.float32), np.full(n, scenes.SHORT_BEAM, np.uint32),
                         np.zeros(n, np.int32), radius)
    return media, o, d, beams


@pytest.mark.gpu
@pytest.mark.parametrize("reach", [0.5, 4.0, 40.0])
def test_end_pieces_culled_only_where_no_rounding_can_make_a_hit(reach):
    media, o, d, beams = end_tie_scene(reach)
    ctx = gpu_context(media)
    bm = native.PhotonBeamsEvaluator(ctx)
    bm.build(beams, leaf_size=64)
    sigs = []
    for start in (0.0, -1e-3):
        print_case("frustum_ends reach %g start %g" % (reach, start))
        n = len(o)
        seg = scenes.segment_values(media, np.zeros(n, np.int32), np.full(n, start), np.full(n, 6.0))
        q = scenes.Queries(o, d, np.arange(n + 1, dtype=np.int64), seg, scenes.LONG_BEAM)
        qv = native.QueryBatchView.to_device(q, order=1)  # as given: one 8 x 8 tile per wave
        sigs.append(native.hit_signatures(ctx, None, bm, qv)[1])
    assert sigs[0][:, 0].sum() > 0, "the scene plants no hit"
    assert np.array_equal(sigs[0], sigs[1])
    bm.destroy()
