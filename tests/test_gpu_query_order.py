"""Photon-only evaluations sort the queries that share query 0's origin along a Hilbert curve over
their directions. The order must not matter: hit sets and values against the oracle for rays over the
whole sphere of directions, for a camera along each axis, and for batches that mix origins, at sizes
around the 64 queries of a wave and where no sort happens."""
import numpy as np
import pytest

from smallupbp_amd import native, scenes

from gpu_helpers import REL_TOL, gpu_context, oracle_photons, print_case, rel_err


def rays(kind, n, seed):
    rng = scenes.rng_for(seed)
    if kind in ("sphere", "mixed"):
        o = np.full((n, 3), 0.5, np.float32)
        d = scenes._isotropic_dirs(rng, n)
        if kind == "mixed":
            other = rng.uniform(size=n) < 0.5
            o[other] = rng.uniform(0, 1, (int(other.sum()), 3)).astype(np.float32)
        return o, d
    axis, sign = "xyz".index(kind[1]), 1.0 if kind[0] == "+" else -1.0
    d = rng.uniform(-0.3, 0.3, (n, 3))
    d[:, axis] = sign
    o = np.full(3, 0.5)
    o[axis] = 0.5 - 2.0 * sign
    return np.tile(o.astype(np.float32), (n, 1)), scenes._unit(d)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [64, 65, 1000])
@pytest.mark.parametrize("kind", ["sphere", "mixed", "+x", "-x", "+y", "-y", "+z", "-z"])
def test_photons_do_not_depend_on_the_query_order(kind, n):
    print_case("query_order", kind=kind, n=n)
    rng = scenes.rng_for(3)
    media = scenes.make_media([((0.1, 0.1, 0.1), (0.5, 0.5, 0.5), 0.0, 0.8), ((0, 0, 0), (0, 0, 0), 0.0, 1.0)])
    ph = scenes.make_photons(rng, 5000, radius=0.03)
    o, d = rays(kind, n, 11)
    off, seg = scenes.ray_segments(media, o, d, (0, 0, 0), (1, 1, 1), 0, 1)
    q = scenes.Queries(o, d, off, seg, scenes.LONG_BEAM)
    w = scenes.Workload("order", media, ph, None, q)
    ref, rsig, _ = oracle_photons(w)
    ctx = gpu_context(media)
    bre = native.EmbreeBre(ctx)
    bre.build(ph)
    qv = native.QueryBatchView.to_device(q)
    assert np.array_equal(native.hit_signatures(ctx, bre, None, qv)[0], rsig)
    assert np.max(rel_err(bre.evalBre(qv).cpu().numpy(), ref)) <= REL_TOL
    bre.destroy()


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [0.0, np.nan, np.inf])
def test_bad_directions_sort_and_are_reported(bad):
    rng = scenes.rng_for(3)
    media = scenes.make_media([((0.1, 0.1, 0.1), (0.5, 0.5, 0.5), 0.0, 0.8)])
    ph = scenes.make_photons(rng, 500, radius=0.03)
    o, d = rays("+z", 200, 11)
    d[[0, 77]] = bad
    seg = scenes.segment_values(media, np.zeros(200, np.int32), np.zeros(200), np.full(200, 4.0))
    q = scenes.Queries(o, d, np.arange(201, dtype=np.int64), seg, scenes.LONG_BEAM)
    ctx = gpu_context(media)
    bre = native.EmbreeBre(ctx)
    bre.build(ph)
    qv = native.QueryBatchView.to_device(q)
    if bad == 0.0:  # finite: no light is gathered along it
        bre.evalBre(qv)
    else:
        with pytest.raises(native.UpbpError):
            bre.evalBre(qv)
    bre.destroy()
