"""Light tails are built by blocks of 256 consecutive light vertices, whose first vertices may continue a
chain of the block before, and merge records by vertex instead of by slot. Vertex merging against the
FP64 oracle with one path, with fewer vertices than a block, and with long paths across many blocks."""
import numpy as np
import pytest

from oracle import pyoracle as po
from smallupbp_amd import native, scenes

from gpu_helpers import REL_TOL, gpu_context, print_case, rel_err


@pytest.mark.gpu
@pytest.mark.parametrize("n_paths,length", [(1, 3), (12, 18), (70, 4), (700, 18), (3000, 9)])
@pytest.mark.parametrize("kind", ["pp3d", "surf"])
def test_merging_with_long_paths(kind, n_paths, length):
    print_case("light_tails", kind=kind, paths=n_paths, length=length)
    make = scenes.pp3d_scene if kind == "pp3d" else scenes.surf_scene
    sc = make(n_paths=n_paths, n_queries=2000, radius=0.1, cell_count=2999, seed=91 + n_paths, max_light_length=length)
    ref, _, cnt = po.vm_eval(po.OracleHashGrid(sc), sc, precision=64)
    ctx = gpu_context(sc.media)
    grid = native.HashGrid(ctx)
    grid.build(sc.positions, sc.mis.light_vertices, sc.radius, sc.cell_count, sc.technique)
    out = grid.eval(sc.queries, sc.mis)
    assert np.max(rel_err(out, ref)) <= REL_TOL
    grid.destroy()
