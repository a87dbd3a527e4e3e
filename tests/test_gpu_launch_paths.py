"""Launch paths chosen by sizes, compared with the oracle or with the general path
at the sizes where they can go wrong."""
import numpy as np
import pytest

from helpers import ModelArrays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ring", [3, 8, 9, 21])
def test_bending_of_vertices_with_any_number_of_triangles(gpu, po, ring):
    """The bending chain takes 8 lanes per vertex: a bipyramid has two vertices with
    `ring` triangles (fewer than the lanes, as many, one more, several rounds) and
    the others with four.  The chain is FP64 on both sides, so only the rounding of
    the force to FP32 (6e-8) and FP64 rounding through the cotangents remain."""
    pfg = gpu
    rng = np.random.default_rng(ring)
    th = 2 * np.pi * np.arange(ring) / ring
    P = np.concatenate([np.stack([3 * np.cos(th), 3 * np.sin(th), 0 * th], 1),
                        [[0, 0, 2.0], [0, 0, -2.0]]])
    P = (P + rng.uniform(-0.1, 0.1, P.shape) + 24).astype(np.float32)
    tri = []
    for k in range(ring):
        j = (k + 1) % ring
        tri += [[k, j, ring], [j, k, ring + 1]]
    tri = np.array(tri, np.int32)
    p = pfg.default_params(nx=48, ny=48, nz=48)
    p.morse_u0, p.kbend = 0.0, 2.0
    ma = ModelArrays(*P.T, plt_elem_start=[0, len(P)], plt_tri_start=[0, len(tri)],
                     tri=tri.ravel(), tri_S0=np.ones(len(tri)), plt_S0=[1.0], plt_V0=[1.0])
    o = po.Oracle(p, model=ma.model)
    with pfg.Solver(p) as s:
        s.load(ma.model)
        for st in (pfg.STAGE_CELLS, pfg.STAGE_MEMBRANE, pfg.STAGE_BONDS, pfg.STAGE_FORCES):
            s.stage(st)
            o.stage(st)
        mk = s.markers()
    for k in ("fx", "fy", "fz"):
        want = o.marker(k)
        assert np.abs(want).max() > 0
        assert np.abs(mk[k] - want).max() < 1e-6 * np.abs(want).max()
