"""Launch paths chosen by sizes, compared with the oracle or with the general path
at the sizes where they can go wrong."""
from concurrent.futures import ThreadPoolExecutor

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


ODD_SIZES = [(1, 1, 1), (1, 7, 5), (2, 100, 4), (5, 7, 3), (21, 3, 2), (33, 70, 4), (63, 2, 9),
             (64, 1, 5), (65, 3, 2), (127, 4, 3), (130, 65, 3)]


@pytest.mark.parametrize("walls", [(0, 0, 0), (1, 1, 1), (0, 1, 2)])
@pytest.mark.parametrize("size", ODD_SIZES, ids=lambda s: "x".join(map(str, s)))
def test_blocks_across_rows_and_planes(gpu, po, size, walls):
    """Blocks of 64 cells run across rows and planes: axes shorter and longer than a
    wavefront, several rows or planes in one block, a last block partly empty, with
    every wall kind and with a tenth of the cells solid (where no velocity face sets
    the cells).  One step of a state 5 % off the weights: FP32 rounding of values
    below 0.5 through some ten operations stays under 2e-7."""
    pfg = gpu
    nx, ny, nz = size
    if walls[2] == 2 and nz < 2:
        pytest.skip("two velocity faces need two planes")
    N = nx * ny * nz
    rng = np.random.default_rng(N)
    flags = None if walls[2] == 2 else (rng.random(N) < 0.1).astype(np.uint8)
    p = pfg.default_params(nx=nx, ny=ny, nz=nz, use_flags=int(flags is not None))
    for a in range(3):
        p.wall[a] = walls[a]
    p.body_force[0] = 1e-5
    p.wall_u_hi[2][0] = 0.02
    p.wall_u_lo[2][1] = 0.01
    w = np.array([po.load().orc_w(d) for d in range(19)])[:, None]
    f = (w * (1 + 0.05 * rng.standard_normal((19, N)))).astype(np.float32)
    with pfg.Solver(p) as s:
        if flags is not None:
            s.upload_flags(flags)
        s.set_f(f)
        s.set_fluid_only(True)
        s.step(1)
        fg, fields = s.f().astype(np.float64), s.fields()
    L = po.lattice(p, flags)
    fo = po.lb_step(L, f.astype(np.float64))
    fluid = np.ones(N, bool) if flags is None else flags == 0
    assert np.abs(fg - fo)[:, fluid].max(initial=0.0) < 2e-7
    for got, want in zip(fields, po.fields(L, fo)):
        assert np.abs(got - want)[fluid].max(initial=0.0) < 1e-6
        assert (got[~fluid] == 0).all()


@pytest.mark.parametrize("solid", [False, True])
@pytest.mark.parametrize("store, half_ulp", [(0, 0.0), (1, 2.0 ** -11)])
@pytest.mark.parametrize("size", [(5, 7, 3), (64, 3, 2), (67, 66, 5), (131, 130, 132)],
                         ids=lambda s: "x".join(map(str, s)))
def test_moving_walls_of_every_axis(gpu, po, size, store, half_ulp, solid):
    """Walls on every side, each with its own velocity, their edges and corners, solid
    cells beside them, in lattices that stay in the cache and in one that does not
    (where FP32 takes the loads in another way).  From the stored state: the rounding
    of one FP32 step (3e-7), and half an ulp of the stored deviation."""
    pfg = gpu
    nx, ny, nz = size
    N = nx * ny * nz
    rng = np.random.default_rng(N + store)
    flags = (rng.random(N) < 0.1).astype(np.uint8) if solid else None
    p = pfg.default_params(nx=nx, ny=ny, nz=nz, store=store, use_flags=int(solid))
    for a in range(3):
        p.wall[a] = pfg.WALL_BOUNCE
        for c in range(3):
            if c != a:
                p.wall_u_lo[a][c], p.wall_u_hi[a][c] = rng.uniform(-0.05, 0.05, 2)
    w = np.array([po.load().orc_w(d) for d in range(19)])[:, None]
    f = (w * (1 + 0.05 * rng.standard_normal((19, N)))).astype(np.float32)
    with pfg.Solver(p) as s:
        if solid:
            s.upload_flags(flags)
        s.set_f(f)
        f = s.f().astype(np.float64)
        s.set_fluid_only(True)
        s.step(1)
        fg = s.f().astype(np.float64)
    fo = po.lb_step(po.lattice(p, flags), f)
    fluid = slice(None) if flags is None else flags == 0
    err = np.abs(fg - fo) - 1.01 * half_ulp * np.abs(fo - w)
    assert err[:, fluid].max(initial=0.0) < 3e-7


@pytest.mark.parametrize("nx", [60, 101])
def test_overlap_equals_serial_on_rows_that_share_blocks(gpu, nx):
    """The blocks that the stencils touch are stamped by cell index: a platelet
    across the periodic x face of a lattice whose rows share blocks.  Only the
    arrival order of the force field's atomics differs."""
    pfg = gpu
    sc = pfg.Scene(pfg.SCENE_SHEAR, nx=nx, ny=33, nz=31, elements=256, receptors=-1, ligands=-1)
    sc.x[:] += nx - 0.25 * nx
    res = []
    for overlap in (False, True):
        with pfg.Solver(sc.params) as s:
            s.load(sc)
            s.set_overlap(overlap)
            s.step(16)
            res.append((s.f(), s.markers()))
    assert np.abs(res[0][0] - res[1][0]).max() < 1e-6
    for k in ("x", "y", "z", "vx", "vy", "vz"):
        assert np.abs(res[0][1][k] - res[1][1][k]).max() < 1e-5, k


def fibrin_cloud(pfg, n, nx=48):
    """n free fibrin nodes without links on a small lattice."""
    rng = np.random.default_rng(n)
    P = (rng.random((3, n)) * nx).astype(np.float32)
    p = pfg.default_params(nx=nx, ny=nx, nz=nx)
    ma = ModelArrays(*P, kind=np.full(n, pfg.MARKER_FIBER), body=np.full(n, -1))
    s = pfg.Solver(p)
    s.load(ma.model)
    s._keep = ma
    return s, P


@pytest.mark.parametrize("n", [1, 3, 29127, 29128, 233017, 300001])
def test_frames_of_any_size(gpu, n):
    """A frame of nine arrays goes through one small pinned buffer (up to 29127
    markers: 1 MiB), one half of a large one (up to 233016: 8 MiB) or several, with
    array and batch boundaries apart: every value arrives, exactly."""
    pfg = gpu
    s, P = fibrin_cloud(pfg, n)
    with s:
        rng = np.random.default_rng(1)
        F, V = (rng.standard_normal((3, n)).astype(np.float32) for _ in range(2))
        s.set_marker_forces(*F)
        s.set_marker_velocities(*V)
        for _ in range(2):
            m = s.markers()
            for names, want in (("xyz", P), (("vx", "vy", "vz"), V), (("fx", "fy", "fz"), F)):
                for k, a in zip(names, want):
                    assert np.array_equal(m[k], a), k


def test_frames_from_several_threads(gpu):
    """Handles in threads of their own download at once (buffers are shared by the
    process, a call holds one): the same values as one after the other."""
    pfg = gpu
    solvers = []
    for k in range(4):
        p = pfg.default_params(nx=96 + 7 * k, ny=90, nz=80, store=k % 3)
        p.body_force[0] = 1e-5
        p.wall[1] = pfg.WALL_BOUNCE
        s = pfg.Solver(p)
        s.step(3 + k)
        solvers.append(s)
    want = [s.fields() for s in solvers]

    def work(k):
        return [all(np.array_equal(a, b) for a, b in zip(solvers[k].fields(), want[k]))
                for _ in range(5)]

    with ThreadPoolExecutor(4) as pool:  # a failed download raises from map
        same = list(pool.map(work, range(4)))
    for s in solvers:
        s.close()
    assert np.all(same)


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("size", [(64, 6, 5), (33, 7, 5), (130, 65, 3)])
def test_fields_of_solid_cells_are_zero(gpu, size, noalloc):
    """Solid cells read 0, in blocks of 64 solid cells, in mixed ones and in a last block
    partly empty, where the buffers still hold the frame of a larger lattice."""
    import ctypes as C
    pfg = gpu
    nx, ny, nz = size
    N = nx * ny * nz

    def fields(s):
        if not noalloc:
            return s.fields()
        out = [np.full(s.N, 7.0, np.float32) for _ in range(4)]
        assert pfg.lib().pfg_download_fields_noalloc(
            C.c_void_p(s._h.value), *[a.ctypes.data_as(C.POINTER(C.c_float)) for a in out]) == 0
        return out

    flags = (np.random.default_rng(N).random(N) < 0.1).astype(np.uint8)
    flags[64:64 * 7] = 1
    flags[N - N % 64 - 64:] = 1
    p = pfg.default_params(nx=nx, ny=ny, nz=nz, use_flags=1)
    big = pfg.default_params(nx=96, ny=64, nz=64)
    for q in (p, big):
        q.body_force[0] = q.body_force[1] = q.body_force[2] = 1e-5
    with pfg.Solver(big) as b, pfg.Solver(p) as s:
        b.step(2)
        s.upload_flags(flags)
        s.step(2)
        assert all((a != 0).all() for a in fields(b))
        for a in fields(s):
            assert (a[flags != 0] == 0).all()
            assert (a[flags == 0] != 0).any()


def test_noalloc_fields_with_velocity_faces(gpu):
    """Both field downloads impose the velocity faces: equal bit for bit."""
    import ctypes as C
    pfg = gpu
    p = pfg.default_params(nx=40, ny=30, nz=20)
    p.wall[0] = p.wall[1] = pfg.WALL_BOUNCE
    p.wall[2] = pfg.WALL_VELOCITY
    p.wall_u_lo[2][2] = p.wall_u_hi[2][2] = 0.04
    with pfg.Solver(p) as s:
        s.step(7)
        want = s.fields()
        got = [np.empty(s.N, np.float32) for _ in range(4)]
        st = pfg.lib().pfg_download_fields_noalloc(
            C.c_void_p(s._h.value), *[a.ctypes.data_as(C.POINTER(C.c_float)) for a in got])
        assert st == 0
        for a, b in zip(got, want):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("by_body", [1, 2])
@pytest.mark.parametrize("staging", [1, 2, 3, 4])
def test_markers_that_left_every_range(gpu, staging, by_body):
    """A run that has diverged ends in numbers, not in a fault: elements far below a
    wall (beyond the range of int), far along a periodic axis, infinite or not a
    number.  The stencil index of such a coordinate used to overflow past its range
    check.  The fluid around the lost elements is lost with them; a platelet far
    from them steps on."""
    pfg = gpu
    sc = pfg.Scene(pfg.SCENE_LARGE, nx=128, ny=64, nz=64, n_platelets=3, elements=200,
                   receptors=16, ligands=256, fibrin_nodes=64, fibrin_links=80)
    x, y, z = sc.x.copy(), sc.y.copy(), sc.z.copy()
    first, lost, healthy = (np.flatnonzero(sc.body == b) for b in range(3))
    z[first] = -3e9
    x[lost[0]], y[lost[1]], x[lost[2]], z[lost[3]] = 1e30, np.inf, np.nan, 3e38
    with pfg.Solver(sc.params) as s:
        s.load(sc)
        s.set_ib_staging(staging)
        s.set_forces_by_body(by_body)
        s.set_forces_lanes(4 if by_body == 1 else 0)
        s.set_markers(x, y, z)
        s.step(2)
        m = s.markers()
    assert all(np.isfinite(m[k][healthy]).all() for k in ("x", "y", "z", "fx", "fy", "fz"))
    assert (m["z"][first] < -2e9).all()


def cloud_model(sizes, nx=48):
    """Platelets of `sizes` elements as random clouds, about 20 Morse partners each."""
    rng = np.random.default_rng(sum(sizes))
    P, body = [], []
    for b, n in enumerate(sizes):
        side = 0.72 * n ** (1 / 3)
        P.append(rng.random((n, 3)) * side + rng.random(3) * (nx - 1))
        body += [b] * n
    P, body = np.concatenate(P), np.array(body)
    start = np.concatenate([[0], np.cumsum(sizes)])
    return ModelArrays(*P.T, body=body, plt_elem_start=start,
                       plt_tri_start=np.zeros(len(sizes) + 1), tri_S0=[],
                       plt_S0=np.ones(len(sizes)), plt_V0=np.ones(len(sizes)))


@pytest.mark.parametrize("sizes", [(1, 2), (63, 64, 65), (127, 1, 128, 129), (4096,), (4097, 70)])
def test_morse_from_runs_of_the_platelet(gpu, sizes):
    """A wavefront per marker takes its Morse candidates from runs of 64 elements
    (part runs, several platelets in turn, the longest platelet that has a lane per
    run), or from the cell lists where a platelet is longer: the forces of the 4-lane
    pass over the cell lists, to the rounding of sums of some 20 terms of up to 80."""
    pfg = gpu
    ma = cloud_model(sizes)
    p = pfg.default_params(nx=48, ny=48, nz=48, bin_cells=2)
    p.morse_u0, p.morse_cutoff = 1.0, 1.2
    p.wall[2] = pfg.WALL_BOUNCE
    F = []
    for lanes in (64, 4):
        with pfg.Solver(p) as s:
            s.load(ma.model)
            s.set_forces_by_body(2)
            s.set_forces_lanes(lanes)
            for st in (pfg.STAGE_CELLS, pfg.STAGE_MEMBRANE, pfg.STAGE_FORCES):
                s.stage(st)
            m = s.markers()
            F.append(np.stack([m["fx"], m["fy"], m["fz"]]))
    assert np.abs(F[0] - F[1]).max() <= 1e-5 * max(1.0, np.abs(F[1]).max())
    assert sum(sizes) < 4 or np.abs(F[1]).max() > 0


@pytest.mark.parametrize("setting, values", [("set_forces_lanes", (4, 64)),
                                             ("set_forces_by_body", (1, 2))])
def test_settings_between_the_cells_and_the_forces(gpu, setting, values):
    """What CELLS leaves serves the force pass of any later setting: the forces of a
    handle that had the setting from the start, in both directions of the change."""
    pfg = gpu
    ma = cloud_model((200, 300))
    p = pfg.default_params(nx=48, ny=48, nz=48, bin_cells=2)
    p.morse_u0, p.morse_cutoff = 1.0, 1.2
    for first, then in (values, values[::-1]):
        F = []
        for before in (first, then):
            with pfg.Solver(p) as s:
                s.load(ma.model)
                s.set_ib_staging(1)
                getattr(s, setting)(before)
                for st in (pfg.STAGE_CELLS, pfg.STAGE_MEMBRANE):
                    s.stage(st)
                getattr(s, setting)(then)
                s.stage(pfg.STAGE_FORCES)
                m = s.markers()
                F.append(np.stack([m["fx"], m["fy"], m["fz"]]))
        assert np.abs(F[1]).max() > 0
        assert np.abs(F[0] - F[1]).max() <= 1e-5 * np.abs(F[1]).max()


DEFAULT, LISTS, BODY = (0, 0, 0), (4, 2, 1), (4, 1, 1)  # lanes, by body, staging


@pytest.mark.parametrize("fibrin_ligands", [0, 1])
@pytest.mark.parametrize("stage, stepped, then", [
    ("FORCES", DEFAULT, LISTS), ("FORCES", LISTS, DEFAULT), ("FORCES", BODY, LISTS),
    ("BONDS", DEFAULT, DEFAULT), ("BONDS", BODY, LISTS), ("SPREAD", DEFAULT, (0, 0, 3))])
def test_stages_after_a_step_that_kept_other_lists(gpu, stage, stepped, then, fibrin_ligands):
    """A step keeps the lists it needs itself; a stage called afterwards gives what it
    gives after a step that keeps the lists of every marker (one step, so that both
    start from the same positions): the bonds exactly, forces to their rounding."""
    pfg = gpu
    sc = pfg.Scene(pfg.SCENE_LARGE, nx=64, ny=48, nz=48, n_platelets=2, elements=300,
                   receptors=64, ligands=256, fibrin_nodes=2000, fibrin_links=2000)
    sc.fibrin_ligands = fibrin_ligands
    m = sc.model()
    p = sc.params
    p.k_on, p.bond_reach, p.detach_rate = 0.5, 2.0, 0.0
    out = []

    def apply(s, lanes, by_body, staging):
        s.set_forces_lanes(lanes)
        s.set_forces_by_body(by_body)
        s.set_ib_staging(staging)

    for first, second in ((LISTS, LISTS if stage == "FORCES" else then), (stepped, then)):
        with pfg.Solver(p) as s:
            s.load(m)
            apply(s, *first)
            s.step(1)
            apply(s, *second)
            s.stage(getattr(pfg, "STAGE_" + stage))
            mk = s.markers()
            out.append((np.stack([mk["fx"], mk["fy"], mk["fz"]]), s.bonds()[0], s.aux()))
    (F0, bonds0, aux0), (F1, bonds1, aux1) = out
    assert np.array_equal(bonds0, bonds1)
    assert stage != "BONDS" or not fibrin_ligands or (bonds0 >= m.n_wall_ligands).any()
    assert np.abs(F0).max() > 0 and (stage != "SPREAD" or np.abs(aux0).max() > 0)
    assert np.abs(F0 - F1).max() <= 1e-5 * np.abs(F0).max()
    assert np.abs(aux0 - aux1).max() <= 1e-5 * np.abs(aux0).max()


@pytest.mark.parametrize("receptors", [-1, 16])
@pytest.mark.parametrize("by_body", [0, 1])
def test_cell_lists_after_steps_without_them(gpu, by_body, receptors):
    """Steps that need no cell lists keep none, and those whose bonds read the fibrin
    nodes' lists keep these without an order; asked for afterwards, they are those
    of the positions the last step started from, as the CELLS stage gives them."""
    pfg = gpu
    sc = pfg.Scene(pfg.SCENE_LARGE, nx=96, ny=64, nz=64, n_platelets=3, elements=200,
                   receptors=receptors, ligands=receptors, fibrin_nodes=128, fibrin_links=150)
    with pfg.Solver(sc.params) as s:
        s.load(sc)
        s.set_forces_by_body(by_body)
        s.set_forces_lanes(4 if by_body else 0)  # 0: a wavefront each, which spreads too
        s.step(3)
        m = s.markers()
        s.step(1)
        got = s.cells()
    with pfg.Solver(sc.params) as s:
        s.load(sc)
        s.set_forces_by_body(by_body)
        s.set_forces_lanes(4 if by_body else 0)
        s.set_markers(m["x"], m["y"], m["z"])
        s.stage(pfg.STAGE_CELLS)
        want = s.cells()
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    n = want[1][-1]
    assert n == (128 if by_body else s.n_markers)
    if not by_body:
        assert np.array_equal(got[2][:n], want[2][:n])
    else:
        assert np.array_equal(np.sort(got[2][:n]), np.sort(want[2][:n]))


@pytest.mark.parametrize("kick", [False, True])
@pytest.mark.parametrize("fibrin", [16, 17, 2049])
def test_scattered_markers_beside_chunks(gpu, fibrin, kick):
    """Scattered fibrin nodes share the launches of the platelets' chunks, 16 or more
    per workgroup by their number: the force field, velocities and moves of the form
    without chunks (sums of FP32 terms in another order)."""
    pfg = gpu
    sc = pfg.Scene(pfg.SCENE_LARGE, nx=128, ny=96, nz=96, n_platelets=4, elements=300,
                   receptors=-1, ligands=-1, fibrin_nodes=fibrin, fibrin_links=8)
    p = sc.params
    if kick:
        p.fiber_move = pfg.FIBER_KICK
    f = np.random.default_rng(2).standard_normal((3, sc.n_markers)).astype(np.float32) * 1e-3
    out = []
    for form in (1, 2):
        with pfg.Solver(p) as s:
            s.load(sc)
            s.set_ib_staging(form)
            s.set_marker_forces(*f)
            s.stage(pfg.STAGE_SPREAD)
            F = s.aux()
            s.stage(pfg.STAGE_LB)
            s.stage(pfg.STAGE_INTERP)
            s.stage(pfg.STAGE_UPDATE)
            m = s.markers()
            out.append([F] + [m[k] for k in ("vx", "vy", "vz", "x", "y", "z")])
    scale = np.abs(out[1][0]).max()
    assert scale > 0
    assert np.abs(out[0][0] - out[1][0]).max() <= 2e-6 * scale
    for a, b in zip(out[0][1:4], out[1][1:4]):
        assert np.abs(a - b).max() <= 2e-6 * max(np.abs(b).max(), 1.0)
    for a, b in zip(out[0][4:], out[1][4:]):
        assert np.abs(a - b).max() <= 1e-5 * 128


@pytest.mark.parametrize("n, spacing", [(15, 2), (16, 2), (17, 2), (33, 3), (5000, 3),
                                        (33000, 2), (66000, 1.5)])
def test_clots_are_cut_until_their_chunks_fit(gpu, n, spacing):
    """Fibrin nodes close together beside as many far apart: chunks halved until their
    boxes fit, part of them listed.  The force field and the velocities of the direct
    form; a node's some 30 terms of at most 0.3 of a force in all, summed in another
    order on both sides, differ by less than 1e-6 of the largest force."""
    pfg = gpu
    rng = np.random.default_rng(n)
    side = int(np.ceil(n ** (1 / 3)))
    nx = int(side * spacing) + 24
    g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    P = np.concatenate([g * spacing + 8 + rng.uniform(-0.3, 0.3, g.shape),
                        rng.random((n, 3)) * nx])
    p = pfg.default_params(nx=nx, ny=nx, nz=nx)
    p.wall[1] = pfg.WALL_BOUNCE
    ma = ModelArrays(*P.T, kind=np.full(2 * n, pfg.MARKER_FIBER), body=np.full(2 * n, -1))
    f = rng.standard_normal((3, 2 * n)).astype(np.float32) * 1e-3
    out = []
    for form in (1, 2):
        with pfg.Solver(p) as s:
            s.load(ma.model)
            s.set_ib_staging(form)
            s.set_marker_forces(*f)
            s.stage(pfg.STAGE_SPREAD)
            F = s.aux()
            s.stage(pfg.STAGE_LB)
            s.stage(pfg.STAGE_INTERP)
            m = s.markers()
            out.append((F, np.stack([m["vx"], m["vy"], m["vz"]])))
    fmax = np.abs(f).max() * abs(p.ib_force_scale)
    assert np.abs(out[1][0]).max() > 0.1 * fmax
    assert np.abs(out[0][0] - out[1][0]).max() <= 1e-6 * fmax
    assert np.abs(out[0][1] - out[1][1]).max() <= 2e-6


def forces_after_a_step(pfg, p, ma, lanes):
    with pfg.Solver(p) as s:
        s.load(ma.model)
        s.set_forces_lanes(lanes)
        s.step(1)
        m = s.markers()
        return np.stack([m["fx"], m["fy"], m["fz"]])


@pytest.mark.parametrize("n, lanes", [(32767, 64), (32768, 4)])
def test_automatic_lanes_of_a_fibrin_network(gpu, n, lanes):
    """A model without platelets takes 4 lanes per node from 32768 nodes: bit for bit
    the forces of the lanes set by hand (eight links a node, summed in another order
    by other lanes)."""
    pfg = gpu
    rng = np.random.default_rng(n)
    P = (rng.random((3, n)) * 96).astype(np.float32)
    a = np.arange(n)
    link = np.stack([np.repeat(a, 4), (np.repeat(a, 4) + np.tile([1, 7, 57, 401], n)) % n], 1)
    d = np.linalg.norm(P[:, link[:, 0]] - P[:, link[:, 1]], axis=0)
    ma = ModelArrays(*P, kind=np.full(n, pfg.MARKER_FIBER), body=np.full(n, -1),
                     link=link.ravel(), link_l0=0.9 * d)
    p = pfg.default_params(nx=96, ny=96, nz=96)
    p.fiber_k = 1e-3
    F = {k: forces_after_a_step(pfg, p, ma, k) for k in (0, 4, 64)}
    assert not np.array_equal(F[4], F[64])
    assert np.array_equal(F[0], F[lanes])


def test_a_wavefront_by_choice_is_the_automatic_one(gpu):
    """64 lanes set by hand take the pass that the library takes by itself between 32768
    and 65535 markers: the same forces bit for bit (other passes sum in another order)."""
    pfg = gpu
    ma = cloud_model((1000,) * 33, nx=96)
    p = pfg.default_params(nx=96, ny=96, nz=96, bin_cells=2)
    p.morse_u0, p.morse_cutoff = 1e-4, 1.2
    F = {k: forces_after_a_step(pfg, p, ma, k) for k in (0, 4, 64)}
    assert not np.array_equal(F[4], F[64])
    assert np.array_equal(F[0], F[64])


@pytest.mark.parametrize("elements", [0, 2559, 2560])
@pytest.mark.parametrize("halt", [False, True])
def test_spreading_of_scattered_models(gpu, elements, halt):
    """The automatic form follows the markers in chunks, not the scattered ones beside
    them: one step of either form from the same state (velocities of order 1e-2 from
    sums in another order, forces through them at most the same)."""
    pfg = gpu
    rng = np.random.default_rng(elements)
    n, nx = 6000, 160
    E = rng.random((elements, 3)) * 0.9 * max(elements, 1) ** (1 / 3) + 70
    P = np.concatenate([E, rng.random((n, 3)) * nx])
    kind = np.repeat([pfg.MARKER_ELEMENT, pfg.MARKER_FIBER], [elements, n])
    kw = dict(plt_elem_start=[0, elements], plt_tri_start=[0, 0], tri_S0=[], plt_S0=[1.0],
              plt_V0=[1.0]) if elements else {}
    ma = ModelArrays(*P.T, kind=kind, body=np.where(kind == pfg.MARKER_ELEMENT, 0, -1), **kw)
    p = pfg.default_params(nx=nx, ny=nx, nz=nx)
    p.morse_u0, p.morse_cutoff = 1e-4, 1.2
    p.body_force[0] = 1e-5
    out = []
    for form in (0, 1, 2):
        with pfg.Solver(p) as s:
            s.load(ma.model)
            s.set_ib_staging(form)
            s.set_halt_on_detach(halt)
            s.step(1)
            m = s.markers()
            out.append(np.stack([m[k] for k in ("vx", "vy", "vz", "x", "y", "z")]))
    for a in out[:2]:
        assert np.abs(a[:3] - out[2][:3]).max() <= 1e-6
        assert np.abs(a[3:] - out[2][3:]).max() <= 1e-6 * nx


@pytest.mark.parametrize("store", [0, 1])
@pytest.mark.parametrize("force", [(1e-3, 0, 0), (0, 0, -1e-30), (0, float("nan"), 0)])
def test_force_field_is_empty_after_the_lb_update(gpu, store, force):
    """The LB update consumes the spread force: every cell that holds one, in any one
    component, however small, holds zero afterwards."""
    pfg = gpu
    sc = pfg.Scene(pfg.SCENE_SHEAR, nx=50, ny=33, nz=35, n_platelets=1, elements=200,
                   receptors=-1, ligands=-1, fibrin_nodes=-1)
    p = sc.params
    p.store = store
    f = np.repeat(np.asarray(force, np.float32)[:, None], sc.n_markers, axis=1)
    with pfg.Solver(p) as s:
        s.load(sc)
        s.set_marker_forces(*f)
        s.stage(pfg.STAGE_SPREAD)
        assert (s.aux() != 0).any()
        s.stage(pfg.STAGE_LB)
        assert (s.aux() == 0).all()
