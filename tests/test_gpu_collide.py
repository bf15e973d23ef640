"""Proximity-query parity: GPU CD2 / CD records against the oracle's brute-force
restatement of btc::pointTriCollision and btc::boxTriCollision.

Bar: bit-exact -- every field of every record (indices, types, and the FP64
distances, normals, positions and weights compared by bit pattern), in the
reference's order."""
import ctypes as C

import numpy as np
import pytest

import eolc
import oracle as O
from eolc import scene

pytestmark = pytest.mark.gpu

FIELDS = ("dist", "nor1", "nor2", "pos1", "pos2", "pos1_", "count1", "count2", "verts1", "verts2",
          "weights1", "weights2", "tri1", "tri2", "nedge1", "edge2", "edgeDir")


def rec_tuple(r):
    out = []
    for f in FIELDS:
        v = getattr(r, f)
        if isinstance(v, float):
            out.append(np.float64(v).tobytes())
        elif isinstance(v, int):
            out.append(v)
        else:
            a = np.array(list(v))
            out.append(a.tobytes() if a.dtype.kind == "f" else tuple(a.tolist()))
    out.append(tuple(list(r.edge1)[: r.nedge1]))
    return tuple(out)


def oracle_cd(thr, pts, nrm, whd, E, x, tri, eol=False, box_npts=8, box_nedges=12):
    n, recs = O.point_tri(thr, pts, nrm, x, tri, eol=eol)
    assert n >= 0
    P = len(pts)
    out = list(recs)
    for b in range(len(whd)):
        nb, br = O.box_tri(thr, whd[b], E[b], x, tri, eol=False)
        assert nb >= 0
        if eol:
            base = P + b * box_npts + b * box_nedges
            for r in br:
                if r.count1 == 1 and r.count2 == 3:
                    r.verts1[0] = base + r.verts1[0]
                for e in range(r.nedge1):
                    r.edge1[e] = base + (box_npts + r.edge1[e])
        out.extend(br)
    return out


def compare(ctx, sc, x, thr, pts, nrm, whd, E, eol=False):
    ctx.set_topology(sc.X, sc.tri, sc.hinge)
    ctx.upload_state(x, np.zeros_like(x))
    g = ctx.collide(thr, pts, nrm, whd, E, eol_points=eol)
    o = oracle_cd(thr, pts, nrm, whd, E, x, sc.tri, eol=eol)
    kinds = {}
    for r in o:
        kinds[(r.count1, r.count2)] = kinds.get((r.count1, r.count2), 0) + 1
    print(f"records gpu {len(g)} oracle {len(o)} kinds {kinds}", flush=True)
    assert len(g) == len(o)
    for k, (a, b) in enumerate(zip(g, o)):
        assert rec_tuple(a) == rec_tuple(b), f"record {k} differs"
    return kinds


def thin_box_scene(n, sigma):
    sc = scene.Scene(n, sigma_x=sigma)
    pts, nrm, whd, E = scene.obstacles(seed=1236, P=64, B=4)
    # one thin box whose corners reach the cloth (V1-T2), one tilted box
    whd = np.vstack([whd, [0.2, 0.15, 0.006]])
    E = list(E) + [np.eye(4)]
    E[-1][0, 3], E[-1][1, 3], E[-1][2, 3] = 0.37, 0.61, 0.0011
    R = np.eye(4)
    c, s = np.cos(0.4), np.sin(0.4)
    R[:3, :3] = [[c, -s, 0], [s * 0.9, c * 0.9, 0.43589], [-s * 0.43589, -c * 0.43589, 0.9]]
    R[:3, :3] = np.linalg.qr(R[:3, :3])[0]
    R[0, 3], R[1, 3], R[2, 3] = 0.7, 0.3, 0.01
    whd = np.vstack([whd, [0.12, 0.1, 0.08]])
    E.append(R)
    return sc, pts, nrm, whd, E


def test_cd2_parity_small(ctx):
    sc, pts, nrm, whd, E = thin_box_scene(96, 1e-3)
    kinds = compare(ctx, sc, sc.x0, 1e-3, pts, nrm, whd, E)
    assert set(kinds) >= {(1, 3), (3, 1), (2, 2)}          # every record type occurs


def test_constraint_rows_from_gpu_records(ctx):
    """Constraints::fill collision rows (Constraints.cpp:417-470) from the GPU's CD2
    records equal the restated loop applied to the oracle's records, exactly."""
    from test_constraints import restated
    sc, pts, nrm, whd, E = thin_box_scene(96, 1e-3)
    ctx.set_topology(sc.X, sc.tri, sc.hinge)
    ctx.upload_state(sc.x0, np.zeros_like(sc.x0))
    g = ctx.collide(1e-3, pts, nrm, whd, E)
    o = oracle_cd(1e-3, pts, nrm, whd, E, sc.x0, sc.tri)
    A = eolc.collision_constraints(g, sc.N)
    R = restated(o, sc.N)
    print(f"constraint rows {A.shape[0]} from {len(g)} records, nnz {A.nnz}", flush=True)
    assert A.shape == R.shape and A.shape[0] > 0
    assert (abs(A - R)).max() == 0.0


def test_cd_eol_points_parity(ctx):
    sc, pts, nrm, whd, E = thin_box_scene(64, 1e-3)
    # points right on the cloth so the EOL vertex-point branch fires
    pts = pts.copy()
    pts[:8, :2] = sc.X[[5, 77, 300, 901, 1500, 2222, 3000, 4000]]
    pts[:8, 2] = 1e-4
    compare(ctx, sc, sc.x0, 2e-3, pts, nrm, whd, E, eol=True)


def test_cd2_no_obstacles_and_far_obstacles(ctx):
    sc = scene.Scene(16, sigma_x=1e-3)
    ctx.set_topology(sc.X, sc.tri, sc.hinge)
    ctx.upload_state(sc.x0, np.zeros_like(sc.x0))
    assert ctx.collide(1e-3) == []
    pts = np.array([[0.5, 0.5, 3.0]]); nrm = np.array([[0, 0, 1.0]])
    assert ctx.collide(1e-3, pts, nrm) == []


def test_overflow_reports_required_size(ctx):
    sc, pts, nrm, whd, E = thin_box_scene(48, 1e-3)
    ctx.set_topology(sc.X, sc.tri, sc.hinge)
    ctx.upload_state(sc.x0, np.zeros_like(sc.x0))
    full = ctx.collide(1e-3, pts, nrm, whd, E)
    assert len(full) > 1
    buf = (eolc.CollisionRec * 1)()
    cnt = C.c_int(0)
    Es = np.concatenate([np.asarray(e).T.reshape(-1) for e in E])
    rc = eolc.lib().eolc_collide(ctx._h, 1e-3, len(pts), pts.ctypes.data_as(C.c_void_p),
                                 nrm.ctypes.data_as(C.c_void_p), len(whd),
                                 np.ascontiguousarray(whd).ctypes.data_as(C.c_void_p),
                                 Es.ctypes.data_as(C.c_void_p), 0, 8, 12, buf, 1, C.byref(cnt))
    assert rc == eolc.ERR_OVERFLOW and cnt.value == len(full)


def test_cd2_parity_config2(ctx):
    """512x512 cloth with noise 1e-3, 64 points and 4 boxes at threshold 1e-3."""
    sc = scene.Scene(512, sigma_x=1e-3)
    pts, nrm, whd, E = scene.obstacles(seed=1236, P=64, B=4)
    compare(ctx, sc, sc.x0, 1e-3, pts, nrm, whd, E)


def _material_layout(verts, tri):
    """A material-space layout with every face CCW (the context requires positive
    areas): the first axis-pair projection of the positions that has one."""
    v = np.asarray(verts, dtype=np.float64)
    for i, j in ((0, 1), (1, 0), (0, 2), (2, 0), (1, 2), (2, 1)):
        X = v[:, [i, j]]
        a, b, c = X[tri[:, 0]], X[tri[:, 1]], X[tri[:, 2]]
        if np.all((b[:, 0] - a[:, 0]) * (c[:, 1] - a[:, 1]) - (b[:, 1] - a[:, 1]) * (c[:, 0] - a[:, 0]) > 0):
            return X
    raise AssertionError("no CCW projection")


@pytest.mark.parametrize("name", ["point_over_triangle", "points_nearest_and_tie", "eol_points",
                                  "corner_under_triangle", "vertex_inside_box", "edge_through_box_edge"])
def test_closed_form_scenes(ctx, name):
    """The hand-worked scenes of the oracle's pins through the GPU path: records bit
    for bit equal to the oracle's, and equal to the closed-form values."""
    import collide_scenes as S
    print(f"closed-form collision scene {name}", flush=True)
    built = getattr(S, name)()
    if len(built) == 4:
        verts, tri, pts, nrm = built
        whd, E = np.zeros((0, 3)), []
    else:
        verts, tri = built
        pts, nrm = np.zeros((0, 3)), np.zeros((0, 3))
        whd, E = S.BOX_WHD[None, :], [S.box_frame(S.BOX_CENTER)]
    eol = name == "eol_points"
    X = _material_layout(verts, tri)
    ctx.set_topology(X, tri, np.zeros((0, 4), dtype=np.int32))
    x = np.asarray(verts, dtype=np.float64).reshape(-1)
    ctx.upload_state(x, np.zeros_like(x))
    g = ctx.collide(S.THR, pts, nrm, whd, E, eol_points=eol)
    o = oracle_cd(S.THR, pts, nrm, whd, E, x, tri, eol=eol)
    assert len(g) == len(o) and len(g) > 0
    for k, (a, b) in enumerate(zip(g, o)):
        assert rec_tuple(a) == rec_tuple(b), f"record {k} differs"
    exp_fn = getattr(S, "expected_" + name, None)
    if exp_fn is not None:
        v2 = S.jittered(verts, O.mt19937_uniform)
        exp = exp_fn(v2)
        S.compare(g[: len(exp)] if eol else g, exp)


@pytest.mark.parametrize("n", [51, 52, 64, 74])
def test_counts_at_the_scan_pieces(ctx, n):
    """Record offsets come from scans over the edges and the grid's buckets in pieces of
    8,192 counts: 7,905 and 8,216 edges (one piece, one and a remainder), 8,192 faces
    (16,384 buckets, two whole pieces) and 16,576 edges; every record bit for bit."""
    sc, pts, nrm, whd, E = thin_box_scene(n, 1e-3)
    assert compare(ctx, sc, sc.x0, 2e-3, pts, nrm, whd, E)


@pytest.mark.parametrize("P,B", [(2048, 0), (2049, 0), (1, 9), (0, 8)])
def test_query_and_box_group_edges(ctx, P, B):
    """Up to 2,048 queries are swept over all faces, more take the grid; boxes run eight to
    a launch.  Both sides of each, with faces too ill-shaped for the box reject (a third
    of the sheet flattened to a line), record for record."""
    sc = scene.Scene(23, sigma_x=1e-3)
    pts, nrm, whd, E = scene.obstacles(seed=40 + P + B, P=P, B=max(B, 1))
    x = sc.x0.reshape(-1, 3).copy()
    x[: sc.N // 3, 1:] = 0.0
    if B:
        compare(ctx, sc, x.reshape(-1), 2e-3, pts, nrm, whd, E)
    else:
        assert compare(ctx, sc, x.reshape(-1), 2e-3, pts, nrm, np.zeros((0, 3)), [])


def test_sweep_list_overflow_takes_the_grid(ctx):
    """More candidates than the sweep keeps (65,536): 1,500 points over 128 faces stacked
    on each other, every point within the band of half of them."""
    k = 64
    X = np.zeros((4 * k, 2))
    tri = np.zeros((2 * k, 3), dtype=np.int32)
    x = np.zeros((4 * k, 3))
    for s in range(k):
        X[4 * s:4 * s + 4] = np.array([[0, 0], [1, 0], [0, 1], [1, 1]]) + [2.0 * s, 0.0]
        x[4 * s:4 * s + 4, :2] = [[0, 0], [1, 0], [0, 1], [1, 1]]
        x[4 * s:4 * s + 4, 2] = 1e-7 * s
        tri[2 * s:2 * s + 2] = np.array([[0, 1, 2], [1, 3, 2]]) + 4 * s
    rng = np.random.default_rng(3)
    P = 1500
    pts = np.concatenate([rng.uniform(0.05, 0.95, size=(P, 2)), np.full((P, 1), 2e-3)], axis=1)
    nrm = np.tile([0.0, 0.0, 1.0], (P, 1))
    ctx.set_topology(X, tri, np.zeros((0, 4), dtype=np.int32))
    ctx.upload_state(x.reshape(-1), np.zeros(x.size))
    g = ctx.collide(1e-3, pts, nrm)
    o = oracle_cd(1e-3, pts, nrm, np.zeros((0, 3)), [], x.reshape(-1), tri)
    print(f"{len(g)} records", flush=True)
    assert len(g) == len(o) == P
    assert all(rec_tuple(a) == rec_tuple(b) for a, b in zip(g, o))


@pytest.mark.parametrize("order", [(0, 6, 1, 6, 0, 2), (6, 6, 6)])
def test_calls_that_share_the_kept_block(ctx, order):
    """Queries of different sizes after one another on one topology (the context's block
    grows, then holds less than it could), a velocity transfer between them: every call's
    records are those of a context that makes this call alone."""
    sc, pts, nrm, whd, E = thin_box_scene(24, 1e-3)
    x, thr = sc.x0, 5e-3

    def on(c):
        c.set_topology(sc.X, sc.tri, sc.hinge)
        c.upload_state(x, np.zeros_like(x))
        return c

    def call(c, nb):
        return [rec_tuple(r) for r in c.collide(thr, pts, nrm, whd[:nb], E[:nb])]

    want = {}
    for nb in set(order):
        with eolc.Context(0) as c:
            want[nb] = call(on(c), nb)
    assert len(want[max(order)]) > 0
    on(ctx)
    new = np.random.default_rng(4).uniform(0.05, 0.95, (500, 2)) * sc.X.max(axis=0)
    moved = None
    for k, nb in enumerate(order):
        print(f"kept block: call {k}, {nb} boxes", flush=True)
        assert call(ctx, nb) == want[nb]
        got = ctx.velocity_transfer(sc.X, sc.v0, sc.tri, new)[1]
        assert moved is None or np.array_equal(got, moved)
        moved = got


def test_kept_block_after_a_call_beyond_its_limit():
    """A query that needs more than the 256 MB a context keeps (1,000,000 points, 316 bytes
    each) leaves the block to the smaller queries after it: their memory (200,000 points)
    is held from the second one on, also over a new topology, and given back with the
    context."""
    sc, pts, nrm, _, _ = thin_box_scene(24, 1e-3)
    rng = np.random.default_rng(6)
    many = np.concatenate([rng.uniform(0.0, 1.0, (1_000_000, 2)), np.full((1_000_000, 1), 5.0)], axis=1)
    up = np.tile([0.0, 0.0, 1.0], (len(many), 1))

    def free():
        now, total = C.c_size_t(0), C.c_size_t(0)
        assert C.CDLL(eolc.LIB_PATH).hipMemGetInfo(C.byref(now), C.byref(total)) == 0   # (the library's own runtime)
        return now.value

    with eolc.Context(0) as c:
        for k in range(2):
            c.set_topology(sc.X, sc.tri, sc.hinge)
            c.upload_state(sc.x0, np.zeros_like(sc.x0))
            if k == 0:
                start = free()
                for n in (1_000_000, 200_000, 200_000):
                    print(f"kept block: {n} points, {(start - free()) >> 20} MB held before", flush=True)
                    assert c.collide(1e-3, many[:n], up[:n]) == []
            held = start - free()
            print(f"kept block: {held >> 20} MB held", flush=True)
            assert 50 << 20 <= held <= 256 << 20
    print(f"kept block: {(start - free()) >> 20} MB held after the context", flush=True)
    assert start - free() <= 8 << 20
