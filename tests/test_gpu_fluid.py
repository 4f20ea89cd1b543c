"""GPU fluid path through the C ABI: FluidModel::step against the reference's
own outputs (via the fixture) and the FP64 oracle, and the frame path's
particle bookkeeping and rendering."""
import ctypes as C

import numpy as np
import pytest

from atomorph_amd import _capi as A
from atomorph_amd import morph as M
from oracle import oracle_py as op
from tests import gpu_util as G
from tests.test_gpu_render import GpuRenderer
from tests.test_oracle import render_inputs

pytestmark = pytest.mark.gpu

# FP32 grid against FP64: positions within 1e-4 cell, velocities 1e-4, colours 1e-4
TOL = {0: 1e-4, 1: 1e-4, 2: 1e-4, 3: 1e-4, 11: 1e-4, 12: 1e-4, 13: 1e-4, 14: 1e-4}


def _model(n, gsx, gsy, W=64, H=64):
    lib = G.lib()
    f = C.c_void_p()
    G.check(lib.amh_fluid_create(C.byref(f), gsx, gsy, n, W, H, 2, G.stream()), "amh_fluid_create")
    return f


def _step_gpu(P, gsx, gsy, steps, radius):
    lib = G.lib()
    n = P.shape[0]
    f = _model(n, gsx, gsy)
    try:
        Q = np.ascontiguousarray(P.copy())
        G.check(lib.amh_fluid_set_particles(f, op.ptr(Q), G.stream()), "set")
        outs = []
        for k in range(steps):
            G.check(lib.amh_fluid_step(f, steps - 1 - k, radius, 0, G.stream()), "step")
            G.check(lib.amh_fluid_get_particles(f, op.ptr(Q), G.stream()), "get")
            outs.append(Q.copy())
        return outs
    finally:
        lib.amh_fluid_destroy(f)


def test_fluid_step_matches_reference_fixture(golden_functions):
    g = golden_functions
    gx, gy, fr = (int(g["fluid_meta"][0]), int(g["fluid_meta"][1]), float(g["fluid_meta"][2]))
    G.log("fluid step vs fixture")
    outs = _step_gpu(g["fluid_in"], gx, gy, 3, fr)
    for k in range(3):
        want = g["fluid_out"][k]
        for col, tol in TOL.items():
            d = np.abs(outs[k][:, col] - want[:, col]).max()
            assert d <= tol * (k + 1), (k, col, d)


@pytest.mark.parametrize("layout", ["uniform", "clustered", "cell_sorted"])
def test_fluid_step_matches_oracle_many_particles(layout):
    """uniform: every block's particles span the grid (direct global
    scatter); clustered: runs of 256 particles around one centre, as chain
    atoms are (the LDS-tiled scatter), with a few wide runs mixed in;
    cell_sorted: the clustered particles ordered by cell, so runs of lanes
    share a stencil and are summed across lanes before they scatter."""
    rng = np.random.default_rng(4)
    n, gsx, gsy = 20480, 276, 276
    P = np.zeros((n, 20))
    if layout == "uniform":
        P[:, 0] = rng.uniform(8, 268, n)
        P[:, 1] = rng.uniform(8, 268, n)
    else:
        centres = rng.uniform(20, 256, (n // 256, 2))
        spread = np.where(np.arange(n // 256) % 10 == 0, 60.0, 3.0)
        P[:, 0] = np.clip(np.repeat(centres[:, 0], 256) + rng.normal(0, 1, n) * np.repeat(spread, 256), 8, 268)
        P[:, 1] = np.clip(np.repeat(centres[:, 1], 256) + rng.normal(0, 1, n) * np.repeat(spread, 256), 8, 268)
    P[:, 2:4] = rng.normal(0, 0.2, (n, 2))
    P[:, 4] = P[:, 0] + rng.normal(0, 3, n)
    P[:, 5] = P[:, 1] + rng.normal(0, 3, n)
    P[:, 6] = 1.0
    P[:, 7:15] = rng.uniform(0, 1, (n, 8))
    P[:, 15] = rng.choice([0.1, 1.0], n)
    P[:, 16] = (rng.uniform(0, 1, n) < 0.9).astype(float)
    P[:, 17] = rng.integers(0, 2, n)
    if layout == "cell_sorted":
        cx, cy = (P[:, 0] - 0.5).astype(int), (P[:, 1] - 0.5).astype(int)
        P = P[np.lexsort((cy, cx))]
    G.log(f"fluid step 20k particles, {layout}")
    outs = _step_gpu(P, gsx, gsy, 3, 20.0)
    Q = P.copy()
    o = op.oracle()
    for k in range(3):
        o.or_fluid_step(op.ptr(Q), n, gsx, gsy, 2 - k, 20.0, 0)
        for col in (0, 1, 2, 3):
            d = np.abs(outs[k][:, col] - Q[:, col]).max()
            assert d <= 2e-3, (k, col, d)
        assert (outs[k][:, 16] == Q[:, 16]).all()


@pytest.mark.parametrize("crowd", [1, 15, 16, 17, 63, 64, 65, 256, 257, 600])
@pytest.mark.parametrize("fill", [150, 6000])  # both sizes of work items
def test_fluid_step_of_crowded_cells_matches_oracle(crowd, fill):
    """Cells of `crowd` particles among thinly filled ones: runs of entries
    that end at, before and after the cuts of the lanes' rows, of a wave and of
    a work item, by a wall and away from it, in tiles that share nodes."""
    rng = np.random.default_rng(crowd)
    gsx, gsy = 64, 40
    xy = [np.array([c]) + rng.uniform(0, 1, (crowd, 2)) for c in ((30.5, 20.5), (31.5, 20.5), (2.5, 3.5), (39.5, 23.5))]
    xy.append(rng.uniform((2, 2), (gsx - 3, gsy - 3), (fill, 2)))
    xy = np.concatenate(xy)[rng.permutation(4 * crowd + fill)]
    n = len(xy)
    P = np.zeros((n, 20))
    P[:, 0:2] = xy
    P[:, 2:4] = rng.normal(0, 0.2, (n, 2))
    P[:, 4:6] = xy + rng.normal(0, 3, (n, 2))
    P[:, 6] = 1.0
    P[:, 7:15] = rng.uniform(0, 1, (n, 8))
    P[:, 15] = 1.0
    P[:, 16] = 1.0
    P[:, 17] = rng.integers(0, 2, n)
    G.log(f"fluid step, {crowd} particles in a cell")
    got = _step_gpu(P, gsx, gsy, 1, 20.0)[0]
    want = P.copy()
    op.oracle().or_fluid_step(op.ptr(want), n, gsx, gsy, 0, 20.0, 0)
    for col, tol in TOL.items():
        d = np.abs(got[:, col] - want[:, col]).max()
        assert d <= tol, (col, d)


def _lone_particle_step(P):
    """One model step of particles whose stencils meet no other's, away from
    the walls and within their freedom radius, in the engine's arithmetic: FP32
    node fields from the FP32 moments e^p h^q of each particle's cell, all else
    FP64 in the oracle's order.  Returns x, y, u, v."""
    f32 = np.float32
    kW = np.array([[0.125, -0.5, 0.5], [0.75, 0, -1], [0.125, 0.5, 0.5]], f32)
    kD = np.array([[0.5, -1, 0], [0, 2, 0], [-0.5, -1, 0]], f32)
    x, y, gravity = P[:, 0], P[:, 1], P[:, 4:6]
    cell = [(c - 0.5).astype(int) for c in (x, y)]
    e, h = x - cell[0] - 1.0, y - cell[1] - 1.0
    M = [[(a * b).astype(f32) for b in (np.ones_like(h), h, h * h)] for a in (np.ones_like(e), e, e * e)]

    def along(k, v):  # sum_p k[p] v[p]
        return (k[0] * v[0] + k[1] * v[1]) + k[2] * v[2]

    m, mx, my = (np.zeros((3, 3, len(P)), f32) for _ in range(3))
    for a in range(3):
        xw = [along(kW[a], [M[p][q] for p in range(3)]) for q in range(3)]
        xd = [along(kD[a], [M[p][q] for p in range(3)]) for q in range(3)]
        for b in range(3):
            m[a, b], mx[a, b], my[a, b] = along(kW[b], xw), along(kW[b], xd), along(kD[b], xw)

    def weights(c, v):
        t = c - v
        w = [0.5 * t * t + 1.5 * t + 1.125]
        d = [t + 1.5]
        t = t + 1.0
        w.append(-t * t + 0.75)
        d.append(-2.0 * t)
        t = t + 1.0
        return w + [0.5 * t * t - 1.5 * t + 1.125], d + [t - 1.5]

    (px, gx), (py, gy) = weights(cell[0], x), weights(cell[1], y)
    ix, iy, n = x.astype(int), y.astype(int), np.arange(len(P))

    def node(f, i, j):
        return f[ix + i - cell[0], iy + j - cell[1], n].astype(float)

    d01, d02, d11, d12 = (node(m, i, j) for i in (0, 1) for j in (0, 1))
    x01, x02, x11, x12 = (node(mx, i, j) for i in (0, 1) for j in (0, 1))
    y01, y02, y11, y12 = (node(my, i, j) for i in (0, 1) for j in (0, 1))
    pdx, pdy = d11 - d01, d02 - d01
    C20, C02 = 3.0 * pdx - x11 - 2.0 * x01, 3.0 * pdy - y02 - 2.0 * y01
    C30, C03 = -2.0 * pdx + x11 + x01, -2.0 * pdy + y02 + y01
    s1, s2 = d01 + y01 + C02 + C03, d01 + x01 + C20 + C30
    C21, C31 = 3.0 * d12 - 2.0 * x02 - x12 - 3.0 * s1 - C20, -2.0 * d12 + x02 + x12 + 2.0 * s1 - C30
    C12, C13 = 3.0 * d12 - 2.0 * y11 - y12 - 3.0 * s2 - C02, -2.0 * d12 + y11 + y12 + 2.0 * s2 - C03
    C11 = x02 - C13 - C12 - x01
    u, v = x - ix, y - iy
    u2, v2 = u * u, v * v
    density = (d01 + x01 * u + y01 * v + C20 * u2 + C02 * v2 + C30 * (u * u2) + C03 * (v * v2) + C21 * u2 * v +
               C31 * (u * u2) * v + C12 * u * v2 + C13 * u * (v * v2) + C11 * u * v)
    pressure = np.minimum(density - 1.0, 2.0)

    def per_mass(f, a, b):
        return np.where(m[a, b] > 0, f / np.where(m[a, b] > 0, m[a, b], f32(1)), f).astype(float)

    A, B = np.abs(y - gravity[:, 1]), np.abs(x - gravity[:, 0])
    C_ = np.sqrt(A * A + B * B)
    dx = np.minimum(0.03, C_) * B / C_
    dy = A * dx / B
    cax, cay = np.where(x <= gravity[:, 0], dx, -dx), np.where(y <= gravity[:, 1], dy, -dy)
    U, V = P[:, 2].copy(), P[:, 3].copy()
    stencil = [(a, b, px[a] * py[b]) for a in range(3) for b in range(3)]
    for a, b, phi in stencil:
        U += phi * (per_mass((-((gx[a] * py[b]) * pressure)).astype(f32), a, b) + cax)
        V += phi * (per_mass((-((px[a] * gy[b]) * pressure)).astype(f32), a, b) + cay)
    gu, gv = np.zeros_like(U), np.zeros_like(V)
    for a, b, phi in stencil:
        gu += phi * per_mass((phi * U).astype(f32), a, b)
        gv += phi * per_mass((phi * V).astype(f32), a, b)
    return np.stack([x + gu, y + gv, gu, gv], 1)


@pytest.mark.parametrize("spacing", [5, 8, 11])
def test_fluid_step_where_weights_vanish(spacing):
    """Particles near a cell's edge, whose weight at the far nodes is 1e-3 to
    1e-13: the node masses there are the FP32 rounding of the cell's moments,
    to the bit, and the velocities divided by them are reproduced.  1e-10 is
    what one FP32 rounding of a node's sums may move a particle (2^-24 of
    velocities of at most 1e-3 from such nodes); masses from the weights'
    products would move most of them by 1e-6 to 1e-4."""
    rng = np.random.default_rng(spacing)
    gsx = gsy = 200
    at = np.arange(10, gsx - 10, spacing)
    cells = np.stack(np.meshgrid(at, at), -1).reshape(-1, 2)
    n = len(cells)
    P = np.zeros((n, 20))
    near = 10.0 ** rng.uniform(-6, -1, (n, 2))  # distance of e and h from -0.5 or 0.5
    P[:, 0:2] = cells + 0.5 + np.where(rng.integers(0, 2, (n, 2)), near, 1.0 - near)
    P[:, 2:4] = rng.normal(0, 0.2, (n, 2))
    P[:, 4:6] = P[:, 0:2] + rng.uniform(0.5, 3, (n, 2))
    P[:, 6] = 1.0
    P[:, 7:15] = rng.uniform(0, 1, (n, 8))
    P[:, 15:18] = 1.0
    want = _lone_particle_step(P)
    G.log(f"fluid step, {n} lone particles {spacing} cells apart")
    got = _step_gpu(P, gsx, gsy, 1, 20.0)[0]
    assert np.abs(got[:, :4] - want).max() <= 1e-10


@pytest.mark.parametrize("n", [1, 63, 65, 32768, 32769, 70000])
def test_fluid_particles_read_back_as_set(n):
    """Around the rows of a workgroup and the particles read back at a time."""
    rng = np.random.default_rng(n)
    P = rng.uniform(0, 1, (n, 20))
    P[:, 16:18] = rng.integers(0, 2, (n, 2))
    lib = G.lib()
    f = _model(n, 64, 64)
    try:
        G.log(f"fluid particles {n}")
        G.check(lib.amh_fluid_set_particles(f, op.ptr(P), G.stream()), "set")
        Q = np.full((n, 20), -7.0)
        G.check(lib.amh_fluid_get_particles(f, op.ptr(Q), G.stream()), "get")
    finally:
        lib.amh_fluid_destroy(f)
    assert (Q[:, :18] == P[:, :18]).all() and (Q[:, 18:] == -7.0).all()


def _clustered(rng, n, lo, hi, shift=0.0):
    """Particles in runs of 256 around random centres in [lo, hi)^2 (moved by
    shift cells), with velocities, attractors and colours."""
    P = np.zeros((n, 20))
    centres = rng.uniform(lo, hi, (n // 256, 2)) + shift
    P[:, 0] = np.clip(np.repeat(centres[:, 0], 256) + rng.normal(0, 3, n), 8, hi + 20)
    P[:, 1] = np.clip(np.repeat(centres[:, 1], 256) + rng.normal(0, 3, n), 8, hi + 20)
    P[:, 2:4] = rng.normal(0, 0.2, (n, 2))
    P[:, 4] = P[:, 0] + rng.normal(0, 3, n)
    P[:, 5] = P[:, 1] + rng.normal(0, 3, n)
    P[:, 6] = 1.0
    P[:, 7:15] = rng.uniform(0, 1, (n, 8))
    P[:, 15] = rng.choice([0.1, 1.0], n)
    P[:, 16] = 1.0
    P[:, 17] = rng.integers(0, 2, n)
    return P


@pytest.mark.parametrize("grid", [276, 600])
def test_fluid_steps_after_new_particles_match_oracle(grid):
    """Work items exist only for tiles with entries, plus one zeroing item
    for each tile that had entries the step before: after a step of one
    particle set, a second set a few cells away (sharing the first one's
    node halos) steps as the oracle steps it from an empty grid.  276^2 has
    1,225 tiles (counts scanned in LDS), 600^2 has 5,625 (scanned on the
    device first)."""
    rng = np.random.default_rng(11)
    n = 20480
    A = _clustered(rng, n, 30, grid - 60)
    B = _clustered(rng, n, 30, grid - 60, shift=4.0)
    lib = G.lib()
    f = _model(n, grid, grid)
    try:
        G.log(f"fluid grid {grid}: one step of the first set, then the second")
        QA = np.ascontiguousarray(A.copy())
        G.check(lib.amh_fluid_set_particles(f, op.ptr(QA), G.stream()), "set A")
        G.check(lib.amh_fluid_step(f, 0, 20.0, 0, G.stream()), "step A")
        Q = np.ascontiguousarray(B.copy())
        G.check(lib.amh_fluid_set_particles(f, op.ptr(Q), G.stream()), "set B")
        outs = []
        for k in range(3):
            G.check(lib.amh_fluid_step(f, 2 - k, 20.0, 0, G.stream()), "step B")
            G.check(lib.amh_fluid_get_particles(f, op.ptr(Q), G.stream()), "get")
            outs.append(Q.copy())
    finally:
        lib.amh_fluid_destroy(f)
    R = B.copy()
    for k in range(3):
        op.oracle().or_fluid_step(op.ptr(R), n, grid, grid, 2 - k, 20.0, 0)
        for col in (0, 1, 2, 3, 11, 12, 13, 14):
            d = np.abs(outs[k][:, col] - R[:, col]).max()
            assert d <= 2e-3, (k, col, d)


def _fluid_frame(g, variant, t, fluidsteps, sp=1.0, reset=True, fluid=None, rend=None, atom_keys=None):
    """Render one fluid frame of the cfg1 chains through the C ABI (atom_keys:
    a device copy of the key points atom-major for the update, or None)."""
    lib = G.lib()
    cfg, keys, off, widths, order, nb, blob_rgba, (lag, slope) = render_inputs(g, variant)
    if rend is None:
        vals = {"bbox": [cfg.bbox_x1, cfg.bbox_y1, cfg.bbox_x2, cfg.bbox_y2], "motion": cfg.motion,
                "fading": cfg.fading, "show": cfg.show_blobs, "density": cfg.density, "feather": cfg.feather,
                "keep_bg": cfg.keep_background}
        rend = GpuRenderer(keys, g["chain_after"], off, widths, order, blob_rgba, vals, lag, slope)
    h = 2
    wtot = int(np.sum(widths))
    pts = g["chain_after"].reshape(-1, h)
    nch = len(widths)
    # activation ranks and blob sizes per key segment, as the engine builds them
    rank = np.zeros((h, wtot), np.int32)
    surf = np.zeros((h, nch), np.int32)
    for y in range(h):
        yn = (y + 1) % h
        for c, (o_, w) in enumerate(zip(off, widths)):
            f1 = (pts[o_:o_ + w, y] >> 48) & 2
            f2 = (pts[o_:o_ + w, yn] >> 48) & 2
            cls = np.where((f1 > 0) & (f2 > 0), 0, np.where(f1 > 0, 1, np.where(f2 > 0, 2, 3)))
            order_x = np.lexsort((np.arange(w), cls))
            rank[y, o_ + order_x] = np.arange(w)
            surf[y, c] = int((f1 > 0).sum())
    keep = [G.to_dev(rank.ravel()), G.to_dev(surf.ravel())]
    fa = A.FluidFrame(C.pointer(rend.args), keep[0].data_ptr(), keep[1].data_ptr(), None, sp, fluidsteps, 0,
                      None if atom_keys is None else atom_keys.data_ptr())
    if fluid is None:
        fluid = C.c_void_p()
        G.check(lib.amh_fluid_create(C.byref(fluid), int(64 * sp) + 20, int(64 * sp) + 20, wtot, 64, 64, h,
                                     G.stream()), "create")
        G.check(lib.amh_fluid_reset(fluid, sp, G.stream()), "reset")
    G.check(lib.amh_fluid_render(fluid, C.byref(fa), float(t), G.dptr(rend.out), G.stream()), "render")
    img = G.to_host(rend.out, np.uint32).view(np.uint8).reshape(64, 64, 4).copy()
    return img, fluid, rend, surf, rank


def test_fluid_frame_without_steps_reproduces_key_frame(golden_cfg1):
    """fluidsteps = 0 at t = 0: each of the |A| active particles of a chain
    sits on its source pixel (grid = pixel + 10, weight 1), so the frame is
    key frame 0 as get_pixel returns it."""
    g = golden_cfg1
    G.log("fluid frame t=0, no steps")
    img, fluid, rend, surf, rank = _fluid_frame(g, "default", 0.0, 0)
    try:
        key = np.ascontiguousarray(g["shown"][0]).view(np.uint8).reshape(64, 64, 4)
        assert (img == key).all()
        # active particles per chain = round((1-t)|A| + t|B|) at t = 0
        lib = G.lib()
        n = int(rank.shape[1])
        Q = np.zeros((n, 20))
        G.check(lib.amh_fluid_get_particles(fluid, op.ptr(Q), G.stream()), "get")
        widths = g["chain_w"]
        off = np.concatenate([[0], np.cumsum(widths)[:-1]])
        for c, (o_, w) in enumerate(zip(off, widths)):
            assert int(Q[o_:o_ + w, 16].sum()) == surf[0, c]
    finally:
        G.lib().amh_fluid_destroy(fluid)


def test_fluid_frames_advance_and_count(golden_cfg1):
    """Frames in order with 4 model steps each: the active count follows the
    interpolated blob areas and the image stays covered and opaque where the
    fluid is."""
    g = golden_cfg1
    fluid = rend = None
    widths = g["chain_w"]
    off = np.concatenate([[0], np.cumsum(widths)[:-1]])
    lib = G.lib()
    try:
        for i in range(16):
            t = i / 16
            G.log(f"fluid frame {i}")
            img, fluid, rend, surf, rank = _fluid_frame(g, "default", t, 4, fluid=fluid, rend=rend)
            n = int(rank.shape[1])
            Q = np.zeros((n, 20))
            G.check(lib.amh_fluid_get_particles(fluid, op.ptr(Q), G.stream()), "get")
            fk = int(t * 2)
            tl = (t - fk / 2) * 2
            for c, (o_, w) in enumerate(zip(off, widths)):
                want = int(np.floor((1 - tl) * surf[fk, c] + tl * surf[(fk + 1) % 2, c] + 0.5))
                assert int(Q[o_:o_ + w, 16].sum()) == want
            cover = int((img[..., 3] > 0).sum())
            assert cover > 0.5 * min(surf[0].sum(), surf[1].sum())
            assert np.isfinite(Q[:, :4]).all()
    finally:
        if fluid is not None:
            lib.amh_fluid_destroy(fluid)


def _renderer(g, variant, swap_tables=False):
    cfg, keys, off, widths, order, nb, blob_rgba, (lag, slope) = render_inputs(g, variant)
    vals = {"bbox": [cfg.bbox_x1, cfg.bbox_y1, cfg.bbox_x2, cfg.bbox_y2], "motion": cfg.motion,
            "fading": cfg.fading, "show": cfg.show_blobs, "density": cfg.density, "feather": cfg.feather,
            "keep_bg": cfg.keep_background}
    if swap_tables:
        lag, slope = slope, lag
    return GpuRenderer(keys, g["chain_after"], off, widths, order, blob_rgba, vals, lag, slope)


def test_fluid_perlin_lag_slope_kept_between_frames(golden_cfg1):
    """A model keeps each atom's PERLIN lag and slope from frame to frame of
    a key segment and computes them again when the noise tables change: the
    colour targets (R, G, B, A) its update sets equal those of a fresh model
    at the same time, and they depend on the tables."""
    g = golden_cfg1
    variant = "spline_perlin_bg_feather2"
    assert int(g[f"render_{variant}_opts"][1]) == 6  # PERLIN
    lib = G.lib()
    n = int(np.sum(g["chain_w"]))
    made = []

    def particles(f):
        Q = np.zeros((n, 20))
        G.check(lib.amh_fluid_get_particles(f, op.ptr(Q), G.stream()), "get")
        return Q

    def same_targets(QA, QB):
        both = (QA[:, 16] > 0) & (QB[:, 16] > 0)
        assert both.sum() > 0.5 * (QB[:, 16] > 0).sum()
        return (QA[both, 7:11] == QB[both, 7:11]).all()

    try:
        rend = _renderer(g, variant)
        swapped = _renderer(g, variant, swap_tables=True)
        fa = None
        for t in (0.0, 0.1, 0.2, 0.3):  # key segment 0: the lag and slope of t = 0 are kept
            G.log(f"perlin memo: frame t={t}")
            _, fa, _, _, _ = _fluid_frame(g, variant, t, 2, fluid=fa, rend=rend)
            if not made:
                made.append(fa)
        _, fb, _, _, _ = _fluid_frame(g, variant, 0.3, 2, rend=rend)
        made.append(fb)
        assert same_targets(particles(fa), particles(fb))
        # other tables: the kept values no longer hold
        _, fa, _, _, _ = _fluid_frame(g, variant, 0.35, 2, fluid=fa, rend=swapped)
        _, fc, _, _, _ = _fluid_frame(g, variant, 0.35, 2, rend=swapped)
        made.append(fc)
        _, fd, _, _, _ = _fluid_frame(g, variant, 0.35, 2, rend=rend)
        made.append(fd)
        assert same_targets(particles(fa), particles(fc))
        assert not same_targets(particles(fd), particles(fc))  # the tables matter at t = 0.35
    finally:
        for f in made:
            lib.amh_fluid_destroy(f)


@pytest.mark.parametrize("variant", ["default", "spline_perlin_bg_feather2"])
def test_fluid_update_from_atom_major_keys(golden_cfg1, variant):
    """amh_fluid_atom_keys transposes the key points atom-major, and frames
    whose update reads an atom's key points from that copy equal frames
    that read them row by row: the same active particles with the same
    colour targets, and (as between any two runs: tiles split over several
    work items add their node sums with FP32 atomics, in no fixed order)
    images within 1 LSB and positions and velocities within 1e-4."""
    g = golden_cfg1
    lib = G.lib()
    T = G.torch()
    h, n = 2, int(np.sum(g["chain_w"]))
    rend = _renderer(g, variant)
    keys = G.zeros(n * h, T.int64)
    G.check(lib.amh_fluid_atom_keys(G.dptr(rend.keep[1]), h, n, G.dptr(keys), G.stream()), "atom keys")
    want = np.ascontiguousarray(G.key_major(g["chain_after"], h)).view(np.uint64).reshape(h, n).T.ravel()
    assert np.array_equal(G.to_host(keys, np.uint64), want)
    made = []
    try:
        fa = fb = None
        for t in (0.0, 0.3, 0.55, 0.8):
            G.log(f"atom-major keys: {variant} t={t}")
            ia, fa, _, _, _ = _fluid_frame(g, variant, t, 2, fluid=fa, rend=rend)
            if len(made) == 0:
                made.append(fa)
            ib, fb, _, _, _ = _fluid_frame(g, variant, t, 2, fluid=fb, rend=rend, atom_keys=keys)
            if len(made) == 1:
                made.append(fb)
            assert np.abs(ia.astype(np.int32) - ib.astype(np.int32)).max() <= 1, t
            QA, QB = np.zeros((n, 20)), np.zeros((n, 20))
            G.check(lib.amh_fluid_get_particles(fa, op.ptr(QA), G.stream()), "get")
            G.check(lib.amh_fluid_get_particles(fb, op.ptr(QB), G.stream()), "get")
            assert np.array_equal(QA[:, 16], QB[:, 16]), t
            act = QA[:, 16] > 0
            assert act.sum() > 0
            assert np.array_equal(QA[act, 7:11], QB[act, 7:11]), t
            assert np.abs(QA[:, :4] - QB[:, :4]).max() <= 1e-4, t
    finally:
        for f in made:
            lib.amh_fluid_destroy(f)


def test_engine_fluid_render():
    """am::morph with set_fluid: frames render through the fluid path and
    differ from the atom path."""
    from atomorph_amd import synth
    frames = synth.workload("ellipses64")
    m = M.Morph()
    m.set(seed=1, cycle_length=1 << 14)
    for i, f in enumerate(frames):
        m.add_frame_rgba(i, f)
    m.set_resolution(64, 64)
    m.run(1)
    m.run(300)
    m.next_state()
    assert m.run(1) == M.STATE_ATOM_MORPHING
    m.run(4)
    atoms = m.render(0.3)
    m.set(fluid=5, feather=1)
    imgs = [m.render(i / 16) for i in range(16)]
    assert all((im[..., 3] > 0).sum() > 100 for im in imgs)
    assert not (imgs[5] == atoms).all()


def test_fluid_activation_ranks():
    """amh_fluid_ranks: per key segment and chain the ranks are a
    permutation of the slots, classes first (HAS_FLUID in both rows, only the
    source, only the destination, neither), and within a class the order of
    the keyed permutation -- equal to a host replay of the definition."""
    T = G.torch()
    lib = G.lib()
    rng = np.random.default_rng(21)
    widths = np.array([1, 2, 3, 64, 255, 256, 257, 700, 1500], np.int64)
    h = 3
    off = np.concatenate([[0], np.cumsum(widths)[:-1]]).astype(np.int64)
    wtot = int(widths.sum())
    flags = rng.integers(0, 4, (h, wtot))
    pts = op.pack_points(rng.integers(0, 64, (h, wtot)), rng.integers(0, 64, (h, wtot)), 0, 0, flags)
    seed = 0x1234ABCD
    # every device buffer stays referenced until the kernel has run: a
    # temporary freed early hands its memory to the next allocation
    dev = G.to_dev(pts.ravel())
    off_d = G.to_dev(off)
    w_d = G.to_dev(widths.astype(np.int32))
    rank = G.zeros(h * wtot, T.int32)
    assert off_d.data_ptr() != w_d.data_ptr()
    G.log(f"fluid ranks: {len(widths)} chains, wtot {wtot}, {h} key frames")
    G.check(lib.amh_fluid_ranks(G.dptr(dev), h, wtot, G.dptr(off_d), G.dptr(w_d), len(widths), seed, G.dptr(rank),
                                G.stream()), "amh_fluid_ranks")
    got = G.to_host(rank, np.int32).reshape(h, wtot)
    orc = op.oracle()
    for y in range(h):
        yn = (y + 1) % h
        for c, (o, w) in enumerate(zip(off, widths)):
            f1 = (flags[y, o:o + w] & 2) > 0
            f2 = (flags[yn, o:o + w] & 2) > 0
            cls = np.where(f1 & f2, 0, np.where(f1, 1, np.where(f2, 2, 3)))
            key = orc.or_hash64((seed ^ (c << 32) ^ y) & ((1 << 64) - 1))
            base = np.concatenate([[0], np.cumsum(np.bincount(cls, minlength=4))[:-1]])
            want = np.zeros(w, np.int64)
            for p in range(w):
                x = orc.or_perm_index(p, int(w), key)
                want[x] = base[cls[x]]
                base[cls[x]] += 1
            seg = got[y, o:o + w]
            assert np.array_equal(np.sort(seg), np.arange(w)), (y, c)
            assert np.array_equal(seg, want), (y, c)


# ------------------------------------------------------------ fluid frames
def _fluid_fixture():
    import os
    return dict(np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "fluid.npz")))


def test_fluid_draw_within_one_lsb_of_reference():
    """The drawing half of draw_fluid (colour relax, bilinear splat, FP64
    resolve, outward feather, background) on the particles the compiled
    reference had after step_fluid, at six frames of the cfg1 fluid morph
    with feather 0-3 and keep_background on and off: frames within 1 LSB of
    the reference's, relaxed colours and maturity equal to its particles."""
    fx = _fluid_fixture()
    lib = G.lib()
    T = G.torch()
    n = fx["fl_pre"].shape[1]
    keys = G.to_dev(np.ascontiguousarray(fx["fl_shown"]).ravel())
    lag, slope = G.to_dev(op.perlin_perm(1)), G.to_dev(op.perlin_perm(2))
    out = G.zeros(64 * 64, T.int32)
    bb = [int(v) for v in fx["fl_bbox"]]
    fluid = C.c_void_p()
    G.check(lib.amh_fluid_create(C.byref(fluid), 84, 84, n, 64, 64, 2, G.stream()), "create")
    try:
        for k, i in enumerate(fx["fl_index"]):
            feather, keep = (int(v) for v in fx["fl_opts"][k])
            t = float(fx["fl_t"][k])
            G.log(f"fluid draw: frame {i} t={t} feather {feather} keep_background {keep}")
            args = A.RenderArgs(64, 64, 2, 0, *bb, 4, 6, 0, 1, feather, keep, 0, 0, 0, keys.data_ptr(), None, None,
                                None, None, None, lag.data_ptr(), slope.data_ptr())
            fa = A.FluidFrame(C.pointer(args), None, None, None, 1.0, 3, 0)
            P = np.ascontiguousarray(fx["fl_pre"][k])
            G.check(lib.amh_fluid_set_particles(fluid, op.ptr(P), G.stream()), "set")
            G.check(lib.amh_fluid_draw(fluid, C.byref(fa), t, G.dptr(out), G.stream()), "amh_fluid_draw")
            img = G.to_host(out, np.uint32).view(np.uint8).reshape(64, 64, 4)
            want = fx["fl_img"][k]
            d = np.abs(img.astype(np.int32) - want.astype(np.int32))
            G.log(f"  worst channel difference {int(d.max())}, differing channels {int((d > 0).sum())}, "
                  f"drawn pixels {int((want[..., 3] > 0).sum())}")
            assert d.max() <= 1, (i, int(d.max()))
            Q = np.zeros((n, 20))
            G.check(lib.amh_fluid_get_particles(fluid, op.ptr(Q), G.stream()), "get")
            post = fx["fl_post"][k]
            assert np.allclose(Q[:, 11:15], post[:, :4], rtol=0, atol=1e-12), i
            assert (Q[:, 17] == post[:, 4]).all(), i
            assert (Q[:, :2] == P[:, :2]).all()  # drawing moves nothing
    finally:
        lib.amh_fluid_destroy(fluid)


@pytest.mark.parametrize("steps", [4, 3])
def test_fluid_frames_replayed_from_a_graph_equal_eager_frames(golden_cfg1, steps):
    """amh_fluid_render on a stream of its own captures a frame's launches
    into a hipGraph once and replays it, the per-frame values coming from
    the parameter block: 12 frames (with other GPU work and host syncs
    between the replays) equal the same frames launched one by one within
    1 LSB, and the particles agree within 1e-4.  With an odd number of
    steps per frame the bins' count parity alternates from frame to frame,
    so the frames replay two graphs in turn."""
    g = golden_cfg1
    lib = G.lib()
    T = G.torch()
    cfg, keys, off, widths, order, nb, blob_rgba, (lag, slope) = render_inputs(g, "spline_perlin_bg_feather2")
    vals = {"bbox": [cfg.bbox_x1, cfg.bbox_y1, cfg.bbox_x2, cfg.bbox_y2], "motion": cfg.motion,
            "fading": cfg.fading, "show": cfg.show_blobs, "density": cfg.density, "feather": cfg.feather,
            "keep_bg": cfg.keep_background}
    rend = GpuRenderer(keys, g["chain_after"], off, widths, order, blob_rgba, vals, lag, slope)
    h, wtot = 2, int(np.sum(widths))
    pts = g["chain_after"].reshape(-1, h)
    rank = np.zeros((h, wtot), np.int32)
    surf = np.zeros((h, len(widths)), np.int32)
    for y in range(h):
        for c, (o_, w) in enumerate(zip(off, widths)):
            f1 = (pts[o_:o_ + w, y] >> 48) & 2
            f2 = (pts[o_:o_ + w, (y + 1) % h] >> 48) & 2
            cls = np.where((f1 > 0) & (f2 > 0), 0, np.where(f1 > 0, 1, np.where(f2 > 0, 2, 3)))
            rank[y, o_ + np.lexsort((np.arange(w), cls))] = np.arange(w)
            surf[y, c] = int((f1 > 0).sum())
    keep = [G.to_dev(rank.ravel()), G.to_dev(surf.ravel())]
    fa = A.FluidFrame(C.pointer(rend.args), keep[0].data_ptr(), keep[1].data_ptr(), None, 1.0, steps, 0)
    stream = C.c_void_p()
    G.check(lib.amh_stream_create(C.byref(stream)), "stream")
    models = []
    try:
        for graphs in (1, 0):
            f = C.c_void_p()
            G.check(lib.amh_fluid_create(C.byref(f), 84, 84, wtot, 64, 64, h, stream), "create")
            G.check(lib.amh_fluid_reset(f, 1.0, stream), "reset")
            G.check(lib.amh_fluid_use_graphs(f, graphs), "graphs")
            models.append(f)
        outs = [T.zeros(12 * 64 * 64, dtype=T.int32, device="cuda") for _ in range(2)]
        G.sync()
        for i in range(12):
            t = i / 12
            G.log(f"fluid graph replay frame {i} ({steps} steps)")
            for f, o in zip(models, outs):
                G.check(lib.amh_fluid_render(f, C.byref(fa), t, C.c_void_p(o.data_ptr() + 4 * 64 * 64 * i), stream),
                        "render")
            G.check(lib.amh_stream_sync(stream), "sync")
            (T.ones(1 << 20, device="cuda") * 2.0).sum().item()  # other work between the replays
        a = G.to_host(outs[0], np.uint32).view(np.uint8).reshape(12, 64, 64, 4)
        b = G.to_host(outs[1], np.uint32).view(np.uint8).reshape(12, 64, 64, 4)
        for i in range(12):
            d = np.abs(a[i].astype(np.int32) - b[i].astype(np.int32))
            G.log(f"  frame {i}: differing channels {int((d > 0).sum())}")
            assert d.max() <= 1, (i, int(d.max()))
            assert (a[i][..., 3] > 0).sum() > 500
        # the float atomics of the model steps may add in another order from
        # one run to the next, so the particles agree to rounding, not bits
        Q = [np.zeros((wtot, 20)) for _ in range(2)]
        for f, q in zip(models, Q):
            G.check(lib.amh_fluid_get_particles(f, op.ptr(q), stream), "get")
        assert np.abs(Q[0][:, :4] - Q[1][:, :4]).max() <= 1e-4
        assert np.array_equal(Q[0][:, 16], Q[1][:, 16])
    finally:
        for f in models:
            lib.amh_fluid_destroy(f)
        lib.amh_stream_destroy(stream)
