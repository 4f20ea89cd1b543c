"""GPU parity of frame rendering (atom path) through the C ABI.

From identical trajectories (the reference's refined cfg1 chains) the GPU
frames are within 1 LSB per channel of the frames the compiled reference
rendered, for six option sets; and equal the oracle's frames except where
the oracle's FP64 weight sums sit on a rounding tie."""
import ctypes as C

import numpy as np
import pytest

from atomorph_amd import _capi as A
from oracle import oracle_py as op
from tests import gpu_util as G
from tests.test_oracle import render_inputs

pytestmark = pytest.mark.gpu

VARIANTS = ["default", "linear_cosine", "none_linear_bg", "spline_perlin_bg_feather2", "average_blobs",
            "distinct_blobs"]


class GpuRenderer:
    """Device buffers for rendering one fixed set of chains."""

    def __init__(self, keys, pts_atom_major, off, widths, order, blob_rgba, cfg_vals, lag, slope):
        T = G.torch()
        lib = G.lib()
        h, H, W = keys.shape[0], keys.shape[1], keys.shape[2]
        self.W, self.H = W, H
        nchains = len(widths)
        nb = order.shape[1]
        rank = -np.ones((h, nchains), np.int32)
        for y in range(h):
            for b in range(nb):
                if order[y, b] >= 0:
                    rank[y, order[y, b]] = b
        self.keep = [G.to_dev(np.ascontiguousarray(keys).view(np.uint32).reshape(-1)),
                     G.to_dev(G.key_major(pts_atom_major, h)), G.to_dev(np.asarray(off, np.int64)),
                     G.to_dev(np.asarray(widths, np.int32)), G.to_dev(rank.ravel()),
                     G.to_dev(np.ascontiguousarray(blob_rgba, np.uint32).ravel()), G.to_dev(lag), G.to_dev(slope)]
        k, p, o, w, r, br, lg, sl = self.keep
        self.args = A.RenderArgs(W, H, h, nb, *cfg_vals["bbox"], cfg_vals["motion"], cfg_vals["fading"],
                                 cfg_vals["show"], cfg_vals["density"], cfg_vals["feather"], cfg_vals["keep_bg"],
                                 0, nchains, int(np.sum(widths)), k.data_ptr(), p.data_ptr(), o.data_ptr(),
                                 w.data_ptr(), r.data_ptr(), br.data_ptr(), lg.data_ptr(), sl.data_ptr())
        self.wsb = lib.amh_render_workspace_bytes(W, H, int(np.sum(widths)))
        self.ws = T.zeros(self.wsb, dtype=T.uint8, device="cuda")
        G.check(lib.amh_render_workspace_init(G.dptr(self.ws), self.wsb, W, H, int(np.sum(widths)), G.stream()),
                "workspace init")
        self.out = G.zeros(W * H, T.int32)

    def frame(self, t):
        G.check(G.lib().amh_render_frame(C.byref(self.args), float(t), G.dptr(self.ws), self.wsb,
                                         G.dptr(self.out), G.stream()), "amh_render_frame")
        return G.to_host(self.out, np.uint32).view(np.uint8).reshape(self.H, self.W, 4).copy()


def _renderer_for(g, variant, density=1):
    cfg, keys, off, widths, order, nb, blob_rgba, (lag, slope) = render_inputs(g, variant, density)
    vals = {"bbox": [cfg.bbox_x1, cfg.bbox_y1, cfg.bbox_x2, cfg.bbox_y2], "motion": cfg.motion,
            "fading": cfg.fading, "show": cfg.show_blobs, "density": cfg.density, "feather": cfg.feather,
            "keep_bg": cfg.keep_background}
    return GpuRenderer(keys, g["chain_after"], off, widths, order, blob_rgba, vals, lag, slope), cfg


@pytest.mark.parametrize("variant", VARIANTS)
def test_render_within_one_lsb_of_reference(golden_cfg1, variant):
    g = golden_cfg1
    rend, cfg = _renderer_for(g, variant)
    worst, differing = 0, 0
    for i, t in enumerate(g[f"render_{variant}_t"]):
        G.log(f"render {variant} frame {i} t={t}")
        got = rend.frame(t)
        want = g[f"render_{variant}"][i]
        d = np.abs(got.astype(np.int32) - want.astype(np.int32))
        worst = max(worst, int(d.max()))
        differing += int((d > 0).sum())
    G.log(f"render {variant}: worst channel difference {worst}, differing channels {differing}")
    assert worst <= 1


def test_render_workspace_is_left_clean(golden_cfg1):
    """Rendering the same frame twice, with other frames between, gives the
    same image (the per-pixel accumulators and overflow counters reset)."""
    rend, _ = _renderer_for(golden_cfg1, "default")
    a = rend.frame(0.3)
    for t in (0.0, 0.55, 0.9):
        rend.frame(t)
    assert (rend.frame(0.3) == a).all()


def test_render_empty_and_negative_time(golden_cfg1):
    rend, _ = _renderer_for(golden_cfg1, "default")
    # normalize_time maps -0.75 to 0.25
    assert (rend.frame(-0.75) == rend.frame(0.25)).all()
    assert (rend.frame(3.25) == rend.frame(0.25)).all()


DENSITY_CASES = [(2, "default"), (2, "spline_perlin_bg_feather2"), (2, "average_blobs"), (3, "default")]


@pytest.mark.parametrize("density,variant", DENSITY_CASES)
def test_render_at_density_within_one_lsb_of_reference(golden_density, density, variant):
    """Chains max_surface * density wide (the reference CLI's default
    density is 2) and alpha round(min(1, taps / density) * mean alpha)
    (morph.cpp:606-612): GPU frames within 1 LSB of the reference's."""
    g = golden_density(density)
    rend, cfg = _renderer_for(g, variant, density)
    assert cfg.density == density
    worst, halved = 0, 0
    for i, t in enumerate(g[f"render_{variant}_t"]):
        G.log(f"render density {density} {variant} frame {i} t={t}")
        got = rend.frame(t)
        want = g[f"render_{variant}"][i]
        worst = max(worst, int(np.abs(got.astype(np.int32) - want.astype(np.int32)).max()))
        halved += int(((want[..., 3] > 0) & (want[..., 3] < 255)).sum())
    G.log(f"density {density} {variant}: worst channel difference {worst}, partial-alpha pixels {halved}")
    if cfg.show_blobs == 0:  # AVERAGE / DISTINCT draw the blob's own alpha (morph.cpp:1321-1334)
        assert halved > 0  # pixels with fewer taps than the density exist
    assert worst <= 1


@pytest.mark.parametrize("variant", ["default", "spline_perlin_bg_feather2"])
def test_render_graph_replays_equal_eager_frames(golden_cfg1, variant):
    """amh_render_graph_frame (arguments and workspace kept by the handle)
    gives the frames of amh_render_frame bit for bit and the reference's within
    1 LSB, time after time, with frames of the other call on the same workspace
    between them, and finishes the frames still queued when it is destroyed."""
    rend, _ = _renderer_for(golden_cfg1, variant)
    lib, T = G.lib(), G.torch()
    ts = [float(t) for t in golden_cfg1[f"render_{variant}_t"]][:6] + [-0.75, 2.3]
    eager = [rend.frame(t) for t in ts]
    outs = [G.zeros(rend.W * rend.H, T.int32) for _ in ts]
    G.sync()
    stream, graph = C.c_void_p(), C.c_void_p()
    G.check(lib.amh_stream_create(C.byref(stream)), "stream")
    try:
        G.check(lib.amh_render_graph_create(C.byref(graph), C.byref(rend.args), G.dptr(rend.ws), rend.wsb, stream),
                "amh_render_graph_create")
        for rep in range(3):
            G.log(f"render handle {variant}: round {rep}")
            for t, o in zip(ts, outs):
                G.check(lib.amh_render_graph_frame(graph, t, G.dptr(o), stream), "amh_render_graph_frame")
            G.check(lib.amh_stream_sync(stream), "sync")
            for t, o, want in zip(ts, outs, eager):
                got = G.to_host(o, np.uint32).view(np.uint8).reshape(rend.H, rend.W, 4)
                assert (got == want).all(), (rep, t)
            for o, want in zip(outs, golden_cfg1[f"render_{variant}"][:6]):
                got = G.to_host(o, np.uint32).view(np.uint8).reshape(rend.H, rend.W, 4)
                assert int(np.abs(got.astype(np.int32) - want.astype(np.int32)).max()) <= 1
            # the other call's frames on the same workspace
            assert (rend.frame(ts[rep]) == eager[rep]).all()
        # destroyed with frames still queued: it waits for them
        for o in outs:
            o.zero_()
        G.sync()
        for t, o in zip(ts, outs):
            G.check(lib.amh_render_graph_frame(graph, t, G.dptr(o), stream), "amh_render_graph_frame")
        G.check(lib.amh_render_graph_destroy(graph), "amh_render_graph_destroy")
        graph = C.c_void_p()
        G.check(lib.amh_stream_sync(stream), "sync")
        for t, o, want in zip(ts, outs, eager):
            got = G.to_host(o, np.uint32).view(np.uint8).reshape(rend.H, rend.W, 4)
            assert (got == want).all(), ("after destroy", t)
    finally:
        lib.amh_render_graph_destroy(graph)
        lib.amh_stream_destroy(stream)


@pytest.mark.parametrize("W,H,nchains,width,spread,feather", [
    (16, 16, 3, 40, 20, 0),      # one image tile, exactly
    (17, 33, 5, 400, 20, 0),     # ragged tiles; more atoms in a tile than its workgroup has threads
    (65, 31, 7, 300, 12, 3),     # feather across tiles, several blobs per pixel
    (48, 20, 40, 60, 1, 0),      # forty blobs around one pixel
    (48, 20, 40, 60, 1, 1),
])
def test_render_tiles_of_overlapping_blobs(W, H, nchains, width, spread, feather):
    """Frames of random overlapping chains, tile edges and dense tiles, are
    within 1 LSB per channel of the oracle's (exact integer sums against its
    FP64 sums, as in the tests above)."""
    rng = np.random.default_rng(W * 1000 + H)
    h = 2
    widths = np.full(nchains, width, np.int64)
    wtot = int(widths.sum())
    off = np.concatenate([[0], np.cumsum(widths)[:-1]]).astype(np.int64)
    x = np.clip(W // 2 + rng.integers(-spread, spread + 1, (wtot, h)), 0, W - 1)
    y = np.clip(H // 2 + rng.integers(-spread, spread + 1, (wtot, h)), 0, H - 1)
    pts = op.pack_points(x, y, rng.integers(0, 256, (wtot, h)), rng.integers(0, 256, (wtot, h)), 3).ravel()
    keys = rng.integers(0, 256, (h, H, W, 4)).astype(np.uint8)
    keys[..., 3] = rng.choice([0, 120, 255], (h, H, W))
    order = np.stack([rng.permutation(nchains) for _ in range(h)]).astype(np.int32)
    lag, slope = op.perlin_perm(3), op.perlin_perm(4)
    vals = {"bbox": [0, 0, W - 1, H - 1], "motion": 3, "fading": 6, "show": 0, "density": 2, "feather": feather,
            "keep_bg": 1}
    rend = GpuRenderer(keys, pts, off, widths, order, np.zeros((h, nchains), np.uint32), vals, lag, slope)
    cfg = op.RenderCfg(W, H, h, 0, 0, W - 1, H - 1, 3, 6, 0, 2, feather, 1, 0, 0, op.ptr(lag), op.ptr(slope))
    want = np.zeros((H, W, 4), np.uint8)
    for t in (0.0, 0.21, 0.5, 0.9):
        G.log(f"render tiles {W}x{H} {nchains} chains of {width}, feather {feather}, t={t}")
        got = rend.frame(t)
        op.oracle().or_render_atoms(C.byref(cfg), op.ptr(keys), op.ptr(pts), op.ptr(off), op.ptr(widths), nchains,
                                    op.ptr(order), nchains, None, t, op.ptr(want))
        assert int(np.abs(got.astype(np.int32) - want.astype(np.int32)).max()) <= 1, t
        assert (rend.frame(t) == got).all()


@pytest.mark.parametrize("W,H", [(1024, 1024), (1040, 1024), (2048, 2048), (2064, 2048)])
def test_render_scattered_atoms_on_many_tiles(W, H):
    """Atoms anywhere in frames of 4,096, 4,160, 16,384 and 16,512 image tiles:
    each way of counting and placing atoms per tile, within 1 LSB of the
    oracle's frame."""
    rng = np.random.default_rng(W + H)
    widths = np.array([700, 3000, 1], np.int64)
    wtot, h = int(widths.sum()), 2
    off = np.concatenate([[0], np.cumsum(widths)[:-1]]).astype(np.int64)
    x, y = rng.integers(0, W, (wtot, h)), rng.integers(0, H, (wtot, h))
    pts = op.pack_points(x, y, rng.integers(0, 256, (wtot, h)), rng.integers(0, 256, (wtot, h)), 3).ravel()
    keys = rng.integers(0, 256, (h, H, W, 4)).astype(np.uint8)
    order = np.stack([rng.permutation(3) for _ in range(h)]).astype(np.int32)
    lag, slope = op.perlin_perm(3), op.perlin_perm(4)
    vals = {"bbox": [0, 0, W - 1, H - 1], "motion": 3, "fading": 6, "show": 0, "density": 1, "feather": 0, "keep_bg": 0}
    rend = GpuRenderer(keys, pts, off, widths, order, np.zeros((h, 3), np.uint32), vals, lag, slope)
    cfg = op.RenderCfg(W, H, h, 0, 0, W - 1, H - 1, 3, 6, 0, 1, 0, 0, 0, 0, op.ptr(lag), op.ptr(slope))
    want = np.zeros((H, W, 4), np.uint8)
    G.log(f"render {W}x{H}, scattered atoms")
    got = rend.frame(0.21)
    op.oracle().or_render_atoms(C.byref(cfg), op.ptr(keys), op.ptr(pts), op.ptr(off), op.ptr(widths), 3, op.ptr(order),
                                3, None, 0.21, op.ptr(want))
    assert int(np.abs(got.astype(np.int32) - want.astype(np.int32)).max()) <= 1
    assert (rend.frame(0.21) == got).all()


@pytest.mark.parametrize("W,H", [(64, 64), (1040, 1024)])
def test_render_more_taps_than_31_bits_count(W, H):
    """2^29 + 999 atoms, each with four taps, so that the tiles' lists start
    beyond 2^31: 131,072 or so per pixel on few tiles, 504 on many.  Every
    pixel is the rounded mean of the up to four key pixels whose atoms reach
    it, exactly (52 GB of device memory)."""
    T, lib = G.torch(), G.lib()
    wtot, h, n = (1 << 29) + 999, 2, W * H
    rng = np.random.default_rng(W)
    keys = rng.integers(0, 256, (h, H, W, 4)).astype(np.uint8)
    keys[..., 3] = 255
    a = T.arange(wtot, device="cuda") % n
    pts = T.empty(h, wtot, dtype=T.int64, device="cuda")
    T.remainder(a, W, out=pts[0])
    pts[0] |= T.div(a, W, rounding_mode="floor") << 16
    del a
    pts[0] |= (128 << 32) | (128 << 40) | (3 << 48)
    pts[1] = pts[0]
    dkeys = G.to_dev(keys.view(np.uint32).reshape(-1))
    off, width, rank = G.to_dev(np.zeros(1, np.int64)), G.to_dev(np.array([wtot], np.int32)), G.zeros(h, T.int32)
    args = A.RenderArgs(W, H, h, 1, 0, 0, W - 1, H - 1, 3, 3, 0, 1, 0, 0, 0, 1, wtot, dkeys.data_ptr(), pts.data_ptr(),
                        off.data_ptr(), width.data_ptr(), rank.data_ptr(), None, None, None)
    wsb = lib.amh_render_workspace_bytes(W, H, wtot)
    ws, out = T.empty(wsb, dtype=T.uint8, device="cuda"), G.zeros(n, T.int32)
    G.check(lib.amh_render_workspace_init(G.dptr(ws), wsb, W, H, wtot, G.stream()), "workspace init")
    G.sync()
    G.log(f"render {W}x{H}, {wtot} atoms")
    G.check(lib.amh_render_frame(C.byref(args), 0.0, G.dptr(ws), wsb, G.dptr(out), G.stream()), "amh_render_frame")
    got = G.to_host(out, np.uint32).view(np.uint8).reshape(H, W, 4).astype(np.int64)
    del ws, pts
    T.cuda.empty_cache()
    per = (wtot // n + (np.arange(n) < wtot % n)).reshape(H, W)
    den, num = np.zeros((H, W), np.int64), np.zeros((H, W, 4), np.int64)
    for dy in (0, 1):
        for dx in (0, 1):
            w = per[:H - dy, :W - dx] * (128 if dx else 127) * (128 if dy else 127)
            den[dy:, dx:] += w
            num[dy:, dx:] += w[..., None] * keys[0, :H - dy, :W - dx].astype(np.int64)
    assert (got == (2 * num + den[..., None]) // (2 * den[..., None])).all()
