"""The engine's measured cases: what a program that morphs images has it do.

Every case goes through the C ABI (include/atomorph_hip.h) as a host program
binds it: key frames in HBM, created streams, workspaces and handles kept
between calls.  The kinds, in the order a morph job runs them:

  detect  one key frame's blobs: ingest, 4-connected labelling, blob count,
          statistics and the pixel lists
  warm    learned warm start of freshly built chains (MLP, sort-and-match)
  refine  batched transport descent, one hipGraph replay of 16 passes
  plain   the default descent: one visit of 2^16 attempts per chain, a sweep
          over all chains
  atoms   output frames on the atom path
  fluid   output frames with the fluid model on, 10 steps each, from a seek
          into the animation; at least half a megapixel and four frames, since
          smaller ones repeat bit for bit too often to compare them
  sim     the fluid model on its own: 10 steps, then the particles on the host
  train   one training step of the proposal MLP (gradients, Adam)

The key frames are thresholded four-octave noise, the largest components
kept, as atomorph_amd.synth makes them, but generated on the GPU and with a
little per-pixel colour noise, as photographs have.
"""
import ctypes as C
import functools
import math

import numpy as np
import torch
import torch.nn.functional as F

from atomorph_amd import _capi as A
from atomorph_amd import learned

REFINE_PASSES, REFINE_ROUNDS = 16, 32
CYCLE = 1 << 16       # swap attempts per visit of the plain descent
FLUID_STEPS = 10
FRAMES_OUT = 60       # frames of the whole animation: frame i is at time i / 60
SEEK = 8              # the frame that the fluid cases start at
DIMS = [8, 128, 128, 128, 128, 2]


def listed():
    scene64 = {"width": 64, "height": 64, "blobs": 6, "cover": 0.4, "keys": 2}
    scene1024 = {"width": 1024, "height": 1024, "blobs": 150, "cover": 0.18, "keys": 4}
    scene2048 = {"width": 2048, "height": 2048, "blobs": 1200, "cover": 0.36, "keys": 2}
    return [
        # the smallest image the tests morph: launches and the count's wait
        {"name": "detect_64", "kind": "detect", "width": 64, "height": 64, "blobs": 6, "cover": 0.4},
        # a 2048^2 key frame of 1,200 blobs, 1.5 M blob pixels
        {"name": "detect_2048", "kind": "detect", "width": 2048, "height": 2048, "blobs": 1200, "cover": 0.36},
        # the benchmark's chains: 4 key frames, 150 chains, about 200,000 atoms
        {"name": "warm_1024", "kind": "warm", **scene1024},
        {"name": "refine_1024", "kind": "refine", "tile": 5, **scene1024},
        # the library's default descent on a pair of 512^2 key frames
        {"name": "plain_512", "kind": "plain", "width": 512, "height": 512, "blobs": 40, "cover": 0.36, "keys": 2},
        # a preview: 8 small frames at the command line's density of 2
        {"name": "atoms_64", "kind": "atoms", "frames": 8, "density": 2, "motion": 4, "fading": 6, "feather": 0,
         "background": 0, **scene64},
        # ragged size, soft edges over the cross-dissolved key frames
        {"name": "atoms_1001x777_bg", "kind": "atoms", "width": 1001, "height": 777, "blobs": 90, "cover": 0.25,
         "keys": 3, "frames": 1, "density": 1, "motion": 3, "fading": 5, "feather": 2, "background": 1},
        # the largest pair: about 2 M atoms per frame
        {"name": "atoms_2048", "kind": "atoms", "frames": 2, "density": 1, "motion": 4, "fading": 6, "feather": 0,
         "background": 0, **scene2048},
        # the fluid model on its own, 20,480 particles read back after 10 steps
        {"name": "sim_20k", "kind": "sim", "particles": 20480, "gsx": 276, "gsy": 276},
        # the benchmark's frames: a 276^2 grid under a 1024^2 image
        {"name": "fluid_1024_276", "kind": "fluid", "frames": 4, "sparseness": 0.25, "feather": 0, "background": 0,
         **scene1024},
        # the same image on the default grid, 1044^2
        {"name": "fluid_1024_1044", "kind": "fluid", "frames": 4, "sparseness": 1.0, "feather": 0, "background": 0,
         **scene1024},
        # the trainer's batch
        {"name": "train_16384", "kind": "train", "batch": 16384},
    ]


def draw(rng):
    """A case of one kind with sizes over its range (64 pixels a side to what
    costs as much as the largest listed cases, batches of 100 to 16,384 rows)."""
    kind = rng.choice(["detect", "warm", "refine", "plain", "atoms", "fluid", "sim", "train"])

    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if kind == "train":
        return {"kind": kind, "batch": log_int(100, 16384)}
    if kind == "sim":
        gsx = log_int(48, 400)
        gsy = min(400, max(48, int(gsx * rng.uniform(0.6, 1.6))))
        n = int(rng.uniform(0.1, 1.5) * gsx * gsy)
        return {"kind": kind, "particles": max(200, min(20480, n)), "gsx": gsx, "gsy": gsy}
    side = {"detect": 1536, "warm": 640, "plain": 512, "fluid": 800}.get(kind, 1024)
    least = 704 if kind == "fluid" else 64
    w = log_int(least, side)
    h = min(side, max(least, int(w * rng.uniform(0.6, 1.6))))
    blobs = log_int(4, max(6, int(w * h / 6000)))
    cover = round(rng.uniform(0.15, 0.29 if kind == "fluid" else 0.4), 3)
    case = {"kind": kind, "width": w, "height": h, "blobs": blobs, "cover": cover}
    if kind == "detect":
        return case
    case["keys"] = rng.choice([2, 2, 3, 4])
    if kind == "refine":
        case["tile"] = rng.randrange(6)
    if kind == "atoms":
        case.update(frames=rng.choice([1, 1, 2, 3]), density=rng.choice([1, 2]), motion=rng.choice([3, 4, 4]),
                    fading=rng.choice([3, 5, 6, 6]), feather=rng.choice([0, 0, 1, 3]), background=rng.choice([0, 1]))
    if kind == "fluid":
        case.update(frames=4, sparseness=rng.choice([0.25, 0.5, 1.0]),
                    feather=rng.choice([0, 0, 2]), background=rng.choice([0, 1]))
    return case


# ------------------------------------------------------------------ helpers
def _p(t, offset=0):
    return C.c_void_p(t.data_ptr() + offset * t.element_size())


def _np(a):
    return a.ctypes.data_as(C.c_void_p)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 2654435761 % (1 << 62) + 1)
    return g


def _empty(n, dtype=torch.int32):
    return torch.empty(max(int(n), 1), dtype=dtype, device="cuda")


@functools.lru_cache(None)
def _stream():
    """The program's one created stream, as am::morph makes one for its work."""
    h = C.c_void_p()
    A.check(A.load().amh_stream_create(C.byref(h)), "stream")
    return h


class _Handle:
    """A C handle and the call that destroys it."""

    def __init__(self, destroy):
        self.h, self.destroy = C.c_void_p(), destroy

    def __del__(self):
        if self.h:
            self.destroy(self.h)


def _noise(W, H, period, g):
    """Gradient noise, four octaves of halving period and amplitude."""
    total = torch.zeros(H, W, device="cuda")
    amp = 1.0
    for _ in range(4):
        p = max(int(round(period)), 2)
        angle = 2 * math.pi * torch.rand(H // p + 2, W // p + 2, generator=g, device="cuda")
        gx, gy = torch.cos(angle), torch.sin(angle)
        y, x = (torch.arange(n, device="cuda") / p for n in (H, W))
        y0, x0 = y.long(), x.long()
        ty, tx = (y - y0)[:, None], (x - x0)[None, :]

        def dot(i, j):
            return gx[y0 + i][:, x0 + j] * (tx - j) + gy[y0 + i][:, x0 + j] * (ty - i)

        sx, sy = (t * t * t * (t * (t * 6 - 15) + 10) for t in (tx, ty))
        a = dot(0, 0) + sx * (dot(0, 1) - dot(0, 0))
        b = dot(1, 0) + sx * (dot(1, 1) - dot(1, 0))
        total += amp * (a + sy * (b - a))
        amp, period = amp * 0.5, period / 2.0
    return total


def _frame(W, H, blobs, cover, g):
    """A key frame (H * W packed RGBA words): the `blobs` largest components
    of the noise above its (1 - cover) quantile, opaque, one colour each plus
    per-pixel noise, on a transparent ground."""
    side = math.sqrt(W * H)
    field = _noise(W, H, max(8, int(side / (math.sqrt(blobs) * 1.5))), g)
    t = torch.sort(field.view(-1))[0][int((1.0 - cover) * (W * H - 1))]
    fg = field.view(-1) > t
    labels = _empty(W * H)
    words = fg.to(torch.int32) * -16777216
    torch.cuda.synchronize()
    A.check(A.load().amh_segment(_p(words), W, H, _p(labels), _stream()), "segment")
    A.load().amh_stream_sync(_stream())
    sizes = torch.bincount(labels[labels >= 0].long(), minlength=W * H)
    keep = torch.zeros(W * H, dtype=torch.bool, device="cuda")
    keep[torch.sort(sizes, descending=True, stable=True)[1][:blobs]] = True
    fg = fg & keep[labels.clamp(min=0).long()]
    base = torch.randint(16, 240, (W * H, 3), generator=g, device="cuda")[labels.clamp(min=0).long()]
    rgb = (base + torch.randint(-12, 13, (W * H, 3), generator=g, device="cuda")).int()
    return torch.where(fg, rgb[:, 0] | (rgb[:, 1] << 8) | (rgb[:, 2] << 16) | -16777216, 0).int().contiguous()


class _Detect:
    """One key frame's detection with its buffers."""

    def __init__(self, words, W, H, blobs, cover):
        self.words, self.W, self.H, self.stream, self.lib = words, W, H, _stream(), A.load()
        n = W * H
        self.stored, self.shown, self.labels, self.bop = _empty(n), _empty(n), _empty(n), _empty(n)
        # room for the blobs and pixels that a frame of this cover can hold
        self.plist = torch.zeros(int(cover * n) + 2, dtype=torch.int32, device="cuda")
        self.ws = _empty(self.lib.amh_blob_workspace_bytes(W, H), torch.uint8)
        self.nb = C.c_int32()
        torch.cuda.synchronize()
        self.label()
        self.stats = torch.zeros(blobs, C.sizeof(A.BlobStat) // 8, dtype=torch.int64, device="cuda")
        self.first = torch.zeros(blobs + 1, dtype=torch.int64, device="cuda")
        self.gws_bytes = self.lib.amh_group_workspace_bytes(n, self.nb)
        self.gws = _empty(self.gws_bytes, torch.uint8)
        torch.cuda.synchronize()

    def label(self):
        L, s, W, H = self.lib, self.stream, self.W, self.H
        A.check(L.amh_ingest_frame(_p(self.words), W, H, 1, _p(self.stored), _p(self.shown), s), "ingest")
        A.check(L.amh_segment(_p(self.words), W, H, _p(self.labels), s), "segment")
        A.check(L.amh_blob_count(_p(self.labels), W, H, _p(self.ws), C.byref(self.nb), s), "count")

    def run(self):
        L, s, W, H = self.lib, self.stream, self.W, self.H
        self.label()
        A.check(L.amh_blob_stats(_p(self.labels), _p(self.stored), W, H, _p(self.ws), self.nb, _p(self.bop),
                                 _p(self.stats), s), "stats")
        A.check(L.amh_group_pixels(_p(self.bop), W * H, self.nb, _p(self.gws), self.gws_bytes, _p(self.first),
                                   _p(self.plist), s), "group")
        return {"stored": self.stored, "shown": self.shown, "labels": self.labels, "blob": self.bop,
                "stats": self.stats, "first": self.first, "list": self.plist}


def _match(stats, bbox, rng):
    """order[y][c] = blob of chain c in key frame y (-1: none): pairwise swap
    descent on distance, colour and size, as the engine's matching."""
    h, nch = len(stats), max(len(s) for s in stats)
    feat = np.zeros((h, nch, 7))
    order = np.full((h, nch), -1, np.int64)
    diag = math.hypot(bbox[2] - bbox[0] + 1, bbox[3] - bbox[1] + 1)
    for y, s in enumerate(stats):
        n = s[:, 0:1].astype(float)
        feat[y, :len(s)] = np.hstack([s[:, 1:3] / n / diag, s[:, 3:7] / n / 510.0, n])
        order[y, :len(s)] = np.arange(len(s))

    def dist(a, b):
        d = np.sqrt(((a[:, :2] - b[:, :2]) ** 2).sum(1)) + np.sqrt(((a[:, 2:6] - b[:, 2:6]) ** 2).sum(1))
        both = (a[:, 6] > 0) & (b[:, 6] > 0)
        total = a[:, 6] + b[:, 6]
        return np.where(both, d, 0.0) + np.abs(a[:, 6] - b[:, 6]) / np.where(total > 0, total, 1.0)

    for r in range(200 * h if nch > 1 else 0):
        y = r % h
        q = rng.permutation(nch)[:nch // 2 * 2].reshape(-1, 2)
        i, j = q[:, 0], q[:, 1]
        p, n = feat[(y - 1) % h], feat[(y + 1) % h]
        now = dist(p[i], feat[y, i]) + dist(n[i], feat[y, i]) + dist(p[j], feat[y, j]) + dist(n[j], feat[y, j])
        then = dist(p[i], feat[y, j]) + dist(n[i], feat[y, j]) + dist(p[j], feat[y, i]) + dist(n[j], feat[y, i])
        q = q[then < now]
        feat[y, q] = feat[y, q[:, ::-1]]
        order[y, q] = order[y, q[:, ::-1]]
    return order


class _Chains:
    """Key frames, detected, matched and built into chains, with the render
    arguments that describe them."""

    def __init__(self, case, seed):
        self.lib, self.stream = A.load(), _stream()
        W, H, h = case["width"], case["height"], case["keys"]
        g, rng = _gen(seed), np.random.default_rng(seed)
        frames = [_frame(W, H, case["blobs"], case["cover"], g) for _ in range(h)]
        found = [_Detect(f, W, H, case["blobs"], case["cover"]) for f in frames]
        for d in found:
            d.run()
        torch.cuda.synchronize()
        stats = [d.stats[:d.nb.value, :7].cpu().numpy() for d in found]
        boxes = torch.cat([d.stats[:d.nb.value].view(torch.int32)[:, 14:18] for d in found]).cpu().numpy()
        self.bbox = [int(v) for v in (*boxes[:, :2].min(0), *boxes[:, 2:].max(0))]
        order = _match(stats, self.bbox, rng)
        nch = order.shape[1]
        size = np.stack([np.where(o >= 0, s[np.maximum(o, 0), 0], 0) for o, s in zip(order, stats)])
        width = size.max(0) * case.get("density", 1)
        mid = [(self.bbox[0] + self.bbox[2]) // 2, (self.bbox[1] + self.bbox[3]) // 2]
        self.W, self.H, self.h, self.nch, self.wtot = W, H, h, nch, int(width.sum())
        self.host_w = np.ascontiguousarray(width, np.int32)
        self.host_off = np.concatenate([[0], np.cumsum(width)[:-1]]).astype(np.int64)
        dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
        self.off, self.w = dev(self.host_off), dev(self.host_w)
        blob = dev(order.T.astype(np.int32))
        exy = dev(np.full(nch * h, mid[0] | (mid[1] << 16), np.int32))
        self.keys = torch.cat([d.shown for d in found])
        # a chain is as wide as its largest blob; the rows sit at the start of
        # a buffer with room for the chains of any key frames of this cover
        room = h * int(case["cover"] * W * H + 2) * case.get("density", 1)
        self.pts = torch.zeros(h * room, dtype=torch.int64, device="cuda")
        ptrs = [(C.c_void_p * h)(*[t.data_ptr() for t in ts])
                for ts in ([d.plist for d in found], [d.first for d in found])]
        torch.cuda.synchronize()
        build = A.ChainBuild(h, nch, self.wtot, W, 0, self.off.data_ptr(), self.w.data_ptr(), blob.data_ptr(),
                             exy.data_ptr(), C.cast(ptrs[0], C.POINTER(C.c_void_p)),
                             C.cast(ptrs[1], C.POINTER(C.c_void_p)), seed)
        A.check(self.lib.amh_build_chains(C.byref(build), _p(self.pts), self.stream), "build")
        # composite order of the chains' blobs, the blob sizes, the noise tables
        self.rank = dev(np.stack([rng.permutation(nch) for _ in range(h)]).astype(np.int32))
        self.surface = dev(size.astype(np.int32))
        self.perm = [dev(np.tile(rng.permutation(256), 2).astype(np.int32)) for _ in range(2)]
        self.queue = torch.zeros(4, dtype=torch.int32, device="cuda")
        self.stats = torch.zeros(4, dtype=torch.int64, device="cuda")
        self.lib.amh_stream_sync(self.stream)
        torch.cuda.synchronize()

    def render_args(self, case):
        return A.RenderArgs(self.W, self.H, self.h, self.nch, *self.bbox, case.get("motion", 4),
                            case.get("fading", 6), 0, case.get("density", 1), case.get("feather", 0),
                            case.get("background", 0), 0, self.nch, self.wtot, self.keys.data_ptr(),
                            self.pts.data_ptr(), self.off.data_ptr(), self.w.data_ptr(), self.rank.data_ptr(), None,
                            self.perm[0].data_ptr(), self.perm[1].data_ptr())

    def items(self, tile):
        n = C.c_int32()
        A.check(self.lib.amh_refine_items(_np(self.host_w), self.nch, tile, None, 0, C.byref(n)), "items")
        items = np.zeros(2 * max(n.value, 1), np.int32)
        A.check(self.lib.amh_refine_items(_np(self.host_w), self.nch, tile, _np(items), n.value, C.byref(n)), "items")
        return torch.from_numpy(items).cuda(), n.value

    def refine(self, passes):
        """A few batched passes, so that frames are drawn from refined chains."""
        items, n = self.items(2)
        torch.cuda.synchronize()
        for k in range(passes):
            A.check(self.lib.amh_refine_batched(_p(self.pts), self.h, self.wtot, _p(self.off), _p(self.w), _p(items),
                                                n, 2, k, REFINE_ROUNDS, 1, _p(self.queue), _p(self.stats),
                                                self.stream), "refine")
        self.lib.amh_stream_sync(self.stream)


# -------------------------------------------------------------------- kinds
class _Warm(_Chains):
    def __init__(self, case, seed):
        super().__init__(case, seed)
        self.mlp = _Handle(self.lib.amh_mlp_destroy)
        A.check(self.lib.amh_mlp_create(C.byref(self.mlp.h), 65536, self.stream), "mlp")
        self.params = learned.load_default()
        A.check(self.lib.amh_mlp_set_params(self.mlp.h, _np(self.params), self.stream), "params")
        self.built = self.pts.clone()
        self.args = self.render_args(case)
        self.ws_bytes = self.lib.amh_warm_workspace_bytes(self.wtot, self.nch, self.h)
        self.ws = _empty(self.ws_bytes, torch.uint8)
        torch.cuda.synchronize()

    def run(self):
        s = self.stream
        A.check(self.lib.amh_memcpy_d2d(_p(self.pts), _p(self.built), self.pts.numel() * 8, s), "copy")
        A.check(self.lib.amh_warm_start(self.mlp.h, C.byref(self.args), _p(self.pts), _p(self.ws), self.ws_bytes, s),
                "warm start")
        return self.pts


class _Refine(_Chains):
    def __init__(self, case, seed):
        super().__init__(case, seed)
        self.it, n = self.items(case["tile"])
        self.graph = _Handle(self.lib.amh_graph_destroy)
        torch.cuda.synchronize()
        A.check(self.lib.amh_refine_graph_create(C.byref(self.graph.h), _p(self.pts), self.h, self.wtot, _p(self.off),
                                                 _p(self.w), _p(self.it), n, case["tile"], REFINE_PASSES,
                                                 REFINE_ROUNDS, seed, _p(self.queue), _p(self.stats), self.stream),
                "graph")

    def run(self):
        A.check(self.lib.amh_graph_launch(self.graph.h, self.stream), "replay")
        return self.pts, self.stats


class _Plain(_Chains):
    def __init__(self, case, seed):
        super().__init__(case, seed)
        self.rng, self.seed, self.visits = np.random.default_rng(seed), seed, 0

    def run(self):
        rows = self.rng.integers(0, self.h, self.nch)
        for c in range(self.nch):
            w = int(self.host_w[c])
            if w < 2:
                continue
            A.check(self.lib.amh_refine_chain(_p(self.pts), self.h, self.wtot, int(self.host_off[c]), w, int(rows[c]),
                                              -(-CYCLE // (w // 2)), self.seed, (c << 32) ^ self.visits,
                                              _p(self.stats), self.stream), "visit")
            self.visits += 1
        return self.pts, self.stats


class _Atoms(_Chains):
    def __init__(self, case, seed):
        super().__init__(case, seed)
        self.refine(8)
        self.n, self.at = case["frames"], seed % FRAMES_OUT
        self.args = self.render_args(case)
        self.out = torch.zeros(self.n, self.H, self.W, dtype=torch.int32, device="cuda")
        self.ws_bytes = self.lib.amh_render_workspace_bytes(self.W, self.H, self.wtot)
        self.ws = _empty(self.ws_bytes, torch.uint8)
        torch.cuda.synchronize()
        A.check(self.lib.amh_render_workspace_init(_p(self.ws), self.ws_bytes, self.W, self.H, self.wtot,
                                                   self.stream), "workspace")
        self.graph = _Handle(self.lib.amh_render_graph_destroy)
        if self.n > 1:
            A.check(self.lib.amh_render_graph_create(C.byref(self.graph.h), C.byref(self.args), _p(self.ws),
                                                     self.ws_bytes, self.stream), "graph")

    def run(self):
        for k in range(self.n):
            t, out = self.at / FRAMES_OUT, _p(self.out[k])
            if self.n > 1:
                rc = self.lib.amh_render_graph_frame(self.graph.h, t, out, self.stream)
            else:
                rc = self.lib.amh_render_frame(C.byref(self.args), t, _p(self.ws), self.ws_bytes, out, self.stream)
            A.check(rc, "frame")
            self.at = (self.at + 1) % FRAMES_OUT
        return self.out.view(torch.uint8)


class _Fluid(_Chains):
    def __init__(self, case, seed):
        super().__init__(case, seed)
        self.refine(8)
        self.n, self.sparseness = case["frames"], case["sparseness"]
        sp = self.sparseness
        L, s = self.lib, self.stream
        self.args = self.render_args(case)
        self.out = torch.zeros(self.n, self.H, self.W, dtype=torch.int32, device="cuda")
        self.order, self.atom_keys = _empty(self.h * self.wtot), _empty(self.h * self.wtot, torch.int64)
        torch.cuda.synchronize()
        A.check(L.amh_fluid_ranks(_p(self.pts), self.h, self.wtot, _p(self.off), _p(self.w), self.nch, seed,
                                  _p(self.order), s), "ranks")
        A.check(L.amh_fluid_atom_keys(_p(self.pts), self.h, self.wtot, _p(self.atom_keys), s), "atom keys")
        self.fluid = _Handle(L.amh_fluid_destroy)
        A.check(L.amh_fluid_create(C.byref(self.fluid.h), int(self.W * sp) + 20, int(self.H * sp) + 20, self.wtot,
                                   self.W, self.H, self.h, s), "fluid")
        self.frame = A.FluidFrame(C.pointer(self.args), self.order.data_ptr(), self.surface.data_ptr(), None, sp,
                                  FLUID_STEPS, 0, self.atom_keys.data_ptr())
        L.amh_stream_sync(s)

    def run(self):
        A.check(self.lib.amh_fluid_reset(self.fluid.h, self.sparseness, self.stream), "reset")
        for k in range(self.n):
            A.check(self.lib.amh_fluid_render(self.fluid.h, C.byref(self.frame), (SEEK + k) / FRAMES_OUT,
                                              _p(self.out[k]), self.stream), "fluid frame")
        return self.out.view(torch.uint8)


SIM_RADIUS = 20.0  # freedom radius, in cells


def _particles(case, seed):
    """Particles (the 20 values each of amh_fluid_set_particles) in runs of 256
    around random centres, as a chain's atoms lie."""
    rng = np.random.default_rng(seed)
    n, size = case["particles"], np.array([case["gsx"], case["gsy"]])
    P = np.zeros((n, 20))
    centres = rng.uniform(0.15, 0.85, (-(-n // 256), 2)) * size
    P[:, :2] = np.clip(np.repeat(centres, 256, 0)[:n] + rng.normal(0, 4, (n, 2)), 8, size - 8)
    P[:, 2:4] = rng.normal(0, 0.2, (n, 2))
    P[:, 4:6] = P[:, :2] + rng.normal(0, 3, (n, 2))
    P[:, 6] = 1.0
    P[:, 7:15] = rng.uniform(0, 1, (n, 8))
    P[:, 15] = rng.choice([0.1, 1.0], n)
    P[:, 16] = rng.uniform(0, 1, n) < 0.9
    P[:, 17] = rng.integers(0, 2, n)
    return P


class _Sim:
    def __init__(self, case, seed):
        self.lib, self.stream = A.load(), _stream()
        P = _particles(case, seed)
        self.fluid = _Handle(self.lib.amh_fluid_destroy)
        A.check(self.lib.amh_fluid_create(C.byref(self.fluid.h), case["gsx"], case["gsy"], len(P), 64, 64, 2,
                                          self.stream), "fluid")
        A.check(self.lib.amh_fluid_set_particles(self.fluid.h, _np(P), self.stream), "particles")
        self.host = np.zeros_like(P)

    def run(self):
        for k in range(FLUID_STEPS):
            A.check(self.lib.amh_fluid_step(self.fluid.h, FLUID_STEPS - 1 - k, SIM_RADIUS, 0, self.stream), "step")
        A.check(self.lib.amh_fluid_get_particles(self.fluid.h, _np(self.host), self.stream), "particles")
        return self.host


def _toward(p, q, a):
    """The move of p towards q by a, no further than q."""
    d = q - p
    dist = torch.sqrt((d * d).sum(1))
    return d * (torch.minimum(a, dist) / torch.where(dist > 0, dist, torch.ones_like(dist)))[:, None]


def _fluid_step(P, gsx, gsy, steps_left):
    """One step of the fluid model (fluidmodel.cpp:165-580) in 64 bits, no
    wall jitter, on the active particles' columns P."""
    xy, gravity, target, colour = P[:, 0:2], P[:, 4:6], P[:, 7:11], P[:, 11:15]
    strength, mature = P[:, 15], P[:, 17] > 0
    size = torch.tensor([gsx, gsy], device=P.device)
    cell = (xy - 0.5).long()
    d = cell - xy
    e = d + 2
    w = torch.stack([0.5 * d * d + 1.5 * d + 1.125, -(d + 1) ** 2 + 0.75, 0.5 * e * e - 1.5 * e + 1.125], 2)
    dw = torch.stack([d + 1.5, -2 * (d + 1), d + 0.5], 2)
    i, j = torch.meshgrid(torch.arange(3, device=P.device), torch.arange(3, device=P.device), indexing="ij")
    i, j = i.reshape(-1), j.reshape(-1)
    node = (cell[:, 0:1] + i) * gsy + cell[:, 1:2] + j
    phi = w[:, 0, i] * w[:, 1, j]
    gx, gy = dw[:, 0, i] * w[:, 1, j], w[:, 0, i] * dw[:, 1, j]

    def to_nodes(v):
        return torch.zeros(gsx * gsy, dtype=P.dtype, device=P.device).index_add_(0, node.reshape(-1), v.reshape(-1))

    def one(v):  # the same value for each of a particle's nodes
        return v[:, None].expand(-1, 9)

    m, mx, my = to_nodes(phi), to_nodes(gx), to_nodes(gy)
    s = torch.where(mature & (strength > 0), strength, 0.0)
    weight = to_nodes(one(s))
    sums = [to_nodes(one(s * colour[:, k])) for k in range(4)]

    # pressure: bicubic density at the particle from the four nodes around it
    c = xy.long()
    at = c[:, 0] * gsy + c[:, 1]
    d01, d02, d11, d12 = (m[at + o] for o in (0, 1, gsy, gsy + 1))
    x01, x02, x11, x12 = (mx[at + o] for o in (0, 1, gsy, gsy + 1))
    y01, y02, y11, y12 = (my[at + o] for o in (0, 1, gsy, gsy + 1))
    px, py = d11 - d01, d02 - d01
    c20, c02 = 3 * px - x11 - 2 * x01, 3 * py - y02 - 2 * y01
    c30, c03 = -2 * px + x11 + x01, -2 * py + y02 + y01
    s1, s2 = d01 + y01 + c02 + c03, d01 + x01 + c20 + c30
    c21, c31 = 3 * d12 - 2 * x02 - x12 - 3 * s1 - c20, -2 * d12 + x02 + x12 + 2 * s1 - c30
    c12, c13 = 3 * d12 - 2 * y11 - y12 - 3 * s2 - c02, -2 * d12 + y11 + y12 + 2 * s2 - c03
    c11 = x02 - c13 - c12 - x01
    u, v = (xy - c).unbind(1)
    density = (d01 + x01 * u + y01 * v + c20 * u * u + c02 * v * v + c30 * u ** 3 + c03 * v ** 3 + c21 * u * u * v
               + c31 * u ** 3 * v + c12 * u * v * v + c13 * u * v ** 3 + c11 * u * v)
    pressure = torch.clamp(density - 1.0, max=2.0)
    wall = torch.clamp(4.0 - xy, min=0.0) + torch.clamp(size - 5 - xy, max=0.0)
    ax = to_nodes(-gx * pressure[:, None] + phi * wall[:, 0:1])
    ay = to_nodes(-gy * pressure[:, None] + phi * wall[:, 1:2])
    mass = torch.where(m > 0, m, 1.0)
    pull = _toward(xy, gravity, torch.full_like(strength, 0.03))
    vel = torch.stack([P[:, 2 + k] + (phi * ((a / mass)[node] + pull[:, k:k + 1])).sum(1)
                       for k, a in enumerate((ax, ay))], 1)
    moved = torch.stack([(phi * (to_nodes(phi * (vel[:, k] * mature)[:, None]) / mass)[node]).sum(1)
                         for k in range(2)], 1)

    wsum = weight[node].sum(1)
    near = torch.stack([(torch.where(weight > 0, q, 0.0))[node].sum(1) for q in sums], 1)
    near = near / torch.where(wsum > 0, wsum, 1.0)[:, None]
    mix = (near - target).abs()
    mixed = torch.where(mature[:, None], (1 - mix) * colour + mix * near, near)
    P[:, 11:15] = torch.where((wsum > 0)[:, None], mixed, colour)

    xy = xy + moved
    dist = torch.sqrt(((xy - gravity) ** 2).sum(1))
    radius = SIM_RADIUS * P[:, 6]
    back = _toward(xy, gravity, dist - radius) / (steps_left + 1)
    xy = torch.where((dist > radius)[:, None], xy + back, xy)
    low, high = xy < 1.0, xy > size - 2
    P[:, 0:2] = torch.where(low, 1.0, torch.where(high, (size - 2).double(), xy))
    P[:, 2:4] = torch.where(low | high, 0.0, moved)


def _training_batch(n, seed):
    """Parameters (as the trainer initialises them) and a batch: positions,
    colours, offsets from the centroid in RMS radii, and targets near them."""
    g = _gen(seed)
    parts = []
    for din, dout in zip(DIMS[:-1], DIMS[1:]):
        parts += [torch.randn(din * dout, generator=g, device="cuda") / math.sqrt(din),
                  0.05 * torch.randn(dout, generator=g, device="cuda")]
    x = torch.rand(n, 8, generator=g, device="cuda")
    x[:, 5] = 1.0
    x[:, 6:] = 0.7 * torch.randn(n, 2, generator=g, device="cuda")
    t = x[:, 6:] + 0.35 * torch.randn(n, 2, generator=g, device="cuda")
    return torch.cat(parts).contiguous(), x.contiguous(), t.contiguous()


class _Train:
    def __init__(self, case, seed):
        self.lib, self.n = A.load(), case["batch"]
        self.params, self.x, self.t = _training_batch(self.n, seed)
        self.stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        self.mlp = _Handle(self.lib.amh_mlp_destroy)
        A.check(self.lib.amh_mlp_create(C.byref(self.mlp.h), self.n, self.stream), "mlp")
        host = self.params.cpu().numpy()
        A.check(self.lib.amh_mlp_set_params(self.mlp.h, _np(host), self.stream), "params")
        self.grad = torch.zeros(A.MLP_PARAMS, device="cuda")
        self.loss = torch.zeros(1, device="cuda")

    def run(self):
        self.loss.zero_()
        A.check(self.lib.amh_mlp_gradients(self.mlp.h, _p(self.x), _p(self.t), self.n, _p(self.grad), _p(self.loss),
                                           self.stream), "gradients")
        A.check(self.lib.amh_mlp_adam_step(self.mlp.h, 1e-3, self.stream), "adam")
        return {"grad": self.grad, "loss": self.loss}


class _DetectFrame(_Detect):
    def __init__(self, case, seed):
        size = case["width"], case["height"]
        scene = case["blobs"], case["cover"]
        super().__init__(_frame(*size, *scene, _gen(seed)), *size, *scene)


KINDS = {"detect": _DetectFrame, "warm": _Warm, "refine": _Refine, "plain": _Plain, "atoms": _Atoms,
         "fluid": _Fluid, "sim": _Sim, "train": _Train}


def prepare(case, seed):
    state = KINDS[case["kind"]](case, seed)
    torch.cuda.synchronize()
    return state


def run(state):
    return state.run()


def work(case):
    """What one pass cannot do without.  A chain's width is its largest blob
    in any key frame, about 1.1 times the blobs' mean cover."""
    kind = case["kind"]
    if kind == "train":
        params = sum(a * b + b for a, b in zip(DIMS[:-1], DIMS[1:]))
        macs = sum(a * b for a, b in zip(DIMS[:-1], DIMS[1:]))
        # x, t in; gradient out; parameters and both moments in and out
        return {"bytes": case["batch"] * 40 + params * 4 * 7, "flops": 6 * macs * case["batch"]}
    if kind == "sim":
        # 18 values of each particle in, out and on the host
        return {"bytes": case["particles"] * 3 * 144, "flops": 600 * FLUID_STEPS * case["particles"]}
    px = case["width"] * case["height"]
    fg = case["cover"] * px
    if kind == "detect":
        # words in; stored, shown, label and blob of each pixel, the lists out;
        # about 60 operations of colour conversion per blob pixel
        return {"bytes": 20 * px + 4 * fg + 88 * case["blobs"], "flops": 60 * fg}
    h, atoms = case["keys"], 1.1 * fg * case.get("density", 1)
    points = 8 * atoms * h
    if kind == "warm":
        macs = sum(a * b for a, b in zip(DIMS[:-1], DIMS[1:]))
        return {"bytes": 2 * points + 4 * atoms * (h - 1), "flops": 2 * macs * atoms * (h - 1)}
    if kind == "refine":
        return {"bytes": 2 * points, "flops": 12 * REFINE_PASSES * REFINE_ROUNDS * atoms / 2}
    if kind == "plain":
        # per visit: three rows of the chain in, one out
        return {"bytes": 32 * atoms, "flops": 12 * CYCLE * case["blobs"]}
    frames = case["frames"]
    if kind == "atoms":
        # per atom its key points (4 at most) and two key pixels, about 400
        # operations of trajectory and fade; the image out
        return {"bytes": frames * (atoms * (8 * min(h, 4) + 8) + 4 * px), "flops": 400 * frames * atoms}
    # fluid: the particle state (18 doubles, 5 integers) in and out, its key
    # points in, the image out; about 600 operations per particle and step
    return {"bytes": frames * (fg * (2 * 164 + 8 * h) + 4 * px), "flops": 600 * FLUID_STEPS * frames * fg}


def exact(case, seed):
    """The fluid model's particles and the training step's gradient and loss
    in 64 bits; every other kind returns whole numbers."""
    if case["kind"] == "sim":
        P = torch.from_numpy(_particles(case, seed)).cuda()
        active = P[:, 16] > 0
        Q = P[active]
        for k in range(FLUID_STEPS):
            _fluid_step(Q, case["gsx"], case["gsy"], FLUID_STEPS - 1 - k)
        P[active] = Q
        return P
    if case["kind"] != "train":
        return None
    params, x, t = _training_batch(case["batch"], seed)
    p = params.double().requires_grad_(True)
    a, o = x.double(), 0
    for k, (din, dout) in enumerate(zip(DIMS[:-1], DIMS[1:])):
        w, b = p[o:o + din * dout].view(din, dout), p[o + din * dout:o + din * dout + dout]
        o += din * dout + dout
        a = a @ w + b
        if k < 4:
            a = F.gelu(a)
    loss = ((a - t.double()) ** 2).sum(1).mean()
    loss.backward()
    return {"grad": p.grad.detach(), "loss": loss.detach().view(1)}
