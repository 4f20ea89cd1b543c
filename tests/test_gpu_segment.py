"""GPU parity of ingest (HSP), segmentation, blob statistics, pixel grouping
and chain build, through the C ABI.  Integer work: bit-exact."""
import ctypes as C

import numpy as np
import pytest

from atomorph_amd import _capi as A
from atomorph_amd import synth
from oracle import oracle_py as op
from tests import gpu_util as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("absent", [0, 97])
def test_ingest_hsp_exhaustive(absent):
    """Every 24-bit colour through rgb_to_hsp and back equals the oracle, which
    equals the compiled reference: in float where the 8-bit rounding is clear
    and in FP64 in the reference's operation order where it is not.  Once with
    every colour present, once with every 97th pixel absent."""
    T = G.torch()
    lib = G.lib()
    words = (np.arange(1 << 24, dtype=np.uint32) | np.uint32(0xFF000000))
    if absent:
        words[::absent] &= np.uint32(0x00FFFFFF)  # (alpha 0)
    st_w, sh_w = op.ingest(words, 1)
    src = G.to_dev(words)
    st = G.zeros(words.size, T.int32)
    sh = G.zeros(words.size, T.int32)
    G.log("ingest 4096x4096 hsp=1")
    G.check(lib.amh_ingest_frame(G.dptr(src), 4096, 4096, 1, G.dptr(st), G.dptr(sh), G.stream()), "ingest")
    assert (G.to_host(st, np.uint32) == st_w).all()
    assert (G.to_host(sh, np.uint32) == sh_w).all()
    G.log("ingest hsp=0")
    G.check(lib.amh_ingest_frame(G.dptr(src), 4096, 4096, 0, G.dptr(st), G.dptr(sh), G.stream()), "ingest")
    st_w, sh_w = op.ingest(words, 0)
    assert (G.to_host(st, np.uint32) == st_w).all() and (G.to_host(sh, np.uint32) == sh_w).all()


def _segment(frame):
    T = G.torch()
    lib = G.lib()
    h, w = frame.shape[:2]
    src = G.to_dev(synth.to_words(frame))
    lab = G.zeros(h * w, T.int32)
    G.check(lib.amh_segment(G.dptr(src), w, h, G.dptr(lab), G.stream()), "amh_segment")
    return src, lab


def _frames():
    rng = np.random.default_rng(5)
    out = []
    for size, p in ((1, 0.9), (5, 0.6), (63, 0.55), (64, 0.6), (65, 0.5), (130, 0.58), (257, 0.6)):
        img = np.zeros((size, size + 3, 4), np.uint8)
        img[..., 3] = (rng.uniform(0, 1, (size, size + 3)) < p) * 255
        img[..., 0] = rng.integers(0, 256, (size, size + 3))
        out.append((f"random{size}", img))
    # worst case for tile merging: one serpentine component across tiles
    s = np.zeros((96, 200, 4), np.uint8)
    s[::2, :, 3] = 255
    s[1::4, -1, 3] = 255
    s[3::4, 0, 3] = 255
    out.append(("serpentine", s))
    out.append(("empty", np.zeros((17, 33, 4), np.uint8)))
    full = np.zeros((70, 70, 4), np.uint8)
    full[..., 3] = 1
    out.append(("full", full))
    return out


@pytest.mark.parametrize("name,frame", _frames(), ids=[n for n, _ in _frames()])
def test_segment_matches_oracle(name, frame):
    G.log(f"segment {name} {frame.shape}")
    _, lab = _segment(frame)
    want, n = op.segment(frame)
    assert (G.to_host(lab, np.int32) == want).all()


def test_segment_reference_blobs(golden_cfg1):
    for f in range(2):
        G.log(f"segment cfg1 frame {f}")
        _, lab = _segment(golden_cfg1["frames"][f])
        assert (G.to_host(lab, np.int32) == golden_cfg1["labels"][f]).all()


def test_segment_blobs512_full_size():
    frames = synth.workload("blobs512")
    for f, fr in enumerate(frames):
        G.log(f"segment blobs512 frame {f}")
        _, lab = _segment(fr)
        want, n = op.segment(fr)
        assert (G.to_host(lab, np.int32) == want).all()
        assert n == 40


def _stats_and_groups(frame):
    T = G.torch()
    lib = G.lib()
    h, w = frame.shape[:2]
    src, lab = _segment(frame)
    stored = G.zeros(h * w, T.int32)
    G.check(lib.amh_ingest_frame(G.dptr(src), w, h, 1, G.dptr(stored), None, G.stream()), "ingest")
    ws = G.zeros(lib.amh_blob_workspace_bytes(w, h) // 4 + 1, T.int32)
    nb = C.c_int32(0)
    G.check(lib.amh_blob_count(G.dptr(lab), w, h, G.dptr(ws), C.byref(nb), G.stream()), "count")
    nb = nb.value
    bop = G.zeros(h * w, T.int32)
    st = T.zeros(max(nb, 1) * C.sizeof(A.BlobStat), dtype=T.uint8, device="cuda")
    G.check(lib.amh_blob_stats(G.dptr(lab), G.dptr(stored), w, h, G.dptr(ws), nb, G.dptr(bop), G.dptr(st),
                               G.stream()), "stats")
    gws_b = lib.amh_group_workspace_bytes(h * w, nb)
    gws = T.zeros(max(gws_b, 4), dtype=T.uint8, device="cuda")
    first = G.zeros(nb + 1, T.int64)
    plist = G.zeros(h * w, T.int32)
    G.check(lib.amh_group_pixels(G.dptr(bop), h * w, nb, G.dptr(gws), gws_b, G.dptr(first), G.dptr(plist),
                                 G.stream()), "group")
    stats = (A.BlobStat * max(nb, 1)).from_buffer_copy(st.cpu().numpy().tobytes())
    return nb, G.to_host(bop, np.int32), stats, G.to_host(first, np.int64), G.to_host(plist, np.int32), stored


@pytest.mark.parametrize("which", ["cfg1", "blobs512"])
def test_blob_stats_and_grouping(which, golden_cfg1):
    frames = golden_cfg1["frames"] if which == "cfg1" else synth.workload("blobs512")
    for f, fr in enumerate(frames):
        G.log(f"blob stats {which} frame {f}")
        h, w = fr.shape[:2]
        nb, bop, stats, first, plist, stored_d = _stats_and_groups(fr)
        lab, n = op.segment(fr)
        assert nb == n
        roots = np.sort(np.unique(lab[lab >= 0]))
        stored, _ = op.ingest(synth.to_words(fr), 1)
        for b, r in enumerate(roots):
            idx = np.nonzero(lab == r)[0]
            assert (bop[idx] == b).all()
            s = stats[b]
            assert s.count == idx.size and s.first == r
            assert s.sum_x == int((idx % w).sum()) and s.sum_y == int((idx // w).sum())
            for k in range(4):
                assert s.sum_c[k] == int(((stored[idx] >> (8 * k)) & 255).sum())
            assert (s.x1, s.y1, s.x2, s.y2) == (int((idx % w).min()), int((idx // w).min()),
                                                int((idx % w).max()), int((idx // w).max()))
            # grouped pixel list: the blob's pixels in row-major order
            assert (plist[first[b]:first[b + 1]] == idx).all()
        assert first[nb] == int((lab >= 0).sum())
        assert (bop[lab < 0] == -1).all()


@pytest.mark.parametrize("w,h,cover", [(64, 64, 0.5), (64, 65, 0.6), (65, 31, 0.6), (129, 33, 0.3), (200, 161, 0.62),
                                       (1, 1, 1.0), (300, 7, 0.45)])
def test_dithered_frames_around_tile_edges(w, h, cover):
    """Random dithers (hundreds of blobs in a tile, blobs across tile edges)
    at one tile, one pixel more, and ragged sizes: labels, statistics and
    grouping are exactly those of the oracle's labels."""
    rng = np.random.default_rng(w * 1000 + h)
    fr = rng.integers(0, 256, (h, w, 4)).astype(np.uint8)
    fr[..., 3] = np.where(rng.uniform(size=(h, w)) < cover, rng.integers(1, 256, (h, w)), 0)
    G.log(f"dither {w}x{h} {cover}")
    _, lab_d = _segment(fr)
    lab, n = op.segment(fr)
    assert (G.to_host(lab_d, np.int32) == lab).all()
    nb, bop, stats, first, plist, _ = _stats_and_groups(fr)
    roots = np.unique(lab[lab >= 0])
    assert nb == n == roots.size
    want = np.where(lab >= 0, np.searchsorted(roots, lab), -1)
    assert (bop == want).all()
    idx = np.flatnonzero(want >= 0)
    order = idx[np.argsort(want[idx], kind="stable")]
    assert (plist[:idx.size] == order).all()
    counts = np.bincount(want[idx], minlength=nb)
    assert (first == np.concatenate([[0], np.cumsum(counts)])).all()
    stored, _ = op.ingest(synth.to_words(fr), 1)
    x, y = idx % w, idx // w
    s = stats[:nb]
    assert [v.count for v in s] == counts.tolist() and [v.first for v in s] == roots.tolist()
    for got, value in (("sum_x", x), ("sum_y", y)):
        assert [getattr(v, got) for v in s] == [int(q) for q in np.bincount(want[idx], value, minlength=nb)]
    for k in range(4):
        sums = np.bincount(want[idx], (stored[idx] >> (8 * k)) & 255, minlength=nb)
        assert [v.sum_c[k] for v in s] == [int(q) for q in sums]
    for b in range(0, nb, max(1, nb // 50)):
        m = want[idx] == b
        assert (s[b].x1, s[b].y1, s[b].x2, s[b].y2) == (x[m].min(), y[m].min(), x[m].max(), y[m].max())


def test_blob_numbers_of_a_frame_beyond_the_summing_blocks():
    """4096 x 2049 pixels, 8,196 blocks of 1,024: from 8,192 on the blocks'
    counts are scanned instead of summed by every block.  Count, numbers and
    statistics are those of the oracle's labels; the last pixel is a blob."""
    T, lib, w, h = G.torch(), G.lib(), 4096, 2049
    rng = np.random.default_rng(8)
    fr = np.zeros((h, w, 4), np.uint8)
    fr[rng.uniform(size=(h, w)) < 0.002] = (10, 200, 30, 255)
    fr[-1, -1] = (9, 8, 7, 255)
    G.log("blob numbers 4096x2049")
    src, lab_d = _segment(fr)
    lab, n = op.segment(fr)
    assert (G.to_host(lab_d, np.int32) == lab).all()
    ws = G.zeros(lib.amh_blob_workspace_bytes(w, h) // 4 + 1, T.int32)
    nb = C.c_int32(0)
    G.check(lib.amh_blob_count(G.dptr(lab_d), w, h, G.dptr(ws), C.byref(nb), G.stream()), "count")
    roots = np.flatnonzero(lab == np.arange(lab.size))
    assert nb.value == n == roots.size and lab[-1] >= 0
    bop = G.zeros(h * w, T.int32)
    st = T.zeros(n * C.sizeof(A.BlobStat), dtype=T.uint8, device="cuda")
    G.check(lib.amh_blob_stats(G.dptr(lab_d), G.dptr(src), w, h, G.dptr(ws), n, G.dptr(bop), G.dptr(st), G.stream()),
            "stats")
    want = np.where(lab >= 0, np.searchsorted(roots, lab), -1)
    assert (G.to_host(bop, np.int32) == want).all()
    stats = (A.BlobStat * n).from_buffer_copy(st.cpu().numpy().tobytes())
    assert [s.first for s in stats] == roots.tolist()
    assert [s.count for s in stats] == np.bincount(want[want >= 0], minlength=n).tolist()


def _group(bop_host, nb):
    T = G.torch()
    lib = G.lib()
    n = bop_host.size
    gws_b = lib.amh_group_workspace_bytes(n, nb)
    gws = T.zeros(max(gws_b, 4), dtype=T.uint8, device="cuda")
    bop = G.to_dev(np.ascontiguousarray(bop_host, np.int32))
    first = G.zeros(nb + 1, T.int64)
    plist = G.zeros(n, T.int32)
    G.check(lib.amh_group_pixels(G.dptr(bop), n, nb, G.dptr(gws), gws_b, G.dptr(first), G.dptr(plist), G.stream()),
            "group")
    return G.to_host(first, np.int64), G.to_host(plist, np.int32), gws_b


@pytest.mark.parametrize("case", ["checkerboard512", "few_blobs", "many_blobs", "sparse_many", "one_blob"])
def test_group_pixels_any_blob_count(case):
    """Stable grouping of pixels by blob for blob counts from 1 to a
    checkerboard's 131,072 single-pixel blobs: the per-(block, blob) table
    for few blobs, the radix sort beyond; both give the pixels of each blob
    in row-major order, and the workspace stays O(pixels + blobs)."""
    rng = np.random.default_rng(9)
    if case == "checkerboard512":
        yy, xx = np.mgrid[0:512, 0:512]
        on = ((xx + yy) % 2 == 0).ravel()
        bop = -np.ones(512 * 512, np.int32)
        bop[on] = np.arange(int(on.sum()))
        nb = int(on.sum())
    elif case == "few_blobs":
        nb = 300
        bop = rng.integers(-1, nb, 256 * 256).astype(np.int32)
    elif case == "many_blobs":
        nb = 5000
        bop = rng.integers(-1, nb, 256 * 256).astype(np.int32)
    elif case == "sparse_many":
        nb = 70000
        bop = np.where(rng.uniform(size=1024 * 512) < 0.6, rng.integers(0, nb, 1024 * 512), -1).astype(np.int32)
    else:
        nb = 1
        bop = np.where(rng.uniform(size=333 * 77) < 0.5, 0, -1).astype(np.int32)
    G.log(f"group pixels {case}: {bop.size} pixels, {nb} blobs")
    first, plist, ws = _group(bop, nb)
    counts = np.bincount(bop[bop >= 0], minlength=nb)
    assert np.array_equal(first, np.concatenate([[0], np.cumsum(counts)]))
    idx = np.flatnonzero(bop >= 0)
    want = idx[np.argsort(bop[idx], kind="stable")]
    assert np.array_equal(plist[:idx.size], want)
    assert ws <= 24 * bop.size + 16 * nb + (1 << 20)


@pytest.mark.parametrize("n,nb,kind", [(4096, 1024, "any"), (4096, 1025, "any"), (4097, 1024, "any"),  # one workgroup
                                       (2048 * 31 + 5, 2048, "band"), (100_003, 3000, "few")])
def test_group_pixels_at_path_edges(n, nb, kind):
    """The one-workgroup grouping's limits and just beyond them; a band of
    pixels of as many blobs as it has pixels; few of many blobs present."""
    rng = np.random.default_rng(n + nb)
    bop = rng.integers(-1, nb, n).astype(np.int32)
    if kind == "band":
        bop[:2048] = rng.permutation(nb)
    elif kind == "few":
        bop = rng.choice([-1, 0, 1, 2, 1500, 2999], n).astype(np.int32)
    G.log(f"group pixels {n}, {nb} blobs, {kind}")
    first, plist, _ = _group(bop, nb)
    idx = np.flatnonzero(bop >= 0)
    assert np.array_equal(first, np.concatenate([[0], np.cumsum(np.bincount(bop[idx], minlength=nb))]))
    assert np.array_equal(plist[:idx.size], idx[np.argsort(bop[idx], kind="stable")])


def test_engine_detects_checkerboard_alpha():
    """A dithered (checkerboard) alpha channel: every present pixel is its
    own blob, 131,072 per 512^2 key frame, through am::morph's detection."""
    from atomorph_amd import morph as M
    yy, xx = np.mgrid[0:512, 0:512]
    frames = []
    for k in range(2):
        f = np.zeros((512, 512, 4), np.uint8)
        on = (xx + yy + k) % 2 == 0
        f[on] = (200, 40 + 100 * k, 90, 255)
        frames.append(f)
    m = M.Morph()
    m.set(seed=1)
    for i, f in enumerate(frames):
        m.add_frame_rgba(i, f)
    m.set_resolution(512, 512)
    G.log("checkerboard alpha: detection")
    assert m.run(1) == M.STATE_BLOB_UNIFICATION, m.error()
    for k in range(2):
        assert m.blob_count(k) == 512 * 512 // 2
        for b in (0, 1, 77777, 131071):
            s = m.blob(k, b)["surface"]
            assert len(s) == 1
