"""The learned warm start on the GPU: sort-and-match keeps every chain row a
permutation of its points, and the trained network lowers the transport
cost the refinement starts from (and ends at for a fixed budget) against the
plain start the reference uses (rows in pixel order) and against the same
sort-and-match driven by an untrained network."""
import ctypes as C

import numpy as np
import pytest

from atomorph_amd import _capi as A
from atomorph_amd import learned as L
from atomorph_amd import morph as M
from atomorph_amd import synth
from oracle import oracle_py as op
from tests import gpu_util as G

pytestmark = pytest.mark.gpu


def _fresh(frames, seed=1):
    return L.build(frames, seed=seed, match_steps=2000)


def _rows(pts, widths):
    off = np.concatenate([[0], np.cumsum(widths)[:-1]])
    return [(o, w) for o, w in zip(off, widths)]


def test_warm_start_rows_stay_permutations():
    frames = synth.workload("blobs512")
    m = _fresh(frames)
    before, widths = m.chains()
    m.set_learned(L.init_params(seed=3))
    G.log("warm start, random network, blobs512")
    ms = m.warm_start()
    after, w2 = m.chains()
    assert np.array_equal(widths, w2) and ms > 0.0
    h = before.shape[0]
    assert np.array_equal(after[0], before[0])  # row 0 keeps its order
    moved = 0
    for y in range(1, h):
        for o, w in _rows(before, widths):
            a, b = np.sort(after[y, o:o + w]), np.sort(before[y, o:o + w])
            assert np.array_equal(a, b), (y, o, w)
            moved += int(np.count_nonzero(after[y, o:o + w] != before[y, o:o + w]))
    assert moved > 0


def test_trained_network_gains_over_plain_and_untrained_start():
    p = L.load_default()
    if p is None:
        pytest.fail("trained parameters missing: run python -m atomorph_amd.learned")
    frames = synth.workload("blobs512")
    base = _fresh(frames)
    c_plain = base.cost()
    pts0, widths = base.chains()
    costs = {}
    for name, params in (("trained", p), ("untrained", L.init_params(seed=3))):
        m = _fresh(frames)
        m.put_chains(pts0)
        m.set_learned(params)
        G.log(f"warm start {name}")
        m.warm_start()
        costs[name] = m.cost()
    G.log(f"start costs: plain {c_plain}, {costs}")
    assert costs["trained"] < 0.97 * c_plain
    assert costs["trained"] < costs["untrained"]
    # after the same batched budget the warm-started chains stay ahead
    ends = {}
    for name, params in (("plain", None), ("trained", p)):
        m = _fresh(frames)
        m.put_chains(pts0)
        if params is not None:
            m.set_learned(params)
            m.warm_start()
        m.set_refine(M.REFINE_BATCHED, rounds=32, tile=4, graph_passes=0)
        m.run(4)
        ends[name] = m.cost()
    G.log(f"after 4 batched passes: {ends}")
    assert ends["trained"] <= ends["plain"]


@pytest.mark.parametrize("width,chains,side", [(1, 1, 64), (1023, 1, 64), (1024, 2, 64), (1025, 1, 2000), (4097, 3, 64),
                                               (70000, 5, 300)])
def test_warm_start_matches_a_stable_sort_of_the_predictions(width, chains, side):
    """Row 1 against the match computed on the host from the same predictions:
    lists that end at, before and after the sort's blocks, keys of 20 to 30
    bits, and points and predictions that coincide (few distinct places)."""
    T, lib = G.torch(), G.lib()
    rng = np.random.default_rng(width)
    wid = np.array([width - (chains - 1) * (width // (chains + 1))] + [width // (chains + 1)] * (chains - 1), np.int64)
    off = np.concatenate([[0], np.cumsum(wid)[:-1]])
    x, y = rng.integers(0, min(side, 40), (2, 2, width))
    fx, fy = 64 * rng.integers(0, 4, (2, 2, width))
    zero = np.zeros(2 * width, np.int64)
    pts = op.pack_points(x.ravel(), y.ravel(), fx.ravel(), fy.ravel(), zero).ravel()
    dev = [G.zeros(2 * side * side, T.int32), G.to_dev(pts), G.to_dev(off), G.to_dev(wid.astype(np.int32)),
           G.zeros(2 * chains, T.int32), G.zeros(512, T.int32), G.zeros(512, T.int32)]
    R = A.RenderArgs(side, side, 2, chains, 0, 0, side - 1, side - 1, 4, 6, 0, 1, 0, 0, 0, chains, width,
                     *[d.data_ptr() for d in dev[:5]], None, dev[5].data_ptr(), dev[6].data_ptr())
    mlp = C.c_void_p()
    G.check(lib.amh_mlp_create(C.byref(mlp), 1024, G.stream()), "create")
    try:
        params = np.ascontiguousarray(L.init_params(seed=3), np.float32)
        G.check(lib.amh_mlp_set_params(mlp, op.ptr(params), G.stream()), "params")
        bytes_ = lib.amh_warm_workspace_bytes(width, chains, 2)
        ws, feat, pred = G.zeros(bytes_, T.uint8), G.zeros(8 * width, T.float32), G.zeros(2 * width, T.float32)
        G.log(f"warm start of {width} atoms in {chains} chains, {side}x{side}")
        G.check(lib.amh_learn_features(C.byref(R), 0, G.dptr(feat), None, G.dptr(ws), bytes_, G.stream()), "features")
        G.check(lib.amh_mlp_forward(mlp, G.dptr(feat), width, G.dptr(pred), G.stream()), "forward")
        G.check(lib.amh_warm_start(mlp, C.byref(R), G.dptr(dev[1]), G.dptr(ws), bytes_, G.stream()), "warm start")
        got, uv = G.to_host(dev[1], np.uint64), G.to_host(pred, np.float32).reshape(width, 2).astype(np.float64)
    finally:
        lib.amh_mlp_destroy(mlp)
    px, py = (x + fx / 256.0)[1], (y + fy / 256.0)[1]
    bits = int(np.ceil(np.log2(16 * side)))
    want = pts.copy()
    for o, w in zip(off, wid):
        at = slice(o, o + w)
        cx, cy = px[at].mean(), py[at].mean()
        s = np.sqrt((px[at] ** 2).mean() - cx * cx + (py[at] ** 2).mean() - cy * cy) + 1.0

        def order(u, v):
            u, v = (np.clip(np.rint(q), 0, 2 ** bits - 1).astype(np.int64) for q in (u, v))
            return np.argsort((v << bits) | u, kind="stable")

        slots = order(16 * (cx + s * uv[at, 0]), 16 * (cy + s * uv[at, 1]))
        held = order(np.floor(16 * px[at]), np.floor(16 * py[at]))
        want[width + o + slots] = pts[width + o + held]
    assert np.array_equal(got, want)
