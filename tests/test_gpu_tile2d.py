"""Several time steps of a 2D plan per launch on register tiles
(csrc/tile2d_kernels.h): equal to single steps, value for value, in traces,
all three field buffers and gradients.

The grids sit at the tiles' edges (48 owned nodes in x; 16 or 48 owned rows),
with sources and receivers on the owned nodes' edges, in the rings tiles
share, on one node, and (receivers) on Dirichlet nodes.  The numbers of steps
cover every remainder of a launch's 8.
"""
import numpy as np
import pytest

import awcpml
from cases import small2d
from test_gpu_two_step import _oracle, _plan, _same, _state

pytestmark = pytest.mark.gpu


def _case(n, halo, freetop, nt):
    case = small2d(n=n, halo=halo, freetop=freetop, nt=nt)
    mid = [10.0 * (v // 2) for v in n]
    case["srcpos"], case["t0s"], case["recpos"] = np.array([mid]), case["t0s"][:1], np.array([mid])
    return case


def _points(n):
    """1-based nodes on and next to tile edges, near the corners, in the middle."""
    xs = sorted({2, 3, n[0] - 1, n[0] // 2} | {v for v in (48, 49, 56, 57, 96, 97) if v < n[0]})
    ys = sorted({2, n[1] - 1, n[1] // 2} | {v for v in (17, 18, 26, 49, 50) if v < n[1]})
    return np.array([[x, y] for x in xs for y in ys], dtype=np.int64)


# the smallest grids, one node around a tile's owned width, no CPML, idle top,
# slabs that touch (n = 2*halo+3) and overlap; shots enough for 64-row tiles
# and for the split into tiles with and without CPML nodes
GRIDS = {
    "tiny": ((5, 4), 0, False, 1), "nohalo": ((101, 67), 0, False, 1), "touch": ((15, 17), 6, False, 1),
    "overlap": ((30, 33), 20, True, 1), "own-1": ((49, 33), 6, True, 2), "own": ((50, 34), 6, False, 1),
    "own+1": ((51, 35), 6, False, 1), "wide": ((213, 61), 9, True, 3), "tall": ((58, 190), 7, False, 2),
    "rows64": ((150, 147), 8, True, 70), "split": ((300, 290), 6, False, 44),
}


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("name", list(GRIDS))
def test_tiles_equal_single_steps(name, dtype):
    n, halo, freetop, shots = GRIDS[name]
    o = _oracle(_case(n, halo, freetop, 29))
    pts = _points(n)
    w = o.dt2srctf()
    srcs = [pts[[(3 * s) % len(pts), (7 * s + 1) % len(pts), (3 * s) % len(pts)]] for s in range(shots)]
    wav = np.asfortranarray(np.concatenate([w, -0.4 * w, 0.7 * w], axis=1))  # two on one node
    P = _plan(o, dtype=dtype, nshots=shots, srcs=srcs, wav=wav)
    rec = np.concatenate([pts, [[1, 1], [n[0], n[1] // 2 + 1], [2, n[1]]], pts[:2]])
    for s in range(shots):
        P.set_receivers(s, rec if s % 2 == 0 else rec[::3])
    show = sorted({0, shots // 2, shots - 1})

    def state():
        return [[P.traces(s)] + [P.field(s, k) for k in range(3)] for s in show]

    def run(splits):
        P.reset()
        for k in splits:
            P.advance(k)
        return state()

    # the plan's own choice, before any setting, against single steps
    splits = [(29,), (1, 2, 3, 4, 5, 6, 8), (10, 19), (11, 18)]
    auto = [run(s) for s in splits]
    P.set_time_block(1)
    one = [run(s) for s in splits]
    for a, b in zip(auto, one):
        _same(a, b)
    assert max(np.abs(t[0]).max() for t in one[0]) > 0
    P.set_time_block(2)
    P.set_graph(True)
    for _ in range(3):
        _same(run((29,)), one[0])
    P.close()


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("n,shots", [((61, 53), 3), ((150, 147), 70)])
def test_gradient_through_tiles(n, shots, dtype):
    """Checkpoint intervals that leave every launch length in the replay."""
    o = _oracle(_case(n, 7, False, 26))
    o.run()
    P = _plan(o, dtype=dtype, nshots=shots, srcs=[o.positions()[0]] * shots)
    obs = [0.5 * o.traces()] * shots
    for every in (1, 3, 9, 26):
        auto = awcpml.fwi.misfit_gradient(P, obs, every=every)
        P.set_time_block(1)
        one = awcpml.fwi.misfit_gradient(P, obs, every=every)
        P.set_time_block(2)
        assert auto[0] == one[0]
        assert np.array_equal(auto[1], one[1])
    P.close()


def test_batch_accepts_plans_that_ran_on_their_own():
    """A plan that ran without any launch setting may join a batch without a
    reset of its own, as one that ran single steps may."""
    o = _oracle(_case((57, 43), 6, True, 30))
    plans = [_plan(o), _plan(o)]
    for P in plans:
        P.reset()
    plans[0].advance(12)
    plans[0].advance(o.nt - 12)
    want = plans[0].traces()
    with awcpml.Batch(plans) as B:
        B.run()
        for P in plans:
            assert np.array_equal(P.traces(), want)
    for P in plans:
        P.close()


# tiles that begin before the corner: the same grid size modulo 48 at different
# halos and idle sides moves the beginning through its whole range
@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("n,halo,freetop", [((171, 150), 8, False), ((200, 163), 11, True), ((207, 197), 20, False),
                                            ((175, 191), 3, True), ((193, 162), 15, False)])
def test_moved_tiles_equal_single_steps(n, halo, freetop, dtype):
    print("[gpu] moved tiles %s %d %s" % (n, halo, dtype), flush=True)
    o = _oracle(_case(n, halo, freetop, 21))
    pts = _points(n)
    shots = 520
    srcs = [pts[[(5 * s) % len(pts)]] for s in range(shots)]
    P = _plan(o, dtype=dtype, nshots=shots, srcs=srcs)
    for s in range(shots):
        P.set_receivers(s, pts[s % 3::3])
    show = range(0, shots, 37)

    def run(k):
        P.reset()
        P.advance(k)
        P.advance(o.nt - k)
        return [[P.traces(s)] + [P.field(s, f) for f in range(3)] for s in show]

    moved = [run(0), run(11)]
    P.set_time_block(1)
    one = run(0)
    for m in moved:
        _same(m, one)
    P.close()


@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_gradient_of_segments_past_the_cache(dtype):
    """q fields of one segment above 256 MiB are stored past the caches."""
    o = _oracle(_case((300, 290), 6, False, 20))
    o.run()
    shots = 60
    P = _plan(o, dtype=dtype, nshots=shots, srcs=[o.positions()[0]] * shots)
    obs = [0.5 * o.traces()] * shots
    assert 300 * 290 * shots * o.nt * (8 if dtype == "f64" else 4) > 256 << 20
    auto = awcpml.fwi.misfit_gradient(P, obs, every=o.nt)
    P.set_time_block(1)
    one = awcpml.fwi.misfit_gradient(P, obs, every=o.nt)
    assert auto[0] == one[0] and np.array_equal(auto[1], one[1])
    P.close()
