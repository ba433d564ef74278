"""3D plans left to the library's choice: launches of two time steps in the
shape that fits the grid and the number of shots, equal to single steps value
for value, in traces, all three field buffers and gradients.

The grids give every kind of chunk list: no CPML, CPML layers that fill the
march axis, idle sides, one chunk and many; few blocks (placed one by one) and
more than 256 per XCD (their mean).  The numbers of steps are odd and even.
"""
import numpy as np
import pytest

import awcpml
from cases import small3d
from test_gpu_two_step import _oracle, _plan, _same, _state

pytestmark = pytest.mark.gpu

GRIDS = {
    "tiny": ((5, 4, 6), 0, False, 1), "layers": ((19, 16, 13), 6, False, 1),
    "freetop": ((37, 29, 23), 5, True, 2), "open": ((70, 35, 27), 5, False, 3),
    "long": ((24, 20, 190), 4, False, 1), "flat": ((150, 90, 12), 3, True, 1),
    "many": ((66, 130, 41), 5, False, 60),
}


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("name", list(GRIDS))
def test_default_equals_single_steps(name, dtype):
    print("[gpu] default 3D launches %s %s" % (name, dtype), flush=True)
    n, halo, freetop, shots = GRIDS[name]
    case = small3d(n=n, halo=halo, freetop=freetop, nt=23)
    mid = [10.0 * (v // 2) for v in n]
    case["srcpos"], case["recpos"] = np.array([mid]), np.array([mid, [0.0, 0.0, 0.0]])
    o = _oracle(case)
    o.run()
    P = _plan(o, dtype=dtype, nshots=shots, srcs=[o.positions()[0]] * shots)

    def run(splits):
        P.reset()
        for k in splits:
            P.advance(k)
        return _state(P, shots)[:: max(1, shots - 1)]

    splits = [(o.nt,), (1, 2, o.nt - 3), (4, 1, o.nt - 5)]
    auto = [run(s) for s in splits]
    steps, rows, march, _ = P.time_block()
    assert steps == 2 and rows in ((8,) if dtype == "f64" else (8, 16)) and 4 <= march <= 96
    P.set_time_block(1)
    assert P.time_block()[0] == 1
    one = [run(s) for s in splits]
    for a, b in zip(auto, one):
        _same(a, b)
    if dtype == "f64":
        assert np.array_equal(one[0][0][0], o.traces())
        assert np.array_equal(auto[0][0][2], o.pend())
    P.close()


def test_default_graph_gradient_and_limits():
    """Replayed graphs, the gradient's forward and replay, and the cases that
    keep single steps: a source on a Dirichlet node, more than 32 sources."""
    print("[gpu] default 3D launches: graphs, gradient, limits", flush=True)
    o = _oracle(small3d(n=(40, 31, 27), halo=5, freetop=False, nt=26))
    o.run()
    P = _plan(o, nshots=2, srcs=[o.positions()[0]] * 2)
    P.advance(o.nt)
    want = _state(P, 2)
    P.set_graph(True)
    for _ in range(3):
        P.reset()
        P.advance(o.nt)
        _same(_state(P, 2), want)
    P.set_graph(False)
    obs = [0.5 * o.traces()] * 2
    auto = [awcpml.fwi.misfit_gradient(P, obs, every=k) for k in (1, 7, 26)]
    P.set_time_block(1)
    for k, g in zip((1, 7, 26), auto):
        one = awcpml.fwi.misfit_gradient(P, obs, every=k)
        assert one[0] == g[0] and np.array_equal(one[1], g[1])
    P.close()
    w = o.dt2srctf()
    ps = o.positions()[0]
    edge = ps.copy()
    edge[:, 2] = 1
    for srcs, wav in ((edge, w), (np.repeat(ps, 33, axis=0), np.asfortranarray(np.repeat(w, 33, axis=1) / 33))):
        P = _plan(o, srcs=[srcs], wav=wav)
        P.advance(o.nt)
        assert P.time_block()[0] == 1
        auto = _state(P, 1)
        P.set_time_block(1)
        P.reset()
        P.advance(o.nt)
        _same(_state(P, 1), auto)
        P.close()


@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_batch_shape_and_plans_that_ran(dtype):
    """Batches in the shape found for all their plans (one plan sets its own
    chunk length), and of plans that ran by themselves before."""
    print("[gpu] default 3D launches: batch %s" % dtype, flush=True)
    os_ = [_oracle(small3d(n=n, halo=h, freetop=f, nt=21))
           for n, h, f in (((37, 29, 23), 5, True), ((70, 19, 41), 4, False), ((24, 50, 90), 3, False))]
    plans = [_plan(o, dtype=dtype, nshots=k) for o, k in zip(os_, (1, 3, 2))]
    nt = min(o.nt for o in os_)
    want = []
    for P in plans:
        P.advance(nt)
        want.append([P.traces(s)[:nt] for s in range(P.nshots)])

    def check():
        with awcpml.Batch(plans) as B:
            B.reset()
            B.advance(nt)
            for P, w in zip(plans, want):
                assert all(np.array_equal(P.traces(s)[:nt], w[s]) for s in range(P.nshots))
            return B.time_block()

    assert check()[0] == 1  # nothing asked for two steps; the plans are not at home
    for P, march in zip(plans, (0, 7, 0)):
        P.reset()
        P.set_time_block(2, 0, march)
    assert check()[:2] == (2, 8 if dtype == "f64" else 16)
    for P in plans:
        P.close()
