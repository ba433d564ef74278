"""Plans and batches left to the library's choice of launches: what a call left
behind, accepted, refused or timed with one step per launch it does with several
(three fields after a gradient, batches whose plans run alone in between, timed
runs, memory that has run short).

Everything is compared value for value with a plan set to single steps, or with
the same call made another way.
"""
import ctypes

import numpy as np
import pytest

import awcpml
from awcpml import _lib
from cases import small2d, small3d
from test_gpu_two_step import _batch_state, _oracle, _plan, _same, _state

pytestmark = pytest.mark.gpu


def _case(nd, nt=30, freetop=True, n=None):
    """One source inside, so that launches of several steps apply."""
    n = n or ((61, 53) if nd == 2 else (37, 29, 23))
    case = (small2d if nd == 2 else small3d)(n=n, halo=5, freetop=freetop, nt=nt)
    case["srcpos"], case["t0s"] = np.array([[10.0 * (v // 2) for v in n]]), case["t0s"][:1]
    return case


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("nd", [2, 3])
def test_state_after_gradient(nd, dtype):
    """All three fields and the step count after a gradient, and the run that
    goes on from there."""
    print("[gpu] state after a gradient %dD %s" % (nd, dtype), flush=True)
    o = _oracle(_case(nd))
    o.run()
    obs = [0.5 * o.traces()] * 2
    plans = [_plan(o, dtype=dtype, nshots=2, srcs=[o.positions()[0]] * 2) for _ in range(2)]
    plans[1].set_time_block(1)
    for every in (1, 2, 3, 4, 5, 9, 11, 17, 30):
        got = []
        for P in plans:
            awcpml.fwi.misfit_gradient(P, obs, every=every)
            left = _state(P, 2)
            at = P.steps_done()
            P.advance(min(4, o.nt - at))
            got.append((at, left, _state(P, 2)))
        assert got[0][0] == got[1][0] == every
        _same(got[0][1], got[1][1])
        _same(got[0][2], got[1][2])
    for P in plans:
        P.close()


@pytest.mark.parametrize("nd", [2, 3])
@pytest.mark.parametrize("own", ["advance", "checkpoint"])
def test_batch_goes_on_after_a_plan_ran_on_its_own(nd, own):
    """A plan's first run of its own, and its reset, leave a batch that holds it
    as it was."""
    print("[gpu] batch after a plan's own run %dD %s" % (nd, own), flush=True)
    os_ = [_oracle(_case(nd, nt)) for nt in (30, 26)]
    ref = [_plan(o) for o in os_]
    for P, o in zip(ref, os_):
        P.set_time_block(1)
        P.advance(o.nt)
    plans = [_plan(o) for o in os_]
    with awcpml.Batch(plans) as B:
        plans[0].reset()
        plans[0].advance(12) if own == "advance" else plans[0].checkpoint_run(6)
        plans[0].reset()
        B.advance(30)
        _same(_batch_state(plans), _batch_state(ref))
        B.set_graph(True)
        for _ in range(2):
            B.run()
            _same(_batch_state(plans), _batch_state(ref))
        B.set_time_block(2)
        B.run()
        _same(_batch_state(plans), _batch_state(ref))
    for P in plans + ref:
        P.close()


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("nd", [2, 3])
@pytest.mark.parametrize("at", [2, 9, 10, 11, 17])
def test_batch_takes_a_plan_that_came_to_its_step_alone(nd, at, dtype):
    """A plan reset and run alone to the batch's step rejoins it there."""
    print("[gpu] batch takes a plan run alone to step %d, %dD %s" % (at, nd, dtype), flush=True)
    os_ = [_oracle(_case(nd, nt)) for nt in (30, 26)]
    ref = [_plan(o, dtype=dtype) for o in os_]
    for P, o in zip(ref, os_):
        P.set_time_block(1)
        P.advance(o.nt)
    plans = [_plan(o, dtype=dtype) for o in os_]
    with awcpml.Batch(plans) as B:
        for graph in (False, True):
            B.set_graph(graph)
            B.reset()
            B.advance(at)
            plans[0].reset()
            plans[0].advance(at)
            if graph:
                assert B.time_advance(30 - at) > 0
            else:
                B.advance(30 - at)
            _same(_batch_state(plans), _batch_state(ref))
        # another step than the batch's, and one more beside it, are refused as ever
        B.reset()
        B.advance(at)
        plans[0].reset()
        plans[0].advance(at)
        plans[0].forward(1)
        with pytest.raises(_lib.AwcpmlError, match="stepped or changed on its own"):
            B.advance(1)
        B.reset()
        B.advance(at)
        plans[0].reset()
        plans[0].advance(at - 1)
        with pytest.raises(_lib.AwcpmlError, match="stepped or changed on its own"):
            B.advance(1)
    for P in plans + ref:
        P.close()


@pytest.mark.parametrize("graph", [False, True])
def test_first_timed_run_holds_no_allocation(graph):
    """time_advance of a plan that has not run yet: the buffers it gets (30 MB
    here) and the graph it captures come before the events, so that a first run
    of one launch takes what the later ones take."""
    print("[gpu] first timed run, graph %s" % graph, flush=True)
    o = _oracle(_case(2, nt=8, n=(300, 290)))
    first, later = [], []
    for _ in range(6):
        P = _plan(o, nshots=44, srcs=[o.positions()[0]] * 44)
        P.set_graph(graph)
        P.reset()
        first.append(P.time_advance(o.nt))
        assert P.time_block()[0] == 2
        for _ in range(3):
            P.reset()
            later.append(P.time_advance(o.nt))
        P.close()
    print(first, later, flush=True)
    assert min(first) < 1.15 * max(later)


@pytest.mark.parametrize("nd", [2, 3])
def test_stencil2_timing_needs_the_request(nd):
    """time_stencil2 stays refused for a plan that never asked for two steps."""
    print("[gpu] time_stencil2 without a request %dD" % nd, flush=True)
    o = _oracle(_case(nd))
    P = _plan(o)
    for ran in (False, True):
        with pytest.raises(_lib.AwcpmlError, match="do not apply"):
            P.time_stencil2(1)
        P.advance(8)
    P.set_time_block(2)
    P.reset()
    assert P.time_stencil2(2) > 0
    P.close()


@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_2d_stencil_timing_is_of_the_launches_that_run(dtype):
    """time_stencil2 of a 2D plan times its steps in launches as long as
    awcpml_advance makes them.  One source and a few receivers add little to
    44 shots of 300 x 290 nodes, so both agree within half (a launch of two
    steps takes three times as long per step)."""
    print("[gpu] 2D stencil timing %s" % dtype, flush=True)
    o = _oracle(_case(2, nt=160, n=(300, 290)))
    P = _plan(o, dtype=dtype, nshots=44, srcs=[o.positions()[0]] * 44)
    P.set_time_block(2)
    stencil, run = [], []
    for _ in range(4):
        P.reset()
        run.append(P.time_advance(160) / 160)
        P.reset()
        stencil.append(P.time_stencil2(80) / 160)
    print(stencil, run, flush=True)
    assert 0.5 < min(stencil) / min(run) < 1.5
    for n in (1, 2, 3):
        P.reset()
        assert P.time_stencil2(n) > 0
    P.reset()
    P.advance(o.nt)
    two = _state(P, 1)
    P.set_time_block(1)
    P.reset()
    P.advance(o.nt)
    _same(two, _state(P, 1))
    P.close()


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("n,shots", [((70, 61), 3), ((40, 37), 5), ((30, 26, 24), 2), ((66, 17, 15), 5)])
def test_gradient_with_wide_offsets(n, shots, dtype):
    """The reverse step with 64-bit offsets (fields of 4 GiB and more per shot)
    forced on small grids: bitwise the 32-bit one."""
    print("[gpu] gradient with wide offsets %s %s" % (n, dtype), flush=True)
    o = _oracle(_case(len(n), nt=110, n=n))
    o.run()
    obs = [0.5 * o.traces()] * shots
    P = _plan(o, dtype=dtype, nshots=shots, srcs=[o.positions()[0]] * shots)
    for group in (0, 1, 2):
        P.set_adjoint_group(group)
        P.set_wide_offsets(False)
        J, g = awcpml.fwi.misfit_gradient(P, obs, every=7)
        P.set_wide_offsets(True)
        Jw, gw = awcpml.fwi.misfit_gradient(P, obs, every=7)
        assert P.time_block()[0] == 1
        assert J == Jw and np.array_equal(g, gw) and np.abs(g).max() > 0
    P.close()


class _Ballast:
    """Device memory taken so that `left` bytes stay free."""

    def __init__(self, left):
        self.hip = ctypes.CDLL("libamdhip64.so.7")
        self.hip.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
        self.hip.hipFree.argtypes = [ctypes.c_void_p]
        self.ptrs = []
        while self.free() > left:
            p = ctypes.c_void_p()
            assert self.hip.hipMalloc(ctypes.byref(p), min(self.free() - left, 32 << 30)) == 0
            self.ptrs.append(p)

    def free(self):
        v, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert self.hip.hipMemGetInfo(ctypes.byref(v), ctypes.byref(t)) == 0
        return v.value

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        for p in self.ptrs:
            self.hip.hipFree(p)


def test_spares_refused_once_are_asked_for_again():
    """A gradient's forward run that keeps single steps for the memory its
    reverse steps would need (here 336 GB) does not bind the runs after it."""
    print("[gpu] spares after a refusal", flush=True)
    K = 25000
    o = _oracle(_case(3, nt=K, n=(160, 150, 140)))
    P = _plan(o, dtype="f32")
    P.checkpoint_run(K)
    assert P.time_block()[0] == 1
    P.reset()
    P.advance(6)
    assert P.time_block()[0] == 2
    P.close()


def test_spares_refused_for_lack_of_memory_come_with_the_next_reset():
    """Little free memory at one run does not bind the runs after a reset."""
    print("[gpu] spares after a shortage", flush=True)
    n, S = (128, 160, 160), 10
    o = _oracle(_case(3, nt=9, n=n))
    P = _plan(o, dtype="f32", nshots=S, srcs=[o.positions()[0]] * S)
    with _Ballast(4 * S * int(np.prod(n)) * 7):  # less than 8 times the spare field
        P.advance(4)
        assert P.time_block()[0] == 1
    P.advance(5)
    assert P.time_block()[0] == 1
    one = _state(P, 1)
    P.reset()
    P.advance(9)
    assert P.time_block()[0] == 2
    _same(_state(P, 1), one)
    P.close()


def test_gradient_takes_the_spares_memory_back():
    """A gradient that fits only without the spare buffers the library took for
    an earlier run still fits."""
    print("[gpu] gradient in the memory of the spares", flush=True)
    n, K, S, h = (128, 160, 160), 10, 10, 5
    case = _case(3, nt=K, n=n, freetop=False)
    case["recpos"] = case["srcpos"] + np.array([[0.0] * 3, [20.0, 10.0, 0.0]])
    o = _oracle(case)
    P = _plan(o, dtype="f32", nshots=S, srcs=[o.positions()[0]] * S)
    P.set_adjoint_group(S)
    tbar = [np.ones((K, P._nrecs[s])) for s in range(S)]
    P.checkpoint_run(K)
    assert P.time_block()[0] == 2
    want = P.adjoint(tbar)
    assert np.abs(want).max() > 0
    fields = _state(P, S)
    # K fields of q, 3 of lam, two sets of slabs, the accumulators
    N = int(np.prod(n))
    slabs = sum((2 * h + 1) * N // v for v in n)
    need = 4 * S * (N * (K + 3) + 4 * slabs) + 12 * N
    spares = 4 * S * (N + 2 * slabs)
    P.checkpoint_run(K)
    with _Ballast(need - spares // 2) as B:
        print("[gpu] free %d of %d needed" % (B.free(), need), flush=True)
        got = P.adjoint(tbar)
    assert P.time_block()[0] == 1
    assert np.array_equal(got, want)
    _same(_state(P, S), fields)
    P.reset()
    P.advance(K)
    assert P.time_block()[0] == 2
    P.close()
