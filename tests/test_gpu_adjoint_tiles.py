"""The reverse step at its tiles' edges: grids whose x tile reaches both CPML
sides, whose last tile holds one node or 64, the thinnest halos, the smallest
n = 2 halo + 4, and block counts on both sides of one block per XCD; several
shots in groups that divide them and that do not.

FP64: the sum over the shots of the oracle's gradients, to 1e-10 relative L2
(the same terms in another order over at most 110 steps and 5 shots; each order
errs by less than 1e-13).  FP32: to 1e-3, as the forward's own FP32 error allows.
"""
import numpy as np
import pytest

from awcpml import fwi
from cases import rel_l2, small2d, small3d
from test_gpu_features import oracle_for, plan_from_oracle

pytestmark = pytest.mark.gpu

GRIDS = {
    "2d-both-sides": ((40, 37), 12, False), "2d-smallest": ((16, 16), 6, False),
    "2d-one-node": ((66, 41), 5, True), "2d-full": ((65, 38), 4, False),
    "2d-two-tiles": ((129, 90), 7, False), "2d-halo1": ((70, 30), 1, False),
    "3d-both-sides": ((30, 26, 24), 8, False), "3d-smallest": ((10, 10, 10), 3, False),
    "3d-one-node": ((66, 17, 15), 2, True), "3d-halo1": ((65, 13, 12), 1, False),
    "3d-classes": ((133, 21, 19), 3, False),
}


@pytest.mark.parametrize("name", list(GRIDS))
def test_reverse_step_tiles(name):
    print("[gpu] reverse step tiles %s" % name, flush=True)
    n, halo, freetop = GRIDS[name]
    case = (small2d if len(n) == 2 else small3d)(n=n, halo=halo, freetop=freetop,
                                                nt=110 if len(n) == 2 else 70)
    mid = [10.0 * (v // 2) for v in n]
    # receivers in the layers' inner ends, the middle and a corner node
    case["srcpos"], case["t0s"] = np.array([mid]), case["t0s"][:1]
    case["recpos"] = np.array([mid, [10.0 * halo] * len(n), [10.0] * len(n)])
    o = oracle_for(case)
    o.run()
    obs = 0.5 * o.traces()
    J, g = o.fwi_gradient(obs)
    for dtype, tol in (("f64", 1e-10), ("f32", 1e-3)):
        P = plan_from_oracle(o, dtype=dtype)
        assert rel_l2(fwi.misfit_gradient(P, obs, every=6)[1], g) <= tol
        P.close()
        P = plan_from_oracle(o, dtype=dtype, nshots=5)
        for group in (0, 1, 2, 5):
            P.set_adjoint_group(group)
            assert rel_l2(fwi.misfit_gradient(P, [obs] * 5, every=9)[1], 5 * g) <= tol, group
        P.close()


@pytest.mark.parametrize("dirichlet", [False, True])
@pytest.mark.parametrize("nd", [2, 3])
def test_checkpoints_of_two_and_three_fields(nd, dirichlet):
    """Segments of 1 and 2 steps and sources on Dirichlet nodes keep the third
    field; the oracle's gradient either way (FP64, 1e-10 as above), and from
    every spacing the same forward state afterwards as from single steps."""
    print("[gpu] checkpoints %dD dirichlet %s" % (nd, dirichlet), flush=True)
    n = (43, 37) if nd == 2 else (23, 21, 19)
    case = (small2d if nd == 2 else small3d)(n=n, halo=5, freetop=True, nt=30)
    case["srcpos"], case["t0s"] = case["srcpos"][:1].copy(), case["t0s"][:1]
    case["srcpos"][0] = [10.0 * (v // 2) for v in n]
    if dirichlet:
        case["srcpos"][0][-1] = 0.0
    o = oracle_for(case)
    o.run()
    obs = 0.5 * o.traces()
    _, g = o.fwi_gradient(obs)
    P, Q = plan_from_oracle(o), plan_from_oracle(o)
    Q.set_time_block(1)
    for every in (1, 2, 3, 4, 17, 30):
        for R in (P, Q):
            assert rel_l2(fwi.misfit_gradient(R, obs, every=every)[1], g) <= 1e-10, every
        assert np.array_equal(P.field(0, 1), Q.field(0, 1))
    P.close()
    Q.close()
