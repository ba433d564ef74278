"""Host transfers of fields, models and traces: the device packs padded rows
into dense FP64 ones and back (csrc/transfer_kernels.h).

The final field a plan returns must hold, at every receiver node, the last
sample of that receiver's trace: both come from the same device value through
different transfers, so they agree exactly.  FP64 fields and traces are also
the oracle's, bit for bit.
"""
import numpy as np
import pytest

from cases import oracle_problem, small2d, small3d

pytestmark = pytest.mark.gpu


def _nodes(n, count, seed):
    """1-based nodes: random ones and every corner row's ends."""
    rng = np.random.Generator(np.random.PCG64(seed))
    pos = [[int(rng.integers(1, v + 1)) for v in n] for _ in range(count)]
    pos += [[1] + list(n[1:]), list(n), [n[0] // 2 + 1] + [1] * (len(n) - 1)]
    return np.array(pos, dtype=np.int64)


# rows shorter and longer than one 1024-element segment, a pitch equal to the
# row (no padding), and a field longer than one 4 Mi-element stage
@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("n", [(57, 43), (64, 40), (1030, 37), (2100, 2050), (33, 29, 31), (32, 27, 26)])
def test_field_and_traces_hold_the_same_values(dtype, n):
    import awcpml
    big = n[0] * n[1] > 1 << 20
    case = (small2d if len(n) == 2 else small3d)(n=n, halo=5, nt=24 if big else 60)
    srcs = awcpml.Sources(case["srcpos"], case["t0s"], [awcpml.rickersource1D] * len(case["srcpos"]), case["f0"])
    S = awcpml.setup(case["l"], case["lt"], case["vel"], srcs, awcpml.Receivers(case["recpos"]),
                     halo=case["halo"], rcoef=case["rcoef"], ppw=case["ppw"], freetop=case["freetop"])
    pos = _nodes(n, 700, 11)  # enough values that wavelet and trace transfers leave the short path
    near = S.possrcs[:1] + np.array([[q % 7 - 3, q // 7] + [0] * (len(n) - 2) for q in range(28)])
    pos = np.concatenate([pos, np.clip(near, 1, np.array(n))])
    with awcpml.Plan.from_setup(S, dtype=dtype) as P:
        P.set_receivers(0, pos)
        P.reset()
        P.advance(S.nt)
        tr, field = P.traces(0), P.field(0)
    at = field[tuple((pos - 1).T)]
    assert np.abs(at).max() > 0
    assert np.array_equal(at, tr[-1])
    if dtype == "f64":
        o = oracle_problem(case)
        o.run()
        assert np.array_equal(field, o.pend())
