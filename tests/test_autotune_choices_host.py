"""CPU tests of the autotuner's 2D branch, its cache and the library's own 3D
choice, with the stand-in plan of
test_autotune_host: launches of several steps are taken where they apply and are
faster, and single steps kept where their buffers do not fit.  Choices that
other kernels were timed for do not count."""
import json

import pytest

from awcpml import _lib
from test_autotune_host import FakePlan, at


class Fake2D(FakePlan):
    """Whole steps of `one` ms, of `multi` ms in launches of several steps."""

    def __init__(self, one=1.0, multi=0.3, applies=True, fits=True):
        super().__init__(ndim=2)
        self.nt, self.one, self.multi, self.applies, self.fits = 100, one, multi, applies, fits

    def set_time_block(self, steps, *shape):
        if steps == 2 and not self.fits:
            raise _lib.AwcpmlError(-3, "out of memory")
        super().set_time_block(steps, *shape)

    def time_block(self):
        return (2 if self.tb[0] == 2 and self.applies else 1, 4, 16, 2)

    def advance(self, n):
        pass

    def time_advance(self, n):
        return n * (self.multi if self.tb[0] == 2 else self.one)

    def time_stencil2(self, n):
        return 0.25 * 2 * n


def test_2d_takes_several_steps_per_launch(tmp_path):
    P = Fake2D()
    best = at.autotune(P, cache=str(tmp_path / "t.json"))
    assert P.tb[0] == 2 and best["time_block"] is not None
    # both figures are measured: whole steps, and the stencil launches alone
    assert best["ms_per_whole_step"] == pytest.approx(0.3)
    assert best["ms_per_step"] == pytest.approx(0.25)
    Q = Fake2D()
    assert at.autotune(Q, cache=str(tmp_path / "t.json"))["cached"] and Q.tb[0] == 2


def test_2d_keeps_single_steps_when_faster(tmp_path):
    P = Fake2D(multi=1.2)
    best = at.autotune(P, cache=str(tmp_path / "t.json"))
    assert P.tb[0] == 1 and best["time_block"] is None
    assert best["ms_per_whole_step"] == pytest.approx(1.0)
    assert best["ms_per_step"] == best["ms_per_launch"]


def test_2d_buffers_that_do_not_fit(tmp_path):
    P = Fake2D(fits=False)
    best = at.autotune(P, cache=str(tmp_path / "t.json"))
    assert P.tb[0] == 1 and best["time_block"] is None


def test_2d_launches_that_do_not_apply(tmp_path):
    """Two identical single-step runs: the second one's luck decides nothing."""
    P = Fake2D(multi=0.99, applies=False)
    best = at.autotune(P, cache=str(tmp_path / "t.json"))
    assert P.tb[0] == 1 and best["time_block"] is None


def test_choices_of_other_kernels_are_timed_anew(tmp_path):
    """An entry without the kernels' digest, or with another, would pin the plan
    to a choice that the present kernels were not timed for."""
    old = {"block_y": 4, "march_len": 64, "prefetch": 3, "shot_group": 1, "ms_per_launch": 1.0,
           "ms_per_step": 1.0, "time_block": None, "tried": 3}
    P = Fake2D()
    plain = "2D:298x298:h20:f32:s8"
    assert at._key(P).startswith(plain + ":")
    cache = tmp_path / "old.json"
    cache.write_text(json.dumps({plain: old, plain + ":0123456789ab": old}))
    best = at.autotune(P, cache=str(cache))
    assert not best["cached"] and P.tb[0] == 2
    assert set(json.loads(cache.read_text())) == {plain, plain + ":0123456789ab", at._key(P)}
    assert at.autotune(Fake2D(), cache=str(cache))["cached"]


def test_3d_library_choice_is_a_candidate(tmp_path):
    cache = str(tmp_path / "t.json")
    ms = {(0, 0, 0, True): 1.3, (0, 0, 0, False): 1.5, (16, 144, 3, True): 1.4}
    P = FakePlan(two_ms=ms, one_ms=0.95)
    best = at.autotune(P, cache=cache)
    assert P.tb == (2, 0, 0, 0) and P.align is True
    assert best["time_block"] == {"block_rows": 0, "march_len": 0, "prefetch": 0, "align": True}
    Q = FakePlan(two_ms=ms, one_ms=0.95)
    assert at.autotune(Q, cache=cache)["cached"] and Q.tb == (2, 0, 0, 0)
