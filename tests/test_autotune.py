"""The autotuner's choices on a context that records what it is asked to do."""
import pytest

from langevina_amd import autotune
from langevina_amd.lgv import PHI_AUTO, PHI_MARCH, PHI_SITE


class Recorder:
    """A context whose launch times do not depend on the tiles: the first timing
    of each class is 1 ms, later ones wander by 2 per cent below it."""

    def __init__(self, N, pairs, scounts=(2, 3)):
        self.N, self.nrep, self.precision = [N], 1, 0
        self.scounts = scounts
        self.pairs_auto, self.kernel = pairs, PHI_AUTO
        self.sweep, self.ideal = [], []
        self.timed = 0
        self.tile = (56, 8)

    def ideal_tile(self, replica=0):
        return self.tile

    def step(self, dt):
        pass

    run = step

    def set_phi_kernel(self, kernel):
        self.kernel = kernel

    def phi_kernel(self):
        return PHI_SITE if self.kernel == PHI_SITE else PHI_MARCH

    def phi_pairs(self):
        return self.pairs_auto if self.kernel == PHI_AUTO else 0


@pytest.fixture
def tuner(monkeypatch):
    monkeypatch.setattr(autotune, "set_sweep_tiles",
                        lambda ctx, r, *t: ctx.sweep.append(t))
    monkeypatch.setattr(autotune, "set_ideal_tile", lambda ctx, r, *t: ctx.ideal.append(t))

    def class_ms(ctx, dt, steps, cls):
        if cls is None:  # whole steps: the size rule's phi kernel is the fastest
            return {PHI_AUTO: 1.0, PHI_SITE: 1.2, PHI_MARCH: 1.1}[ctx.kernel]
        ctx.timed += 1
        return 1.0 - 0.02 * (ctx.timed % 3 == 2)

    monkeypatch.setattr(autotune, "_class_ms", class_ms)
    return autotune


def test_march_tiles_are_not_tuned_where_steps_run_pairs(tuner):
    ctx = Recorder(256, pairs=2)
    chosen = tuner.autotune_sweeps(ctx, 0.04)
    assert ctx.kernel == PHI_AUTO
    assert chosen[256][:2] == (0, 0)
    assert all(t[:2] == (0, 0) for t in ctx.sweep)


@pytest.mark.parametrize("pairs,scounts", [(0, (2, 3)), (2, (1, 3))])
def test_march_tiles_are_tuned_where_steps_run_half_sweeps(tuner, pairs, scounts):
    ctx = Recorder(256, pairs, scounts)
    tuner.autotune_sweeps(ctx, 0.04)
    assert any(t[:2] != (0, 0) for t in ctx.sweep)


def test_the_ideal_tile_in_use_is_the_incumbent(tuner, monkeypatch):
    """No tile is faster than another: the context keeps the one it had."""
    monkeypatch.setattr(tuner, "_class_ms", lambda *a: 1.0)
    ctx = Recorder(208, pairs=0)
    chosen = tuner.autotune_ideal(ctx, 0.04)
    assert chosen[208] == (56, 8, 1.0)
    assert ctx.ideal[0] == ctx.ideal[-1] == (56, 8)
    assert len(set(ctx.ideal)) == len(ctx.ideal) // 2  # each candidate once a round
