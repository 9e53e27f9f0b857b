"""What the autotuner times: every configuration once, by what it runs as and not by its
setting, and steps only, without the capture of the graphs that replay them.

The times themselves are not compared with bounds: the first test looks at which of the
settings that are one configuration is reported, the second at whether replay from graphs,
a few percent faster than launches for this system, is ever found to be."""
import pytest

from openmm_sdm_plugin_amd import _native, systems

pytestmark = pytest.mark.gpu


def _context(s, replicas):
    ctx = _native.NativeContext(s, replicas)
    for r in range(replicas):
        p = systems.params_config1()
        p.seed = r + 1
        ctx.set_params(r, p)
        ctx.set_positions(r, s.positions)
        ctx.set_velocities(r, s.velocities)
    return ctx


@pytest.mark.parametrize("waters,box,replicas", [(60, 1.9, 1), (60, 1.9, 8), (400, 3.0, 1), (400, 3.0, 2)])
def test_one_setting_for_each_configuration(hip_device, waters, box, replicas):
    """Up to 32 blocks every pair_split but 1 gives the same parts, and without restraints and
    force-field terms every side_fork the same step: the first of each is reported."""
    s = systems.make_small(waters, 6, box=box, frame=1)
    ctx = _context(s, replicas)
    print(f"case n={s.n} replicas={replicas}", flush=True)
    for _ in range(2):
        t = ctx.autotune(8)
        assert t["pair_split"] in (1, 2) and t["side_fork"] == 1
        assert ctx.get_tuning() == t


def test_graphs_are_not_timed_with_their_capture(hip_device):
    s = systems.make_config1(frame=0)
    picks = []
    for k in range(6):
        picks.append(_context(s, 1).autotune(20)["use_graph"])
        print(f"case autotune {k}: use_graph={picks[-1]}", flush=True)
    assert any(picks)
