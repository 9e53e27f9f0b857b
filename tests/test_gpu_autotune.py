"""What the autotuner times: every configuration once, by what it runs as and not by its
setting.  The times are not compared; the test looks at which of the settings that are one
configuration is reported."""
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
