"""Steps replayed from graphs, several at a time, against the same steps launched one kernel
after the other: the kernels and their order are the same, so every bit is."""
import numpy as np
import pytest

from openmm_sdm_plugin_amd import _native, systems

pytestmark = pytest.mark.gpu


def _run(s, use_graph, interval, every, calls):
    ctx = _native.NativeContext(s, 2)
    ctx.set_tuning(use_graph=use_graph, sort_interval=interval, energy_every_step=every)
    for r in range(2):
        p = systems.params_config1()
        p.seed = 5 + r
        ctx.set_params(r, p)
        ctx.set_positions(r, s.positions)
        ctx.set_velocities(r, s.velocities)
    out = []
    for n in calls:  # the context's own evaluations and waits lie between the replays
        ctx.step(n)
        out.append((ctx.get_positions(0), ctx.get_velocities(1), ctx.energies()))
        ctx.compute()
        out.append((ctx.forces(1), ctx.energies()))
    return out


@pytest.mark.parametrize("interval,every", [(1, 0), (7, 0), (9, 1), (50, 0)])
def test_runs_of_steps_are_the_same_bits(hip_device, interval, every):
    s = systems.make_small(60, 6, frame=1)
    calls = (1, 8, 9, 10, 33, 3)
    print(f"case interval={interval} every={every}", flush=True)
    for a, b in zip(_run(s, 1, interval, every, calls), _run(s, 0, interval, every, calls)):
        assert all(np.array_equal(x, y) for x, y in zip(a[:-1], b[:-1]))
        assert a[-1] == b[-1]
