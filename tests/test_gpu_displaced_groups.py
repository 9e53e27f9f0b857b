"""The displaced-state pairs at the edges of their split: displaced atoms by groups of eight
and blocks of 64, more candidate blocks than have waves of their own, atoms of the block
excluded from displaced ones; against the FP64 oracle, and the same bits from a batch so
large that a wave takes all groups of a block.

Tolerance: FP64 sums of a few thousand terms in another order than the oracle's, 1e-10 of
the largest summed magnitudes (taken as 1e3 times the result's scale at most)."""
import numpy as np
import pytest

from openmm_sdm_plugin_amd import _native, systems
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _run(s, replicas):
    ctx = _native.NativeContext(s, replicas)
    for r in range(replicas):
        ctx.set_params(r, systems.params_config1())
        ctx.set_positions(r, s.positions)
    ctx.compute_components()
    e = ctx.energies()
    F = [ctx.forces(r, _native.FORCE_STATE1) for r in (0, replicas - 1)]
    dF = [ctx.forces(r, _native.FORCE_STATE2) - F[k] for k, r in enumerate((0, replicas - 1))]
    return ctx, e, dF, F


@pytest.mark.parametrize("displaced", [1, 7, 8, 9, 63, 64, 65, 131])
def test_groups_and_batches(hip_device, displaced):
    s = systems.make_small(60, 7, frame=displaced)
    # the first atoms move: part of the chain, or waters too, the last one in part
    d = s.displacement[0].copy()
    s.displacement[:] = 0.0
    s.displacement[:displaced] = d
    print(f"case n={s.n} displaced={displaced}", flush=True)
    _, u, _, dF, _, nd = O.sdm_direct(O.Topology(s), s.positions)
    ctx, e, got, F = _run(s, 1)
    assert e[0]["flags"] == 0
    assert abs(e[0]["u"] - u) <= 1e-10 * max(1e3, 1e3 * abs(u))
    # forces are read back as differences of two FP64 sums with fixed-point parts (2^-32)
    assert np.max(np.abs(got[0] - dF)) <= 1e-9 * (1.0 + np.max(np.abs(dF))) + 4 * 2.0 ** -32
    assert int(ctx.count_pairs()[1][0]) == nd
    nb = (s.n + 63) // 64
    _, eb, gb, Fb = _run(s, 25000 // (64 * nb) + 1)
    for k in ("u", "U0", "Ub", "pot_energy"):
        assert eb[0][k] == eb[-1][k]
    assert np.array_equal(Fb[0], F[0]) and np.array_equal(Fb[1], F[0])
    assert eb[0]["u"] == e[0]["u"] and np.array_equal(gb[0], got[0]) and np.array_equal(gb[1], got[0])


def test_more_candidate_blocks_than_waves(hip_device):
    s = systems.make_small(1400, 12, box=4.2, cutoff=0.9, frame=1)
    s.cutoff, s.periodic = 15.0, False  # every block is a candidate
    print(f"case n={s.n}", flush=True)
    _, u, _, dF, _, nd = O.sdm_direct(O.Topology(s), s.positions)
    ctx, e, got, _ = _run(s, 1)
    assert e[0]["flags"] == 0
    assert abs(e[0]["u"] - u) <= 1e-10 * max(1e3, 1e3 * abs(u))
    assert np.max(np.abs(got[0] - dF)) <= 1e-9 * (1.0 + np.max(np.abs(dF))) + 4 * 2.0 ** -32
    assert int(ctx.count_pairs()[1][0]) == nd
