"""Runs of eight steps in the kept order, replayed from one graph, against the same steps
launched kernel by kernel, in the forms that change a step's kernels or streams: tile lists
kept with a skin (the fused update then also keeps the displacement record that decides their
reuse), centre-of-mass removal, force-field terms and restraints on the side stream, pair
energies of every step on a stream of their own (batches of several generations of waves),
constraints and virtual sites (which have no fused update); 47 blocks of 64 atoms (4 with
virtual sites), the last one partly filled, in one replica and in batches on both sides of the
rules that choose by the number of blocks (2,048) and of waves (24,576).  The same kernels and data: the same bits."""
import numpy as np
import pytest

from openmm_sdm_plugin_amd import _native, systems
from test_gpu_restraints import _restrained
from test_gpu_terms import _terms
from vsite_cases import four_site

pytestmark = pytest.mark.gpu

CALLS = (1, 9, 10, 19)


def _context(s, replicas, **tuning):
    ctx = _native.NativeContext(s, replicas)
    ctx.set_tuning(**tuning)
    rng = np.random.default_rng(3)
    for r in range(replicas):
        p = systems.params_config1()
        p.seed = 5 + r
        ctx.set_params(r, p)
        ctx.set_positions(r, s.positions)
        v = rng.normal(size=(s.n, 3)) * np.sqrt(2.494353 / np.maximum(s.mass, 1.0))[:, None]
        ctx.set_velocities(r, np.where(np.asarray(s.mass)[:, None] > 0.0, v, 0.0))
    return ctx


def _steps(ctx, replicas):
    out = []
    for n in CALLS:  # the context's own evaluations and waits lie between the replays
        ctx.step(n)
        out += [ctx.get_positions(r) for r in (0, replicas - 1)]
        out += [ctx.get_velocities(replicas - 1), ctx.energies()]
        ctx.compute()
        out += [ctx.forces(0), ctx.energies()]
    return out


def _same(a, b):
    return all(np.array_equal(x, y) if isinstance(x, np.ndarray) else x == y for x, y in zip(a, b))


def _system(form):
    """The system and what is set on its context."""
    s = systems.make_config1(frame=1)
    if form in ("terms", "constraints"):
        ff = _terms(s, np.random.default_rng(7), constraints=form == "constraints")
        return s, lambda ctx: ctx.set_forcefield_terms(ff)
    if form == "restraints":
        s = _restrained()
        return s, lambda ctx: ctx.set_restraints(s.restraints)
    if form == "sites":
        return four_site(), lambda ctx: None
    if form == "cm":
        return s, lambda ctx: ctx.set_cm_motion_removal(3)
    return s, lambda ctx: None


@pytest.mark.parametrize("replicas", [1, 34, 44])
@pytest.mark.parametrize("form,skin,every", [
    ("plain", 0.0, 1), ("plain", 0.02, 0), ("plain", 0.1, 0), ("plain", 0.02, 1), ("cm", 0.0, 0),
    ("cm", 0.1, 0), ("terms", 0.0, 0), ("terms", 0.02, 1), ("restraints", 0.0, 0),
    ("restraints", 0.1, 1), ("constraints", 0.0, 0), ("constraints", 0.1, 0), ("sites", 0.0, 0)])
def test_replayed_and_launched_steps(hip_device, form, skin, every, replicas):
    runs = []
    for use_graph in (1, 0):
        s, extra = _system(form)
        print(f"case {form} n={s.n} replicas={replicas} skin={skin} every={every} graph={use_graph}", flush=True)
        ctx = _context(s, replicas, use_graph=use_graph, sort_interval=50, list_skin=skin,
                       energy_every_step=every)
        extra(ctx)
        runs.append(_steps(ctx, replicas))
    assert runs[0][3][0]["flags"] == 0
    assert _same(*runs)


@pytest.mark.parametrize("replicas", [1, 44])
@pytest.mark.parametrize("use_graph", [0, 1])
def test_kept_lists_take_the_same_pairs(hip_device, use_graph, replicas):
    """With one part per block the same pairs are added in the same order with and without a
    skin: a list kept for too long would leave some out."""
    s, _ = _system("plain")
    runs = []
    for skin in (0.0, 0.02, 0.1):
        print(f"case replicas={replicas} graph={use_graph} skin={skin}", flush=True)
        ctx = _context(s, replicas, use_graph=use_graph, sort_interval=50, pair_split=1, list_skin=skin)
        ctx.step(1)
        for n in (8, 17, 16):
            ctx.step(n)
        runs.append([ctx.get_positions(0), ctx.get_velocities(replicas - 1)])
    assert _same(runs[0], runs[1]) and _same(runs[0], runs[2])
