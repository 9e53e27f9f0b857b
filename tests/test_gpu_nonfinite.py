"""Atoms at coordinates that are not finite, or beyond the range of FP32, as a replica that
blows up leaves them: the slot order stays an order of all atoms (the order along the curve
and the one within a block of 64, empty slots last), so the pairs of all other atoms are
computed as without them and nothing is read or written out of range.  Systems of fewer
atoms than a block, and of some blocks with a last one that is partly empty or full.

The reference is the FP64 oracle for the same system in which the lost molecules are without
charge and Lennard-Jones energy: their pairs are at no distance below the cutoff.  Tolerance:
FP32 pair arithmetic, 2e-5 of the RMS force (as for the pair kernel's edges)."""
import numpy as np
import pytest
import torch

from openmm_sdm_plugin_amd import _native, systems
from oracle import oracle as O

pytestmark = pytest.mark.gpu

KINDS = {"nan": [np.nan] * 3, "one nan": [0.3, np.nan, 0.1], "inf": [np.inf] * 3,
         "mixed": [np.inf, -np.inf, np.nan], "beyond fp32": [1e39, 0.2, -1e39]}


def _molecules(s):
    """Waters (O, H, H) of the system."""
    lig = set(int(a) for a in s.ligand)
    return [(o, h1, h2) for h1, o, h2 in np.asarray(s.angles).reshape(-1, 3).tolist()
            if o not in lig]


def _system(waters, ligand, periodic):
    s = systems.make_small(waters, ligand, frame=waters)
    s.periodic = periodic
    return s


def _lost(s, which, value):
    x = np.array(s.positions)
    mols = _molecules(s)
    atoms = [a for m in which for a in mols[m % len(mols)]]
    x[atoms] = value
    return x, sorted(set(atoms))


def _context(s, x, replicas=1):
    ctx = _native.NativeContext(s, replicas)
    for r in range(replicas):
        p = systems.params_config1()
        p.seed = 3 + r
        ctx.set_params(r, p)
        ctx.set_velocities(r, s.velocities)
    t = torch.tensor(x, dtype=torch.float64, device="cuda").contiguous()
    torch.cuda.synchronize()
    ctx.set_positions_device(t.data_ptr())
    return ctx


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("waters,ligand", [(2, 3), (19, 6), (20, 4), (41, 6), (62, 6)])
def test_other_atoms_keep_their_pairs(hip_device, waters, ligand, kind, periodic):
    s = _system(waters, ligand, periodic)
    x, atoms = _lost(s, [0, waters // 2, waters - 1] if waters > 3 else [0], KINDS[kind])
    print(f"case n={s.n} {kind} periodic={periodic}", flush=True)
    q = _system(waters, ligand, periodic)
    q.charge, q.epsilon = np.array(q.charge), np.array(q.epsilon)
    q.charge[atoms] = 0.0
    q.epsilon[atoms] = 0.0
    _, u, F0, _, _, _ = O.sdm_direct(O.Topology(q), s.positions)
    ctx = _context(s, x[None])
    ctx.compute_components()
    keep = np.setdiff1d(np.arange(s.n), atoms)
    got = ctx.forces(0, _native.FORCE_STATE1)[keep]
    rms = np.sqrt(np.mean(F0[keep] ** 2)) + 1e-12
    assert np.sqrt(np.mean((got - F0[keep]) ** 2)) <= 2e-5 * rms
    assert abs(ctx.energies()[0]["u"] - u) <= 1e-9 * max(1.0, abs(u))


@pytest.mark.parametrize("kind", ["nan", "mixed", "beyond fp32"])
@pytest.mark.parametrize("waters", [41, 62])
def test_steps_of_a_batch_with_a_lost_molecule(hip_device, waters, kind):
    """Runs of steps with a molecule lost in one replica: the other replica takes the steps it
    takes beside a sound one, bit by bit, the lost one's other molecules stay finite, and sound
    coordinates set afterwards are evaluated as in a new context."""
    s = _system(waters, 6, True)
    x, atoms = _lost(s, [1], KINDS[kind])
    print(f"case n={s.n} {kind}", flush=True)
    a = _context(s, np.stack([x, s.positions]), 2)
    b = _context(s, np.stack([s.positions, s.positions]), 2)
    for n in (1, 9, 25):
        a.step(n)
        b.step(n)
        assert np.array_equal(a.get_positions(1), b.get_positions(1))
        assert np.array_equal(a.get_velocities(1), b.get_velocities(1))
    keep = np.setdiff1d(np.arange(s.n), atoms)
    assert np.all(np.isfinite(a.get_positions(0)[keep]))
    for r in range(2):
        a.set_positions(r, s.positions)
        b.set_positions(r, s.positions)
    a.compute()
    b.compute()
    assert all(np.array_equal(a.forces(r), b.forces(r)) for r in range(2))
