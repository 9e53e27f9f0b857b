"""One constrained step with clusters of every kind the constraint kernel tells apart: rigid
three-site molecules in the order that is worked on in registers and in another order, two
constraints or one of a molecule, and a chain of the largest cluster size, in counts around
the 64 clusters of a workgroup; against the oracle's Newton solution.

Tolerance: the forces are FP32 pair arithmetic (2e-5 of the RMS force, here a few 1e3
kJ/mol/nm), which moves an atom of 1 amu by at most 1e-7 nm in a step of 1 fs; SHAKE stops
1e-10 off in d^2, far below that."""
import types

import numpy as np
import pytest

from openmm_sdm_plugin_amd import _native, systems
from oracle import oracle as O
from oracle import terms as OT

pytestmark = pytest.mark.gpu


def _constraints(s, chain):
    lig = [int(a) for a in s.ligand]
    pairs = list(zip(lig[:chain - 1], lig[1:chain])) if chain else []
    first = [a for a in range(s.n) if a not in set(lig) and abs(s.mass[a] - 15.9994) < 1e-6]
    for k, o in enumerate(first):
        pairs += [[(o, o + 1), (o, o + 2), (o + 1, o + 2)], [(o, o + 2), (o, o + 1), (o + 1, o + 2)],
                  [(o, o + 1), (o, o + 2)], [(o, o + 1)]][k % 4 if chain else 0]
    return np.array(pairs, dtype=np.int32)


@pytest.mark.parametrize("waters,chain", [(63, 0), (64, 16), (65, 3), (130, 8)])
def test_constraint_clusters(hip_device, waters, chain):
    s = systems.make_small(waters, 16, frame=waters)
    print(f"case n={s.n} chain={chain}", flush=True)
    x0 = np.asarray(s.positions)
    cons = _constraints(s, chain)
    length = np.linalg.norm(x0[cons[:, 0]] - x0[cons[:, 1]], axis=1)
    none, at2, at4 = np.zeros(0), np.zeros((0, 2), int), np.zeros((0, 4), int)
    ff = types.SimpleNamespace(
        torsions=at4, torsion_n=none, torsion_phase=none, torsion_k=none, impropers=at4,
        improper_t0=none, improper_k=none, posre_fb_atoms=none, posre_fb_x0=none,
        posre_fb_hk=none, posre_fb_tol=none, posre_h_atoms=none, posre_h_x0=none,
        posre_h_hk=none, exception_pairs=at2, exception_qq=none, exception_sigma=none,
        exception_epsilon=none, constraints=cons, constraint_r=length)
    p = systems.params_config1()
    p.temperature = 0.0
    ctx = _native.NativeContext(s, 1)
    ctx.set_forcefield_terms(ff)
    ctx.set_params(0, p)
    ctx.set_positions(0, x0)
    ctx.set_velocities(0, s.velocities)
    ctx.step(1)
    topo = O.Topology(s)
    E1, E2, Eb, F1, F2, Fb = O.reference_eval(topo, x0)
    sc = O.execute_scalars(O.make_params(p), E1, E2, Eb, 0.0)
    F = (1 - sc.sp) * F1 + sc.sp * F2 + Fb
    xu, _ = O.langevin_update(x0, s.velocities, F, s.mass, p.step_size, p.friction, 0.0,
                              np.zeros_like(x0), form="cl")
    xc = OT.constrain(x0, xu, s.mass, cons, length)
    assert np.max(np.abs(ctx.get_positions(0) - xc)) < 1e-7
    assert ctx.energies()[0]["flags"] == 0
