"""How many FP32 terms the force on one atom is added up from before it goes to the 64-bit
accumulator: an atom alone in the last block of 64, with 8,192 others all on one side of it,
so that its terms add up and do not cancel.

Every term is exact but for some FP32 roundings of its own (charges whose product with
sqrt(k_e) is an FP32 number, coordinates that are FP32 numbers, no box, no reaction field, no
Lennard-Jones energy); these are independent from term to term, 3e-7 / sqrt(8192) < 4e-9 of
the sum, and 2e-8 for a reciprocal square root that is off to one side by a sixth of a last
place.  A chain of n additions of like terms is off by rms 0.29 2^-23.5 sqrt(n / 3) (uniform
errors of half a last place of sums that grow evenly): 1.2e-7 for chains of 72, of
which the eight lanes of an atom make eight in each of at least 4,096 / 576 sums: 1.6e-8 of the
half of the force that comes from the atom's own tiles, 8e-9 of the force (and less for
shorter chains).  Added up: below 3e-8 rms.  Chains of 512 (sums over 4,096 pairs) are off by
6e-8."""
import numpy as np
import pytest

from openmm_sdm_plugin_amd import _native, systems

pytestmark = pytest.mark.gpu

K_E = 138.935456


def _system(seed, blocks=128):
    rng = np.random.default_rng([17, seed])
    n = 64 * blocks + 1
    x = np.float32(rng.uniform(0.0, 2.0, (n, 3))).astype(np.float64)
    # in the upper half of the sort grid along x, which the curve takes last
    x[-1] = [5.0, 1.0, 1.0]
    q = np.full(n, 0.25)
    q[-1] = 1.0
    z, e2 = np.zeros(n), np.zeros((0, 2), dtype=np.int32)
    s = systems.SDMSystem(
        box=np.full(3, 100.0), cutoff=40.0, eps_rf=1.0, charge=q / np.sqrt(K_E), sigma=z, epsilon=z,
        mass=np.full(n, 16.0), exclusions=e2, bonds=e2, bond_r0=z[:0], bond_k=z[:0],
        angles=np.zeros((0, 3), dtype=np.int32), angle_t0=z[:0], angle_k=z[:0],
        displacement=np.zeros((n, 3)), positions=x, velocities=np.zeros((n, 3)),
        ligand=np.zeros(0, dtype=np.int32), name="one side")
    s.periodic = False
    d = x[-1] - x[:-1]
    r = np.sqrt((d * d).sum(1))
    return s, (q[:-1, None] * d / r[:, None] ** 3).sum(0)


@pytest.mark.parametrize("split", [1, 4])
def test_force_of_many_like_terms(hip_device, split):
    err = []
    for seed in range(12):
        s, want = _system(seed)
        ctx = _native.NativeContext(s, 1)
        ctx.set_tuning(cell_cells_per_dim=16, pair_split=split)
        ctx.set_params(0, systems.params_config1())
        ctx.set_positions(0, s.positions)
        ctx.compute()
        got = ctx.forces(0)[-1]
        err.append((got[0] - want[0]) / want[0])
        assert ctx.energies()[0]["flags"] == 0
    rms = float(np.sqrt(np.mean(np.square(err))))
    print(f"case split={split} rms={rms:.2e} mean={np.mean(err):.2e}", flush=True)
    assert rms <= 3e-8
