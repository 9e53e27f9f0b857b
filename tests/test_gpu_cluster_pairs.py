"""The pair, energy and tile kernels at the edges of their 64-atom blocks and 8-atom clusters
(fewer atoms than a cluster, one more or less than a block or two), with every number of
waves per block, where each pair takes its own minimum image (box of about two cutoffs),
without periodic images, and with the geometric sigma rule; against the FP64 oracle.

Tolerances: U0 is an FP64 sum (1e-10 of the summed magnitudes' scale, as pair energies of
opposite sign cancel); forces are FP32 pair arithmetic on coordinates rounded to 1.2e-7 nm at most:
|dF/F| <= 13 * 1.2e-7 / 0.1 nm for the steepest term of the closest pairs, plus a few FP32
roundings, so 2e-5 of the RMS force; the pair count is exact except for pairs whose distance
is within FP32 rounding of the cutoff."""
import numpy as np
import pytest

from openmm_sdm_plugin_amd import _native, systems
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _check(s, tuning):
    topo = O.Topology(s)
    U0, u, F0, dF, n0, nd = O.sdm_direct(topo, s.positions)
    ctx = _native.NativeContext(s, 1)
    ctx.set_tuning(**tuning)
    p = systems.params_config1()
    ctx.set_params(0, p)
    # the atoms of a molecule stay whole, some of them outside the box
    ctx.set_positions(0, s.positions)
    ctx.compute_components()
    e = ctx.energies()[0]
    assert e["flags"] == 0
    assert abs(e["U0"] - U0) <= 1e-10 * max(1.0, abs(U0), 100.0 * s.n)
    assert abs(e["u"] - u) <= 1e-9 * max(1.0, abs(u))
    got = ctx.forces(0, _native.FORCE_STATE1)
    rms = np.sqrt(np.mean(F0 ** 2)) + 1e-12
    assert np.sqrt(np.mean((got - F0) ** 2)) <= 2e-5 * rms
    p0, pd = ctx.count_pairs()
    assert abs(int(p0[0]) - n0) <= 1 and int(pd[0]) == nd


@pytest.mark.parametrize("split", [1, 2, 32])
@pytest.mark.parametrize("waters,ligand", [(1, 2), (1, 4), (2, 2), (19, 6), (20, 4), (20, 5),
                                           (40, 7), (40, 8), (41, 6), (63, 6)])
def test_block_and_cluster_edges(hip_device, waters, ligand, split):
    s = systems.make_small(waters, ligand, frame=waters)
    print(f"case n={s.n} split={split}", flush=True)
    _check(s, dict(pair_split=split))


@pytest.mark.parametrize("cells", [1, 3, 9])
@pytest.mark.parametrize("geometric", [0, 1])
@pytest.mark.parametrize("cutoff,periodic", [(0.94, True), (0.5, True), (15.0, False)])
def test_image_modes(hip_device, cutoff, periodic, geometric, cells):
    s = systems.make_small(61, 5, cutoff=0.8, frame=3)
    s.cutoff, s.periodic, s.lj_rule = cutoff, periodic, geometric
    print(f"case n={s.n} cutoff={cutoff} periodic={periodic} geo={geometric} cells={cells}", flush=True)
    # a coarse sort grid gives blocks as wide as the box
    _check(s, dict(cell_cells_per_dim=cells, pair_split=2))


@pytest.mark.parametrize("skin", [0.0, 0.02])
@pytest.mark.parametrize("waters,box", [(60, 1.9), (700, 3.3), (11000, 7.0)])
def test_parts_take_every_pair_once(hip_device, waters, box, skin):
    """However the tiles of a block are shared out, also in parts of falling size (from 512
    blocks on): the same pairs, the same energy to FP64 rounding, and forces that differ by
    FP32 sums in another order (some hundred terms, 1e-6 of the RMS force)."""
    s = systems.make_small(waters, 6, box=box, cutoff=0.8, frame=2)
    ref = None
    for split in (1, 2, 16, 32):
        print(f"case n={s.n} split={split} skin={skin}", flush=True)
        ctx = _native.NativeContext(s, 1)
        ctx.set_tuning(pair_split=split, list_skin=skin)
        ctx.set_params(0, systems.params_config1())
        ctx.set_positions(0, s.positions)
        ctx.compute_components()
        got = (int(ctx.count_pairs()[0][0]), ctx.energies()[0]["U0"], ctx.forces(0, _native.FORCE_STATE1))
        ref = ref or got
        assert got[0] == ref[0] and abs(got[1] - ref[1]) <= 1e-12 * max(abs(ref[1]), 1e3 * s.n)
        rms = np.sqrt(np.mean(ref[2] ** 2))
        assert np.sqrt(np.mean((got[2] - ref[2]) ** 2)) <= 1e-6 * rms


@pytest.mark.parametrize("cells", [10, 20, 21, 33])
def test_sort_grid_sizes(hip_device, cells):
    """Sort grids of fewer and more cells than one round of the scan (8 x 1,024) takes."""
    print(f"case cells={cells}", flush=True)
    _check(systems.make_small(40, 7, frame=5), dict(cell_cells_per_dim=cells))
