"""The numbers of parts that an i-block's tiles are shared out in (1, 4, 10, 16, 32, 64), each
at a size whose rule gives it: the same pairs as with one part per block, the same energy to
FP64 rounding, and forces that differ by FP32 sums in other groups and by their rounding to
2^-32 (some hundred terms, 1e-6 of the RMS force)."""
import numpy as np
import pytest

from openmm_sdm_plugin_amd import _native, systems

pytestmark = pytest.mark.gpu


# waters, box: blocks; pair_split: parts
@pytest.mark.parametrize("skin", [0.0, 0.05])
@pytest.mark.parametrize("waters,box,split,parts", [
    (300, 2.6, 2, 64), (400, 2.9, 4, 32), (900, 3.6, 8, 16), (900, 3.6, 32, 32),
    (6000, 5.8, 4, 10), (6000, 5.8, 16, 16), (11000, 7.0, 4, 4), (11000, 7.0, 8, 8)])
def test_parts_by_size(hip_device, waters, box, split, parts, skin):
    s = systems.make_small(waters, 7, box=box, cutoff=0.8, frame=4)
    blocks = (s.n + 63) // 64
    rule = 64 if blocks <= 16 else 32 if blocks <= 32 else 16 if blocks < 256 else 10 if blocks < 512 else 4
    assert max(split, rule) == parts
    got = []
    for n in (1, split):
        print(f"case n={s.n} blocks={blocks} split={n} skin={skin}", flush=True)
        ctx = _native.NativeContext(s, 1)
        ctx.set_tuning(pair_split=n, list_skin=skin)
        ctx.set_params(0, systems.params_config1())
        ctx.set_positions(0, s.positions)
        ctx.compute_components()
        e = ctx.energies()[0]
        assert e["flags"] == 0
        got.append((int(ctx.count_pairs()[0][0]), e["U0"], ctx.forces(0, _native.FORCE_STATE1)))
    (n1, u1, f1), (n2, u2, f2) = got
    assert n1 == n2 and abs(u1 - u2) <= 1e-12 * max(abs(u1), 1e3 * s.n)
    assert np.sqrt(np.mean((f1 - f2) ** 2)) <= 1e-6 * np.sqrt(np.mean(f1 ** 2))
