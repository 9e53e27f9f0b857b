"""The adjoint kernels at the edges of their tiles: selections of 1 to 130 atoms, displaced
and undisplaced, one displaced class and two; u and du/d(q, sigma, eps) against the FP64
oracle.  All arithmetic is FP64, so the tolerances are those of sums of a few thousand terms
that partly cancel: 1e-10 of u, 1e-9 of the largest gradient."""
import math

import numpy as np
import pytest
import torch

from openmm_sdm_plugin_amd import _native, systems
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsel", [1, 16, 17, 32, 33, 64, 65, 130])
@pytest.mark.parametrize("two_guests", [False, True])
def test_selection_tiles_match_oracle(hip_device, nsel, two_guests):
    """Selections at the edges of the gradient kernel's 16, 32 and 64 lanes, of displaced and
    undisplaced atoms mixed, with one displaced class or two (the second one 70 of the
    waters, so that a class has more than 64 atoms), more than 256 atoms."""
    s = systems.make_small(100, 7, box=2.3, frame=nsel)
    s.displacement = s.displacement.copy()
    if two_guests:
        s.displacement[7:7 + 210] = (0.0, -0.7, 0.4)
    rng = np.random.default_rng(nsel)
    sel = np.concatenate([s.ligand, rng.permutation(np.arange(7, s.n))])[:nsel]
    sel = rng.permutation(sel).astype(np.int32)
    print(f"case adjoint tiles n={s.n} nsel={nsel} two_guests={two_guests}", flush=True)
    ctx = _native.NativeContext(s, 1)
    X = torch.tensor(np.stack([s.positions, s.positions + 0.013]), device="cuda")
    grad = torch.full((2, nsel, 3), float("nan"), dtype=torch.float64, device="cuda")
    u = torch.full((2,), float("nan"), dtype=torch.float64, device="cuda")
    ctx.du_dparams_frames(X.data_ptr(), 2, sel, grad.data_ptr(), u.data_ptr())
    topo = O.Topology(s)
    for f, x in enumerate((s.positions, s.positions + 0.013)):
        _, uref, *_ = O.sdm_direct(topo, x)
        assert math.isclose(float(u[f]), uref, rel_tol=1e-10, abs_tol=1e-8)
        ref = np.stack(O.du_dparams(topo, x, sel), 1)
        assert np.allclose(grad[f].cpu().numpy(), ref, rtol=1e-9, atol=1e-9 * np.max(np.abs(ref)))
