"""Transforms of the reciprocal sum on axes of every radix (2, 3, 4, 5, 7, 8 and
their mixes) and on lines long enough that a wave takes one at a time (over 64
butterflies of a pass), in each form of the convolution, against the FP64
oracle: forces within the reciprocal force contract (relative RMS 1e-5),
energy within 1e-6."""
import sys

import numpy as np
import pytest

import oracle
from sponge_amd import system

pytestmark = pytest.mark.gpu

GRIDS = [
    (20, 20, 20),      # 4 x 5
    (25, 49, 27),      # odd radices alone, odd z
    (35, 21, 14),
    (4, 8, 6),         # one pass, fewer points than lanes
    (64, 40, 45),
    (10, 500, 8),      # 4 x 5 x 5 x 5: 125 and 100 butterflies
    (375, 9, 10),      # 3 x 5 x 5 x 5: 125 and 75
    (9, 12, 500),
]


@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "x".join(map(str, g)))
def test_reciprocal_of_every_radix(grid):
    import torch
    from sponge_amd import nb
    s = system.small_random(200, (12.0, 13.0, 14.0), seed=11, cutoff=4.5, skin=1.0, fft=grid)
    eng = nb.NonbondedEngine(s, refresh_interval=20)
    eng.crd_to_uint()
    torch.cuda.synchronize()
    u = eng.uint_crd.cpu().numpy().view(np.uint32)
    ref = oracle.pme_reciprocal(s, u, grid, float(np.float32(eng.pme.beta)))
    lib = nb.load_library()
    for form in (0, 1, 2):
        if lib.sponge_pme_set_tuning(eng.pme.h, -1, form) != 0:
            continue            # the form's lines do not fit the LDS
        print(f"[case] grid {grid} form {form}", flush=True)
        sys.stdout.flush()
        frc = torch.zeros(s.n, 3, device="cuda")
        eng.pme.PME_Reciprocal_Force_With_Energy_And_Virial(eng.uint_crd, eng.charge, frc, 0, 0)
        torch.cuda.synchronize()
        f = frc.cpu().numpy().astype(np.float64)
        err = float(np.sqrt(((f - ref["frc"]) ** 2).sum() / (ref["frc"] ** 2).sum()))
        e = eng.pme.Get_Energy(eng.uint_crd, eng.charge, None, eng.scaler, eng.excl_start, eng.excl_list,
                               eng.excl_numbers, which_part=eng.pme.RECIPROCAL)
        print(f"    force {err:.2e} energy {abs(e / ref['e_rec'] - 1):.2e}", flush=True)
        assert err < 1e-5, form
        assert abs(e - ref["e_rec"]) < 1e-6 * abs(ref["e_rec"]), form
