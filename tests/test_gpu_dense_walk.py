"""The walk that queues the pairs inside the cutoff for full waves, where it
can go wrong: boxes so small that the displacement from a cluster's first atom
no longer names the nearest image (every batch takes the exact test), systems
of fewer clusters than the launch has waves, clusters with padding slots,
beta * cutoff past the erfc table's last row, and no perturbed charges. The
pair sums are FP64 on both sides from the same integer displacements: 1e-9."""
import sys

import numpy as np
import pytest

import oracle
from sponge_amd import system

pytestmark = pytest.mark.gpu

TOL = 1e-9


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


# waters before the solute, cutoff, skin, beta (None: the PME module's)
CASES = [
    (216, 8.0, 1.0, None),    # 18.6 A box: cutoff + a cluster's extent passes half of it
    (216, 9.2, 0.1, None),    # cutoff at half the box
    (343, 5.0, 0.5, 1.7),     # beta * cutoff 8.5: past the table's end
    (343, 5.0, 0.5, 0.02),    # 8 rows
    (343, 5.0, 0.5, 0.002),   # the fewest: 2 rows
    (2197, 9.0, 2.0, None),
]


@pytest.mark.parametrize("waters,cutoff,skin,beta", CASES)
def test_windows(waters, cutoff, skin, beta):
    import torch
    from sponge_amd import nb
    fs = system.fep_mixed(system.fep_system(waters, 0.35, seed=5, cutoff=cutoff, skin=skin))
    say(f"[case] waters {waters} n {fs.n} box {fs.box[0]:.3f} cutoff {cutoff} beta {beta}")
    eng = nb.NonbondedEngine(fs, refresh_interval=0)
    eng.update_neighbor_list(forced=1)
    eng.crd_to_uint()
    torch.cuda.synchronize()
    eng.nl.check()
    u = eng.uint_crd.cpu().numpy().view(np.uint32)
    pairs = oracle.nl_brute(fs, u)
    b = float(np.float32(beta if beta is not None else eng.pme.beta))
    dq_h = (fs.charge_B.astype(np.float64) - fs.charge_A.astype(np.float64)).astype(np.float32)
    lams = [0.0, 0.35, 1.0]
    lam0 = float(np.float32(fs.lam))
    for dq in (dq_h, None):
        got = eng.lj.lambda_windows(eng.nl, eng.uint_crd, eng.charge,
                                    None if dq is None else torch.as_tensor(dq, device="cuda"), b, lams)
        ref = oracle.fep_windows(fs, u, pairs, b, lams, dq=dq, lambda0=lam0)
        err = np.abs(got[:, :7] - ref) / np.maximum(1.0, np.abs(ref))
        say(f"    dq {dq is not None}: worst relative error {err.max():.2e}")
        assert err.max() <= TOL, (dq is not None, np.unravel_index(err.argmax(), err.shape))


@pytest.mark.parametrize("waters,cutoff,skin", [(27, 3.5, 0.5), (216, 9.2, 0.1), (729, 7.0, 1.0)])
@pytest.mark.parametrize("soft", [False, True])
def test_energies(waters, cutoff, skin, soft):
    """Per-atom energies, totals and pair count of an energy step, and the
    same forces bit for bit as a force-only step's. Per-atom arrays are FP32
    sums of FP64 terms: 1e-6 of their size; totals 1e-9 of the terms' scale,
    for soft-core handles 2^-23 of it (their pair records are FP32, the
    oracle's FP64: half an ulp in lambda-mixed A, B and sigma^6 terms)."""
    import torch
    from sponge_amd import nb
    length = (waters * system.WATER_VOLUME) ** (1.0 / 3.0)
    if soft:
        if waters < 100:
            pytest.skip("no room for the solute")
        s = system.fep_mixed(system.fep_system(waters, 0.35, seed=5, cutoff=cutoff, skin=skin))
    else:
        s = system.water_box(waters, round(length, 3), seed=3, cutoff=cutoff, skin=skin)
    say(f"[case] energies waters {waters} n {s.n} box {s.box[0]:.3f} cutoff {cutoff} soft {soft}")
    eng = nb.NonbondedEngine(s, refresh_interval=0)
    eng.update_neighbor_list(forced=1)
    eng.force_step(0, 0, from_crd=True, overwrite=True)
    torch.cuda.synchronize()
    eng.nl.check()
    f = eng.frc.cpu().numpy()
    eng.lj.LJ_PME_Direct_Force_With_Atom_Energy_And_Virial(
        eng.nl, eng.uint_crd, eng.charge, eng.frc.zero_(), eng.pme.beta, 1, eng.atom_energy, 1, eng.atom_virial,
        eng.atom_direct)
    g = eng.frc.cpu().numpy()
    eng.lj.LJ_PME_Direct_Force_With_Atom_Energy_And_Virial(eng.nl, eng.uint_crd, eng.charge, eng.frc.zero_(),
                                                           eng.pme.beta)
    assert np.array_equal(g, eng.frc.cpu().numpy()) and np.isfinite(f).all()
    u = eng.uint_crd.cpu().numpy().view(np.uint32)
    pairs = oracle.nl_brute(s, u)
    ref = (oracle.direct_soft if soft else oracle.direct)(s, u, pairs, eng.pme.beta)
    for got, want in ((eng.atom_energy, ref["atom_energy"]), (eng.atom_virial, ref["atom_virial"]),
                      (eng.atom_direct, ref["atom_direct"])):
        got = got.cpu().numpy().astype(np.float64)
        assert np.abs(got - want).max() <= 1e-6 * np.abs(want).max()
    eng.force_step(1, 1, from_crd=True, overwrite=True)
    p = eng.energy_parts()
    scale = np.abs(ref["atom_energy"]).sum()
    assert p["pairs_in"] == ref["n_in"]
    for k, v in (("lj", ref["e_lj"]), ("direct", ref["e_direct"])):
        assert abs(p[k] - v) <= (2.0 ** -23 if soft else 1e-9) * scale, (k, p[k], v)


@pytest.mark.parametrize("waters,cutoff,skin,ntypes", [(27, 3.5, 0.5, 1), (216, 9.2, 0.1, 4), (343, 6.0, 1.0, 5),
                                                       (729, 7.0, 1.0, 8)])
def test_gradients(waters, cutoff, skin, ntypes):
    """Both gradients at the edges of the type count (4 and 8 accumulators)
    against the FP64 oracle. Table gradients are FP64 sums of FP64 terms, with
    FP32 weights F - T on the loss side: 1e-9 and 1e-6 of the sum of the
    entries' sizes; charge gradients are FP32 terms: 1e-5 of their norm."""
    import dataclasses
    import torch
    from sponge_amd import nb
    rng = np.random.default_rng(ntypes)
    length = (waters * system.WATER_VOLUME) ** (1.0 / 3.0)
    base = system.water_box(waters, round(length, 3), seed=3, cutoff=cutoff, skin=skin)
    A, B = system._lb_table(rng.uniform(2.0, 3.2, ntypes), rng.uniform(0.05, 0.2, ntypes))
    s = dataclasses.replace(base, lj_type=rng.integers(0, ntypes, base.n).astype(np.int32), lj_A=A, lj_B=B)
    say(f"[case] gradients waters {waters} n {s.n} cutoff {cutoff} types {ntypes}")
    eng = nb.NonbondedEngine(s, refresh_interval=0)
    eng.update_neighbor_list(forced=1)
    eng.force_step(0, 0, from_crd=True, overwrite=True)
    P = len(A)
    gq, gA, gB = (torch.zeros(k, dtype=torch.float64, device="cuda") for k in (s.n, P, P))
    loss = torch.zeros(1, dtype=torch.float64, device="cuda")
    target = torch.as_tensor(rng.normal(0.0, 5.0, (s.n, 3)).astype(np.float32), device="cuda")
    u = eng.uint_crd.cpu().numpy().view(np.uint32)
    pairs = oracle.nl_brute(s, u)
    K = (eng.pme.fftx, eng.pme.ffty, eng.pme.fftz)
    eng.energy_gradient(gq, gA, gB)
    e = oracle.energy_grad(s, u, pairs, eng.pme.beta, K)
    got = [t.cpu().numpy().copy() for t in (gq, gA, gB)]
    eng.force_matching_gradient(eng.frc, target, loss, gq, gA, gB)
    f = oracle.loss_grad(s, u, pairs, eng.pme.beta, K, eng.frc.cpu().numpy().astype(np.float64),
                         target.cpu().numpy().astype(np.float64))
    more = [t.cpu().numpy().copy() for t in (gq, gA, gB)]
    for name, g, ref, tol in (("energy", got, e, (1e-9, 2.0 ** -23)), ("loss", more, f[1:], (1e-6, 1e-6))):
        err = np.linalg.norm(g[0] - ref[0]) / np.linalg.norm(ref[0])
        say(f"    {name}: charges {err:.2e}")
        assert err <= 1e-5, name
        for k in (1, 2):
            d = np.abs(g[k] - ref[k]).max() / np.abs(ref[k]).sum()
            say(f"    {name}: table {k} {d:.2e}")
            assert d <= tol[k - 1], (name, k)


@pytest.mark.parametrize("waters,cutoff,skin", [(1, 0.9, 0.1), (27, 3.5, 0.5), (216, 9.2, 0.1), (700, 4.0, 0.3),
                                                (1500, 12.0, 2.0)])
def test_list(waters, cutoff, skin):
    """The rebuild's z tables, runs and exclusion marks: the listed pairs are
    the oracle's, bit for bit, with a second rebuild after every atom moved
    across the faces of the box."""
    import torch
    from sponge_amd import nb
    length = (waters * system.WATER_VOLUME) ** (1.0 / 3.0)
    s = system.water_box(waters, round(length, 3), seed=waters, cutoff=cutoff, skin=skin, fft=(20, 20, 20))
    say(f"[case] list waters {waters} box {s.box[0]:.3f} list radius {cutoff + skin}")
    eng = nb.NonbondedEngine(s, refresh_interval=0)
    x0 = eng.crd.clone()
    for shift in (0.0, 0.37):
        x = torch.remainder(x0 + shift * float(s.box[0]), float(s.box[0]))
        eng.crd.copy_(torch.where(x >= float(s.box[0]), torch.zeros_like(x), x))
        eng.update_neighbor_list(forced=1)
        eng.crd_to_uint()
        torch.cuda.synchronize()
        eng.nl.check()
        u = eng.uint_crd.cpu().numpy().view(np.uint32)
        got, ref = eng.nl.pairs(), oracle.nl_brute(s, u)
        say(f"    {len(got)} pairs, status {eng.nl.status()['pairs']}")
        assert np.array_equal(got, ref)
        assert eng.nl.status()["pairs"] == len(ref)
