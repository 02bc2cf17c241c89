"""The work a program that uses this library has it do, as cases to be timed.

Every case is a periodic box of rigid TIP3P water (with ions, or with one
12-atom solute for the free-energy kinds) at 1.0 g/cm^3, at the sizes of
`sponge_amd.system` and between them:

md      one neighbor-list period of NVE dynamics: coordinates and velocities
        set, the list rebuilt, `steps` steps (force, leap-frog + SETTLE),
        replayed from one graph as a program that runs dynamics keeps it
batch   the same period for a batch of independent free-energy windows and
        replicas (`md.BatchedMD`)
calls   the calls of one step of SPONGE's main loop, each on its own, with
        the skin-triggered list check (a host program that keeps its loop)
print   a step that reports: forces, per-atom energies and virials, the
        energy parts on the host, the pressure
score   a structure seen for the first time: list, forces, energies
frame   one trajectory frame at `windows` lambda windows (FEP / MBAR)
ti      one trajectory frame's dH/dlambda (thermodynamic integration)
egrad   the energy and its gradient in the charges and the LJ tables
fgrad   a force-matching loss and its gradients (one training step)

`exact` evaluates the same in 64 bits with plain torch: the energy below is
differentiated by autograd where forces or gradients are asked for.
"""
import math

import numpy as np
import torch

from sponge_amd import grad, md, nb, system

GRIDS = [g for g in range(20, 110) if system.check_2357(g)]


def _grid(length):
    """The PME grid: the smallest size of at least one point per Angstrom
    (108 for the 96,120-atom box, 64 for the 23,570-atom one)."""
    return next(g for g in GRIDS if g >= length)


def _length(waters):
    return round((waters * 29.915) ** (1.0 / 3.0), 3)


def _case(kind, waters, cutoff, **more):
    length = more.pop("box", None) or _length(waters)
    return dict(kind=kind, waters=waters, cutoff=float(cutoff), box=length,
                grid=more.pop("grid", None) or _grid(length), **more)


def listed():
    return [
        # dynamics of the three benchmark boxes: latency, the ordinary size, the largest
        dict(_case("md", 216, 8, box=18.64, grid=20, ions=0, steps=20), name="md_648"),
        dict(_case("md", 7850, 10, box=61.9, grid=64, ions=10, steps=20), name="md_23570"),
        dict(_case("md", 32000, 10, box=98.6, grid=108, ions=60, steps=20), name="md_96120"),
        # 16 lambda windows and 5 uneven replicas, as the benchmark's batch
        dict(_case("batch", 1000, 9, windows=16, replicas=5, steps=20), name="batch_21"),
        # a host program's own loop over a small box: launches and latency
        dict(_case("calls", 216, 8, box=18.64, grid=20, ions=0), name="calls_648"),
        # a reporting step, and a new structure of an odd size
        dict(_case("print", 7850, 10, box=61.9, grid=64, ions=10), name="print_23570"),
        dict(_case("score", 3333, 10, ions=7), name="score_10013"),
        # post-processing of a trajectory frame
        dict(_case("frame", 7850, 9, grid=64, windows=16), name="frame_23496"),
        dict(_case("ti", 1500, 9), name="ti_4446"),
        # fitting charges and LJ tables
        dict(_case("egrad", 7850, 10, box=61.9, grid=64, ions=10), name="egrad_23570"),
        dict(_case("fgrad", 1000, 10, ions=3), name="fgrad_3006"),
        dict(_case("egrad", 32000, 10, box=98.6, grid=108, ions=60), name="egrad_96120"),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["md", "md", "md", "batch", "calls", "print", "score", "frame", "ti", "egrad", "fgrad"])
    hi = {"md": 24000, "batch": 1000, "calls": 20000, "print": 30000, "score": 30000, "frame": 8000, "ti": 8000,
          "egrad": 20000, "fgrad": 8000}[kind]
    waters = log(400 if kind in ("frame", "ti", "batch") else 216, hi)
    cutoff = 8.0 if waters < 700 else rng.choice([8.0, 9.0, 10.0] if waters > 1100 else [8.0, 9.0])
    if kind in ("frame", "ti"):
        more = dict(windows=rng.randint(2, 24)) if kind == "frame" else {}
    elif kind == "batch":
        more = dict(windows=rng.randint(2, 16), replicas=rng.randint(0, 4), steps=rng.randint(10, 20))
    else:
        more = dict(ions=rng.randint(0, max(1, waters // 500)))
        if kind == "md":
            more["steps"] = rng.randint(10, 25)
    return _case(kind, waters, cutoff, **more)


# --------------------------------------------------------------------------
# inputs


def _box_system(c, seed):
    return system.water_box(c["waters"], c["box"], c["ions"], c["ions"], seed=int(seed) % (1 << 31),
                            cutoff=c["cutoff"], skin=2.0, fft=(c["grid"],) * 3)


def _fep_system(c, seed, lam, waters=None):
    fs = system.fep_system(waters or c["waters"], lam, seed=int(seed) % (1 << 31), cutoff=c["cutoff"], skin=2.0)
    g = c["grid"] if waters in (None, c["waters"]) else _grid(float(fs.box[0]))
    fs.fft = (g, g, g)
    return fs


def _batch_systems(c, seed):
    """Windows of one solute at evenly spaced lambdas, and replicas of 1/2, 1,
    3/2, ... times the windows' size (the benchmark's 1,500, 3,000, ... atoms
    for 1,000 waters) at other lambdas. The molecules are the same ones for
    every seed (so are the atom counts), placed anew: turned and shifted."""
    rng = np.random.default_rng(int(seed))
    out = [_fep_system(c, 11, k / max(1, c["windows"] - 1)) for k in range(c["windows"])]
    for r in range(c["replicas"]):
        out.append(_fep_system(c, 12 + r, (0.37 * (r + 1)) % 1.0, max(400, c["waters"] * (r + 1) // 2)))
    for s in out:
        x = s.crd[:, rng.permutation(3)].astype(np.float64) + rng.uniform(0.0, 1.0, 3) * s.box
        s.crd = np.mod(x, s.box.astype(np.float64)).astype(np.float32)
        s.crd[s.crd >= s.box] = 0.0
    return out


def _velocities(s, seed):
    return system.rigid_velocities(s, 300.0, (int(seed) + 5) % (1 << 31)).astype(np.float32)


def _target(n, seed):
    """Reference forces to fit to: normal, 10 kcal/mol/A a component."""
    return np.random.default_rng(int(seed)).normal(0.0, 10.0, (n, 3)).astype(np.float32)


def _dev(a, dt=torch.float32):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device="cuda")


class State:
    pass


def prepare(case, seed):
    c, st = case, State()
    st.case = c
    kind = c["kind"]
    if kind in ("md", "batch"):
        systems = [_box_system(c, seed)] if kind == "md" else _batch_systems(c, seed)
        st.engines = [md.MDEngine(s, vel=_velocities(s, seed + k), refresh_interval=20) for k, s in
                      enumerate(systems)]
        one = md.BatchedMD(st.engines) if kind == "batch" else st.engines[0]
        st.start = [e.crd.clone() for e in st.engines] + [e.vel.clone() for e in st.engines]
        now = [e.crd for e in st.engines] + [e.vel for e in st.engines]
        st.out = (now, [e.nb.frc for e in st.engines])
        st.owner = one
        one.prepare()
        one.step(forced_update=0)      # eager: sizes what a first step sizes
        torch.cuda.synchronize()
        st.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st.graph):
            s = torch.cuda.current_stream()
            torch._foreach_copy_(now, st.start)
            if kind == "md":
                one.nb.update_neighbor_list(forced=1, stream=s)
            else:
                one.batch.neighbor_list_update(forced=1, stream=s)
            for _ in range(c["steps"]):
                one.step(forced_update=0, stream=s)
        return st
    if kind in ("frame", "ti"):
        fs = _fep_system(c, seed, 0.5)
        st.eng = nb.NonbondedEngine(fs, refresh_interval=0)
        st.frame = st.eng.crd.clone()
        st.dq = _dev(fs.charge_B.astype(np.float64) - fs.charge_A.astype(np.float64))
        st.lams = np.linspace(0.0, 1.0, c.get("windows", 2))
        return st
    s = _box_system(c, seed)
    if kind == "print":
        st.md = md.MDEngine(s, vel=_velocities(s, seed), refresh_interval=20)
        st.md.prepare()
        return st
    st.eng = nb.NonbondedEngine(s, refresh_interval=0)
    st.eng.update_neighbor_list(forced=1)
    st.eng.crd_to_uint()
    if kind in ("calls", "score"):
        st.structure = st.eng.crd.clone()
    if kind in ("egrad", "fgrad"):
        st.q, st.A, st.B = st.eng.charge.clone(), torch.tensor(s.lj_A), torch.tensor(s.lj_B)
        st.target = _dev(_target(s.n, seed))
    return st


# --------------------------------------------------------------------------
# one pass


def run(st):
    kind = st.case["kind"]
    if kind in ("md", "batch"):
        st.graph.replay()
        return st.out
    if kind == "calls":
        e = st.eng
        e.frc.zero_()
        nb.crd_to_uint(e.crd, e.box, e.uint_crd)
        e.lj.LJ_PME_Direct_Force_With_Atom_Energy_And_Virial(e.nl, e.uint_crd, e.charge, e.frc, e.pme.beta)
        e.pme.PME_Excluded_Force_With_Atom_Energy(e.uint_crd, e.scaler, e.charge, e.excl_start, e.excl_list,
                                                  e.excl_numbers, e.frc)
        e.pme.PME_Reciprocal_Force_With_Energy_And_Virial(e.uint_crd, e.charge, e.frc)
        e.update_neighbor_list()
        return e.frc
    if kind == "print":
        m = st.md
        e = m.nb
        e.atom_energy.zero_()
        e.atom_virial.zero_()
        m.force(need_energy=1, need_virial=1)
        m.calculate_pressure()
        return e.frc, e.atom_energy, e.atom_virial, e.energy_parts(), m.pressure, m.ek
    if kind == "score":
        e = st.eng
        e.crd.copy_(st.structure)
        e.atom_energy.zero_()
        e.atom_virial.zero_()
        e.update_neighbor_list(forced=1)
        e.force_step(need_energy=1, need_virial=1, from_crd=True, overwrite=True)
        return e.frc, e.atom_energy, e.atom_virial, e.energy_parts()
    if kind in ("frame", "ti"):
        e = st.eng
        e.crd.copy_(st.frame)
        e.update_neighbor_list(forced=1)
        e.crd_to_uint()
        ex = (e.excl_start, e.excl_list, e.excl_numbers)
        if kind == "frame":
            return (e.lj.lambda_windows(e.nl, e.uint_crd, e.charge, st.dq, e.pme.beta, st.lams),
                    e.pme.lambda_windows(e.uint_crd, e.charge, st.dq, e.scaler, *ex, 0.5, st.lams))
        lj = e.lj.Get_Partial_H_Partial_Lambda_With_Columb_Direct(e.uint_crd, e.charge, e.nl, st.dq, 1, e.pme.beta)
        cross = e.pme.cross_dhdl(e.nl, e.uint_crd, e.charge, st.dq, e.scaler, *ex, lj_pertubated=1)
        return lj, e.lj.h_sigma_of_dH_dlambda_direct, cross["reciprocal"], cross["self"], cross["correction"]
    q, A, B = (t.detach().requires_grad_() for t in (st.q, st.A, st.B))
    if kind == "egrad":
        value = grad.nonbonded_energy(st.eng, q, A, B)
    else:
        value = grad.force_matching_loss(st.eng, q, A, B, st.target)
    value.backward()
    return value.detach(), q.grad, A.grad, B.grad


# --------------------------------------------------------------------------
# what a pass cannot do without


def _atoms(c):
    if c["kind"] == "batch":
        sizes = [c["waters"]] * c["windows"] + [max(400, c["waters"] * (r + 1) // 2) for r in range(c["replicas"])]
        return 3 * sum(sizes), [float(_length(w)) for w in sizes]
    return 3 * c["waters"] + 2 * c.get("ions", 0), [c["box"]]


def work(case):
    """Per evaluation: coordinates, charges, types and exclusions in, forces
    out; 50 operations per pair inside the cutoff and 2 x 2.5 G log2 G for
    the transforms of G grid points. Dynamics add the coordinates and
    velocities in and out of each step; gradients two more pair passes."""
    c = case
    n, boxes = _atoms(c)
    grid = sum((c["grid"] if c["kind"] != "batch" else _grid(b)) ** 3 for b in boxes)
    pairs = n * 0.5 * 4.0 / 3.0 * math.pi * c["cutoff"] ** 3 * 3.0 / 29.915
    flops = 50.0 * pairs + 5.0 * grid * math.log2(grid)
    step = n * (12 + 4 + 4 + 12 + 12)
    kind = c["kind"]
    if kind in ("md", "batch"):
        return {"bytes": c["steps"] * (step + n * (12 + 24 + 8)), "flops": c["steps"] * flops}
    if kind in ("frame", "ti"):
        return {"bytes": n * (12 + 4 + 4 + 4 + 12), "flops": 1.5 * flops}
    if kind in ("egrad", "fgrad"):
        return {"bytes": 2 * step, "flops": 3 * flops}
    return {"bytes": step + 8 * n, "flops": flops}


def tolerance(case):
    """About four times the difference from the 64-bit result over the sizes
    above. In 20 steps of dynamics the float32 coordinates' rounding (4e-6 A
    in 60, which the constraints turn into velocities by 1/dt) leaves 1e-4 to
    2e-4; one evaluation's 32-bit forces 7e-7; the 64-bit pair sums of frames
    stand beside a 32-bit reciprocal part, and in ti alone with a cancelling
    sum of it."""
    return {"md": {"rel": 1e-3}, "batch": {"rel": 1e-3}, "calls": {"rel": 4e-6}, "print": {"rel": 4e-6},
            "score": {"rel": 4e-6}, "frame": {"rel": 1e-6}, "ti": {"rel": 2e-5}, "egrad": {"rel": 4e-6},
            "fgrad": {"rel": 4e-6}}[case["kind"]]


# --------------------------------------------------------------------------
# the same in 64 bits


def _beta(rc):
    lo, hi = 0.0, 4.0
    for _ in range(100):
        b = 0.5 * (lo + hi)
        lo, hi = (b, hi) if math.erfc(b * rc) / rc >= 1e-5 else (lo, b)
    return float(np.float32(b))


class Exact:
    """Energies of one system in 64 bits, differentiable in the coordinates,
    the charges and the LJ tables."""

    def __init__(self, s):
        d = dict(device="cuda")
        self.s, self.n, self.rc = s, s.n, float(s.cutoff)
        self.box32 = torch.tensor(s.box, dtype=torch.float32, **d)
        self.box = self.box32.double()
        self.V = float(np.prod(s.box.astype(np.float64)))
        self.beta = _beta(self.rc)
        self.q = torch.tensor(s.charge, **d).double()
        tri = lambda t: torch.tensor(np.maximum(t[:, None], t[None]) * (np.maximum(t[:, None], t[None]) + 1) // 2 +
                                     np.minimum(t[:, None], t[None]), **d)
        self.tri = tri(np.arange(64))
        self.type = torch.tensor(s.lj_type, **d).long()
        self.A, self.B = (torch.tensor(t, **d).double() for t in (s.lj_A, s.lj_B))
        self.soft = getattr(s, "lj_type_B", None) is not None
        if self.soft:
            self.typeB = torch.tensor(s.lj_type_B, **d).long()
            self.A2, self.B2 = (torch.tensor(t, **d).double() for t in (s.lj_A_B, s.lj_B_B))
            self.mask = torch.tensor(s.mask, **d)
        i = np.repeat(np.arange(s.n), s.excl_numbers)
        self.ei, self.ej = torch.tensor(i, **d), torch.tensor(s.excl_list[:len(i)], **d).long()
        K = [int(k) for k in s.fft]
        self.K = K
        B1 = []
        for k in K:      # |b(m)|^2 of the order-4 exponential spline
            m = torch.arange(k, dtype=torch.float64, **d) * (2 * math.pi / k)
            z = torch.exp(1j * m)
            B1.append(1.0 / ((1 + 4 * z + z * z) / 6).abs() ** 2)
        f = [torch.fft.fftfreq(k, 1.0 / k, dtype=torch.float64, **d) / b for k, b in zip(K, self.box.tolist())]
        msq = f[0][:, None, None] ** 2 + f[1][None, :, None] ** 2 + f[2][None, None, :] ** 2
        msq[0, 0, 0] = 1.0
        self.bc = torch.exp(-math.pi ** 2 * msq / self.beta ** 2) / (math.pi * msq * self.V) * \
            B1[0][:, None, None] * B1[1][None, :, None] * B1[2][None, None, :]
        self.bc[0, 0, 0] = 0.0

    def fixed(self, crd):
        """The library's fixed-point coordinates of float32 ones."""
        cof = torch.tensor(0.25 * 4294967296.0, dtype=torch.float32, device="cuda") / self.box32
        return (crd.float() * cof).to(torch.int32).long() * 4

    def displace(self, u, i, j):
        w = ((u[j] - u[i]) + (1 << 31)) % (1 << 32) - (1 << 31)
        return w.double() * (self.box / 4294967296.0)

    def near(self, u, radius):
        """Pairs i < j within the radius, exclusions left out."""
        x = (u.double() / 4294967296.0).float()
        out = []
        step = max(1, min(self.n, 200_000_000 // self.n))
        for a in range(0, self.n, step):
            r2 = torch.zeros((min(step, self.n - a), self.n - a), device="cuda")
            for k in range(3):
                w = x[a:a + step, k, None] - x[None, a:, k]
                r2 += ((w - w.round()) * self.box32[k]) ** 2
            p = torch.nonzero(r2 < (radius + 0.01) ** 2)
            out.append(p[p[:, 0] < p[:, 1]] + a)
        p = torch.cat(out)
        key, gone = p[:, 0] * self.n + p[:, 1], self.ei * self.n + self.ej
        p = p[~torch.isin(key, gone)]
        return p[:, 0].contiguous(), p[:, 1].contiguous()

    def inside(self, u, near):
        """Those of the pairs inside the cutoff, by the list's float32 rule."""
        i, j = near
        w = (((u[j] - u[i]) + (1 << 31)) % (1 << 32) - (1 << 31)).to(torch.int32)
        r = w.float() * (torch.tensor(1.0 / 4294967296.0, device="cuda") * self.box32)
        r2 = (r[:, 0] * r[:, 0] + r[:, 1] * r[:, 1]) + r[:, 2] * r[:, 2]
        keep = r2 < torch.tensor(self.rc, device="cuda") ** 2
        return i[keep], j[keep]

    def pair_terms(self, r2, i, j, q, A, B, lam=None, cut_soft=False):
        """(LJ, Coulomb) energy of each pair at squared distances r2."""
        qq = q[i] * q[j]
        if not self.soft:
            p = self.tri[self.type[i], self.type[j]]
            i6 = r2 ** -3
            r = r2.sqrt()
            return (A[p] / 12 * i6 - B[p] / 6) * i6, qq * torch.erfc(self.beta * r) / r
        s = self.s
        pa, pb = self.tri[self.type[i], self.type[j]], self.tri[self.typeB[i], self.typeB[j]]
        aa, ab, ba, bb = A[pa], B[pa], self.A2[pb], self.B2[pb]
        soft = (self.mask[i] != self.mask[j]) | ((ba > 1e-6) & (aa < 1e-6)) | ((ba < 1e-6) & (aa > 1e-6))
        s6 = float(s.sc_sigma) ** 6
        one = torch.ones_like(aa)

        def sig(a, b):
            no = (a < 1e-6) | (b < 1e-6)
            return torch.where(no, one * s6, torch.clamp(0.5 * a / torch.where(no, one, b),
                                                         min=float(s.sc_sigma_min) ** 6))
        uA = torch.where(soft, r2 ** 3 + s.sc_alpha * lam ** s.sc_p * sig(aa, ab), r2 ** 3)
        uB = torch.where(soft, r2 ** 3 + s.sc_alpha * (1 - lam) ** s.sc_p * sig(ba, bb), r2 ** 3)
        sA, sB = uA ** (1 / 6), uB ** (1 / 6)
        inA = (~soft | (sA < self.rc)).double() if cut_soft else 1.0
        inB = (~soft | (sB < self.rc)).double() if cut_soft else 1.0
        lj = (1 - lam) * inA * (aa / 12 / uA - ab / 6) / uA + lam * inB * (ba / 12 / uB - bb / 6) / uB
        return lj, qq * ((1 - lam) * inA * torch.erfc(self.beta * sA) / sA +
                         lam * inB * torch.erfc(self.beta * sB) / sB)

    def excluded(self, d, q):
        r = d.norm(dim=1)
        return -q[self.ei] * q[self.ej] * torch.erf(self.beta * r) / r

    def spread(self, u, shift, q):
        """Charge grid; `shift` (differentiable, zero) moves the atoms."""
        idx, wgt = [], []
        for k in range(3):
            t = u[:, k] * self.K[k]
            base = t // (1 << 32)
            f = (t - base * (1 << 32)).double() / 4294967296.0 + shift[:, k] * (self.K[k] / self.box[k])
            w = [f ** 3 / 6, (-3 * f ** 3 + 3 * f ** 2 + 3 * f + 1) / 6, (3 * f ** 3 - 6 * f ** 2 + 4) / 6,
                 (1 - f) ** 3 / 6]
            wgt.append(torch.stack(w, 1))
            idx.append((base[:, None] - torch.arange(4, device="cuda")) % self.K[k])
        at = (idx[0][:, :, None, None] * self.K[1] + idx[1][:, None, :, None]) * self.K[2] + idx[2][:, None, None, :]
        val = q[:, None, None, None] * wgt[0][:, :, None, None] * wgt[1][:, None, :, None] * wgt[2][:, None, None, :]
        Q = torch.zeros(self.K[0] * self.K[1] * self.K[2], dtype=torch.float64, device="cuda")
        return Q.index_add(0, at.reshape(-1), val.reshape(-1)).reshape(self.K)

    def convolve(self, Q):
        return torch.fft.ifftn(torch.fft.fftn(Q) * self.bc).real * Q.numel()

    def self_energy(self, q):
        return -self.beta / math.sqrt(math.pi) * (q * q).sum() - \
            math.pi / (2 * self.beta ** 2 * self.V) * q.sum() ** 2

    def lrc(self, B=None, lam=None):
        c = (-2.0 / 3.0) * math.pi / self.rc ** 3 / 6.0 / self.V

        def total(t, B):
            m = torch.bincount(t, minlength=64).double()
            T = int(t.max()) + 1
            return (m[:T, None] * m[None, :T] * B[self.tri[:T, :T]]).sum()
        if not self.soft:
            return c * total(self.type, self.B if B is None else B)
        a, b = total(self.type, self.B), total(self.typeB, self.B2)
        return c * ((1 - lam) * a + lam * b), c * (b - a)

    def evaluate(self, u, near, q=None, A=None, B=None, graph=False):
        """Energy parts, per-pair terms and forces."""
        q, A, B = (self.q if q is None else q), (self.A if A is None else A), (self.B if B is None else B)
        i, j = self.inside(u, near)
        lam = float(np.float32(self.s.lam)) if self.soft else None
        d = self.displace(u, i, j).requires_grad_()
        e = self.displace(u, self.ei, self.ej).requires_grad_()
        shift = torch.zeros((self.n, 3), dtype=torch.float64, device="cuda", requires_grad=True)
        lj, co = self.pair_terms((d * d).sum(1), i, j, q, A, B, lam)
        cor = self.excluded(e, q)
        Q = self.spread(u, shift, q)
        rec = 0.5 * (Q * self.convolve(Q)).sum()
        gd, ge, gs = torch.autograd.grad(lj.sum() + co.sum() + cor.sum() + rec, (d, e, shift), retain_graph=True,
                                         create_graph=graph)
        f = (-gs).index_add(0, i, gd).index_add(0, j, -gd).index_add(0, self.ei, ge).index_add(0, self.ej, -ge)
        lrc = self.lrc(B, lam)
        parts = dict(lj=lj.sum(), direct=co.sum(), correction=cor.sum(), self=self.self_energy(q), reciprocal=rec,
                     lrc=lrc[0] if self.soft else lrc, pairs_in=torch.tensor(float(len(i)), device="cuda").double())
        return f, parts, (i, j, d, lj, co)


def _nve(s, x, v, steps, dt):
    """Leap-frog with the waters' bonds held, coordinates kept as the library
    keeps them between steps (float32 inputs of each force)."""
    ex = Exact(s)
    m = torch.tensor(s.mass, device="cuda").double()
    im = 1.0 / m
    nw = s.waters
    w = torch.arange(3 * nw, device="cuda").reshape(nw, 3)
    bond = [(0, 1), (0, 2), (1, 2)]
    rHH = 2 * system.TIP3P_ROH * math.sin(math.radians(system.TIP3P_HOH_DEG) / 2)
    want = torch.tensor([system.TIP3P_ROH, system.TIP3P_ROH, rHH], device="cuda").float().double() ** 2
    wi = im[w]
    C = torch.zeros((nw, 3, 3), dtype=torch.float64, device="cuda")
    for a, (p, q) in enumerate(bond):
        for b, (r, t) in enumerate(bond):
            C[:, a, b] = (q == t) * wi[:, q] - (q == r) * wi[:, q] - (p == t) * wi[:, p] + (p == r) * wi[:, p]
    near = ex.near(ex.fixed(x), ex.rc + 3.0)
    for _ in range(steps):
        u = ex.fixed(x)
        f = ex.evaluate(u, near)[0].detach()
        v = v + dt * im[:, None] * f
        y = x + dt * v
        if nw:
            old = torch.stack([ex.displace(u, w[:, p], w[:, q]) for p, q in bond], 1)
            r0 = torch.stack([y[w[:, q]] - y[w[:, p]] for p, q in bond], 1)
            r0 = r0 - ex.box * (r0 / ex.box).round()
            for b in (0, 1):         # a water cut by the box's face comes out whole, at its oxygen
                y[w[:, b + 1]] = y[w[:, 0]] + r0[:, b]
            g = torch.zeros((nw, 3), dtype=torch.float64, device="cuda")
            for _ in range(8):
                r = r0 + torch.einsum("nab,nbd->nad", C, g[:, :, None] * old)
                jac = 2 * C * torch.einsum("nad,nbd->nab", r, old)
                g = g - torch.linalg.solve(jac, ((r * r).sum(2) - want))
            move = torch.zeros((nw, 3, 3), dtype=torch.float64, device="cuda")
            for b, (p, q) in enumerate(bond):
                move[:, p] -= wi[:, p, None] * g[:, b, None] * old[:, b]
                move[:, q] += wi[:, q, None] * g[:, b, None] * old[:, b]
            y = y.index_add(0, w.reshape(-1), move.reshape(-1, 3))
            v = v.index_add(0, w.reshape(-1), move.reshape(-1, 3) / dt)
        x = y
    return x, v, f


def exact(case, seed):
    c, kind = case, case["kind"]
    dt = float(np.float32(0.002 * system.TIME_UNIT_PER_PS))
    if kind in ("md", "batch"):
        systems = [_box_system(c, seed)] if kind == "md" else _batch_systems(c, seed)
        got = [_nve(s, torch.tensor(s.crd, device="cuda").double(),
                    torch.tensor(_velocities(s, seed + k), device="cuda").double(), c["steps"], dt)
               for k, s in enumerate(systems)]
        return [g[0] for g in got] + [g[1] for g in got], [g[2] for g in got]
    if kind in ("frame", "ti"):
        return _exact_fep(c, seed)
    s = _box_system(c, seed)
    ex = Exact(s)
    u = ex.fixed(torch.tensor(s.crd, device="cuda"))
    near = ex.near(u, ex.rc)
    if kind in ("egrad", "fgrad"):
        q, A, B = (t.clone().requires_grad_() for t in (ex.q, ex.A, ex.B))
        f, parts, _ = ex.evaluate(u, near, q, A, B, graph=kind == "fgrad")
        if kind == "egrad":
            value = sum(parts[k] for k in ("lj", "direct", "correction", "self", "reciprocal", "lrc"))
        else:
            value = ((f - torch.tensor(_target(s.n, seed), device="cuda").double()) ** 2).sum()
        value.backward()
        return value.detach(), q.grad, A.grad.cpu(), B.grad.cpu()
    f, parts, (i, j, d, lj, co) = ex.evaluate(u, near)
    if kind == "calls":
        return f
    p = ex.tri[ex.type[i], ex.type[j]]
    i6 = (d.detach() ** 2).sum(1) ** -3
    vir = (ex.A[p] * i6 - ex.B[p]) * i6
    zero = torch.zeros(s.n, dtype=torch.float64, device="cuda")
    energy, virial = zero.index_add(0, i, (lj + co).detach()), zero.index_add(0, i, vir)
    parts = {k: float(t) for k, t in parts.items()}
    parts["lj_virial"] = float(vir.sum())
    if kind == "score":
        return f, energy, virial, parts
    v = torch.tensor(_velocities(s, seed), device="cuda").double()
    ek = 0.5 * (torch.tensor(s.mass, device="cuda").double()[:, None] * v * v).sum()
    W = parts["lj_virial"] + 6 * parts["lrc"] + sum(parts[k] for k in ("direct", "correction", "self", "reciprocal"))
    return f, energy, virial, parts, ((2 * ek + W) / (3 * ex.V)).reshape(1), ek.reshape(1)


def _exact_fep(c, seed):
    s = _fep_system(c, seed, 0.5)
    ex = Exact(s)
    u = ex.fixed(torch.tensor(s.crd, device="cuda"))
    i, j = ex.inside(u, ex.near(u, ex.rc))
    r2 = (ex.displace(u, i, j) ** 2).sum(1)
    e = ex.displace(u, ex.ei, ex.ej)
    dq = torch.tensor((s.charge_B.astype(np.float64) - s.charge_A.astype(np.float64)).astype(np.float32),
                      device="cuda").double()
    no = torch.zeros((s.n, 3), dtype=torch.float64, device="cuda")
    same = ex.mask[i] == ex.mask[j]
    fields, longs = [], []
    for lam in np.linspace(0.0, 1.0, c["windows"]) if c["kind"] == "frame" else [0.5]:
        l = torch.tensor(float(lam), dtype=torch.float64, device="cuda", requires_grad=True)
        q = ex.q + (l - 0.5) * dq
        with torch.no_grad():
            lj, co = ex.pair_terms(r2, i, j, q, ex.A, ex.B, l, cut_soft=True)
        lj2, co2 = ex.pair_terms(r2, i, j, q, ex.A, ex.B, l)
        dlj, = torch.autograd.grad(lj2.sum(), l, retain_graph=True)
        dco, = torch.autograd.grad(co2.sum(), l, retain_graph=True)
        # the reference's form leaves the 1/r out of an ordinary pair's charge term
        qd = q.detach()
        pa, pb = ex.tri[ex.type[i], ex.type[j]], ex.tri[ex.typeB[i], ex.typeB[j]]
        aa, ba = ex.A[pa], ex.A2[pb]
        hard = same & ~((ba > 1e-6) & (aa < 1e-6)) & ~((ba < 1e-6) & (aa > 1e-6))
        r = r2.sqrt()
        cross = hard.double() * (dq[i] * qd[j] + qd[i] * dq[j]) * torch.erfc(ex.beta * r)
        dref = dco + (cross - cross / r).sum()
        tail, dtail = ex.lrc(lam=float(lam))
        fields.append(torch.stack([lj[~same].sum(), lj[same].sum(), co[~same].sum(), co[same].sum(), dlj, dref, dco,
                                   tail, dtail]).detach())
        Q = ex.spread(u, no, q)
        rec, own, cor = 0.5 * (Q * ex.convolve(Q)).sum(), ex.self_energy(q), ex.excluded(e, q).sum()
        longs.append(torch.stack([rec, own, cor]).detach())
        if c["kind"] == "ti":
            g = [torch.autograd.grad(t, l, retain_graph=True)[0] for t in (rec, own, cor)]
            return float(dlj), float(dref), float(g[0]), float(g[1]), float(g[2])
    return torch.stack(fields).cpu().numpy(), torch.stack(longs).cpu().numpy()
