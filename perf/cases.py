"""Measured cases: what a user of this framework has it do, over its range of sizes.

Kinds of pass:
  steps      a propagation segment through the propagator API: the fields of `steps`
             phaseless steps drawn from the key, the steps, QR, resampling, overlaps
  block      one sampler call (propagate_phaseless: blocks of `steps` steps with QR, local
             energies, block statistics, then resampling), its energy read back
  energy     the trial's local energies of a population
  fragments  one block of a fragment batch (grouped steps, block ends), from one graph,
             its statistics read back

Walker types: "rhf" (restricted walkers and trial), "uhf" (unrestricted), "spin"
(unrestricted with one set of Cholesky vectors per spin).  Hamiltonians are the
synthetic ones of cs_afqmc_amd.problems (symmetric Gaussian vectors with exp(-g / 80)
decay, Haar-random trial), made on the GPU.
"""

import math

import numpy as np
import torch

from cs_afqmc_amd import batch, hamiltonian, propagation, rng, sampling, wavefunctions
from cs_afqmc_amd.prop_unrestricted import propagation as spin_propagation
from cs_afqmc_amd.prop_unrestricted import wavefunctions_unrestricted as spin_wavefunctions

DT = 0.005
N_EXP = 6


def _case(name, kind, walkers, norb, nup, ndn, nchol, n, precision, steps=5, blocks=1, count=1):
    return {"name": name, "kind": kind, "walkers": walkers, "norb": norb, "nup": nup,
            "ndn": ndn, "nchol": nchol, "n_walkers": n, "precision": precision, "steps": steps,
            "blocks": blocks, "count": count}


def listed():
    return [
        # the smallest calls: an H10 chain's sizes (minimal basis, 200 walkers), where
        # launches and latency count; QR every 5 steps, through the propagator API ...
        _case("h10_steps_fp64", "steps", "rhf", 10, 5, 5, 27, 200, "fp64"),
        # ... and as the driver runs it: a captured block of 50 steps per sampler call
        _case("h10_block_fp64", "block", "rhf", 10, 5, 5, 27, 200, "fp64", 5, 10),
        # a spin-resolved open-shell system of odd sizes, small
        _case("spin_n37_steps_fp64", "steps", "spin", 37, 9, 7, 149, 333, "fp64"),
        # the ordinary closed-shell problem, in the default precision ...
        _case("rhf_n100_steps_fp64", "steps", "rhf", 100, 20, 20, 400, 1024, "fp64"),
        # ... in the mixed precision of production runs ...
        _case("rhf_n100_steps_bf16x3", "steps", "rhf", 100, 20, 20, 400, 1024, "bf16x3"),
        # ... and a ragged one with float32 contractions
        _case("rhf_n73_steps_fp32", "steps", "rhf", 73, 17, 17, 301, 600, "fp32"),
        # its local energies, the other half of a block
        _case("rhf_n100_energy_fp64", "energy", "rhf", 100, 20, 20, 400, 1024, "fp64"),
        # an open-shell molecule of odd sizes past 128 orbitals, default precision
        _case("uhf_n131_steps_fp64", "steps", "uhf", 131, 29, 26, 523, 777, "fp64"),
        # the largest single problem, mixed precision: propagation and local energies
        _case("uhf_n200_steps_bf16x3", "steps", "uhf", 200, 40, 40, 1000, 2048, "bf16x3"),
        _case("uhf_n200_energy_bf16x3", "energy", "uhf", 200, 40, 40, 1000, 2048, "bf16x3"),
        # uneven fragments (norb 20 to 120, 256 walkers each) as one batch: a small job in
        # the default precision and the full job in mixed precision
        _case("fragments16_fp64", "fragments", "rhf", 120, 24, 24, 480, 256, "fp64", 50, 1, 16),
        _case("fragments64_bf16x3", "fragments", "rhf", 120, 24, 24, 480, 256, "bf16x3", 50, 1,
              64),
    ]


def _log_int(r, lo, hi):
    return int(round(math.exp(r.uniform(math.log(lo), math.log(hi)))))


#: seconds per flop, roughly, of each precision: only bounds what a drawn case costs
_COST = {"fp64": 1 / 4e13, "fp32": 1 / 5e13, "bf16x3": 1 / 2e14}


def _cost(case):
    return work(case)["flops"] * _COST[case["precision"]]


def draw(r):
    """One problem of the listed range: 10 to 250 orbitals, 24 to 2048 walkers."""
    kind = r.choice(["steps", "steps", "steps", "steps", "energy", "energy", "block"])
    walkers = r.choice(["rhf", "rhf", "uhf", "spin"])
    precision = r.choice(["fp64", "fp64", "bf16x3", "bf16x3", "fp32"])
    n = _log_int(r, 24, 2048)
    norb = _log_int(r, 10, 250)
    steps, blocks = r.choice([2, 5, 10]), 1
    if kind == "block":
        norb, blocks = min(norb, 120), r.choice([2, 5])
    nup = max(1, min(50, int(norb * r.uniform(0.15, 0.3))))
    ndn = nup if walkers == "rhf" else max(1, nup - r.randint(0, 3))
    nchol = max(8, int(norb * r.uniform(3.0, 5.0)))
    c = _case("", kind, walkers, norb, nup, ndn, nchol, n, precision, steps, blocks)
    del c["name"]
    most = 0.5 * max(_cost(x) for x in listed())
    while _cost(c) > most and c["n_walkers"] > 24:
        c["n_walkers"] = max(24, c["n_walkers"] * 2 // 3 | 1)
    return c


# ------------------------------------------------------------------------------ inputs
def _sym(a):
    return (a + a.transpose(-1, -2)) / math.sqrt(2.0)


def _vectors(norb, nchol, gen):
    """Symmetric Cholesky vectors (nchol, norb^2) and the one-body matrix (norb, norb)."""
    a = torch.randn((nchol, norb, norb), generator=gen, device="cuda", dtype=torch.float64)
    a = _sym(a) / norb
    a *= torch.exp(-torch.arange(nchol, device="cuda", dtype=torch.float64) / 80.0).view(-1, 1, 1)
    h1 = _sym(0.1 * torch.randn((norb, norb), generator=gen, device="cuda", dtype=torch.float64))
    return a.view(nchol, norb * norb), h1.cpu().numpy()


def _haar(norb, gen):
    q, r = np.linalg.qr(gen.standard_normal((norb, norb)))
    return q * np.sign(np.diag(r))[None, :]


def _problem(case, seed):
    """ham_data, wave_data of a case: the same arrays for the same seed."""
    norb, nup, ndn, nchol = case["norb"], case["nup"], case["ndn"], case["nchol"]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    host = np.random.default_rng(seed)
    chol, h1 = _vectors(norb, nchol, gen)
    h1 = np.array([h1, h1])
    if case["walkers"] == "spin":
        other, h1b = _vectors(norb, nchol, gen)
        chol = torch.stack([chol, 0.8 * chol + 0.6 * other])
        h1[1] = 0.8 * h1[0] + 0.6 * h1b
    up = _haar(norb, host)[:, :nup]
    if case["walkers"] == "rhf":
        wave = {"mo_coeff": up, "rdm1": np.array([up @ up.T] * 2)}
    else:
        dn = _haar(norb, host)[:, :ndn]
        wave = {"mo_coeff": [up, dn], "rdm1": np.array([up @ up.T, dn @ dn.T])}
    return {"h0": 0.0, "h1": h1, "chol": chol, "ene0": 0.0}, wave


def _at_trial(case, wave):
    """Every walker at the trial determinant, where a run starts: complex (W, norb, n), a
    list of two for unrestricted walkers."""
    def one(mo):
        return torch.from_numpy(mo + 0j).cuda().unsqueeze(0).repeat(case["n_walkers"], 1, 1)

    mo = wave["mo_coeff"]
    return [one(m) for m in mo] if isinstance(mo, list) else one(mo)


def _near_trial(case, wave, seed):
    """Walkers around the trial determinant, as during a run."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed + 1)

    def one(mo):
        z = torch.randn((case["n_walkers"],) + mo.shape, generator=gen, device="cuda",
                        dtype=torch.complex128)
        return (0.1 * z + torch.from_numpy(mo).cuda()).contiguous()

    mo = wave["mo_coeff"]
    return [one(m) for m in mo] if isinstance(mo, list) else one(mo)


def _fragment_cases(case):
    """The members of a fragment batch: norb uniform in [20, case's norb], nocc = norb / 5,
    nchol = 4 norb; the sizes are the case's, the seed gives their values."""
    host = np.random.default_rng(0)
    out = []
    for _ in range(case["count"]):
        norb = int(host.integers(20, case["norb"] + 1))
        out.append(dict(case, norb=norb, nup=norb // 5, ndn=norb // 5, nchol=4 * norb))
    return out


def _pair(case):
    """The trial and the propagator of a case."""
    if case["walkers"] == "rhf":
        trial, prop = wavefunctions.rhf, propagation.propagator_restricted
    elif case["walkers"] == "uhf":
        trial, prop = wavefunctions.uhf, propagation.propagator_unrestricted
    else:
        trial, prop = spin_wavefunctions.uhf, spin_propagation.propagator_unrestricted
    return (trial(case["norb"], (case["nup"], case["ndn"])),
            prop(DT, case["n_walkers"], N_EXP, precision=case["precision"]))


def prepare(case, seed):
    if case["kind"] == "fragments":
        frags = []
        for i, m in enumerate(_fragment_cases(case)):
            hd, wd = _problem(m, seed + 1000 * i)
            frags.append(batch.Fragment(hd, wd, "rhf", (m["nup"], m["ndn"]), m["n_walkers"],
                                        dt=DT, seed=seed + i, precision=m["precision"],
                                        n_prop_steps=m["steps"]))
        return {"kind": "fragments", "frags": frags,
                "batch": batch.FragmentBatch(frags, tune=True, use_graph=True)}
    hd, wave = _problem(case, seed)
    trial, prop = _pair(case)
    ham = hamiltonian.hamiltonian(case["norb"])
    hd = ham.build_measurement_intermediates(hd, trial, wave)
    hd = ham.build_propagation_intermediates(hd, prop, trial, wave)
    st = {"kind": case["kind"], "ham": ham, "ham_data": hd, "wave_data": wave, "trial": trial,
          "prop": prop}
    if case["kind"] == "energy":
        st["walkers"] = _near_trial(case, wave, seed)
        return st
    st["prop_data"] = prop.init_prop_data(trial, wave, hd, _at_trial(case, wave))
    st["prop_data"]["key"] = rng.PRNGKey(seed)
    if case["kind"] == "block":
        st["sampler"] = sampling.sampler(case["steps"], case["blocks"], 1)
    else:
        st["fields"] = torch.empty((case["steps"], case["n_walkers"], case["nchol"]),
                                   dtype=torch.float64, device="cuda")
    return st


def run(st):
    if st["kind"] == "energy":
        return st["trial"].calc_energy(st["walkers"], st["ham_data"], st["wave_data"])
    if st["kind"] == "fragments":
        st["batch"].run_block()
        frags = st["frags"]
        # the block energies and weights go to the host, as after a sampler call
        return {"stats": torch.stack([f.slot for f in frags]).cpu(),
                "energies": torch.cat([f.energies for f in frags]),
                "weights": torch.cat([f.prop_data["weights"] for f in frags]),
                "overlaps": torch.cat([f.prop_data["overlaps"] for f in frags]),
                "walkers": torch.cat([f.prop_data["walkers"].view(-1) for f in frags])}
    prop, trial, hd, wave, pd = (st[k] for k in ("prop", "trial", "ham_data", "wave_data",
                                                 "prop_data"))
    if st["kind"] == "block":
        e, pd = st["sampler"].propagate_phaseless(st["ham"], hd, prop, pd, trial, wave)
        return {"energy": e, "stats": pd["block_stats"], "weights": pd["weights"],
                "overlaps": pd["overlaps"], "walkers": pd["walkers"]}
    pd["key"], key = rng.split(pd["key"])
    fields = hd["_afqmc_device"].fields_normal(key[0], key[1], None, out=st["fields"])
    for s in range(fields.shape[0]):
        pd = prop.propagate(trial, hd, pd, fields[s], wave)
    pd = prop.orthonormalize_walkers(pd)
    pd = prop.stochastic_reconfiguration_local(pd)
    pd["overlaps"] = trial.calc_overlap(pd["walkers"], wave)
    return {"walkers": pd["walkers"], "weights": pd["weights"], "overlaps": pd["overlaps"],
            "shift": pd["pop_control_ene_shift"]}


# -------------------------------------------------------------------------------- work
def _work_one(c):
    """Bytes and flops of one pass of one problem: Cholesky vectors and V as symmetric
    matrices, real x complex products 4 flops, complex ones 8."""
    N, G, W = c["norb"], c["nchol"], c["n_walkers"]
    ns = [c["nup"]] if c["walkers"] == "rhf" else [c["nup"], c["ndn"]]
    sets = 2 if c["walkers"] == "spin" else 1
    nv = N * (N + 1) // 2
    walkers = 16.0 * W * N * sum(ns)
    chol, rot = 8.0 * sets * G * nv, 8.0 * G * N * sum(ns)
    energy = sum(4.0 * G * N * n * n + 8.0 * G * n * n + 12.0 * N * n * n + 8.0 * n**3
                 for n in ns)
    if c["kind"] == "energy":
        return walkers + rot + 16.0 * W, W * energy
    step = 4.0 * sets * G * nv + 40.0 * G + sum(
        4.0 * G * N * n + (8.0 + 8.0 * (N_EXP - 1)) * N * N * n + 12.0 * N * n * n + 8.0 * n**3
        for n in ns)
    ends = sum(16.0 * N * n * n for n in ns)
    blocks = c["blocks"]
    flops = W * blocks * (c["steps"] * step + ends)
    nbytes = 2.0 * walkers + chol + rot + 64.0 * W
    if c["kind"] in ("block", "fragments"):
        flops += W * blocks * energy
    return nbytes, flops


def work(case):
    members = [case]
    if case["kind"] == "fragments":  # the mean batch: norb evenly over its range
        k = case["count"]
        norbs = [20 + round((case["norb"] - 20) * (i + 0.5) / k) for i in range(k)]
        members = [dict(case, norb=n, nup=n // 5, ndn=n // 5, nchol=4 * n) for n in norbs]
    each = [_work_one(m) for m in members]
    return {"bytes": sum(e[0] for e in each), "flops": sum(e[1] for e in each)}


# ------------------------------------------------------------------------ 64-bit values
def _philox(c0, c1, c2, c3, k0, k1):
    """Philox4x32-10 (Salmon et al., SC'11) on int64 tensors or ints holding 32 bits."""
    m = 0xFFFFFFFF
    for _ in range(10):
        p0, p1 = c0 * 0xD2511F53, c2 * 0xCD9E8D57
        c0, c1, c2, c3 = (((p1 >> 32) & m) ^ c1 ^ k0, p1 & m, ((p0 >> 32) & m) ^ c3 ^ k1, p0 & m)
        k0, k1 = (k0 + 0x9E3779B9) & m, (k1 + 0xBB67AE85) & m
    return c0, c1, c2, c3


def _normals(seed, counter, count):
    """Box-Muller pairs of 53-bit uniforms: the field draw of a key."""
    pair = torch.arange((count + 1) // 2, device="cuda", dtype=torch.int64)
    r = _philox(pair & 0xFFFFFFFF, pair >> 32, torch.full_like(pair, counter),
                torch.zeros_like(pair), seed, 0)
    bits = [((r[i + 1] & 0xFFFFFFFF) << 21 | r[i] >> 11).double() for i in (0, 2)]
    u1, u2 = (bits[0] + 1.0) * 2.0**-53, bits[1] * 2.0**-53
    rad, ang = torch.sqrt(-2.0 * torch.log(u1)), 2.0 * math.pi * u2
    return torch.stack([rad * torch.cos(ang), rad * torch.sin(ang)], 1).view(-1)[:count]


def _uniform(seed, counter):
    r = _philox(0, 0xFFFFFFFF, counter, 0, seed, 0)
    return (((r[1] << 32) | r[0]) >> 11) * 2.0**-53


def _host(f, t):
    return torch.from_numpy(np.ascontiguousarray(f(t.cpu().numpy()))).cuda()


class _Exact:
    """The phaseless step of one problem in complex128, walkers as lists over spins."""

    def __init__(self, case, seed):
        self.c = case
        hd, wave = _problem(case, seed)
        N = case["norb"]
        self.rhf = case["walkers"] == "rhf"
        mo = wave["mo_coeff"]
        self.wave = wave
        self.mo = [torch.from_numpy(np.ascontiguousarray(m)).cuda()
                   for m in ([mo] if self.rhf else mo)]
        self.S = len(self.mo)
        chol = hd["chol"].view(-1, case["nchol"], N, N)
        self.chol = [chol[0], chol[-1]][:self.S]
        self.sets = chol.shape[0]
        h1 = torch.from_numpy(hd["h1"]).cuda()
        rdm = torch.from_numpy(wave["rdm1"]).cuda()
        if self.sets == 1:
            mf = (chol[0] * (rdm[0] + rdm[1])).sum((1, 2))
        else:
            mf = (chol[0] * rdm[0]).sum((1, 2)) + (chol[1] * rdm[1]).sum((1, 2))
        self.mf = 1j * mf
        self.h0_prop = float((mf * mf).sum()) / 2.0
        self.expE, self.rot_h1, self.rot = [], [], []
        for s in range(self.S):
            L = self.chol[s]
            v0 = 0.5 * torch.bmm(L, L.transpose(1, 2).contiguous()).sum(0)
            v1 = -(mf @ L.reshape(-1, N * N)).view(N, N)
            self.expE.append(torch.linalg.matrix_exp(-DT / 2.0 * (h1[s] - v0 - v1)))
            self.rot_h1.append(self.mo[s].T @ h1[s])
            self.rot.append(torch.matmul(self.mo[s].T.contiguous(), L))

    def init(self):
        W = self.c["n_walkers"]
        phi = _at_trial(self.c, self.wave)
        self.phi = [phi] if self.rhf else phi
        self.e_est = float(self.energy(self.phi).real.sum()) / W
        self.shift = self.e_est
        self.w = torch.ones(W, dtype=torch.float64, device="cuda")
        self.ovlp = self.overlap(self.phi)

    def _o(self, phi, s):
        return torch.matmul(self.mo[s].T.contiguous().to(torch.complex128), phi[s])

    def overlap(self, phi):
        d = [_host(np.linalg.det, self._o(phi, s)) for s in range(self.S)]
        return d[0] * d[-1]

    def green(self, phi):
        return [torch.matmul(phi[s], _host(np.linalg.inv, self._o(phi, s))).transpose(1, 2)
                .contiguous() for s in range(self.S)]

    def force_bias(self, green):
        G, W = self.c["nchol"], green[0].shape[0]
        fb = sum(torch.matmul(green[s].reshape(W, -1),
                              self.rot[s].reshape(G, -1).T.contiguous().to(torch.complex128))
                 for s in range(self.S))
        return 2.0 * fb if self.rhf else fb

    def energy(self, phi):
        green = self.green(phi)
        mult = 2.0 if self.rhf else 1.0
        e1 = sum(mult * (green[s] * self.rot_h1[s]).sum((1, 2)) for s in range(self.S))
        fb = self.force_bias(green)
        e2 = (fb * fb).sum(1) / 2.0
        W, G = self.c["n_walkers"], self.c["nchol"]
        for s in range(self.S):
            n, N = self.rot[s].shape[1:]
            rot = self.rot[s].reshape(G * n, N).to(torch.complex128)
            step = max(1, int(2e8 // (G * n * n)))
            for w0 in range(0, W, step):
                g = green[s][w0:w0 + step]
                k = g.shape[0]
                # f[g, i, w, j] = sum_p rot[g, i, p] green[w, j, p]
                f = torch.matmul(rot, g.reshape(k * n, N).T.contiguous()).view(G, n, k, n)
                e2[w0:w0 + step] -= mult / 2.0 * (f * f.transpose(1, 3)).sum((0, 1, 3))
        return e1 + e2

    def step(self, x):
        N, W = self.c["norb"], self.c["n_walkers"]
        sq = math.sqrt(DT)
        fs = -sq * (1j * self.force_bias(self.green(self.phi)) - self.mf)
        xt = x - fs
        shift_term = (xt * self.mf).sum(1)
        fb_term = (x * fs - fs * fs / 2.0).sum(1)
        for s in range(self.S):
            if s == 0 or self.sets == 2:
                L = self.chol[s].reshape(-1, N * N)
                V = torch.complex(-sq * (xt.imag @ L), sq * (xt.real @ L)).view(W, N, N)
            E = self.expE[s].to(torch.complex128)
            t = torch.matmul(E, self.phi[s])
            acc = t.clone()
            for k in range(1, N_EXP):
                t = torch.matmul(V, t) / k
                acc += t
            self.phi[s] = torch.matmul(E, acc)
        new = self.overlap(self.phi)
        ratio = new / self.ovlp
        imp = torch.exp(-sq * shift_term + fb_term + DT * (self.shift + self.h0_prop)) * ratio
        theta = torch.angle(torch.exp(-sq * shift_term) * ratio)
        f = torch.nan_to_num(imp.abs() * torch.cos(theta), nan=0.0)
        f = torch.where((f < 1e-3) | (f > 100.0), 0.0, f)
        self.w = self.w * f
        self.w = torch.where(self.w > 100.0, 0.0, self.w)
        self.shift = self.e_est - 0.1 * math.log(float(self.w.sum()) / W) / DT
        self.ovlp = new

    def block(self, fields):
        for x in fields:
            self.step(x)
        self.phi = [_host(lambda a: np.linalg.qr(a)[0], p) for p in self.phi]

    def resample(self, zeta):
        W = self.c["n_walkers"]
        w = np.abs(self.w.cpu().numpy())
        cum = np.cumsum(w)
        idx = np.minimum(np.searchsorted(cum, cum[-1] * (np.arange(W) + zeta) / W), W - 1)
        idx = torch.from_numpy(idx).cuda()
        self.phi = [p[idx] for p in self.phi]
        self.w = torch.full_like(self.w, cum[-1] / W)
        self.ovlp = self.overlap(self.phi)

    def walkers(self):
        return self.phi[0] if self.rhf else self.phi


def exact(case, seed):
    # a batch's members are the other cases' steps, many times over: too long here
    if case["kind"] == "fragments":
        return None
    x = _Exact(case, seed)
    if case["kind"] == "energy":
        phi = _near_trial(case, x.wave, seed)
        return x.energy([phi] if x.rhf else phi)
    x.init()
    shape = (case["steps"], case["n_walkers"], case["nchol"])
    stats = []
    for b in range(case["blocks"]):
        x.block(_normals(seed, b, shape[0] * shape[1] * shape[2]).view(shape))
        if case["kind"] == "block":
            x.ovlp = x.overlap(x.phi)
            e = x.energy(x.phi).real
            far = (e - x.e_est).abs() > math.sqrt(2.0 / DT)
            e = torch.where(far, torch.full_like(e, x.e_est), e)
            bw = float(x.w.sum())
            be = float((e * x.w).sum()) / bw
            stats.append([be, bw, float((x.w == 0).sum()), float(far.sum())])
            x.shift = 0.9 * x.shift + 0.1 * be
    x.resample(_uniform(seed, case["blocks"]))
    out = {"walkers": x.walkers(), "weights": x.w, "overlaps": x.ovlp}
    if case["kind"] == "steps":
        out["shift"] = torch.tensor(x.shift, dtype=torch.float64)
    else:
        s = torch.tensor(stats, dtype=torch.float64)
        out["stats"] = s
        out["energy"] = float((s[:, 0] * s[:, 1]).sum() / s[:, 1].sum())
    return out
