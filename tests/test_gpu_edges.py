"""One phaseless step, the force bias and the local energies at sizes on the edges of the
kernels' tiles and chunks (odd row lengths, remainders of 16 and 64, one walker, both GEMM
tile edges), against the CPU oracle.  The float64 path is held to the suite's 1e-10
relative: a step's products sum at most a few thousand terms of O(1) rounding 2^-53."""

import numpy as np
import pytest
import torch

from cs_afqmc_amd import hamiltonian, problems, propagation, wavefunctions
from cs_afqmc_amd.device import DeviceStep
from cs_afqmc_amd.prop_unrestricted import propagation as spin_propagation
from cs_afqmc_amd.prop_unrestricted import wavefunctions_unrestricted as spin_wavefunctions
from oracle import afqmc_oracle as o

pytestmark = pytest.mark.gpu

DT = 0.005
TOL = 1e-10

# walker_type, norb, nelec, nchol, n_walkers
CASES = [
    ("rhf", 1, (1, 1), 1, 1),
    ("rhf", 5, (2, 2), 3, 3),
    ("uhf", 17, (4, 3), 33, 65),
    ("rhf", 33, (5, 5), 131, 70),
    ("uhf", 65, (9, 8), 71, 33),
    ("rhf", 115, (9, 9), 37, 260),  # 128-wide GEMM tiles, partly filled
    ("uhf", 49, (33, 25), 9, 4),    # four-wave measurement, edges of its tile counts
    ("uhf", 66, (64, 49), 7, 3),
]


def rel(a, b):
    if isinstance(b, (list, tuple)):
        return max(rel(x, y) for x, y in zip(a, b))
    a = a.detach().cpu().numpy() if isinstance(a, torch.Tensor) else np.asarray(a)
    s = np.max(np.abs(b))
    return np.max(np.abs(a - b)) / (s if s > 0 else 1.0)


def to_dev(x, dev):
    if isinstance(x, (list, tuple)):
        return [to_dev(y, dev) for y in x]
    return torch.as_tensor(np.ascontiguousarray(x), device=dev)


def make(wt, norb, nelec, nchol, W, hd, wd, precision="fp64"):
    trial = (wavefunctions.rhf if wt == "rhf" else wavefunctions.uhf)(norb, nelec)
    cls = propagation.propagator_restricted if wt == "rhf" else propagation.propagator_unrestricted
    prop = cls(dt=DT, n_walkers=W, precision=precision)
    ham = hamiltonian.hamiltonian(norb)
    wave = dict(wd)
    hdat = ham.build_measurement_intermediates(dict(hd), trial, wave)
    hdat = ham.build_propagation_intermediates(hdat, prop, trial, wave)
    oh = o.build_measurement_intermediates(wt, dict(hd), wd, norb)
    oh = o.build_propagation_intermediates(wt, oh, wd["rdm1"], norb, nelec, DT)
    return trial, prop, hdat, wave, oh


def problem(wt, norb, nelec, nchol, seed=11):
    cs = 0.5 / np.sqrt(norb)
    if wt == "rhf":
        return problems.synthetic_rhf(norb, nelec[0], nchol, seed=seed, chol_std=cs)
    return problems.synthetic_uhf(norb, nelec[0], nelec[1], nchol, seed=seed, chol_std=cs)


def one_step(wt, trial, prop, hdat, wave, oh, wd, walkers, fields, dev, norb):
    """The device's and the oracle's state after one step with the same fields."""
    W = fields.shape[0]
    pd = {"walkers": to_dev(walkers, dev),
          "weights": torch.ones(W, dtype=torch.float64, device=dev),
          "e_estimate": torch.tensor(-0.5, dtype=torch.float64, device=dev),
          "pop_control_ene_shift": torch.tensor(-0.5, dtype=torch.float64, device=dev)}
    pd["overlaps"] = trial.calc_overlap(pd["walkers"], wave)
    pd = prop.propagate(trial, hdat, pd, to_dev(fields, dev), wave)
    od = {"walkers": walkers, "weights": np.ones(W), "e_estimate": -0.5,
          "overlaps": o.calc_overlap(wt, walkers, wd), "pop_control_ene_shift": -0.5}
    od = o.propagate(wt, wt, oh, od, fields, wd, DT, 6, norb)
    return pd, od


@pytest.mark.parametrize("wt,norb,nelec,nchol,W", CASES)
def test_step_force_bias_and_energy(gpu, wt, norb, nelec, nchol, W):
    print(f"edges {wt} N={norb} nelec={nelec} G={nchol} W={W}", flush=True)
    hd, wd, nelec = problem(wt, norb, nelec, nchol)
    trial, prop, hdat, wave, oh = make(wt, norb, nelec, nchol, W, hd, wd)
    rng = np.random.default_rng(3)
    walkers = problems.random_walkers(wt, norb, nelec, W, rng, near=wd["mo_coeff"], noise=0.1)
    fields = rng.standard_normal((W, nchol))
    dw = to_dev(walkers, gpu)
    assert rel(trial.calc_force_bias(dw, hdat, wave),
               o.calc_force_bias(wt, walkers, oh, wd)) < TOL
    assert rel(trial.calc_energy(dw, hdat, wave), o.calc_energy(wt, walkers, oh, wd)) < TOL
    pd, od = one_step(wt, trial, prop, hdat, wave, oh, wd, walkers, fields, gpu, norb)
    assert rel(pd["walkers"], od["walkers"]) < TOL
    assert rel(pd["overlaps"], od["overlaps"]) < TOL
    assert rel(pd["weights"], od["weights"]) < TOL


@pytest.mark.parametrize("asym,packed", [(0.0, True), (2.0**-53, True), (1e-7, False)])
@pytest.mark.parametrize("wt,norb,nelec,nchol,W", [("rhf", 33, (5, 5), 21, 9),
                                                   ("uhf", 131, (5, 3), 18, 5)])
def test_vhs_layout_follows_symmetry(gpu, wt, norb, nelec, nchol, W, asym, packed):
    """V is kept as its upper triangle for Cholesky vectors that are symmetric up to the
    rounding of an orbital rotation, and whole for any larger asymmetry; both layouts give
    the oracle's step (register and streaming Taylor kernel)."""
    print(f"symmetry {wt} N={norb} asym={asym}", flush=True)
    hd, wd, nelec = problem(wt, norb, nelec, nchol)
    chol = np.array(hd["chol"]).reshape(nchol, norb, norb)
    skew = np.random.default_rng(5).uniform(-1.0, 1.0, (norb, norb))
    chol += asym * np.max(np.abs(chol)) * np.triu(skew, 1)[None]
    hd = dict(hd, chol=chol.reshape(nchol, norb * norb))
    trial, prop, hdat, wave, oh = make(wt, norb, nelec, nchol, W, hd, wd)
    entries = norb * (norb + 1) // 2 if packed else norb * norb
    assert hdat["_afqmc_device"].vhs_entries() == entries
    rng = np.random.default_rng(3)
    walkers = problems.random_walkers(wt, norb, nelec, W, rng, near=wd["mo_coeff"], noise=0.1)
    fields = rng.standard_normal((W, nchol))
    pd, od = one_step(wt, trial, prop, hdat, wave, oh, wd, walkers, fields, gpu, norb)
    assert rel(pd["walkers"], od["walkers"]) < TOL
    assert rel(pd["weights"], od["weights"]) < TOL


@pytest.mark.parametrize("scale", [1.0, 1e140, 1e-140])
@pytest.mark.parametrize("norb,n", [(1, 1), (9, 9), (64, 16), (65, 17), (129, 33), (193, 49),
                                    (250, 50), (256, 64)])
def test_orthonormalize_columns_and_scales(gpu, norb, n, scale):
    """Q of LAPACK's Householder QR, at each count of waves, columns per wave and rows per
    lane, with all reflectors in LDS and in batches, and where the squared norms leave the
    fast root's range.  Q of a Gaussian matrix moves by about its condition number (below
    1e4 here) times 2^-53 per rounding: 1e-11."""
    print(f"qr N={norb} n={n} scale={scale}", flush=True)
    hd, wd, nelec = problem("rhf", norb, (n, n), 1)
    trial, prop, hdat, wave, _ = make("rhf", norb, nelec, 1, 3, hd, wd)
    rng = np.random.default_rng(17)
    w = rng.standard_normal((3, norb, n)) + 1j * rng.standard_normal((3, norb, n))
    got = hdat["_afqmc_device"].orthonormalize(to_dev(scale * w, gpu))
    ref = np.array([np.linalg.qr(x)[0] for x in w])
    assert np.max(np.linalg.cond(w)) < 1e4
    assert rel(got, ref) < 1e-11


# float32 carries 24 bits.  Split-bf16 drops lo * lo and rounds each lo, at most 3 * 2^-18 of
# a product, twice that for tr f f: 2.3e-5 of sums of magnitudes up to four times the energy
@pytest.mark.parametrize("precision,tol", [("fp64", TOL), ("fp32", 2e-5), ("bf16x3", 1e-4)])
@pytest.mark.parametrize("norb,nelec,nchol,W", [
    (3, (1, 1), 5, 200), (5, (2, 1), 9, 70), (18, (16, 8), 240, 77), (25, (22, 13), 61, 170),
    (27, (24, 20), 61, 163), (33, (29, 17), 83, 130), (43, (40, 33), 31, 50),
    (66, (64, 50), 19, 60)])
def test_energy_at_each_exchange_tile(gpu, norb, nelec, nchol, W, precision, tol):
    """Local energies at every row and column count of the exchange tile, with partly filled
    last tiles in both directions, one and several passes and walker groups."""
    print(f"exchange N={norb} nelec={nelec} G={nchol} W={W} {precision}", flush=True)
    hd, wd, nelec = problem("uhf", norb, nelec, nchol)
    trial, prop, hdat, wave, oh = make("uhf", norb, nelec, nchol, W, hd, wd, precision)
    walkers = problems.random_walkers("uhf", norb, nelec, W, np.random.default_rng(3),
                                      near=wd["mo_coeff"], noise=0.1)
    got = trial.calc_energy(to_dev(walkers, gpu), hdat, wave)
    assert rel(got, o.calc_energy("uhf", walkers, oh, wd)) < tol


@pytest.mark.parametrize("asym", [0.0, 1e-7])
@pytest.mark.parametrize("wt,norb,nelec,nchol,W", [
    ("rhf", 1, (1, 1), 1, 1), ("rhf", 10, (5, 5), 27, 200), ("uhf", 9, (8, 1), 33, 65),
    ("uhf", 17, (8, 7), 65, 300), ("rhf", 32, (8, 8), 63, 9), ("uhf", 31, (7, 3), 5, 512)])
def test_step_in_one_launch_matches_separate_launches(gpu, wt, norb, nelec, nchol, W, asym):
    """Steps of small problems run as one launch, or as one launch per phase while phases are
    timed: the same walkers, weights, overlaps and shift over steps that reuse the Green's
    function and one that does not, for V kept whole and as its upper triangle."""
    print(f"one launch {wt} N={norb} nelec={nelec} G={nchol} W={W} asym={asym}", flush=True)
    hd, wd, nelec = problem(wt, norb, nelec, nchol)
    chol = np.array(hd["chol"]).reshape(nchol, norb, norb)
    skew = np.random.default_rng(5).uniform(-1.0, 1.0, (norb, norb))
    chol += asym * np.max(np.abs(chol)) * np.triu(skew, 1)[None]
    hd = dict(hd, chol=chol.reshape(nchol, norb * norb))
    trial, prop, hdat, wave, _ = make(wt, norb, nelec, nchol, W, hd, wd)
    dev = hdat["_afqmc_device"]
    rng = np.random.default_rng(3)
    walkers = problems.random_walkers(wt, norb, nelec, W, rng, near=wd["mo_coeff"], noise=0.1)
    fields = to_dev(rng.standard_normal((4, W, nchol)), gpu)
    got = []
    for timed in (False, True):
        dev.prof_enable(timed)
        w = to_dev(walkers, gpu)
        weights = torch.ones(W, dtype=torch.float64, device=gpu)
        overlaps = dev.overlap(w)
        scalars = torch.tensor([-0.5, -0.5], dtype=torch.float64, device=gpu)
        for s in range(4):
            dev.propagate(w, weights, overlaps, fields[s], scalars, reuse_green=s in (1, 3),
                          keep_green=s != 1)
        got.append((w, weights, overlaps, scalars))
    dev.prof_enable(False)
    one, many = got
    for a, b in zip(one, many):
        b = [x.cpu().numpy() for x in b] if isinstance(b, list) else b.cpu().numpy()
        assert rel(a, b) < TOL


@pytest.mark.parametrize("norb,n", [(1, 1), (9, 9), (64, 16), (65, 17), (128, 64)])
def test_orthonormalize_mixed(gpu, norb, n):
    """The mixed mode's QR of up to 128 orbitals; the bound of the test above."""
    print(f"qr mixed N={norb} n={n}", flush=True)
    hd, wd, nelec = problem("rhf", norb, (n, n), 1)
    trial, prop, hdat, wave, _ = make("rhf", norb, nelec, 1, 3, hd, wd, "bf16x3")
    rng = np.random.default_rng(17)
    w = rng.standard_normal((3, norb, n)) + 1j * rng.standard_normal((3, norb, n))
    got = hdat["_afqmc_device"].orthonormalize(to_dev(w, gpu))
    assert np.max(np.linalg.cond(w)) < 1e4
    assert rel(got, np.array([np.linalg.qr(x)[0] for x in w])) < 1e-11


@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16x3"])
@pytest.mark.parametrize("wt,norb,nelec,W", [("rhf", 10, (5, 5), 7), ("uhf", 30, (27, 8), 5)])
def test_energy_with_overlaps_matches_both(gpu, wt, norb, nelec, W, precision):
    """The block end's combined call gives the bits of the separate ones."""
    print(f"energy with overlaps {wt} N={norb} {precision}", flush=True)
    hd, wd, nelec = problem(wt, norb, nelec, 9)
    trial, prop, hdat, wave, _ = make(wt, norb, nelec, 9, W, hd, wd, precision)
    dev = hdat["_afqmc_device"]
    w = to_dev(problems.random_walkers(wt, norb, nelec, W, np.random.default_rng(3),
                                       near=wd["mo_coeff"], noise=0.1), gpu)
    overlaps = torch.zeros(W, dtype=torch.complex128, device=gpu)
    energies = dev.energy(w, overlaps=overlaps)
    assert torch.equal(overlaps, dev.overlap(w))
    assert torch.equal(energies, dev.energy(w))


@pytest.mark.parametrize("wt,nchol,W,one", [
    ("rhf", 9800, 5, True), ("rhf", 10400, 5, False), ("rhf", 25000, 3, False),
    ("uhf", 16666, 3, False), ("rhf", 4800, 300, True), ("rhf", 5200, 300, False)])
def test_step_with_few_orbitals_and_many_vectors(gpu, wt, nchol, W, one):
    """One orbital with as many vectors as a workgroup's LDS holds, or half of it where two
    workgroups share a CU, takes one launch, more vectors the separate ones."""
    print(f"vectors {wt} G={nchol} W={W}", flush=True)
    make_problem = problems.synthetic_rhf if wt == "rhf" else problems.synthetic_uhf
    occ = (1,) if wt == "rhf" else (1, 1)
    # sum_g L_g^2 of order one, without decay: every vector counts
    hd, wd, nelec = make_problem(1, *occ, nchol, seed=11, decay=1e9, chol_std=0.5 / nchol**0.5)
    trial, prop, hdat, wave, oh = make(wt, 1, nelec, nchol, W, hd, wd)
    assert hdat["_afqmc_device"].step_in_one_launch() == one
    rng = np.random.default_rng(3)
    walkers = problems.random_walkers(wt, 1, nelec, W, rng, near=wd["mo_coeff"], noise=0.1)
    fields = rng.standard_normal((W, nchol))
    pd, od = one_step(wt, trial, prop, hdat, wave, oh, wd, walkers, fields, gpu, 1)
    assert np.all(od["weights"] > 0.0)
    assert rel(pd["walkers"], od["walkers"]) < TOL
    assert rel(pd["overlaps"], od["overlaps"]) < TOL
    assert rel(pd["weights"], od["weights"]) < TOL


@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16x3"])
@pytest.mark.parametrize("entries", [
    {(40, 3): np.nan}, {(3, 40): np.nan}, {(7, 7): np.nan}, {(40, 3): np.inf},
    {(3, 40): np.inf, (40, 3): np.inf}, {(7, 7): -np.inf}])
def test_vectors_that_are_not_finite_keep_v_whole(gpu, entries, precision):
    """An entry that is not finite has no mirror image to stand for it, nor does it widen
    the asymmetry that counts as rounding: V is kept whole."""
    norb, nchol, W = 41, 5, 3
    hd, wd, nelec = problem("rhf", norb, (4, 4), nchol)
    trial, prop, hdat, wave, oh = make("rhf", norb, nelec, nchol, W, hd, wd, precision)
    dev = hdat["_afqmc_device"]
    assert dev.vhs_entries() == norb * (norb + 1) // 2
    chol = np.array(hd["chol"]).reshape(nchol, norb, norb)
    for at, value in entries.items():
        chol[(2,) + at] = value
    zeros = np.zeros
    ctx = DeviceStep("rhf", norb, nelec, W, DT, 6, 0.0, 0.0, chol, wd["mo_coeff"],
                     zeros((4, norb)), zeros((nchol, 4, norb)), zeros(nchol), np.eye(norb),
                     precision=precision)
    assert ctx.vhs_entries() == norb * norb


# both sides of the rule's lines: the cost per spin is entries + 20 norb^2 n against 125000, or
# 85000 past 256 walkers
@pytest.mark.parametrize("wt,norb,nelec,nchol,W,asym,one", [
    ("rhf", 28, (7, 7), 20, 256, 0.0, True), ("rhf", 28, (7, 7), 30, 256, 0.0, False),
    ("rhf", 28, (7, 7), 20, 257, 0.0, False), ("rhf", 24, (5, 5), 40, 512, 0.0, True),
    ("rhf", 24, (5, 5), 70, 512, 0.0, False), ("rhf", 24, (5, 5), 40, 513, 0.0, False),
    ("rhf", 29, (1, 1), 5, 9, 0.0, False), ("rhf", 10, (9, 9), 5, 9, 0.0, False),
    ("rhf", 28, (4, 4), 55, 9, 1e-7, True), ("rhf", 28, (4, 4), 58, 9, 1e-7, False),
    ("uhf", 28, (8, 1), 60, 33, 0.0, True), ("uhf", 29, (1, 1), 5, 9, 0.0, False),
    ("uhf", 24, (8, 8), 70, 200, 0.0, True),
    ("spin", 20, (8, 7), 69, 300, 0.0, True), ("spin", 20, (8, 7), 45, 300, 1e-7, True)])
def test_step_route_follows_size(gpu, wt, norb, nelec, nchol, W, asym, one):
    """Steps take one launch up to the sizes where it is the better way, and there agree
    with the launches of the separate phases (which steps that are timed take)."""
    print(f"route {wt} N={norb} nelec={nelec} G={nchol} W={W} asym={asym}", flush=True)
    cs = 0.5 / np.sqrt(norb)
    if wt == "spin":
        hd, wd, nelec = problems.synthetic_uhf_spin(norb, *nelec, nchol, seed=11, chol_std=cs)
    else:
        hd, wd, nelec = problem(wt, norb, nelec, nchol)
    chol = np.array(hd["chol"]).reshape(-1, norb, norb)
    skew = np.random.default_rng(5).uniform(-1.0, 1.0, (norb, norb))
    chol += asym * np.max(np.abs(chol)) * np.triu(skew, 1)[None]
    hd = dict(hd, chol=chol.reshape(np.shape(hd["chol"])))
    if wt == "spin":
        trial, prop = spin_wavefunctions.uhf(norb, nelec), spin_propagation.propagator_unrestricted(
            DT, W, precision="fp64")
        ham = hamiltonian.hamiltonian(norb)
        hdat = ham.build_measurement_intermediates(hd, trial, wd)
        hdat = ham.build_propagation_intermediates(hdat, prop, trial, wd)
    else:
        trial, prop, hdat, _, _ = make(wt, norb, nelec, nchol, W, hd, wd)
    dev = hdat["_afqmc_device"]
    assert dev.vhs_entries() == (norb * norb if asym else norb * (norb + 1) // 2)
    assert dev.step_in_one_launch() == one
    if not one:
        return
    rng = np.random.default_rng(3)
    walkers = problems.random_walkers("rhf" if wt == "rhf" else "uhf", norb, nelec, W, rng,
                                      near=wd["mo_coeff"], noise=0.1)
    fields = to_dev(rng.standard_normal((3, W, nchol)), gpu)
    got = []
    for timed in (False, True):
        dev.prof_enable(timed)
        w = to_dev(walkers, gpu)
        weights = torch.ones(W, dtype=torch.float64, device=gpu)
        overlaps = dev.overlap(w)
        scalars = torch.tensor([-0.5, -0.5], dtype=torch.float64, device=gpu)
        for s in range(3):
            dev.propagate(w, weights, overlaps, fields[s], scalars, reuse_green=s > 0,
                          keep_green=s < 2)
        got.append((w, weights, overlaps, scalars))
    dev.prof_enable(False)
    assert float(got[1][1].sum()) > 0.0
    for a, b in zip(*got):
        b = [x.cpu().numpy() for x in b] if isinstance(b, list) else b.cpu().numpy()
        assert rel(a, b) < TOL


@pytest.mark.parametrize("precision,tol", [("fp64", TOL), ("fp32", 2e-5), ("bf16x3", 1e-4)])
@pytest.mark.parametrize("norb,n,nchol,W", [(115, 9, 37, 850), (115, 9, 32, 896)])
def test_step_with_128_wide_gemm_tiles(gpu, norb, n, nchol, W, precision, tol):
    """V from 128-wide GEMM tiles with partly filled last tiles in all three directions (and
    with whole ones in rows and k), the first and last walkers against the oracle.  The
    bounds of the reduced precisions are those their steps are held to elsewhere."""
    print(f"128-wide tiles N={norb} n={n} G={nchol} W={W} {precision}", flush=True)
    hd, wd, nelec = problem("rhf", norb, (n, n), nchol)
    trial, prop, hdat, wave, oh = make("rhf", norb, nelec, nchol, W, hd, wd, precision)
    assert hdat["_afqmc_device"].vhs_gemm_tile() == 128
    rng = np.random.default_rng(3)
    walkers = problems.random_walkers("rhf", norb, nelec, W, rng, near=wd["mo_coeff"], noise=0.1)
    fields = rng.standard_normal((W, nchol))
    pd = {"walkers": to_dev(walkers, gpu),
          "weights": torch.ones(W, dtype=torch.float64, device=gpu),
          "e_estimate": torch.tensor(-0.5, dtype=torch.float64, device=gpu),
          "pop_control_ene_shift": torch.tensor(-0.5, dtype=torch.float64, device=gpu)}
    pd["overlaps"] = trial.calc_overlap(pd["walkers"], wave)
    pd = prop.propagate(trial, hdat, pd, to_dev(fields, gpu), wave)
    some = np.r_[0:4, 60:68, W - 40:W]  # walkers do not depend on one another
    od = {"walkers": walkers[some], "weights": np.ones(len(some)), "e_estimate": -0.5,
          "overlaps": o.calc_overlap("rhf", walkers[some], wd), "pop_control_ene_shift": -0.5}
    od = o.propagate("rhf", "rhf", oh, od, fields[some], wd, DT, 6, norb)
    for name in ("walkers", "overlaps", "weights"):
        assert rel(pd[name][torch.as_tensor(some, device=gpu)], od[name]) < tol


@pytest.mark.parametrize("precision,tol", [("fp64", TOL), ("fp32", 2e-5), ("bf16x3", 1e-4)])
@pytest.mark.parametrize("norb,nelec,nchol,W", [(4, (1, 1), 150, 131), (7, (2, 1), 140, 70),
                                                (9, (4, 3), 53, 41), (12, (7, 5), 40, 65)])
def test_energy_of_few_electrons(gpu, norb, nelec, nchol, W, precision, tol):
    """Exchange tiles of more than eight walkers, whose sums add up over the passes, with
    partly filled last groups of eight."""
    print(f"exchange N={norb} nelec={nelec} G={nchol} W={W} {precision}", flush=True)
    hd, wd, nelec = problem("uhf", norb, nelec, nchol)
    trial, prop, hdat, wave, oh = make("uhf", norb, nelec, nchol, W, hd, wd, precision)
    walkers = problems.random_walkers("uhf", norb, nelec, W, np.random.default_rng(3),
                                      near=wd["mo_coeff"], noise=0.1)
    got = trial.calc_energy(to_dev(walkers, gpu), hdat, wave)
    assert rel(got, o.calc_energy("uhf", walkers, oh, wd)) < tol
