"""What a user of the sampler has it do, as measurable cases.

A case is one pass of a program through the public entry points (the Carlo
plugin mirror, DeviceSampler, MixedBatch, GradientSampler) on a Kagome
cluster of 3 L^2 sites: pi-flux orbitals (real), or orbitals at a flux phase
or ansatz parameters drawn with the seed (complex).  Kinds:

  chain    montecarlo.run on few walkers (the reference's job script)
  step     n_occupied sweeps of every walker, then their local energies
  eloc     the local energies alone, of walkers in the middle of a run
  restore  configurations from the host (a checkpoint), W rebuilt, energies
  grad     n_occupied sweeps, then energies and log-derivatives
  mixed    one step of five cluster sizes at once (one graph launch)

Every pass continues the walkers' chains, as in a run; except for `chain`,
`prepare` first takes the walkers from their random starts through THERM
intervals.  `exact` replays the chains from the documented start and draw rules
in 64 bits with torch.  It has no value for chains of float W: one near tie
decided differently makes another chain.
"""
import functools
import math
import os
import random
import sys
import warnings

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "kagomedsl.jl_amd"))

from kagome_vmc import montecarlo  # noqa: E402
from kagome_vmc import _native as nat  # noqa: E402
from kagome_vmc.batch import MixedBatch, flux_cluster  # noqa: E402
from kagome_vmc.gradient import GradientSampler, THETA0, ansatz_family, orbital_derivatives  # noqa: E402
from kagome_vmc.hamiltonian import Hamiltonian  # noqa: E402
from kagome_vmc.lattice import DoubleKagome  # noqa: E402

# boundary conditions that close the shell at half filling
BC = {4: (False, True), 6: (False, False), 8: (False, True), 10: (False, False), 12: (False, True)}
MIXED_L = (4, 6, 8, 10, 12)
MIXED_SHARE = (4, 2, 2, 1, 1)            # walkers per size, in units of the case's walkers
PREC = {"fp64": nat.PREC_FP64, "fp32": nat.PREC_FP32}
POLICY = {"reference": nat.REFRESH_REFERENCE, "every_k": nat.REFRESH_EVERY_K, "at_end": nat.REFRESH_AT_END}
KERNEL = {"reference": nat.KERNEL_REFERENCE, "unbiased": nat.KERNEL_UNBIASED}

THERM = 3               # measurement intervals between a random start and the first pass
SETTLE, SETTLE_EACH = 3, 8   # FP64: first, W is rebuilt so many times, after so many sweeps each

# the four counters of a sweep call that follow from the chains (the library
# also counts its own launches and flushes)
COUNTERS = ("sweeps", "moves", "accepted", "refreshes")


def _case(kind, L, walkers, n_up=0, flux=False, prec="fp64", policy="reference", k=0, delay=1, kernel="reference",
          graph=False, intervals=1):
    """n_up 0: half filling; k: accepted moves per refresh of the every_k and
    at_end policies; delay: pending rank-1 terms; intervals: measurements per
    pass of a chain."""
    return {"kind": kind, "L": L, "walkers": walkers, "n_up": n_up, "flux": flux, "prec": prec, "policy": policy,
            "k": k, "delay": delay, "kernel": kernel, "graph": graph, "intervals": intervals}


def listed():
    return [
        # the reference's job script: one chain of the 48-site cluster in
        # FP64, ten measurements; every call is launch latency
        dict(_case("chain", 4, 1, intervals=10), name="chain_L4_fp64_1walker"),
        # a spin-imbalanced cluster and a ragged batch, default options
        dict(_case("step", 6, 777, n_up=57), name="step_L6_fp64_777walkers_57up"),
        # a wide batch of the smallest cluster, float W and delayed updates
        dict(_case("step", 4, 4096, prec="fp32", policy="every_k", k=64, delay=12),
             name="step_L4_fp32_4096walkers_k64"),
        # the FP64 sampler with the reference's refresh cadence, mid size
        dict(_case("step", 8, 4096), name="step_L8_fp64_4096walkers"),
        # the same at the largest cluster: the precision reference of a run
        dict(_case("step", 12, 8192), name="step_L12_fp64_8192walkers"),
        # production sampling: float W, rare refreshes
        dict(_case("step", 12, 8192, prec="fp32", policy="every_k", k=216, delay=12),
             name="step_L12_fp32_8192walkers_k216"),
        # the same with W rebuilt often, for a tight bound on its drift
        dict(_case("step", 12, 8192, prec="fp32", policy="every_k", k=16, delay=12),
             name="step_L12_fp32_8192walkers_k16"),
        # measurement alone: more than one quantity per interval, or a rerun
        dict(_case("eloc", 12, 8192, prec="fp32", policy="every_k", k=216, delay=12), name="eloc_L12_fp32_8192walkers"),
        # resuming from a checkpoint: kappa from the host, W by LU
        dict(_case("restore", 10, 1500), name="restore_L10_fp64_1500walkers"),
        # variational optimisation away from the pi-flux point: complex W
        dict(_case("grad", 8, 2048, flux=True, kernel="unbiased"), name="grad_L8_fp64_2048walkers_flux"),
        # the same at the pi-flux point, large cluster, with the float sampler
        dict(_case("grad", 12, 1000, prec="fp32", kernel="unbiased", delay=8), name="grad_L12_fp32_1000walkers"),
        # finite-size scaling in one job: five sizes, a flux phase for each
        dict(_case("mixed", 12, 1024, flux=True, prec="fp32", policy="every_k", k=64, delay=8, graph=True),
             name="mixed_L4to12_fp32_1024walkers_k64"),
    ]


def _sites(L):
    return 3 * L * L


def _fillings(case, L):
    n = case["n_up"] or _sites(L) // 2
    return n, _sites(L) - n


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any kind and size, walkers over the logarithm of their
    range (odd counts among them), the options in earnest use."""
    kind = rng.choice(["step"] * 6 + ["chain", "eloc", "restore", "grad", "grad", "mixed"])
    L = rng.choice(list(BC))
    n = _sites(L) // 2
    prec = rng.choice(["fp64", "fp32"])
    if kind == "chain":
        return _case("chain", L, rng.choice([1, 1, 2, 3, 7, 16]), prec=prec, delay=1 if prec == "fp64" else 8,
                     intervals=rng.randint(2, 10))
    if kind == "mixed":
        return _case("mixed", 12, _log_int(rng, 16, 1024), flux=True, prec="fp32", policy="every_k",
                     k=rng.choice([64, 216]), delay=rng.choice([4, 8, 12]), graph=rng.random() < 0.7)
    if kind == "grad":
        hi = {4: 8192, 6: 4096, 8: 2048, 10: 1024, 12: 1000}[L]
        flux = rng.random() < 0.5
        return _case("grad", L, _log_int(rng, 16, hi), flux=flux, prec="fp64" if flux else prec, kernel="unbiased",
                     delay=1 if prec == "fp64" else rng.choice([4, 8]))
    # complex W costs up to eight times the refresh of a real one
    flux = rng.random() < (0.25 if kind == "step" else 0.15)
    walkers = _log_int(rng, 16, 1024 if flux else 8192)
    policy = rng.choice(["reference", "every_k", "every_k", "at_end"])
    k = 0 if policy == "reference" else rng.choice([16, 64, n])
    delay = rng.choice([1, 4, 8]) if prec == "fp64" else rng.choice([4, 8, 12, 16])
    n_up = n + rng.choice([0, 0, 0, 1, 2, 3, 5]) if not flux else 0
    return _case(kind, L, walkers, n_up=0 if n_up == n else n_up, flux=flux, prec=prec, policy=policy, k=k,
                 delay=delay, kernel=rng.choice(["reference", "reference", "unbiased"]),
                 graph=kind == "step" and rng.random() < 0.2)


# --- inputs ------------------------------------------------------------------


@functools.lru_cache(maxsize=None)
def _lattice(L):
    return DoubleKagome.build(1.0, L, L, (True, True), BC[L])


@functools.lru_cache(maxsize=None)
def _pi_flux(L, n_up):
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")   # an open shell at an odd filling
        return Hamiltonian.build(n_up, _sites(L) - n_up, _lattice(L))


# flux phases at which enough uniform starts of float handles are far from
# singular (beyond, a start of the largest cluster may need over 64 draws)
PHI = (0.1, 1.2)


def _phases(case, seed):
    rng = random.Random("phase %d" % seed)
    return [rng.uniform(*PHI) for _ in MIXED_L]


def _cluster(case, seed, L):
    """The pi-flux cluster, or the one at a flux phase drawn with the seed."""
    if case["flux"]:
        return flux_cluster(L, _phases(case, seed)[MIXED_L.index(L)])
    return _pi_flux(L, _fillings(case, L)[0])


@functools.lru_cache(maxsize=None)
def _family(L):
    return ansatz_family(_lattice(L))


def _theta(case, seed):
    """(phi, ratio, m, t2): the pi-flux point, or parameters of an optimisation under way."""
    if not case["flux"]:
        return THETA0.copy()
    rng = random.Random("theta %d" % seed)
    return np.array([rng.uniform(*PHI), rng.uniform(0.8, 1.2), rng.uniform(0.0, 0.2),
                     rng.uniform(-0.1, 0.1)])


def _sampler(case, ham, seed):
    return nat.DeviceSampler(ham.bonds_array(), ham.U_up, ham.U_down, case["walkers"], precision=PREC[case["prec"]],
                             kernel=KERNEL[case["kernel"]], refresh_policy=POLICY[case["policy"]],
                             refresh_k=case["k"], delay=case["delay"], seed=seed)


def _thermalise(case, ds, n):
    """A random start can be nearly singular, and what its W has lost stays
    until W is rebuilt.  Float handles redraw such starts."""
    if case["prec"] == "fp64":
        for _ in range(SETTLE):
            ds.sweep(SETTLE_EACH)
            ds.refresh()
    for _ in range(THERM):
        ds.sweep(n)


def prepare(case, seed):
    """The program's handle with walkers at seeded starts.  Refresh phases are
    spread as in a long run where the policy counts accepted moves."""
    kind, L = case["kind"], case["L"]
    if kind == "chain":
        up, dn = _fillings(case, L)
        mc = montecarlo.MC({"n1": L, "n2": L, "PBC": (True, True), "antiPBC": BC[L], "N_up": up, "N_down": dn,
                            "nwalkers": case["walkers"], "precision": case["prec"], "delay": case["delay"],
                            "kernel": case["kernel"], "seed": seed})
        ctx = montecarlo.MCContext(seed=seed)
        montecarlo.init(mc, ctx)
        return {"case": case, "mc": mc, "ctx": ctx}
    if kind == "grad":
        up, dn = _fillings(case, L)
        gs = GradientSampler(_family(L), _theta(case, seed), up, dn, case["walkers"], seed=seed,
                             precision=PREC[case["prec"]], delay=case["delay"])
        gs.sampler.init_random(seed)
        _thermalise(case, gs.sampler, min(up, dn))
        return {"case": case, "ds": gs.sampler, "sweeps": min(up, dn)}
    if kind == "mixed":
        mb = MixedBatch([(_cluster(case, seed, l), m * case["walkers"]) for l, m in zip(MIXED_L, MIXED_SHARE)],
                        graph=case["graph"], precision=PREC[case["prec"]], kernel=KERNEL[case["kernel"]],
                        refresh_policy=POLICY[case["policy"]], refresh_k=case["k"], delay=case["delay"], seed=seed)
        mb.init_random(seed)
        for g in mb.groups:
            g.sampler.stagger_refresh(seed)
        mb.step(THERM)
        return {"case": case, "batch": mb}
    ham = _cluster(case, seed, L)
    ds = _sampler(case, ham, seed)
    ds.init_random(seed)
    state = {"case": case, "ds": ds, "sweeps": min(ham.N_up, ham.N_down)}
    ds.stagger_refresh(seed)
    if case["graph"]:
        ds.enable_graph(True)
    _thermalise(case, ds, state["sweeps"])
    if kind == "restore":
        state["kappa"] = ds.get_configs()
    return state


# --- the measured pass --------------------------------------------------------


def _kept(counters):
    return {k: counters[k] for k in COUNTERS}


def run(state):
    kind = state["case"]["kind"]
    if kind == "chain":
        mc, ctx = state["mc"], state["ctx"]
        ctx.observables = {}
        montecarlo.run(mc, ctx, state["case"]["intervals"] * mc.n_occupied)
        return {"OL": np.stack(ctx.observables["OL"]), "acc": np.array(ctx.observables["acc"])}
    if kind == "mixed":
        return [{"counters": _kept(cnt), "eloc": energies[0]} for cnt, energies in state["batch"].step(1)]
    ds = state["ds"]
    if kind == "restore":
        ds.set_configs(*state["kappa"])
        eloc, nap = ds.measure()
        return {"eloc": eloc, "nap": nap, "logdet": ds.logdet()}
    if kind == "eloc":
        eloc, nap = ds.measure()
        return {"eloc": eloc, "nap": nap}
    cnt, _ = ds.sweep(state["sweeps"])
    if kind == "grad":
        eloc, O = ds.measure_grad()
        return {"counters": _kept(cnt), "eloc": eloc, "O": O}
    eloc, nap = ds.measure()
    return {"counters": _kept(cnt), "eloc": eloc, "nap": nap}


# --- what a pass cannot do without ---------------------------------------------


def _work_one(case, L, walkers):
    """One cluster size.  W (the rows of the empty sites; the others are unit
    rows) is read and written once by a pass that moves electrons and written
    once by one that rebuilds it; a local energy reads two elements per
    antiparallel bond."""
    up, dn = _fillings(case, L)
    ns, kind = _sites(L), case["kind"]
    cplx = case["flux"] or kind == "grad"                   # the flux derivative is complex everywhere
    s = (8 if case["prec"] == "fp64" else 4) * (2 if cplx else 1)
    mul = 8 if cplx else 2                                  # operations of a multiply-add
    sweeps = min(up, dn) * case["intervals"]
    rows = 2 * up * dn                                      # elements of W, both spins
    refresh = sum(mul * (n**3 / 3 + (ns - n) * n * n) for n in (up, dn))
    accepts, passing = 0.13 * sweeps, 0.4                   # per walker; sweeps past both early returns
    nap = 1.25 * ns
    if kind == "eloc":
        return walkers * (8 * ns + 2 * s * nap), walkers * mul * nap
    if kind == "restore":
        return walkers * (8 * ns + s * rows), walkers * (refresh + mul * nap)
    refreshes = passing * case["intervals"] if case["policy"] == "reference" else accepts / case["k"]
    flops = accepts * mul * rows + refreshes * refresh + mul * nap * case["intervals"]
    nbytes = 2 * s * rows + 16 * ns + 2 * s * nap * case["intervals"]
    if kind == "grad":
        flops += 4 * mul * rows
        nbytes += s * rows
    return walkers * nbytes, walkers * flops


def work(case):
    sizes = zip(MIXED_L, MIXED_SHARE) if case["kind"] == "mixed" else [(case["L"], 1)]
    parts = [_work_one(case, L, m * case["walkers"]) for L, m in sizes]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


# --- the same in 64 bits ---------------------------------------------------------


def _philox(c0, c1, c2, c3, key):
    """Philox4x32-10 (Salmon et al., SC'11) over arrays of counters."""
    m32 = np.uint64(0xFFFFFFFF)
    c = [np.asarray(x, dtype=np.uint64) & m32 for x in np.broadcast_arrays(c0, c1, c2, c3)]
    k0, k1 = key & 0xFFFFFFFF, (key >> 32) & 0xFFFFFFFF
    for r in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & m32,
             (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & m32]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return c


def _draw_configs(seed, walkers, attempt, ns, n_up):
    """Seeded permutations of the sites (Fisher-Yates, one Philox stream per
    walker and attempt); the first n_up sites hold the up electrons."""
    perm = np.tile(np.arange(ns), (len(walkers), 1))
    at = np.arange(len(walkers))
    words = []
    for q, i in enumerate(range(ns - 1, 0, -1)):
        if q % 4 == 0:
            words = _philox(np.full(len(walkers), q // 4), attempt, walkers, 1, seed)
        j = ((words[q % 4] * np.uint64(i + 1)) >> np.uint64(32)).astype(np.int64)
        pi = perm[:, i].copy()
        perm[:, i] = perm[at, j]
        perm[at, j] = pi
    return perm[:, :n_up], perm[:, n_up:]


BATCH = 512   # walkers eliminated at a time


def _eliminate(A, invert=False):
    """Gaussian elimination with row pivoting of a batch of square matrices
    (Gauss-Jordan where the inverse is wanted): the inverses or None, and the
    pivots' moduli."""
    A = A.clone()
    B, N = A.shape[0], A.shape[1]
    at, pivots = torch.arange(B, device=A.device), []
    perm = torch.arange(N, device=A.device).repeat(B, 1)
    for k in range(N):
        p = A[:, k:, k].abs().argmax(1) + k
        row, order = A[at, p].clone(), perm[at, p].clone()
        A[at, p], perm[at, p] = A[:, k].clone(), perm[:, k].clone()
        perm[:, k] = order
        piv = row[:, k].clone()
        pivots.append(piv.abs())
        if not invert:
            A[:, k + 1:, k + 1:] -= (A[:, k + 1:, k] / piv[:, None])[:, :, None] * row[:, None, k + 1:]
            continue
        row = row / piv[:, None]
        row[:, k] = 1 / piv
        col = A[:, :, k].clone()
        col[:, k] = 0
        A[:, :, k] = 0
        A -= col[:, :, None] * row[:, None, :]
        A[:, k] = row
    if not invert:
        return None, torch.stack(pivots, 1)
    out = torch.empty_like(A)
    out.scatter_(2, perm[:, None, :].expand(-1, N, -1), A)
    return out, torch.stack(pivots, 1)


class _Walkers:
    """Every walker's chain in 64 bits: sites of the labels, W = U tildeU^-1."""

    def __init__(self, bonds, U_up, U_dn, walkers, start_seed, prec, dev):
        cplx = np.iscomplexobj(U_up) or np.iscomplexobj(U_dn)
        self.dev, self.nw, self.ns = dev, walkers, U_up.shape[0]
        self.bonds = torch.as_tensor(np.asarray(bonds, dtype=np.int64) - 1, device=dev)
        self.U = [torch.as_tensor(np.ascontiguousarray(u),
                                  dtype=torch.complex128 if cplx else torch.float64, device=dev) for u in (U_up, U_dn)]
        self.cplx = cplx
        tol = 1e-4 if prec == "fp32" else 1e-10
        sites = [torch.zeros((walkers, u.shape[1]), dtype=torch.int64, device=dev) for u in self.U]
        bad, attempt = np.arange(walkers), 0
        while len(bad) and attempt < 64:
            new = _draw_configs(start_seed, bad, attempt, self.ns, U_up.shape[1])
            ok = torch.ones(len(bad), dtype=torch.bool, device=dev)
            for spin in (0, 1):
                at = torch.as_tensor(new[spin], device=dev)
                sites[spin][torch.as_tensor(bad, device=dev)] = at
                ok &= self._pivots_fine(self.U[spin], at, tol)
            bad, attempt = bad[~ok.cpu().numpy()], attempt + 1
        self.sites = sites
        self.rebuild()
        w = torch.arange(walkers, device=dev)[:, None]
        self.kap = []                       # label + 1 of the electron at a site, 0: none
        for spin in (0, 1):
            k = torch.zeros((walkers, self.ns), dtype=torch.int64, device=dev)
            k[w, sites[spin]] = torch.arange(sites[spin].shape[1], device=dev)[None, :] + 1
            self.kap.append(k)
        self.sweeps = 0

    def _pivots_fine(self, U, sites, tol):
        """The spread of the pivots (of the real form, where U is complex)."""
        ok = []
        for a in range(0, len(sites), BATCH):
            t = U[sites[a:a + BATCH]]
            if self.cplx:
                t = torch.cat([torch.cat([t.real, -t.imag], 2), torch.cat([t.imag, t.real], 2)], 1)
            piv = _eliminate(t)[1]
            ok.append(piv.min(1)[0] >= tol * piv.max(1)[0])
        return torch.cat(ok)

    def rebuild(self):
        self.W = []
        for U, sites in zip(self.U, self.sites):
            W = torch.empty((self.nw, *U.shape), dtype=U.dtype, device=self.dev)
            for a in range(0, self.nw, BATCH):
                W[a:a + BATCH] = U @ _eliminate(U[sites[a:a + BATCH]], invert=True)[0]
            self.W.append(W)

    def _antiparallel(self):
        i, j = self.bonds[:, 0], self.bonds[:, 1]
        up, dn = self.kap[0] != 0, self.kap[1] != 0
        return (up[:, i] & dn[:, j]) | (up[:, j] & dn[:, i])

    def sweep(self, n, seed, kernel):
        """n exchange proposals on every walker: uniform u and bond from
        Philox keyed by the seed at (sweep, walker)."""
        nb, at = len(self.bonds), torch.arange(self.nw, device=self.dev)
        accepted = torch.zeros(n, dtype=torch.int64, device=self.dev)
        for t in range(n):
            x = _philox(self.sweeps & 0xFFFFFFFF, self.sweeps >> 32, np.arange(self.nw), 0, seed)
            u = ((x[0] >> np.uint64(5)).astype(np.float64) * 67108864.0 +
                 (x[1] >> np.uint64(6)).astype(np.float64)) / 9007199254740992.0
            u = torch.as_tensor(u, device=self.dev)
            b = torch.as_tensor(((x[2] * np.uint64(nb)) >> np.uint64(32)).astype(np.int64), device=self.dev)
            i, j = self.bonds[b, 0], self.bonds[b, 1]
            iu, ju, idn, jd = self.kap[0][at, i], self.kap[0][at, j], self.kap[1][at, i], self.kap[1][at, j]
            one = (iu != 0) & (jd != 0)          # up moves i -> j, down j -> i
            two = (ju != 0) & (idn != 0)
            lu = torch.where(one, iu, ju).clamp(min=1) - 1
            ld = torch.where(one, jd, idn).clamp(min=1) - 1
            Ku, Kd = torch.where(one, j, i), torch.where(one, i, j)
            p = (self.W[0][at, Ku, lu] * self.W[1][at, Kd, ld]).abs() ** 2
            if kernel == "reference":
                zr = self._antiparallel().sum(1).double() / nb
                acc = ~(u > zr) & (((p >= 1) & (u < zr)) | ((p < 1) & (u < zr * p)))
            else:
                acc = u < p
            a = ((one | two) & acc).nonzero()[:, 0]
            accepted[t] = len(a)
            for spin, K, l, old in ((0, Ku, lu, Kd), (1, Kd, ld, Ku)):
                K, l, old = K[a], l[a], old[a]
                for c in range(0, len(a), 256):
                    q, k, m = a[c:c + 256], K[c:c + 256], l[c:c + 256]
                    n0 = torch.arange(len(q), device=self.dev)
                    W = self.W[spin][q]
                    row = W[n0, k].clone()
                    row[n0, m] -= 1
                    self.W[spin][q] = W - W[n0, :, m][:, :, None] * (row / W[n0, k, m][:, None])[:, None, :]
                self.kap[spin][a, old] = 0
                self.kap[spin][a, K] = l + 1
                self.sites[spin][a, l] = K
            self.sweeps += 1
        return accepted

    def eloc(self):
        """Heisenberg J1 local energies: +-1/4 per bond, and -1/2 times the
        two ratios of the exchange on every antiparallel bond."""
        at = torch.arange(self.nw, device=self.dev)[:, None]
        i, j = self.bonds[:, 0].expand(self.nw, -1), self.bonds[:, 1].expand(self.nw, -1)
        iu, ju, idn, jd = (self.kap[s].gather(1, x) for s, x in ((0, i), (0, j), (1, i), (1, j)))
        one, ap = (iu != 0) & (jd != 0), self._antiparallel()
        lu = torch.where(one, iu, ju).clamp(min=1) - 1
        ld = torch.where(one, jd, idn).clamp(min=1) - 1
        Ku, Kd = torch.where(one, j, i), torch.where(one, i, j)
        exch = -0.5 * self.W[0][at, Ku, lu] * self.W[1][at, Kd, ld] * ap
        diag = torch.where((iu != 0) == (ju != 0), 0.25, -0.25)
        return exch.sum(1) + diag.sum(1)

    def log_det(self):
        """log |det tildeU| of both spins."""
        out = torch.zeros(self.nw, dtype=torch.float64, device=self.dev)
        for U, s in zip(self.U, self.sites):
            for a in range(0, self.nw, BATCH):
                out[a:a + BATCH] += _eliminate(U[s[a:a + BATCH]])[1].log().sum(1)
        return out

    def log_derivs(self, dU):
        """O_k = sum over spins of tr(tildeU^-1 d tildeU / d theta_k)."""
        P = len(dU[0])
        O = torch.zeros((self.nw, P), dtype=self.W[0].dtype, device=self.dev)
        for spin in (0, 1):
            d = torch.as_tensor(np.stack(dU[spin]), device=self.dev).to(O.dtype)
            for a in range(0, self.nw, BATCH):
                s = self.sites[spin][a:a + BATCH]
                inv = _eliminate(self.U[spin][s], invert=True)[0]
                for k in range(P):
                    O[a:a + BATCH, k] += (d[k][s] * inv.transpose(1, 2)).sum((1, 2))
        return O


def _exact_one(case, ham, bonds, walkers, seed, dev):
    W = _Walkers(bonds, ham[0], ham[1], walkers, seed, case["prec"], dev)
    kind, n = case["kind"], min(ham[0].shape[1], ham[1].shape[1])
    if kind == "chain":
        acc, ol = [], []
        for _ in range(case["intervals"]):
            acc.append(int(W.sweep(n, seed, case["kernel"]).sum()) / (n * walkers))
            ol.append(W.eloc().real.cpu().numpy())
        return {"OL": np.stack(ol), "acc": np.array(acc)}
    for _ in range(SETTLE):
        W.sweep(SETTLE_EACH, seed, case["kernel"])
        W.rebuild()
    W.sweep(THERM * n, seed, case["kernel"])
    if kind == "restore":
        return {"eloc": W.eloc().real.cpu().numpy(), "nap": None, "logdet": W.log_det().cpu().numpy()}
    if kind != "eloc":
        W.sweep(n, seed, case["kernel"])
    e = W.eloc()
    if kind == "grad":
        return {"counters": None, "eloc": e.cpu().numpy(), "O": W.log_derivs(ham[2:]).cpu().numpy()}
    return {"counters": None, "eloc": e.real.cpu().numpy(), "nap": None}


def exact(case, seed):
    """None in the place of the whole numbers, which have to be the same anyway."""
    if case["prec"] == "fp32":
        return None
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    L, walkers = case["L"], case["walkers"]
    if case["kind"] == "grad":
        fam, theta = _family(L), _theta(case, seed)
        H, G = fam.hamiltonian(theta), fam.generators(theta)
        (u, du, _), (d, dd, _) = (orbital_derivatives(H, G, n) for n in _fillings(case, L))
        # derivatives in the flux phase are complex: so are the orbitals
        ham = (u + 0j, d + 0j, [x + 0j for x in du], [x + 0j for x in dd])
        return _exact_one(case, ham, fam.nn, walkers, seed, dev)
    ham = _cluster(case, seed, L)
    return _exact_one(case, (ham.U_up, ham.U_down), ham.nn, walkers, seed, dev)
