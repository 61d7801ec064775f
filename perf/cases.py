"""Performance cases of the phaseless-AFQMC library: the work its users have it do, through the public Python
entry points (vmc_amd.afqmc.Context, Batch, run_long_prop).

Every case runs on synthetic Hamiltonians of the repository's own kind (diagonal ramp plus a random symmetric
one-body part, random symmetric Cholesky vectors), with the extensive coupling sigma = 1/N for which the walk is
as quiet as a molecular one.  Kinds of case:

  walk      one block of a walk through Context: `nsteps` propagations, the re-orthonormalisation, the local
            energies and the comb, with the driver's energy-shift feedback on the host.  In FP64 the population
            walks on from block to block.  With reduced precision the block starts from the trial determinant
            (as a run or a restarted population does) and ends with the energies.
  run       a whole small run: run_long_prop with the host random stream, the library's one-call driver
  batch     one block of a captured multi-system walk: `nsteps` Batch steps over systems of uneven size
  evaluate  energies and overlaps of given determinants (ham_and_overlap): trial comparison, truncation search
  restore   a saved population loaded back (set_walkers) and its force bias and overlaps read
  surrogate the learned exchange surrogate: the gradient of one minibatch, and the prediction for a population
"""
import math

import numpy as np
import torch

from vmc_amd.abi import AFQ_ENERGY_SURROGATE, AFQ_PREC_BF16, AFQ_PREC_BF16X3, AFQ_SURR_EXCHANGE, HamArrays
from vmc_amd.afqmc import Batch, Context, run_long_prop

DT = 0.005
ORTHO = 5          # propagations between re-orthonormalisations
KEY = 20261202     # Philox key of the device's field draws
F64, C128 = torch.float64, torch.complex128


# ---------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest population the benchmark names: every call is short, launches and latency count
        walk("walk_n10", 10, 5, 5, 40, 128, "rhf"),
        # a run of a small molecule's size (13 orbitals, 5+5 electrons, 64 vectors), as `python -m vmc_amd.dqmc` does it
        dict(name="run_n13", kind="run", norb=13, nalpha=5, nbeta=5, nchol=64, nwalk=20, nranks=4, trial="rhf", blocks=5, nsteps=10),
        # an open-shell molecule with unrestricted integrals: odd sizes, unequal spins, a propagator per spin
        walk("walk_n51_unrestricted", 51, 13, 11, 205, 256, "uhf", ints="u"),
        # the medium system of the benchmark in FP64, with the one-body density matrix accumulated
        walk("walk_n100", 100, 20, 20, 400, 1024, "uhf", rdm=True),
        # the same size, odd and ragged, with the contractions in split BF16 and every energy measured on that level
        walk("walk_n101_mixed", 101, 21, 19, 405, 1000, "uhf", prec="mixed"),
        # the largest shape in FP64 (fewer walkers: the plain reference path that results are checked against)
        walk("walk_n300", 300, 60, 60, 1200, 256, "uhf"),
        # the headline: the largest shape and population, split BF16 with the control-variate energies
        walk("walk_n300_mixed", 300, 60, 60, 1200, 4096, "uhf", prec="mixed", energy="cv"),
        # many systems of uneven size advanced by one captured step
        dict(name="batch_24", kind="batch", nsys=24, nmin=20, nmax=120, nwalk=256, nsteps=5),
        # a handful of determinants evaluated on the medium system, all vectors in the energy
        dict(name="evaluate_n100", kind="evaluate", norb=100, nalpha=20, nbeta=20, nchol=400, ndet=16, trial="uhf", keep=1.0),
        # a checkpointed population of the medium system loaded back
        dict(name="restore_n100", kind="restore", norb=100, nalpha=20, nbeta=20, nchol=400, nwalk=512, trial="uhf"),
        # the learned surrogate on the medium system: one large minibatch's gradient and a prediction for the population
        dict(name="surrogate_n100", kind="surrogate", norb=100, nalpha=20, nbeta=20, nchol=400, nwalk=1024, trial="uhf", hidden=256, rows=4096),
    ]


def walk(name, norb, nalpha, nbeta, nchol, nwalk, trial, ints="r", prec="fp64", energy="exact", rdm=False, nsteps=5):
    return dict(name=name, kind="walk", norb=norb, nalpha=nalpha, nbeta=nbeta, nchol=nchol, nwalk=nwalk, trial=trial, ints=ints,
                prec=prec, energy=energy, rdm=rdm, nsteps=nsteps)


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def system(lo, hi, same=None):
        norb = spread(lo, hi)
        nalpha = max(2, min(64, int(norb * rng.uniform(0.15, 0.45))))
        nbeta = nalpha if same or rng.random() < 0.4 else max(1, nalpha - rng.randint(1, 3))
        return dict(norb=norb, nalpha=nalpha, nbeta=nbeta, nchol=max(8, int(norb * rng.uniform(2.5, 5.0))))

    kind = rng.choice(["walk", "walk", "walk", "walk", "walk", "run", "batch", "evaluate", "restore", "surrogate"])
    if kind == "walk":
        prec = rng.choice(["fp64", "fp64", "mixed"])
        rhf = rng.random() < 0.3
        s = system(8, 240 if prec == "mixed" else 160, same=rhf)
        # the population shrinks with the system, as memory and time make it in use
        nwalk = max(16, min(4096, int(spread(64, 4096) * min(1.0, (60.0 / s["norb"]) ** 2))))
        c = walk("", nwalk=nwalk, trial="rhf" if rhf else "uhf", prec=prec, nsteps=rng.choice([1, 2, 5]), **s)
        if prec == "mixed":
            c["energy"] = rng.choice(["exact", "cv"])
        elif not rhf and rng.random() < 0.25:
            c["ints"] = "u"
        elif rng.random() < 0.3:
            c["rdm"] = True
        del c["name"]
        return c
    if kind == "run":
        return dict(kind="run", nwalk=spread(5, 100), nranks=rng.choice([1, 2, 4]), trial=rng.choice(["rhf", "uhf"]), blocks=rng.randint(3, 6),
                    nsteps=rng.choice([5, 10]), **system(8, 40, same=True))
    if kind == "batch":
        return dict(kind="batch", nsys=rng.randint(3, 24), nmin=rng.randint(10, 30), nmax=rng.randint(40, 100), nwalk=spread(16, 256), nsteps=5)
    if kind == "evaluate":
        return dict(kind="evaluate", ndet=spread(1, 64), trial="uhf", keep=rng.choice([0.3, 0.5, 0.7, 1.0]), **system(10, 160))
    if kind == "restore":
        return dict(kind="restore", nwalk=spread(16, 512), trial="uhf", **system(10, 120))
    return dict(kind="surrogate", nwalk=spread(64, 1024), trial="uhf", hidden=rng.choice([64, 128, 256]), rows=spread(64, 1024), **system(10, 100, same=True))


# ---------------------------------------------------------------------------------------------- inputs
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _generator(seed, stream):
    g = torch.Generator(device=_device())
    g.manual_seed((int(seed) * 1000003 + stream) & 0x7FFFFFFFFFFFFFFF)
    return g


def _vectors(norb, nchol, gen):
    L = torch.randn(nchol, norb, norb, generator=gen, device=_device(), dtype=F64) / norb
    return torch.tril(L) + torch.tril(L, -1).transpose(1, 2)


def _one_body(norb, gen):
    a = torch.randn(norb, norb, generator=gen, device=_device(), dtype=F64)
    return 0.5 * (a + a.T) / norb + torch.diag(torch.linspace(-2.0, 0.0, norb, device=_device(), dtype=F64))


def _square(L):
    """sum_g L_g L_g for symmetric L_g."""
    m = L.reshape(-1, L.shape[-1])
    return m.T @ m


def _lowest(fock, n):
    return torch.from_numpy(np.ascontiguousarray(np.linalg.eigh(fock.cpu().numpy())[1][:, :n])).to(fock.device)


def _mean_field(hs, Ls, ns, spins):
    """Orbitals of a few self-consistent mean-field iterations from the core guess (spins: 1 closed shell, 2 open)."""
    cs = [_lowest(hs[s], ns[s]) for s in range(spins)]
    for _ in range(4):
        js, ks = [], []
        for s in range(spins):
            g, n = Ls[s].shape[0], Ls[s].shape[1]
            js.append(torch.einsum("gij,ij->g", Ls[s], cs[s] @ cs[s].T))
            lc = (Ls[s].reshape(g * n, n) @ cs[s]).reshape(g, n, -1).transpose(0, 1).reshape(n, -1)
            ks.append(lc @ lc.T)
        tot = js[0] + js[1] if spins == 2 else 2.0 * js[0]
        cs = [_lowest(hs[s] + torch.einsum("g,gij->ij", tot, Ls[s]) - ks[s], ns[s]) for s in range(spins)]
    return cs


def _hamiltonian(case, seed, stream=0):
    """The system's tensors: h and L per spin (one entry with restricted integrals), trial orbitals per spin."""
    n, na, nb, g = case["norb"], case["nalpha"], case["nbeta"], case["nchol"]
    gen = _generator(seed, stream)
    Ls = [_vectors(n, g, gen)]
    hs = [_one_body(n, gen)]
    if case.get("ints") == "u":   # the down spin's integrals: the up spin's, slightly changed
        Ls.append(Ls[0] + 0.1 * _vectors(n, g, gen))
        hs.append(hs[0] + 0.05 * _one_body(n, gen))
    rhf = case["trial"] == "rhf"
    two = [hs[0], hs[-1]], [Ls[0], Ls[-1]]
    cs = _mean_field(*two, [na, nb], 1 if rhf else 2)
    phi = [cs[0], cs[0][:, :nb] if rhf else cs[1]]
    return dict(h=hs, L=Ls, phi=phi, rhf=rhf)


def _arrays(case, sys):
    """The host arrays a program hands to the library."""
    def host(x):
        return x.cpu().numpy()

    mod = [h - 0.5 * _square(L) for h, L in zip(sys["h"], sys["L"])]
    more = {}
    if len(sys["h"]) == 2:
        more = dict(h1_dn=host(sys["h"][1]), h1_mod_dn=host(mod[1]), chol_dn=host(sys["L"][1]))
    return HamArrays(case["norb"], case["nalpha"], case["nbeta"], 0.0, host(sys["h"][0]), host(mod[0]), host(sys["L"][0]),
                     host(sys["phi"][0]), host(sys["phi"][1]), trial_rhf=sys["rhf"], **more)


def _start(case, seed, phi, stream=1):
    """The determinant a walk starts from: the trial with its orbitals slightly rotated, so that overlaps are not one."""
    gen = _generator(seed, stream)
    out = []
    for s, p in enumerate(phi):
        if s == 1 and case["trial"] == "rhf":
            out.append(out[0])
            break
        out.append(p + 0.02 * torch.randn(p.shape, generator=gen, device=p.device, dtype=F64) / math.sqrt(p.shape[0]))
    return out


def _determinants(case, seed, phi, count, stream=2):
    """Walkers met in the middle of a walk: the trial plus complex noise, one determinant per row (serial layout)."""
    gen = _generator(seed, stream)
    parts = []
    for p in phi:
        z = torch.randn(count, *p.shape, 2, generator=gen, device=p.device, dtype=F64)
        parts.append((p + 0.3 / math.sqrt(p.shape[0]) * torch.view_as_complex(z)).reshape(count, -1))
    return torch.cat(parts, dim=1)


def _uniforms(seed, count, stream=3):
    return np.random.default_rng([int(seed), stream]).uniform(size=count)


def _batch_cases(case, seed):
    rng = np.random.default_rng([int(seed), 4])
    sizes = rng.integers(case["nmin"], case["nmax"] + 1, size=case["nsys"])
    return [dict(norb=int(n), nalpha=max(1, round(int(n) / 5)), nbeta=max(1, round(int(n) / 5)), nchol=4 * int(n), trial="uhf", nwalk=case["nwalk"])
            for n in sizes]


def _mlp_rows(case, seed):
    """Network inputs and (standardised) targets of one minibatch."""
    rng = np.random.default_rng([int(seed), 5])
    width = case["nchol"] + 2 * case["norb"]
    x = rng.standard_normal((case["rows"], width)).astype(np.float32)
    return x, (x[:, :7].sum(axis=1) / 3 + 0.2 * rng.standard_normal(case["rows"])).astype(np.float32)


def _mlp_params(case, seed):
    """Weights and biases of a network part-way through training, then the input's and the target's mean and deviation."""
    rng = np.random.default_rng([int(seed), 6])
    width, hidden = case["nchol"] + 2 * case["norb"], case["hidden"]
    dims = [width, hidden, hidden, hidden, 1]
    parts = []
    for a, b in zip(dims, dims[1:]):
        parts += [rng.standard_normal(a * b) / math.sqrt(a), 0.1 * rng.standard_normal(b)]
    parts += [np.zeros(width), np.ones(width), [0.0], [1.0]]
    return dims, np.concatenate(parts).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        members = _batch_cases(case, seed)
        systems = [_hamiltonian(m, seed, 10 + i) for i, m in enumerate(members)]
        hams = [_arrays(m, s) for m, s in zip(members, systems)]
        batch = Batch(hams, False, case["nwalk"])
        guess = []
        for i, (ctx, h, m, s) in enumerate(zip(batch.ctx, hams, members, systems)):
            up, dn = (x.cpu().numpy() for x in _start(m, seed, s["phi"], 100 + i))
            ctx.prep_prop(h.phi_up, h.phi_dn, DT)
            ctx.set_walkers_uniform(h.serial_det(up, dn))
            guess.append(float(ctx.measure(want_ho=False)[0]))
        batch.capture(KEY, ORTHO, math.sqrt(2.0 / DT), first_step=1)
        return dict(kind=kind, batch=batch, step=0, nwalk=case["nwalk"], nsteps=case["nsteps"], estimate=np.array(guess), shift=np.array(guess),
                    uniforms=_uniforms(seed, (64, len(hams))))
    sys = _hamiltonian(case, seed)
    ham = _arrays(case, sys)
    start = [x.cpu().numpy() for x in _start(case, seed, sys["phi"])]
    if kind == "run":
        return dict(kind=kind, ham=ham, start=start, case=case)
    rhf = case["trial"] == "rhf"
    ctx = Context(ham, case.get("nwalk", 1), rhf)
    state = dict(kind=kind, ctx=ctx, case=case)
    if kind == "evaluate":
        state.update(dets=_determinants(case, seed, sys["phi"], case["ndet"]).cpu().numpy(), keep=int(case["keep"] * case["nchol"]))
        return state
    if kind == "restore":
        rng = np.random.default_rng([int(seed), 7])
        state.update(dets=_determinants(case, seed, sys["phi"], case["nwalk"]).cpu().numpy(), weights=np.exp(0.1 * rng.standard_normal(case["nwalk"])))
        return state
    ctx.prep_prop(ham.phi_up, ham.phi_dn, DT)
    if kind == "surrogate":
        ctx.set_walkers(_determinants(case, seed, sys["phi"], case["nwalk"]).cpu().numpy())
        ctx.surrogate_init(hidden=case["hidden"], seed=1, capacity=0)
        ctx.surrogate_params(_mlp_params(case, seed)[1])
        state["x"], state["t"] = _mlp_rows(case, seed)
        return state
    if case["prec"] == "mixed":
        ctx.set_precision(AFQ_PREC_BF16X3, AFQ_PREC_BF16X3, AFQ_PREC_BF16X3)
        ctx.set_prop_precision(AFQ_PREC_BF16X3)
    if case["energy"] == "cv":
        ctx.set_surrogate_kind(AFQ_SURR_EXCHANGE, AFQ_PREC_BF16)
        ctx.set_cv(subset_inv=16, risk_frac=0.0, seed=3)
    det = ham.serial_det(*start)
    ctx.set_walkers_uniform(det)
    guess = float(ctx.measure(want_ho=False)[0])
    state.update(det=det, step=0, block=0, estimate=guess, guess=guess, shift=guess, uniforms=_uniforms(seed, 64))
    return state


# ---------------------------------------------------------------------------------------------- one pass
def run(state):
    return {"walk": _run_walk, "run": _run_driver, "batch": _run_batch, "evaluate": _run_evaluate, "restore": _run_restore,
            "surrogate": _run_surrogate}[state["kind"]](state)


def _feedback(estimate, total, nwalk):
    return estimate - 0.1 * math.log(total / nwalk) / DT


def _run_walk(state):
    ctx, case = state["ctx"], state["case"]
    nwalk, mixed = case["nwalk"], case["prec"] == "mixed"
    if mixed:
        ctx.set_walkers_uniform(state["det"])
        state["shift"] = state["estimate"] = state["guess"]
    for _ in range(case["nsteps"]):
        state["step"] += 1
        ctx.propagate(None, state["shift"], seed=KEY, step=state["step"], want_factors=False)
        state["shift"] = _feedback(state["estimate"], ctx.step_stats()["total_weight"], nwalk)
    ctx.orthogonalize()
    out = {}
    if case["rdm"]:
        ctx.rdm_reset()
        ctx.rdm_accumulate()
        out["rdm"] = ctx.one_rdm(case["trial"] == "rhf")[0]
    weights = ctx.weights()
    if case["energy"] == "cv":
        energies = ctx.measure(mode=AFQ_ENERGY_SURROGATE, want_ho=False)
    else:
        energies, out["ham_overlap"] = ctx.measure()
    out.update(weights=weights, energies=energies)
    state["estimate"] = 0.9 * state["estimate"] + 0.1 * float(np.dot(weights, energies) / weights.sum())
    if mixed:
        # FP32 accumulation gives these values single precision, and the program keeps them so
        return {k: v.astype(np.complex64 if np.iscomplexobj(v) else np.float32) for k, v in out.items()}
    total = ctx.comb(state["uniforms"][state["block"] % 64])
    state["block"] += 1
    state["shift"] = _feedback(state["estimate"], total, nwalk)
    return out


def _run_driver(state):
    case, ham = state["case"], state["ham"]
    weights, energies, _ = run_long_prop(ham, ham.phi_up, ham.phi_dn, *state["start"], seed=1234, dt=DT, nsteps=case["nsteps"], nsweeps=case["blocks"],
                                         ortho_steps=ORTHO, nwalk=case["nwalk"], nranks=case["nranks"], walker_rhf=case["trial"] == "rhf")
    return dict(weights=weights, energies=energies)


def _run_batch(state):
    center = state["estimate"].copy()
    totals = []
    for _ in range(state["nsteps"]):
        state["step"] += 1
        tot = state["batch"].step(state["step"], state["shift"], state["uniforms"][state["step"] % 64], center)
        state["estimate"] = 0.9 * state["estimate"] + 0.1 * tot[:, 1] / tot[:, 0]
        state["shift"] = state["estimate"] - 0.1 * np.log(tot[:, 0] / state["nwalk"]) / DT
        totals.append(tot)
    return np.stack(totals)


def _run_evaluate(state):
    return state["ctx"].ham_and_overlap(state["dets"], state["keep"])


def _run_restore(state):
    ctx = state["ctx"]
    ctx.set_walkers(state["dets"], weights=state["weights"])
    return dict(force_bias=ctx.force_bias(), overlaps=ctx.overlaps())


def _run_surrogate(state):
    loss, grads = state["ctx"].surrogate_grad(state["x"], state["t"])
    return dict(loss=loss, grads=grads, predicted=state["ctx"].surrogate_predict().astype(np.float32))


# ---------------------------------------------------------------------------------------------- required work
def _propagate_work(c):
    """(flops, bytes) of one propagation of every walker; real * complex = 4, complex * complex = 8 flops a product."""
    n, g, w = c["norb"], c["nchol"], c["nwalk"]
    spins, props = ([2 * c["nalpha"]], [c["nalpha"]]) if c["trial"] == "rhf" else ([c["nalpha"], c["nbeta"]],) * 2
    tri, vhs = n * (n + 1) / 2, 2 if c.get("ints") == "u" else 1
    cols = [s / 2 if c["trial"] == "rhf" else s for s in spins]
    flops = vhs * 4 * tri * g
    flops += sum(2 * 4 * n * n * p + 5 * 8 * n * n * p for p in props)                    # one-body factors, Taylor terms
    flops += sum(4 * p * p * n + 16 * p ** 3 + 8 * n * p * p + 4 * n * p * g for p in cols)  # overlap, inverse, theta, force bias
    state = 16 * n * sum(props) + 16 * g
    return w * flops, w * 2 * state + 8 * g * (vhs * tri + n * sum(cols))


def _energy_work(c, count, keep=1.0):
    n, g = c["norb"], c["nchol"] * keep
    cols = [c["nalpha"]] if c["trial"] == "rhf" else [c["nalpha"], c["nbeta"]]
    flops = count * sum(4 * g * n * p * p + 8 * g * p * p for p in cols)
    return flops, 8 * g * n * sum(cols) + 16 * count * n * sum(cols)


def work(case):
    kind = case["kind"]
    if kind == "walk":
        pf, pb = _propagate_work(case)
        ef, eb = _energy_work(case, case["nwalk"])
        props = [case["nalpha"]] if case["trial"] == "rhf" else [case["nalpha"], case["nbeta"]]
        qf = case["nwalk"] * sum(16 * (2 * case["norb"] * p * p - 2 * p ** 3 / 3) / 2 for p in props)
        return dict(bytes=case["nsteps"] * pb + eb, flops=case["nsteps"] * pf + ef + qf)
    if kind == "run":
        c = dict(case, nwalk=case["nwalk"] * case["nranks"])
        pf, pb = _propagate_work(c)
        ef, eb = _energy_work(c, c["nwalk"])
        steps = case["blocks"] * case["nsteps"] - 1
        return dict(bytes=steps * (pb + 8 * c["nwalk"] * c["nchol"]) + case["blocks"] * eb, flops=steps * pf + case["blocks"] * ef)
    if kind == "batch":
        # the mean system of the range stands for the drawn ones
        n = (case["nmin"] + case["nmax"]) / 2
        c = dict(norb=n, nalpha=n / 5, nbeta=n / 5, nchol=4 * n, nwalk=case["nwalk"], trial="uhf")
        pf, pb = _propagate_work(c)
        ef, eb = _energy_work(c, case["nwalk"])
        return dict(bytes=case["nsys"] * case["nsteps"] * (pb + eb), flops=case["nsys"] * case["nsteps"] * (pf + ef))
    n, cols = case["norb"], case["nalpha"] + case["nbeta"]
    if kind == "evaluate":
        ef, eb = _energy_work(case, case["ndet"], case["keep"])
        g = case["nchol"]
        green = case["ndet"] * sum(4 * p * p * n + 16 * p ** 3 + 8 * n * p * p + 4 * n * p * g * case["keep"] for p in (case["nalpha"], case["nbeta"]))
        return dict(bytes=eb + 32 * case["ndet"], flops=ef + green)
    if kind == "restore":
        w, g = case["nwalk"], case["nchol"]
        green = w * sum(4 * p * p * n + 16 * p ** 3 + 8 * n * p * p + 4 * n * p * g for p in (case["nalpha"], case["nbeta"]))
        return dict(bytes=16 * w * n * cols + 16 * w * g + 8 * g * n * cols, flops=green)
    width, hidden = case["nchol"] + 2 * n, case["hidden"]
    params = width * hidden + 2 * hidden * hidden + hidden
    return dict(bytes=4 * case["rows"] * width + 8 * params + 4 * case["nwalk"] * width,
                flops=2 * case["rows"] * (3 * params - width * hidden) + 2 * case["nwalk"] * params)


# ---------------------------------------------------------------------------------------------- 64-bit values
class _Exact:
    """The method in plain FP64 tensor operations over a whole population."""

    def __init__(self, case, sys, nwalk):
        self.n, self.g, self.w = case["norb"], case["nchol"], nwalk
        self.rhf, self.phi, self.L, self.h = sys["rhf"], sys["phi"], sys["L"], sys["h"]
        self.spins = [0] if self.rhf else [0, 1]       # spins propagated; a closed shell counts its one twice
        self.mult = 2 if self.rhf else 1
        self.rot = [torch.einsum("mi,gmk->gik", self.phi[s], self.L[min(s, len(self.L) - 1)]) for s in self.spins]

    def prepare(self, dt):
        self.dt = dt
        dens = [p @ torch.linalg.solve(p.T @ p, p.T) for p in self.phi]
        a = sum(torch.einsum("gij,ij->g", self.L[min(s, len(self.L) - 1)], dens[s]) for s in (0, 1))
        self.mf = a                                    # the mean-field shift is i a
        self.const = 0.5 * float((a * a).sum())
        self.E = []
        for h, L in zip(self.h, self.L):
            self.E.append(torch.linalg.matrix_exp(-0.5 * dt * (h - 0.5 * _square(L) + torch.einsum("g,gij->ij", a, L))))

    def set(self, psi):
        """psi: per spin, (W, N, n) complex."""
        self.psi = [psi[s].contiguous() for s in self.spins]
        self.weights = torch.ones(self.w, dtype=F64, device=self.phi[0].device)
        self.logo = self.green()

    def chunks(self, per):
        step = max(1, int(2 ** 28 // max(1, per)))
        return [slice(i, min(self.w, i + step)) for i in range(0, self.w, step)]

    def green(self):
        """theta and the force bias of every walker; returns the log overlap."""
        self.theta, logo = [], 0.0
        fb = torch.zeros(self.w, self.g, dtype=C128, device=self.phi[0].device)
        for s in self.spins:
            S = self.phi[s].T.to(C128) @ self.psi[s]
            sign, logabs = torch.linalg.slogdet(S)
            logo = logo + self.mult * torch.complex(logabs, sign.angle())
            th = self.psi[s] @ torch.linalg.inv(S)
            self.theta.append(th)
            flat = torch.view_as_real(th.transpose(1, 2).reshape(self.w, -1))
            r = self.rot[s].reshape(self.g, -1).T
            fb += self.mult * torch.complex(flat[..., 0] @ r, flat[..., 1] @ r)
        self.fb = fb
        return logo

    def propagate(self, x, shift, cap):
        sq = math.sqrt(self.dt)
        s = -sq * (1j * self.fb - 1j * self.mf)
        p = x - s
        move = (p * (1j * self.mf)).sum(1)
        term = (x * s - 0.5 * s * s).sum(1)
        new = []
        for k, sp in enumerate(self.spins):
            L = self.L[min(sp, len(self.L) - 1)].reshape(self.g, -1)
            E = self.E[min(sp, len(self.E) - 1)].to(C128)
            out = torch.empty_like(self.psi[k])
            for c in self.chunks(3 * self.n * self.n):
                v = torch.complex(p[c].real @ L, p[c].imag @ L).reshape(-1, self.n, self.n) * (1j * sq)
                t = E @ self.psi[k][c]
                acc = t.clone()
                for q in range(1, 6):
                    t = torch.bmm(v, t) / q
                    acc += t
                out[c] = E @ acc
            new.append(out)
        self.psi = new
        logo = self.green()
        d = logo - self.logo
        f = torch.exp((-sq * move.real + term.real + self.dt * (shift + self.const)) + d.real) * torch.cos(-sq * move.imag + d.imag)
        f = torch.where((f >= 1e-3) & (f <= 100.0), f, torch.zeros_like(f))
        w = self.weights * f
        self.weights = torch.where(w > cap, torch.zeros_like(w), w)
        self.logo = logo

    def orthogonalize(self):
        live = self.weights != 0   # a walker of weight zero is left alone
        for k in range(len(self.spins)):
            q, r = np.linalg.qr(self.psi[k].cpu().numpy())
            logr = np.log(np.einsum("wii->wi", r).astype(np.complex128)).sum(1)
            self.logo = torch.where(live, self.logo - self.mult * torch.from_numpy(logr).to(self.logo.device), self.logo)
            self.psi[k] = torch.where(live[:, None, None], torch.from_numpy(q).to(self.logo.device), self.psi[k])

    def energies(self, keep=None):
        keep = self.g if keep is None else keep
        e = 0.5 * (self.fb[:, :keep] ** 2).sum(1)
        for k, s in enumerate(self.spins):
            hphi = (self.h[min(s, len(self.h) - 1)] @ self.phi[s]).to(C128)
            th = self.theta[k]
            e = e + self.mult * torch.einsum("wki,ki->w", th, hphi)
            n = self.phi[s].shape[1]
            r = self.rot[s][:keep].reshape(keep * n, self.n)
            for c in self.chunks(4 * keep * n * n):
                t = th[c]
                flat = torch.view_as_real(t.permute(1, 0, 2).reshape(self.n, -1).contiguous()).reshape(self.n, -1)
                f = torch.view_as_complex((r @ flat).reshape(keep, n, t.shape[0], n, 2))
                e[c] = e[c] - 0.5 * self.mult * (f * f.permute(0, 3, 2, 1)).sum((0, 1, 3))
        return e

    def comb(self, zeta):
        cum = torch.from_numpy(np.cumsum(self.weights.cpu().numpy())).to(self.weights.device)
        total = float(cum[-1])
        teeth = (torch.arange(self.w, device=cum.device, dtype=F64) + zeta) / self.w * total
        at = torch.searchsorted(cum, teeth).clamp(max=self.w - 1)
        self.psi = [p[at] for p in self.psi]
        self.theta = [t[at] for t in self.theta]
        self.fb, self.logo = self.fb[at], self.logo[at]
        self.weights = torch.full_like(self.weights, total / self.w)
        return total


def _normals(key, step, nwalk, nchol):
    """Field draws: Philox4x32-10 (Salmon et al., SC'11) with counter (pair, step, walker), Box-Muller on two 53-bit uniforms."""
    pairs = (nchol + 1) // 2
    mask = np.uint64(0xFFFFFFFF)
    c = [np.tile(np.arange(pairs, dtype=np.uint64), nwalk), np.full(nwalk * pairs, step & 0xFFFFFFFF, np.uint64),
         np.full(nwalk * pairs, step >> 32, np.uint64), np.repeat(np.arange(nwalk, dtype=np.uint64), pairs)]
    k = [key & 0xFFFFFFFF, (key >> 32) & 0xFFFFFFFF]
    for _ in range(10):
        p0, p1 = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k[0]), p1 & mask, (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k[1]), p0 & mask]
        k = [(k[0] + 0x9E3779B9) & 0xFFFFFFFF, (k[1] + 0xBB67AE85) & 0xFFFFFFFF]
    a = (c[0] << np.uint64(32)) | c[1]
    b = (c[2] << np.uint64(32)) | c[3]
    u1 = ((a >> np.uint64(11)).astype(np.float64) + 1.0) * 2.0 ** -53
    u2 = (b >> np.uint64(11)).astype(np.float64) * 2.0 ** -53
    r = np.sqrt(-2.0 * np.log(u1))
    x = np.stack([r * np.cos(2.0 * np.pi * u2), r * np.sin(2.0 * np.pi * u2)], axis=1).reshape(nwalk, 2 * pairs)
    return torch.from_numpy(x[:, :nchol].copy()).to(_device())


def _uniform_population(x, start):
    x.set([s.to(C128).expand(x.w, *s.shape) for s in start])


def exact(case, seed):
    kind = case["kind"]
    if kind == "run":
        return None   # its draws come from the C++ library's random stream
    if kind == "surrogate":
        return _exact_surrogate(case, seed)
    if kind == "batch":
        return _exact_batch(case, seed)
    sys = _hamiltonian(case, seed)
    if kind in ("evaluate", "restore"):
        count = case["ndet"] if kind == "evaluate" else case["nwalk"]
        x = _Exact(case, sys, count)
        d = _determinants(case, seed, sys["phi"], count)
        cut = case["norb"] * case["nalpha"]
        x.set([d[:, :cut].reshape(count, case["norb"], -1), d[:, cut:].reshape(count, case["norb"], -1)])
        o = torch.exp(x.logo)
        if kind == "restore":
            return dict(force_bias=x.fb.cpu().numpy(), overlaps=o.cpu().numpy())
        return torch.stack([x.energies(int(case["keep"] * case["nchol"])) * o, o], dim=1).cpu().numpy()
    if work(case)["flops"] > 1e14:
        return None
    x = _Exact(case, sys, case["nwalk"])
    x.prepare(DT)
    _uniform_population(x, _start(case, seed, sys["phi"]))
    estimate = shift = _first_energy(case, sys, seed)
    cap = max(100.0, case["nwalk"] / 10.0)
    for step in range(1, case["nsteps"] + 1):
        x.propagate(_normals(KEY, step, x.w, x.g), shift, cap)
        shift = _feedback(estimate, float(x.weights.sum()), x.w)
    if case["energy"] != "cv":   # energies do not depend on it, overlaps do
        x.orthogonalize()
    e = x.energies()
    live = x.weights != 0
    out = {}
    if case["rdm"]:
        mats = [(p @ torch.einsum("w,wje->je", x.weights, t.real).T / x.weights.sum()).cpu().numpy() for p, t in zip([x.phi[s] for s in x.spins], x.theta)]
        out["rdm"] = 2 * mats[0] if x.rhf else np.stack(mats)
    if case["energy"] != "cv":
        o = torch.exp(x.logo)
        out["ham_overlap"] = torch.stack([torch.where(live, e * o, torch.zeros_like(o)), o], dim=1).cpu().numpy()
    out.update(weights=x.weights.cpu().numpy(), energies=torch.where(live, e.real, torch.zeros_like(e.real)).cpu().numpy())
    return out


def _first_energy(case, sys, seed, stream=1):
    one = _Exact(case, sys, 1)
    _uniform_population(one, _start(case, seed, sys["phi"], stream))
    return float(one.energies().real[0])


def _exact_batch(case, seed):
    out = np.zeros((case["nsteps"], case["nsys"], 2))
    uniforms = _uniforms(seed, (64, case["nsys"]))
    half = math.sqrt(2.0 / DT)
    for i, m in enumerate(_batch_cases(case, seed)):
        sys = _hamiltonian(m, seed, 10 + i)
        x = _Exact(m, sys, case["nwalk"])
        x.prepare(DT)
        _uniform_population(x, _start(m, seed, sys["phi"], 100 + i))
        center = estimate = shift = _first_energy(m, sys, seed, 100 + i)
        cap = max(100.0, case["nwalk"] / 10.0)
        for step in range(1, case["nsteps"] + 1):
            x.propagate(_normals(KEY + 7919 * i, step, x.w, x.g), shift, cap)
            if step % ORTHO == 0:
                x.orthogonalize()
            e = x.energies().real.clamp(center - half, center + half)
            out[step - 1, i] = float(x.weights.sum()), float((x.weights * e).sum())
            estimate = 0.9 * estimate + 0.1 * out[step - 1, i, 1] / out[step - 1, i, 0]
            shift = _feedback(estimate, out[step - 1, i, 0], x.w)
            x.comb(uniforms[step % 64, i])
    return out


def _exact_surrogate(case, seed):
    dims, flat = _mlp_params(case, seed)
    rows, targets = _mlp_rows(case, seed)
    params, at = [], 0
    for a, b in zip(dims, dims[1:]):
        for shape in ((a, b), (b,)):
            n = int(np.prod(shape))
            params.append(torch.from_numpy(flat[at:at + n].reshape(shape)).to(_device(), F64).requires_grad_())
            at += n

    def net(v):
        for q in range(4):
            v = v @ params[2 * q] + params[2 * q + 1]
            v = torch.nn.functional.gelu(v) if q < 3 else v
        return v[:, 0]

    y, t = net(torch.from_numpy(rows).to(_device(), F64)), torch.from_numpy(targets).to(_device(), F64)
    loss = 0.5 * ((y - t) ** 2).mean()
    grads = torch.autograd.grad(loss, params)
    sys = _hamiltonian(case, seed)
    x = _Exact(case, sys, case["nwalk"])
    d = _determinants(case, seed, sys["phi"], case["nwalk"])
    cut = case["norb"] * case["nalpha"]
    x.set([d[:, :cut].reshape(x.w, x.n, -1), d[:, cut:].reshape(x.w, x.n, -1)])
    diag = [torch.einsum("wki,ki->wk", th, x.phi[s].to(C128)).real for s, th in zip(x.spins, x.theta)]
    with torch.no_grad():
        predicted = net(torch.cat([x.fb.real] + diag, dim=1))
    return dict(loss=float(loss), grads=torch.cat([g.reshape(-1) for g in grads]).cpu().numpy(), predicted=predicted.cpu().numpy())
