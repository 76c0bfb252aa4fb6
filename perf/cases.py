"""Performance cases of the CCSD engine: what a user has it do, over the sizes it is used at.

Five kinds of work, each through the public Python surface:

  solve     create a closed-shell solver on resident integrals, run it (to convergence, or a stated
            number of iterations for the large systems), read T1, T2 and the energies
  contract  one tensor contraction of the CCSD equations, the amplitude operand new on every call
            (as it is in an iteration), the integral operand constant
  sums      the permuting tensor sums of one iteration (symmetrisation, spin adaptation, reordering)
  hbar      the similarity-transformed Hamiltonian products after a solve
  serve     a burst of jobs of uneven size through the serving loop, with the caller's integrals

The systems are the synthetic closed-shell construction (orbital energies and symmetric
three-index factors), with (o, v) from the molecules, the benchmark and the serving stream.
"""
import math

import numpy as np
import torch

import aquarius_amd as aq

# Contractions of the iteration: (A labels, B labels, C labels, alpha, beta).  a-h are virtual, i-n
# occupied; A is the constant integral (or intermediate), B the amplitudes.
FORMS = {
    "ladder": ("abef", "efij", "abij", 0.5, 1.0),   # particle-particle ladder into the doubles residual
    "ring": ("amie", "ebmj", "abij", 0.5, 1.0),     # particle-hole ring
    "xring": ("amej", "ebim", "abij", -1.0, 1.0),   # crossed ring, permuted operands
    "single": ("abej", "ei", "abij", 1.0, 1.0),     # three-virtual integral dressed with T1
    "wamij": ("efam", "efij", "amij", 1.0, 1.0),    # long inner extent, medium output
    "wmnij": ("efmn", "efij", "mnij", 0.5, 1.0),    # long inner extent, small output
    "fae": ("efmn", "afmn", "ae", -1.0, 1.0),       # very long inner extent, tiny output
}

SYSTEM_SHAPES = {"fAI": "vo", "fAB": "vv", "fIJ": "oo", "VABCD": "vvvv", "VABCI": "vvvo", "VABIJ": "vvoo",
                 "VAIBJ": "vovo", "VAIJB": "voov", "VAIJK": "vooo", "VIJKL": "oooo"}


def listed():
    return [
        # water in cc-pVDZ: the smallest real solve, launches and latency
        solve("solve_h2o_fp64", 5, 19, "fp64"),
        # small job of the serving stream, mixed precision (BF16x3 bulk, FP64 refinement)
        solve("solve_small_mixed", 8, 43, "bf16x3"),
        # ordinary odd-sized system of the serving stream in FP64
        solve("solve_medium_fp64", 13, 75, "fp64"),
        # the benchmark's second system (o=20, v=140), mixed precision, GEMM tuner on as there
        solve("solve_o20v140_mixed", 20, 140, "bf16x3", autotune=True),
        # large system in FP64: iterations of the refinement phase
        solve("iterate_large_fp64", 32, 192, "fp64", iterations=4),
        # eight waters in cc-pVDZ: iterations of the BF16x3 bulk phase
        solve("iterate_water8_bf16x3", 40, 152, "bf16x3", iterations=6, autotune=True),
        # the operator surface: the full (unpacked) ladder as a host program issues it
        contract("contract_ladder_fp64", "ladder", 24, 112, "fp64"),
        # the operator surface: a ring term in BF16x3, amplitude operand split anew on every call
        contract("contract_ring_bf16x3", "ring", 29, 171, "bf16x3"),
        # the operator surface: T1 dressing of a three-virtual integral, bound by memory
        contract("contract_single_fp64", "single", 27, 150, "fp64"),
        # the operator surface: symmetrisation, spin adaptation and reordering of doubles amplitudes
        {"name": "sums_doubles", "kind": "sums", "o": 31, "v": 189},
        # what the equation-of-motion consumers read, with the three-virtual product
        {"name": "hbar_medium", "kind": "hbar", "o": 14, "v": 81},
        # eight jobs of the serving stream's smaller half, as a burst on four slots
        {"name": "serve_burst", "kind": "serve", "jobs": 8, "o_min": 4, "o_max": 14, "slots": 4, "pick": 4},
    ]


def solve(name, o, v, precision, iterations=0, autotune=False):
    """iterations = 0: to convergence."""
    c = {"kind": "solve", "o": o, "v": v, "precision": precision, "iterations": iterations, "autotune": autotune}
    return dict(c, name=name) if name else c


def contract(name, form, o, v, precision):
    c = {"kind": "contract", "form": form, "o": o, "v": v, "precision": precision}
    return dict(c, name=name) if name else c


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "iterate", "contract", "contract", "sums", "hbar", "serve"])
    ratio = rng.uniform(3.8, 8.0)   # v / o of the molecules and the serving stream
    precision = rng.choice(["fp64", "bf16x3"])
    if kind == "solve":
        o = log_int(rng, 4, 18)
        return solve("", o, min(int(round(o * ratio)), 140), precision)
    if kind == "iterate":
        o = log_int(rng, 20, 36)
        return solve("", o, min(int(round(o * ratio)), 180), precision, rng.randint(2, 4), rng.random() < 0.5)
    if kind == "contract":
        form = rng.choice(sorted(FORMS))
        o = log_int(rng, 4, 28)
        v = min(int(round(o * ratio)), 110 if form == "ladder" else 165)
        return contract("", form, o, v, precision)
    if kind == "sums":
        o = log_int(rng, 4, 30)
        return {"kind": "sums", "o": o, "v": min(int(round(o * ratio)), 189)}
    if kind == "hbar":
        o = log_int(rng, 4, 16)
        return {"kind": "hbar", "o": o, "v": min(int(round(o * ratio)), 90)}
    return {"kind": "serve", "jobs": rng.randint(2, 8), "o_min": 4, "o_max": rng.randint(6, 13),
            "slots": rng.randint(1, 4), "pick": rng.randrange(1000)}


# ---------------------------------------------------------------- inputs

def generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


class System:
    """Orbital energies and three-index factors of one synthetic closed-shell system (o occupied, v
    virtual): <pq|rs> = sum_Q B(Q,p,r) B(Q,q,s), occupied orbitals first."""

    def __init__(self, o, v, seed):
        g = generator(seed)
        n, nq = o + v, 3 * (o + v)
        kw = {"device": "cuda", "dtype": torch.float64, "generator": g}
        self.o, self.v = o, v
        self.occ = torch.sort(torch.rand(o, **kw) * 1.2 - 1.5).values
        self.vir = torch.sort(torch.rand(v, **kw) * 4.8 + 0.2).values
        b = torch.randn(nq, n, n, **kw) * (0.05 * math.sqrt(150.0 / (v * math.sqrt(nq))))
        self.b = torch.triu(b) + torch.triu(b, 1).transpose(1, 2)

    def fill(self, name, out):
        """Write block `name` into `out`, whose dimensions run last index first (the library's
        column-major order)."""
        sl = {"v": slice(self.o, None), "o": slice(0, self.o)}
        kinds = SYSTEM_SHAPES[name]
        if len(kinds) == 2:
            out.zero_()
            if name != "fAI":
                out.copy_(torch.diag(self.vir if name == "fAB" else self.occ))
            return out
        # letters of <pq|rs> in tensor order
        p, q, r, s = (sl[k] for k in kinds)
        left = self.b[:, p, r].permute(2, 0, 1).contiguous()    # [r, Q, p]
        right = self.b[:, q, s].permute(2, 1, 0).contiguous()   # [s, q, Q]
        for k in range(out.shape[0]):
            torch.matmul(right[k].expand(left.shape[0], -1, -1), left, out=out[k])   # [r, q, p]
        return out


class DeviceArray:
    """A library tensor's device memory, dimensions last index first."""

    def __init__(self, t):
        self.__cuda_array_interface__ = {"shape": tuple(reversed(t.shape)), "typestr": "<f8",
                                         "data": (t.data_ptr(), False), "version": 2}


def view(t, owner=None):
    """The library tensor `t` as a torch tensor on the same memory; `owner`, which frees that memory
    when it is dropped, lives at least as long as the view."""
    x = torch.as_tensor(DeviceArray(t), device="cuda")
    x.owner = owner
    return x


def integrals(ctx, o, v, seed):
    system = System(o, v, seed)
    size = {"o": o, "v": v}
    tensors = {name: ctx.tensor(tuple(size[k] for k in kinds), zero=False) for name, kinds in SYSTEM_SHAPES.items()}
    ctx.sync()
    for name, t in tensors.items():
        system.fill(name, view(t))
    torch.cuda.synchronize()
    for t in tensors.values():
        t.touch()
    return aq.Integrals(ctx, tensors)


def operand(ctx, shape, values):
    t = ctx.tensor(shape, zero=False)
    ctx.sync()
    view(t).copy_(values)
    torch.cuda.synchronize()
    t.touch()
    return t


def lengths(labels, o, v):
    return tuple(v if c < "i" else o for c in labels)


def normal(g, shape, scale):
    """Values of a tensor of lengths `shape`, dimensions last index first."""
    return torch.randn(tuple(reversed(shape)), device="cuda", dtype=torch.float64, generator=g) * scale


def contract_values(case, seed):
    ia, ib, ic, alpha, beta = FORMS[case["form"]]
    g = generator(seed)
    return [normal(g, lengths(lab, case["o"], case["v"]), scale) for lab, scale in ((ia, 0.02), (ib, 0.01), (ic, 0.01))]


def sums_values(case, seed):
    g = generator(seed)
    shape = lengths("abij", case["o"], case["v"])
    return normal(g, shape, 0.01), normal(g, shape, 0.01)


def jobs_of(case):
    """(o, v, precision) of a burst's jobs: o and v as the serving stream draws them."""
    r = np.random.default_rng(case["pick"])
    out = []
    for k in range(case["jobs"]):
        o = int(r.integers(case["o_min"], case["o_max"] + 1))
        out.append((o, int(round(o * r.uniform(4.0, 8.0))), "bf16x3"))
    return out


def config(case):
    over = {"diis_order": 8, "max_iterations": 100, "precision": case["precision"]}
    if case["iterations"]:
        over.update(max_iterations=case["iterations"], convergence=0.0, refine_below=0.0)
    return aq.default_config(**over)


class State(dict):
    """What the program keeps; its device memory goes back when it is dropped."""

    def __del__(self):
        for close in self.pop("close", []):
            close()


class Solver:
    """A solver on a state's integrals: closed when nothing refers to it or to its tensors, and
    before the state is."""

    def __init__(self, state, cfg):
        self.state = state
        self.cc = None
        self.cc = aq.RHFCCSD(state["ctx"], state["ints"], cfg)

    def __del__(self):
        if self.cc is not None:
            self.cc.close()

    def tensors(self, names):
        return {n: view(self.cc.tensor(n), self) for n in names}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "serve":
        ctx = aq.Context()
        ints = [integrals(ctx, o, v, seed + 1000 * k) for k, (o, v, p) in enumerate(jobs_of(case))]
        server = aq.Server(slots=case["slots"], hbm_budget=24 << 30)
        server.set_grouping(50)
        return State(case=case, server=server, ints=ints, close=[server.close] + [i.free for i in ints] + [ctx.close])
    # 60 GB: the memory that a program with several solvers gives each
    ctx = aq.Context(hbm_budget=60 << 30)
    if kind in ("solve", "hbar"):
        ints = integrals(ctx, case["o"], case["v"], seed)
        st = State(case=case, ctx=ctx, ints=ints, close=[ints.free, ctx.close])
        if kind == "solve":
            ctx.set_autotune(case["autotune"])
            return st
        solver = Solver(st, aq.default_config(diis_order=8, max_iterations=3, convergence=0.0))
        solver.cc.run()
        return {"case": case, "solver": solver}
    if kind == "contract":
        ctx.set_precision(case["precision"])
        shapes = [lengths(lab, case["o"], case["v"]) for lab in FORMS[case["form"]][:3]]
        t = [operand(ctx, s, x) for s, x in zip(shapes, contract_values(case, seed))]
    else:
        z, x = sums_values(case, seed)
        o, v = case["o"], case["v"]
        t = [operand(ctx, (v, v, o, o), z), operand(ctx, (v, v, o, o), x), ctx.tensor((v, v, o, o)),
             ctx.tensor((v, o, o, v))]
    return State(case=case, ctx=ctx, t=t, close=[a.free for a in t] + [ctx.close])


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "solve":
        # a new solver on the resident integrals
        solver = Solver(state, config(case))
        r = solver.cc.run()
        return {"energies": np.array([solver.cc.mp2, r["energy"]]), **solver.tensors(("T1", "T2"))}
    if kind == "contract":
        ctx, (a, b, c) = state["ctx"], state["t"]
        ia, ib, ic, alpha, beta = FORMS[case["form"]]
        b.touch()   # the amplitudes are new in every iteration
        ctx.contract(alpha, a, ia, b, ib, beta, c, ic)
        return view(c, state)
    if kind == "sums":
        ctx, (z, x, s, r) = state["ctx"], state["t"]
        ctx.sum(0.5, z, "baji", 0.5, z, "abij")     # symmetrise in place
        ctx.sum(2.0, x, "abij", 0.0, s, "abij")     # spin adaptation
        ctx.sum(-1.0, x, "abji", 1.0, s, "abij")
        ctx.sum(1.0, x, "abij", 0.0, r, "aijb")     # amplitudes in the ring terms' order
        return [view(z, state), view(s, state), view(r, state)]
    if kind == "hbar":
        state["solver"].cc.hbar(with_wabej=True)
        return state["solver"].tensors(HBAR)
    server = state["server"]
    ids = []
    for ints, (o, v, precision) in zip(state["ints"], jobs_of(case)):
        ids.append(server.submit(0, o, v, inputs=ints, diis_order=8, max_iterations=100, precision=precision))
    got = [server.wait(i) for i in ids]
    if any(r["status"] != aq.JOB_DONE for r in got):
        raise RuntimeError("a served job failed: " + "; ".join(r["error"] for r in got if r["error"]))
    return np.array([[r["mp2"], r["energy"]] for r in got])


HBAR = ("FAE", "FMI", "FME", "WMNIJ", "WMNEJ", "WAMIJ", "WAMEI", "WAMIE", "WABEJ")


# ---------------------------------------------------------------- what a pass cannot do without

def iteration_flops(o, v):
    """One iteration's contractions, the ladder on (anti)symmetric pairs (a quarter of 2 o^2 v^4)."""
    return (0.5 * o**2 * v**4 + 12 * o**3 * v**3 + 14 * o**2 * v**3 + 4 * o * v**3 + 4 * o**4 * v**2
            + 20 * o**3 * v**2)


def iteration_bytes(o, v, per):
    """Integrals read once (`per` bytes a value; the four-virtual block as its two pair matrices,
    half of v^4), the amplitudes read and written once."""
    return per * (0.5 * v**4 + v**3 * o + 3 * o * o * v * v) + 8 * 4.0 * o * o * v * v


def solve_work(o, v, precision, iterations):
    reduced = precision == "bf16x3"
    n = iterations or (22 if reduced else 16)     # typical counts to 1e-9
    per = 4 if reduced else 8                     # two 16-bit planes, or 64 bits
    integrals_once = 8.0 * (v**4 + v**3 * o + 4 * o * o * v * v)
    return {"bytes": integrals_once + n * iteration_bytes(o, v, per), "flops": n * iteration_flops(o, v)}


def work(case):
    kind = case["kind"]
    if kind == "serve":
        parts = [solve_work(o, v, p, 0) for o, v, p in jobs_of(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    o, v = case["o"], case["v"]
    if kind == "solve":
        return solve_work(o, v, case["precision"], case["iterations"])
    if kind == "contract":
        ia, ib, ic = FORMS[case["form"]][:3]
        count = [math.prod(lengths(lab, o, v)) for lab in (ia, ib, ic)]
        every = "".join(sorted(set(ia + ib + ic)))
        a = count[0] * (8 if case["precision"] == "fp64" else 4)   # the constant operand as it is kept
        return {"bytes": float(a + 8 * count[1] + 16 * count[2]), "flops": 2.0 * math.prod(lengths(every, o, v))}
    if kind == "sums":
        return {"bytes": 8.0 * 5 * o * o * v * v, "flops": 5.0 * o * o * v * v}
    outputs = sum(math.prod(lengths(lab, o, v)) for lab in ("ae", "mi", "me", "mnij", "mnej", "amij", "amei", "amie",
                                                             "abej"))
    flops = (2.0 * o * v**4 + 6 * o**2 * v**4 + 2 * o**3 * v**3 * 8 + 4 * o**2 * v**3 * 4 + 2 * o**4 * v**2 * 2)
    return {"bytes": 8.0 * (v**4 + 2 * v**3 * o + 4 * o * o * v * v + outputs), "flops": flops}


# ---------------------------------------------------------------- 64-bit values

def ein(spec, a, b):
    """einsum in the library's label order on arrays whose dimensions run last index first."""
    (ia, ib), ic = spec.split("->")[0].split(","), spec.split("->")[1]
    return torch.einsum("%s,%s->%s" % (ia[::-1], ib[::-1], ic[::-1]), a, b)


def perm(spec, x):
    ia, ic = spec.split("->")
    return torch.einsum("%s->%s" % (ia[::-1], ic[::-1]), x)


class Plain:
    """Closed-shell CCSD in plain 64-bit torch: the equations as published for the spin-adapted
    form, DIIS over (T1, T2) and their increments."""

    def __init__(self, o, v, seed):
        s = System(o, v, seed)
        size = {"o": o, "v": v}
        for name, kinds in SYSTEM_SHAPES.items():
            out = torch.empty(tuple(size[k] for k in reversed(kinds)), device="cuda", dtype=torch.float64)
            setattr(self, name, s.fill(name, out))
        self.d1 = s.occ[:, None] - s.vir[None, :]                                        # [i, a]
        self.d2 = self.d1[None, :, None, :] + self.d1[:, None, :, None]                  # [j, i, b, a]
        self.T1, self.T2 = self.fAI / self.d1, self.VABIJ / self.d2
        self.SA = 2 * self.VABIJ - perm("abji->abij", self.VABIJ)
        self.VSA = 2 * self.VAIJB - perm("aibj->aijb", self.VAIBJ)
        self.mp2 = self.energy()

    def tau(self):
        return self.T2 + ein("ai,bj->abij", self.T1, self.T1)

    def energy(self):
        return float(2 * (self.fAI * self.T1).sum() + (self.SA * self.tau()).sum())

    def residual(self):
        T1, T2, I, J, K = self.T1, self.T2, self.VABCI, self.VABIJ, self.VAIJK
        tau = self.tau()
        tsa, t2sa = 2 * tau - perm("abji->abij", tau), 2 * T2 - perm("abji->abij", T2)
        fme = perm("em->me", self.fAI) + ein("efmn,fn->me", self.SA, T1)
        fmi = (self.fIJ + ein("efmn,efin->mi", self.SA, T2) + ein("me,ei->mi", fme, T1) + 2 * ein("finm,fn->mi", K, T1)
               - ein("fimn,fn->mi", K, T1))
        fae = (self.fAB - ein("efmn,afmn->ae", self.SA, T2) - ein("me,am->ae", fme, T1) + 2 * ein("efam,fm->ae", I, T1)
               - ein("feam,fm->ae", I, T1))
        w = 0.5 * self.VIJKL + 0.5 * ein("efmn,efij->mnij", J, tau) + ein("ejmn,ei->mnij", K, T1)
        wmnij = w + perm("nmji->mnij", w)
        wmnej = perm("ejmn->mnej", K) + ein("efmn,fj->mnej", J, T1)
        wamij = (K + ein("efam,efij->amij", I, tau) + ein("amej,ei->amij", self.VAIBJ, T1)
                 + ein("amie,ej->amij", self.VAIJB, T1))
        wamie = (self.VSA + 0.5 * ein("efmn,afin->amie", self.SA, t2sa) + 2 * ein("feam,fi->amie", I, T1)
                 - ein("efam,fi->amie", I, T1) - 2 * ein("mnei,an->amie", wmnej, T1) + ein("nmei,an->amie", wmnej, T1))
        wamei = (self.VAIBJ - 0.5 * ein("efnm,afni->amei", J, T2) + ein("efam,fi->amei", I, T1)
                 - ein("nmei,an->amei", wmnej, T1))
        z1 = (self.fAI + ein("ae,ei->ai", self.fAB, T1) - ein("mi,am->ai", fmi, T1) + ein("amie,em->ai", self.VSA, T1)
              + ein("me,aeim->ai", fme, t2sa) + ein("efam,efim->ai", I, tsa) - ein("mnei,eamn->ai", wmnej, t2sa))
        z2 = (0.5 * J + ein("abej,ei->abij", I, T1) - ein("amij,bm->abij", wamij, T1) + ein("ae,ebij->abij", fae, T2)
              - ein("mi,abmj->abij", fmi, T2) + 0.5 * ein("abef,efij->abij", self.VABCD, tau)
              + 0.5 * ein("mnij,abmn->abij", wmnij, tau) + 0.5 * ein("amie,ebmj->abij", wamie, t2sa)
              - 0.5 * ein("amei,ebjm->abij", wamei, T2) - ein("amej,ebim->abij", wamei, T2))
        return z1, z2 + perm("baji->abij", z2)

    def solve(self, iterations, convergence=1e-9, order=8):
        xs, es = [], []
        gram = np.zeros((0, 0))
        e = self.mp2
        for _ in range(iterations):
            z1, z2 = self.residual()
            z1, z2 = z1 / self.d1, z2 / self.d2
            self.T1, self.T2 = self.T1 + z1, self.T2 + z2
            e = self.energy()
            conv = max(float(z1.abs().max()), float(z2.abs().max()))
            xs, es = [(self.T1, self.T2)] + xs[:order - 1], [(z1, z2)] + es[:order - 1]
            k = len(es)
            row = np.array([float((z1 * a).sum() + (z2 * b).sum()) for a, b in es])
            old, gram = gram[:k - 1, :k - 1], np.zeros((k, k))
            gram[1:, 1:], gram[0], gram[:, 0] = old, row, row
            if k > 1:
                m = np.zeros((k + 1, k + 1))
                m[:k, :k], m[k, :k], m[:k, k] = gram, -1.0, -1.0
                c = np.linalg.solve(m, np.append(np.zeros(k), -1.0))
                self.T1 = sum(ck * x[0] for ck, x in zip(c, xs))
                self.T2 = sum(ck * x[1] for ck, x in zip(c, xs))
            if conv < convergence:
                break
        return e

    def hbar(self):
        T1, T2, I, J, K = self.T1, self.T2, self.VABCI, self.VABIJ, self.VAIJK
        tau, t2sa = self.tau(), 2 * T2 - perm("abji->abij", T2)
        fme = perm("em->me", self.fAI) + ein("efmn,fn->me", self.SA, T1)
        fmi = (self.fIJ + ein("efmn,efin->mi", self.SA, T2) + ein("me,ei->mi", fme, T1) + 2 * ein("finm,fn->mi", K, T1)
               - ein("fimn,fn->mi", K, T1))
        fae = (self.fAB - ein("efmn,afmn->ae", self.SA, T2) - ein("me,am->ae", fme, T1) + 2 * ein("efam,fm->ae", I, T1)
               - ein("feam,fm->ae", I, T1))
        w = 0.5 * self.VIJKL + 0.5 * ein("efmn,efij->mnij", J, tau) + ein("ejmn,ei->mnij", K, T1)
        wmnij = w + perm("nmji->mnij", w)
        wmnej = perm("ejmn->mnej", K) + ein("efmn,fj->mnej", J, T1)
        wamij = (K + ein("efam,efij->amij", I, tau) + ein("amej,ei->amij", self.VAIBJ, T1)
                 + ein("amie,ej->amij", self.VAIJB, T1) - ein("nmij,an->amij", wmnij, T1)
                 + ein("nmej,aein->amij", wmnej, t2sa) - ein("mnej,aein->amij", wmnej, T2)
                 - ein("mnei,aenj->amij", wmnej, T2) + ein("me,aeij->amij", fme, T2))
        wamie = (self.VSA + ein("efmn,afin->amie", self.SA, t2sa) + 2 * ein("feam,fi->amie", I, T1)
                 - ein("efam,fi->amie", I, T1))
        wamei = self.VAIBJ - ein("efnm,afni->amei", J, T2) + ein("efam,fi->amei", I, T1)
        wabej = (I + ein("mnej,abmn->abej", wmnej, tau) - 0.5 * ein("bmje,am->abej", wamie, T1)
                 - 0.5 * ein("bmej,am->abej", wamei, T1) - ein("amej,bm->abej", wamei, T1)
                 + ein("abef,fj->abej", self.VABCD, T1) + ein("efam,fbmj->abej", I, t2sa)
                 - ein("feam,fbmj->abej", I, T2) - ein("febm,afmj->abej", I, T2) - ein("me,abmj->abej", fme, T2))
        wamie = wamie - 2 * ein("mnei,an->amie", wmnej, T1) + ein("nmei,an->amie", wmnej, T1)
        wamei = wamei - ein("nmei,an->amei", wmnej, T1)
        return dict(zip(HBAR, (fae, fmi, fme, wmnij, wmnej, wamij, wamei, wamie, wabej)))


def exact(case, seed):
    kind = case["kind"]
    if kind == "serve":
        out = []
        for k, (o, v, precision) in enumerate(jobs_of(case)):
            p = Plain(o, v, seed + 1000 * k)
            out.append([p.mp2, p.solve(100)])
        return np.array(out)
    if kind == "contract":
        a, b, c = contract_values(case, seed)
        ia, ib, ic, alpha, beta = FORMS[case["form"]]
        return alpha * ein("%s,%s->%s" % (ia, ib, ic), a, b) + beta * c
    if kind == "sums":
        z, x = sums_values(case, seed)
        return [0.5 * (z + perm("baji->abij", z)), 2 * x - perm("abji->abij", x), perm("abij->aijb", x).contiguous()]
    p = Plain(case["o"], case["v"], seed)
    if kind == "hbar":
        p.solve(3, convergence=0.0)
        return p.hbar()
    if case["iterations"]:
        e = p.solve(case["iterations"], convergence=0.0)
    else:
        e = p.solve(100)
    return {"energies": np.array([p.mp2, e]), "T1": p.T1, "T2": p.T2}
