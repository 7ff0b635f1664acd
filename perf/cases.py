"""Performance cases: what users of this framework have it compute.

A case is one pass through the public entry points of ``imsrg_mi355x``: a
derivative for an ODE solver on the host, a whole or partial Magnus flow (one
Hamiltonian or a batch), a Hartree-Fock solution, an observable or a tensor
operator transformed by e^Omega, or the gradient of the flow's energy.  Sizes
are harmonic-oscillator bases from emax = 2 (12 orbits) to emax = 8 (90
orbits), the range of the repository's own workloads, with closed-shell
references of equal or different proton and neutron holes.

``exact`` recomputes the small cases in 64 bits from the textbook expressions:
scalar operators as dense J-coupled tensors over ordered orbit pairs, tensor
operators in the m-scheme.
"""
import functools
import math
import os
import sys

import numpy as np
import torch
import torch.utils.checkpoint

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "eom-imsrg_full_amd"))

from imsrg_mi355x import Basis  # noqa: E402
from imsrg_mi355x import engine as E  # noqa: E402
from imsrg_mi355x.autograd import flow_e0  # noqa: E402
from imsrg_mi355x.basis import closed_shell_con, hk_orbits  # noqa: E402

PRECISION = {"fp64": E.PREC_FP64, "int8x5": E.PREC_INT8X5, "int8x4": E.PREC_INT8X4}
SHELLS = (1, 3, 6)  # orbits per isospin that fill the 0s, 0p and 1s0d shells


def listed():
    return [
        # one right-hand side for an ODE solver that keeps its state on the host: the smallest call
        dict(name="ode-emax4", op="ode", emax=4, kp=3, kn=3, gen="white"),
        # the whole Magnus flow of a light nucleus in the smallest basis: launch latency, many short series
        dict(name="flow-emax2", op="flow", emax=2, kp=1, kn=1, gen="white", prec="fp64", ds=0.5, steps=200),
        # a whole flow in a small basis, other denominators
        dict(name="flow-emax4-atan", op="flow", emax=4, kp=3, kn=3, gen="atan", prec="fp64", ds=0.5, steps=200),
        # a whole flow in the ordinary basis of a survey over nuclei
        dict(name="flow-emax6", op="flow", emax=6, kp=3, kn=3, gen="white", prec="fp64", ds=0.5, steps=200),
        # the leading steps of the flow in the largest basis, in FP64 and with sliced products
        dict(name="flow-emax8", op="flow", emax=8, kp=6, kn=6, gen="white", prec="fp64", ds=0.5, steps=8),
        dict(name="flow-emax8-int8x4", op="flow", emax=8, kp=6, kn=6, gen="white", prec="int8x4", ds=0.5, steps=8),
        # an ensemble of interactions flowed together (uncertainty estimates)
        dict(name="batch16-emax6", op="batch", emax=6, kp=3, kn=3, gen="white", prec="fp64", ds=0.5, steps=4, nbatch=16),
        # the set-up before a flow: Hartree-Fock, and an observable taken to its basis
        dict(name="hf-emax8", op="hf", emax=8, kp=6, kn=6),
        # a scalar observable (a radius) in an odd-sized basis with a neutron excess, after a flow
        dict(name="observable-emax7", op="bch", emax=7, kp=3, kn=6, prec="fp64"),
        # electromagnetic operators after a flow: E1 in a small basis, E2 in the largest
        dict(name="tensor-e1-emax4", op="tensor", emax=4, kp=3, kn=3, rank=2, dpar=2),
        dict(name="tensor-e2-emax8", op="tensor", emax=8, kp=6, kn=6, rank=4, dpar=0),
        # sensitivities of the energy to every matrix element (forward and backward)
        dict(name="gradient-emax5", op="gradient", emax=5, kp=3, kn=3, gen="white", ds=0.5, steps=3),
    ]


def draw(rng):
    op = rng.choice(["ode", "flow", "flow", "batch", "hf", "bch", "tensor", "tensor", "gradient"])
    emax = rng.randint(2, {"batch": 6, "gradient": 6}.get(op, 8))
    fit = [k for k, e in zip(SHELLS, range(3)) if e < emax]
    c = dict(op=op, emax=emax, kp=rng.choice(fit), kn=rng.choice(fit))
    if op in ("ode", "flow", "batch"):
        c["gen"] = rng.choice(["white", "atan", "w2"])
    if op == "gradient":
        c["gen"] = rng.choice(["white", "atan"])
    if op in ("flow", "batch", "bch"):
        c["prec"] = rng.choice(["fp64", "int8x5", "int8x4"]) if emax > 6 else "fp64"
    if op in ("flow", "batch", "gradient"):
        c["ds"] = round(rng.uniform(0.2, 0.5), 3)
        c["steps"] = rng.randint(1, 3) if op == "gradient" else rng.randint(1, 4 if emax > 6 or op == "batch" else 12)
    if op == "batch":
        c["nbatch"] = rng.randint(2, 16)
    if op == "tensor":
        c["rank"], c["dpar"] = rng.choice([(2, 0), (2, 2), (4, 0), (6, 2)][: 3 if emax > 5 else 4])
    if op in ("ode", "hf", "bch", "tensor"):
        c["hw"] = round(rng.uniform(16.0, 24.0), 2)
    return c


# ---------------------------------------------------------------- inputs
def _orbits(case):
    orb = hk_orbits(case["emax"])
    cp, cn = (closed_shell_con(orb, case[k]) for k in ("kp", "kn"))
    return orb, [p if o[3] < 0 else n for o, p, n in zip(orb, cp, cn)]


@functools.lru_cache(maxsize=2)
def _plan(emax, kp, kn, prec, nbatch, graphs):
    """The context a program keeps for a basis, and where its streams are not zero: (basis, context, scale)."""
    basis = Basis.from_orbits(*_orbits(dict(emax=emax, kp=kp, kn=kn)))
    ctx = E.Context(basis, precision=PRECISION[prec], nbatch=nbatch)
    if graphs:
        ctx.set_graphs(True)
    allowed = [np.outer(basis.pauli_mask(b), basis.pauli_mask(b)).astype(float) for b in basis.blocks]
    scale = basis.vec_from_full(0.0, np.zeros((basis.nsp, basis.nsp)), allowed)
    return basis, ctx, scale


def _plan_of(case):
    return _plan(case["emax"], case["kp"], case["kn"], case.get("prec", "fp64"), case.get("nbatch", 1), case["op"] == "batch")


def _stream(basis, scale, rng, diag, s1, s2, herm=1):
    """An operator stream: one-body diagonal `diag` plus noise of width s1 within (l, j, tz), two-body noise of width s2."""
    n = basis.nsp
    up = np.triu(rng.normal(0.0, s1, (n, n)), 0 if herm == 1 else 1)
    f = np.where(basis.same_ljt(), up + herm * np.triu(up, 1).T, 0.0)
    if diag is not None:
        np.fill_diagonal(f, diag)
    v = scale * rng.normal(0.0, s2, basis.neq)
    h, p = basis.holes, basis.parts
    one = np.concatenate([f[np.ix_(a, b)].reshape(-1, order="F") for a, b in ((h, h), (p, p), (p, h))])
    v[0], v[1:1 + one.size] = 0.0, one
    return v


def _hamiltonian(basis, scale, rng, case):
    # Gaussian matrix elements as in the repository's workloads, narrower where more holes sum up in the mean
    # field, so that the gap above the filled shells stays open for every seed and the flow decouples
    width = {1: 1.0, 3: 0.5, 6: 0.3}[max(case["kp"], case["kn"])]
    return _stream(basis, scale, rng, case.get("hw", 20.0) * (2 * basis.n + basis.l + 1.5), 0.5, width)


def _tensor_stream(basis, rank, dpar, rng):
    """A hermitian tensor: selection rules, Pauli zeros, and the conjugate of every stored half where both halves are stored."""
    jj, l, tz = basis.jj.astype(int), basis.l.astype(int), basis.tz.astype(int)
    ok = ((abs(jj[:, None] - jj) <= rank) & (jj[:, None] + jj >= rank) & (tz[:, None] == tz)
          & ((l[:, None] + l + dpar // 2) % 2 == 0))
    up = np.triu(rng.uniform(-1, 1, ok.shape))
    f = np.where(ok, up + np.triu(up, 1).T * (1 - 2 * ((abs(jj[:, None] - jj) // 2) % 2)), 0.0)
    h, p = basis.holes, basis.parts
    out = [np.zeros(1)] + [f[np.ix_(a, b)].reshape(-1, order="F") for a, b in ((h, h), (p, p), (p, h))]
    blocks, square = {(b.J, b.Tz, b.P): b for b in basis.blocks}, {}
    for J1, J2, Tz, P1 in _tensor_blocks(max(b.J for b in basis.blocks), rank):
        P2 = P1 ^ (dpar // 2)
        b1, b2 = blocks[J1, Tz, P1], blocks[J2, Tz, P2]
        if b1.dim * b2.dim == 0:
            continue
        m = rng.uniform(-1, 1, (b1.dim, b2.dim))
        m[~basis.pauli_mask(b1)] = 0.0
        m[:, ~basis.pauli_mask(b2)] = 0.0
        if J1 == J2 and P1 == P2:
            m = 0.5 * (m + m.T)
        elif J1 == J2:
            m = square.pop((J1, Tz, P2)).T if (J1, Tz, P2) in square else square.setdefault((J1, Tz, P1), m)
        s1, s2 = ([0, b.npp, b.npp + b.nph, b.dim] for b in (b1, b2))
        out += [m[s1[r]:s1[r + 1], s2[c]:s2[c + 1]].reshape(-1, order="F") for r, c in TENSOR_PARTS]
    return np.concatenate(out)


#: row and column pair classes (pp, ph, hh) of a tensor block's nine parts
TENSOR_PARTS = ((0, 0), (0, 1), (0, 2), (1, 1), (2, 2), (1, 2), (2, 0), (1, 0), (2, 1))


def _tensor_blocks(jmax, rank):
    for J1 in range(0, jmax + 1, 2):
        for J2 in range(max(abs(J1 - rank), J1), min(J1 + rank, jmax) + 1, 2):
            for Tz in (-1, 0, 1):
                for P1 in (0, 1):
                    yield J1, J2, Tz, P1


def _inputs(case, seed, basis, scale):
    """The host streams of a case."""
    rng = np.random.default_rng([seed, case["emax"], case["kp"], case["kn"]])
    op = case["op"]
    if op == "batch":
        return {"h": np.stack([_hamiltonian(basis, scale, rng, case) for _ in range(case["nbatch"])])}
    d = {"h": _hamiltonian(basis, scale, rng, case)}
    if op in ("hf", "bch"):
        d["o"] = _stream(basis, scale, rng, None, 1.0, 0.1)
    if op == "tensor":
        d["t"] = _tensor_stream(basis, case["rank"], case["dpar"], rng)
    return d


def prepare(case, seed):
    basis, ctx, scale = _plan_of(case)
    d, op = _inputs(case, seed, basis, scale), case["op"]
    s = {"case": case, "ctx": ctx}
    if op == "gradient":
        s["h"] = torch.from_numpy(d["h"])
        return s
    h = ctx.op(1, d["h"])
    if op != "hf":
        h.normal_order()
    if op == "ode":
        s.update(y=h.download(), h=h, dh=ctx.op(1))
    elif op in ("flow", "batch"):
        s.update(h0=h, h=ctx.op(1), omega=ctx.op(-1))
    elif op == "hf":
        s.update(h0=h, h=ctx.op(1), o0=ctx.op(1, d["o"]), o=ctx.op(1))
    else:
        omega = ctx.generator("white", h)
        omega.scale(0.5)
        s.update(omega=omega)
        if op == "bch":
            s.update(o0=ctx.op(1, d["o"]), o=ctx.op(1))
        else:
            s.update(t0=ctx.tensor(case["rank"], case["dpar"], 1, d["t"]), t=ctx.tensor(case["rank"], case["dpar"], 1))
    ctx.sync()
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    c, ctx = s["case"], s["ctx"]
    op = c["op"]
    if op == "ode":
        s["h"].upload(s["y"])
        return ctx.dhds(s["h"], c["gen"], s["dh"]).download()
    if op == "flow":
        s["h"].copy_from(s["h0"])
        r = ctx.magnus_flow(s["h"], c["gen"], c["ds"], c["steps"], G=s["omega"])
        return {"steps": r["steps"], "e0": float(r["e0"][-1]), "h": s["h"].download(), "omega": s["omega"].download()}
    if op == "batch":
        s["h"].copy_from(s["h0"])
        flow = ctx.flow(s["h"], c["gen"], c["ds"], s["omega"])
        e0 = [[r["e0"] for r in flow.step()] for _ in range(c["steps"])]
        flow.close()
        return {"e0": np.array(e0), "h": s["h"].download(), "omega": s["omega"].download()}
    if op == "hf":
        s["h"].copy_from(s["h0"])
        s["o"].copy_from(s["o0"])
        D, e, _ = s["h"].hartree_fock()
        s["o"].to_hf(D)
        return {"D": D, "e": e, "h": s["h"].download(), "o": s["o"].download()}
    if op == "bch":
        s["o"].copy_from(s["o0"])
        n = ctx.transform_bch(s["o"], s["omega"])
        return {"n": n, "o": s["o"].download()}
    if op == "tensor":
        s["t"].copy_from(s["t0"])
        n = ctx.bch_tensor(s["omega"], s["t"])
        return {"n": n, "t": s["t"].download()}
    h = s["h"].detach().requires_grad_()
    e0 = flow_e0(h, ctx, c["gen"], c["ds"], c["steps"], ncheck=c["steps"])
    e0.backward()
    return {"e0": e0.detach(), "grad": h.grad}


# ---------------------------------------------------------------- work
def work(case):
    orb, con = _orbits(case)
    basis = Basis.from_orbits(orb, con)
    op, neq = case["op"], 8.0 * basis.neq
    ladder = sum(2.0 * b.dim * b.dim * (b.npp + b.nhh) for b in basis.blocks)
    comm = 2.2 * ladder  # ladders and Pandya products of one commutator (about equal)
    if op == "hf":
        # V' = U^T V U with U's few non-zero entries per column, for the Hamiltonian and the observable
        return {"bytes": 4 * neq, "flops": sum(2 * 2.0 * 2 * b.dim * b.dim * min(b.dim, 25) for b in basis.blocks)}
    if op == "tensor":
        blocks = {(b.J, b.Tz, b.P): b for b in basis.blocks}
        n = fl = 0.0
        for J1, J2, Tz, P1 in _tensor_blocks(max(b.J for b in basis.blocks), case["rank"]):
            b1, b2 = blocks[J1, Tz, P1], blocks[J2, Tz, P1 ^ (case["dpar"] // 2)]
            n += b1.dim * b2.dim
            fl += 2.0 * b1.dim * b2.dim * (b1.npp + b1.nhh + b2.npp + b2.nhh)
        return {"bytes": neq + 16.0 * n, "flops": 8 * 2 * fl}  # about 8 commutators, Pandya products like the ladders
    steps = {2: 15, 4: 26}.get(case["emax"], 26) if case.get("steps", 0) >= 200 else case.get("steps", 1)
    count = {"ode": 1 + (case.get("gen") == "w2"), "flow": 15 * steps, "batch": 15 * steps * case.get("nbatch", 1),
             "bch": 9, "gradient": 15 * 5 * steps}[op]
    return {"bytes": (3 if op in ("flow", "batch", "bch") else 2) * neq * case.get("nbatch", 1), "flops": count * comm}


# ---------------------------------------------------------------- 64-bit values
def _sixj(js, nJ):
    """{a b J; c d K} over the doubled j's in js and integer J, K < nJ, indexed [J, K, a, b, c, d] (Racah's sum)."""
    j = np.array(js) / 2.0
    J, K, a, b, c, d = np.meshgrid(np.arange(nJ), np.arange(nJ), j, j, j, j, indexing="ij", sparse=True)
    lf = np.array([math.lgamma(n + 1.0) for n in range(200)])
    fact = lambda x: lf[np.clip(np.rint(x).astype(int), 0, 199)]  # noqa: E731

    def delta(x, y, z):
        good = (x + y >= z) & (abs(x - y) <= z)
        return good, 0.5 * (fact(x + y - z) + fact(x - y + z) + fact(y + z - x) - fact(x + y + z + 1))

    tri = [delta(a, b, J), delta(c, d, J), delta(a, d, K), delta(c, b, K)]
    good = tri[0][0] & tri[1][0] & tri[2][0] & tri[3][0]
    lead = tri[0][1] + tri[1][1] + tri[2][1] + tri[3][1]
    lows, highs = (a + b + J, c + d + J, a + d + K, c + b + K), (a + b + c + d, b + J + d + K, J + a + K + c)
    out = np.zeros(good.shape)
    for t in range(4 * nJ + 4):
        term = lead + fact(t + 1)
        ok = good
        for x in lows:
            ok, term = ok & (t >= x - 1e-9), term - fact(t - x)
        for x in highs:
            ok, term = ok & (t <= x + 1e-9), term - fact(x - t)
        out += np.where(ok, (-1.0) ** t * np.exp(np.where(ok, term, 0.0)), 0.0)
    return out


class _Dense:
    """Scalar operators (e0, f[a, b], V[J, a, b, c, d] over ordered pairs, unnormalised) of one basis."""

    def __init__(self, orbits, con):
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        orb = np.array(orbits)
        self.n, self.l, self.j, self.tz = orb.T
        self.con, self.N, self.nJ = np.array(con), len(orb), int(self.j.max()) + 1
        N, j, nJ = self.N, self.j, self.nJ
        self.hol, self.par = np.flatnonzero(self.con == 1), np.flatnonzero(self.con == 0)
        self.blocks = self._pairs()
        kind = (self.l * 2 + (self.tz > 0)) * 100 + j
        self.same = self._t(kind[:, None] == kind[None, :])
        # where the entries of a stream go: position, factor, and whether the entry is a mirror image
        h, p = self.hol, self.par
        fpos, fmir = np.zeros((N, N), np.int64), np.zeros((N, N), bool)
        k = 1
        for rows, cols in ((h, h), (p, p), (p, h)):
            m = len(rows) * len(cols)
            fpos[np.ix_(rows, cols)] = k + np.arange(m).reshape(len(cols), len(rows)).T
            k += m
        fpos[np.ix_(h, p)], fmir[np.ix_(h, p)] = fpos[np.ix_(p, h)].T, True
        vpos, vfac = np.zeros((nJ, N, N, N, N), np.int64), np.zeros((nJ, N, N, N, N))
        vmir = np.zeros((nJ, N, N, N, N), bool)
        back, inv = [], []
        for (J, _, _), cls in self.blocks.items():
            dims = np.cumsum([0] + [len(x) for x in cls])
            pr = np.concatenate(cls)
            pos, mir = np.zeros((dims[3], dims[3]), np.int64), np.zeros((dims[3], dims[3]), bool)
            for r, c in ((0, 0), (0, 1), (0, 2), (1, 1), (2, 2), (1, 2)):
                R, C = np.meshgrid(np.arange(dims[r], dims[r + 1]), np.arange(dims[c], dims[c + 1]), indexing="ij")
                R, C = R.T.reshape(-1), C.T.reshape(-1)  # column by column
                if r == c:
                    R, C = R[R >= C], C[R >= C]
                at = k + np.arange(len(R))
                k += len(R)
                pos[C, R], mir[C, R] = at, True
                pos[R, C], mir[R, C] = at, False
                a, b, x, y = pr[R, 0], pr[R, 1], pr[C, 0], pr[C, 1]
                back.append((((J * N + a) * N + b) * N + x) * N + y)
                inv.append(1.0 / (np.where(a == b, 2 ** 0.5, 1.0) * np.where(x == y, 2 ** 0.5, 1.0)))
            a, b = pr.T
            norm = np.where(a == b, 2 ** 0.5, 1.0)
            flip = np.where((((j[a] + j[b]) // 2 - J) % 2) == 0, -1.0, 1.0) * norm
            sides = ((b, a, flip), (a, b, norm))
            for s1, s2, sp in sides:
                for t1, t2, tp in sides:
                    at = (J, s1[:, None], s2[:, None], t1[None, :], t2[None, :])
                    vpos[at], vfac[at], vmir[at] = pos, sp[:, None] * tp[None, :], mir
        self.neq = k
        self.fpos, self.vpos, self.vfac = self._t(fpos), self._t(vpos), self._t(vfac)
        self.fmir, self.vmir = self._t(fmir), self._t(vmir)
        self.back, self.inv = self._t(np.concatenate(back)), self._t(np.concatenate(inv))
        self.fback = self._t(np.concatenate([(a[:, None] * N + b).T.reshape(-1) for a, b in ((h, h), (p, p), (p, h))]))
        self.occ = self._t(self.con.astype(float))
        self.J1 = self._t(2.0 * np.arange(nJ) + 1.0)
        self.d = self._t(j + 1.0)
        ph = (j[:, None] + j[None, :]) // 2 - np.arange(nJ)[:, None, None]
        self.swap = self._t(np.where(ph % 2 == 0, 1.0, -1.0))  # (-1)^(ja + jb - J)
        self.nn = self.occ[:, None] - self.occ[None, :]

    def _t(self, x):
        return torch.from_numpy(np.ascontiguousarray(x)).to(self.dev)

    def _pairs(self):
        N, j, l, tz, out = self.N, self.j, self.l, self.tz, {}
        a, b = np.triu_indices(N)
        cls = self.con[a] + self.con[b]
        for J in range(self.nJ):
            for T in (-1, 0, 1):
                for P in (0, 1):
                    ok = ((tz[a] + tz[b] == 2 * T) & ((l[a] + l[b]) % 2 == P) & (abs(j[a] - j[b]) <= 2 * J)
                          & (j[a] + j[b] >= 2 * J))
                    if ok.any():
                        out[J, T, P] = [np.stack([a, b], 1)[ok & (cls == c)] for c in (0, 1, 2)]
        return out

    @functools.cached_property
    def six(self):
        js = sorted(set(self.j.tolist()))
        at = self._t(np.array([js.index(x) for x in self.j.tolist()]))
        s = self._t(_sixj(js, self.nJ))
        for dim in (2, 3, 4, 5):
            s = s.index_select(dim, at)
        return s

    def op(self, v, herm=1):
        """A stream as an operator."""
        f = v[self.fpos] * torch.where(self.fmir, float(herm), 1.0)
        return v[0], f, v[self.vpos] * self.vfac * torch.where(self.vmir, float(herm), 1.0)

    def vec(self, A):
        return torch.cat([A[0].reshape(1), A[1].reshape(-1)[self.fback], A[2].reshape(-1)[self.back] * self.inv])

    def recouple(self, X):
        X = X.permute(0, 1, 4, 3, 2) * self.J1.view(-1, 1, 1, 1, 1)
        return -torch.stack([(self.six[J] * X).sum(0) for J in range(self.nJ)])

    def commutator(self, A, B):
        if any(x.requires_grad for x in A + B):  # keep the operands alone for the backward pass
            return torch.utils.checkpoint.checkpoint(lambda *x: self._commutator(x[:3], x[3:]), *A, *B, use_reentrant=False)
        return self._commutator(A, B)

    def _commutator(self, A, B):
        occ, N, nJ = self.occ, self.N, self.nJ
        un, w = 1 - occ, self.J1
        m = lambda X: X.reshape(nJ, N * N, N * N)  # noqa: E731
        (_, fa, va), (_, fb, vb) = A, B
        hh, pp = torch.outer(occ, occ).reshape(-1), torch.outer(un, un).reshape(-1)
        e0 = torch.einsum("a,ab,ba->", self.d, self.nn * fa, fb)
        ab = (m(va) * hh.view(1, -1, 1)) @ (m(vb) * pp.view(1, -1, 1))
        ba = (m(vb) * hh.view(1, -1, 1)) @ (m(va) * pp.view(1, -1, 1))
        e0 = e0 + 0.25 * (w * (torch.diagonal(ab - ba, dim1=1, dim2=2) * hh).sum(1)).sum()
        # one body
        f = fa @ fb - fb @ fa
        f = f + torch.einsum("J,ab,Jbiaj->ij", w, self.nn * fa, vb) / self.d[:, None]
        f = f - torch.einsum("J,ab,Jbiaj->ij", w, self.nn * fb, va) / self.d[:, None]
        mid = (m(va) * pp) @ m(vb) - (m(vb) * pp) @ m(va)
        mih = (m(va) * hh) @ m(vb) - (m(vb) * hh) @ m(va)
        Mp, Mh = (x.reshape(nJ, N, N, N, N) for x in (mid, mih))
        s = torch.einsum("J,c,Jcicj->ij", w, occ, Mp) + torch.einsum("J,c,Jcicj->ij", w, un, Mh)
        f = torch.where(self.same, f + 0.5 * s / self.d[:, None], 0.0)
        # two body: one-body parts, ladders, particle-hole
        V = 0.5 * (Mp - Mh)
        for g, X, sg in ((fa, vb, 1.0), (fb, va, -1.0)):
            V = V + sg * (torch.einsum("ia,Jajkl->Jijkl", g, X) + torch.einsum("ja,Jiakl->Jijkl", g, X)
                          - torch.einsum("ak,Jijal->Jijkl", g, X) - torch.einsum("al,Jijka->Jijkl", g, X))
        Pa, Pb = self.recouple(va), self.recouple(vb)
        Z = ((m(Pa) * self.nn.reshape(-1)) @ m(Pb)).reshape(nJ, N, N, N, N)
        Z = self.recouple(Z)
        bra, ket = self.swap.view(nJ, N, N, 1, 1), self.swap.view(nJ, 1, 1, N, N)
        Z = Z - bra * Z.transpose(1, 2)
        return e0, f, V - Z + ket * Z.transpose(3, 4)

    def axpy(self, a, X, Y):
        return tuple(a * x + y for x, y in zip(X, Y))

    def norm(self, A):
        return float(((A[1] ** 2).sum() + 0.25 * (A[2] ** 2).sum()).detach()) ** 0.5

    def normal_order(self, A):
        _, f, V = A
        occ, w = self.occ, self.J1
        e = (self.d * occ * torch.diagonal(f)).sum() + 0.5 * torch.einsum("J,a,b,Jabab->", w, occ, occ, V)
        g = torch.einsum("J,h,Jahbh->ab", w, occ, V) / self.d[:, None]
        return e, torch.where(self.same, f + g, 0.0), V

    def generator(self, kind, H, num=None):
        num = num or H
        if kind == "w2":
            e1 = self.generator("atan", H)
            e2 = self.generator("atan", H, self.commutator(e1, H))
            return tuple(1.5 * x + 0.5 * y for x, y in zip(e1, e2))
        _, f, V = H
        mono = torch.einsum("J,Jabab->ab", self.J1, V) / torch.outer(self.d, self.d)
        eps, ph = torch.diagonal(f), torch.outer(1 - self.occ, self.occ) > 0
        dis = lambda x, den: x / den if kind == "white" else 0.5 * torch.atan(2 * x / den)  # noqa: E731
        one = torch.where(ph & self.same, eps[:, None] - eps[None, :] - mono, 1.0)
        E1 = torch.where(ph & self.same, dis(num[1], one), 0.0)
        v4 = lambda x, *at: x.reshape([self.N if k in at else 1 for k in range(4)])  # noqa: E731
        den = (v4(mono, 0, 1) + v4(mono, 2, 3) - v4(mono, 0, 2) - v4(mono, 0, 3) - v4(mono, 1, 2) - v4(mono, 1, 3)
               + v4(eps, 0) + v4(eps, 1) - v4(eps, 2) - v4(eps, 3))
        un = 1 - self.occ
        two = v4(un, 0) * v4(un, 1) * v4(self.occ, 2) * v4(self.occ, 3) > 0
        same = torch.eye(self.N, dtype=torch.float64, device=self.dev) * (2 ** 0.5 - 1) + 1
        size = v4(same, 0, 1) * v4(same, 2, 3)  # the generator acts on normalised elements
        E2 = torch.where(two, size * dis(num[2] / size, torch.where(two, den, 1.0)), 0.0)
        return 0.0 * H[0], E1 - E1.T, E2 - E2.permute(0, 3, 4, 1, 2)

    def mbpt2(self, H):
        eps, h, p = torch.diagonal(H[1]), self._t(self.hol), self._t(self.par)
        X = H[2].index_select(1, p).index_select(2, p).index_select(3, h).index_select(4, h)
        den = eps[h].view(1, 1, -1, 1) + eps[h] - eps[p].view(-1, 1, 1, 1) - eps[p].view(1, -1, 1, 1)
        return 0.25 * (self.J1.view(-1, 1, 1, 1, 1) * X ** 2 / den).sum()

    def bch(self, G, H):
        out, ad, coef, n = H, H, 1.0, 0
        while n < 39:
            ad, n = self.commutator(G, ad), n + 1
            coef /= n
            out = self.axpy(coef, ad, out)
            if self.norm(ad) * coef < 1e-6:
                break
        return out, n

    def magnus(self, D, G):
        cof, size, full = (1.0, -0.5, 1.0 / 12, 0.0, -1.0 / 720, 0.0, 1.0 / 30240), [self.norm(D)], self.norm(G)
        out, ad, q = D, D, 1
        for i in range(1, 7):
            if full < 1e-9 or size[i - q] / full < 1e-6:
                break
            q = 1 if cof[i] else 2
            ad = self.commutator(G, ad)
            out = self.axpy(cof[i], ad, out)
            size.append(self.norm(ad) * abs(cof[i]))
        return out[0] * 0.0, out[1], out[2]

    def flow(self, H0, kind, ds, steps):
        D = self.generator(kind, H0)
        G, H = tuple(0.0 * x for x in D), H0
        e0, crit = [], [abs(float(self.mbpt2(H0).detach()))]
        while crit[-1] > 1e-6 and len(e0) < steps:
            G = self.axpy(ds, self.magnus(D, G), G)
            H, _ = self.bch(G, H0)
            D = self.generator(kind, H)
            e0.append(H[0])
            crit.append(abs(float(self.mbpt2(H).detach())))
        return torch.stack(e0), H, G

    def rotate(self, A, D):
        V = A[2]
        for dim in range(1, 5):
            V = torch.tensordot(V, D, ([dim], [0])).movedim(-1, dim)
        return A[0], D.T @ A[1] @ D, V

    def hartree_fock(self, A):
        groups, eig, D = {}, None, torch.eye(self.N, dtype=torch.float64, device=self.dev)
        for k in range(self.N):
            groups.setdefault((self.l[k], self.j[k], self.tz[k]), []).append(k)
        K = torch.einsum("J,Jabcd->abcd", self.J1, A[2])
        while True:
            g = torch.einsum("abcd,bx,dx,x->ac", K, D, D, self.occ) / self.d[:, None]
            F = torch.where(self.same, A[1] + g, 0.0)
            last, eig, D = eig, torch.zeros(self.N, dtype=torch.float64, device=self.dev), torch.zeros_like(D)
            for at in groups.values():
                e, u = torch.linalg.eigh(F[at][:, at])
                for c, k in enumerate(at):
                    D[at, k] = u[:, c]
                eig[at] = e
            if last is not None and sum(float(((eig - last)[at] ** 2).sum()) ** 0.5 for at in groups.values()) <= 1e-6:
                break
        D = D * torch.where(torch.diagonal(D) < 0, -1.0, 1.0)
        rot = self.rotate((A[0], F, A[2]), D)
        T = torch.diagonal(D.T @ A[1] @ D)
        e = (self.d * self.occ * (T + 0.5 * (torch.diagonal(rot[1]) - T))).sum()
        return D, e, (e, rot[1], rot[2])


def _clebsch(ja, ma, jb, mb, J, M):
    """<ja ma jb mb | J M>, everything doubled."""
    if ma + mb != M or not abs(ja - jb) <= J <= ja + jb or abs(M) > J:
        return 0.0
    f = lambda x: math.factorial(x // 2)  # noqa: E731
    pre = ((J + 1) * f(J + ja - jb) * f(J - ja + jb) * f(ja + jb - J) / f(ja + jb + J + 2)
           * f(J + M) * f(J - M) * f(ja - ma) * f(ja + ma) * f(jb - mb) * f(jb + mb))
    s = 0.0
    for k in range(0, ja + jb + J + 2, 2):
        den = (k, ja + jb - J - k, ja - ma - k, jb + mb - k, J - jb + ma + k, J - ja - mb + k)
        if min(den) >= 0:
            s += (-1) ** (k // 2) / math.prod(f(x) for x in den)
    return math.sqrt(pre) * s


class _MScheme:
    """The commutator of a scalar with the zero component of a rank-lambda tensor over single-particle m-states."""

    def __init__(self, d, rank):
        self.d, self.rank = d, rank
        st = [(a, m) for a in range(d.N) for m in range(-d.j[a], d.j[a] + 1, 2)]
        self.n, dev = len(st), d.dev
        self.orb = d._t(np.array([a for a, _ in st]))
        self.occ = d.occ[self.orb]
        n, js = self.n, sorted(set(d.j.tolist()))
        small = {(ja, ma, jb, mb, J): _clebsch(ja, ma, jb, mb, 2 * J, ma + mb) for ja in js for jb in js
                 for ma in range(-ja, ja + 1, 2) for mb in range(-jb, jb + 1, 2) for J in range(d.nJ)}
        self.C = []
        for J in range(d.nJ):
            c = np.zeros((n, n, 2 * J + 1))
            for x, (a, ma) in enumerate(st):
                for y, (b, mb) in enumerate(st):
                    M = (ma + mb) // 2
                    if abs(M) <= J:
                        c[x, y, M + J] = small[d.j[a], ma, d.j[b], mb, J]
            self.C.append(d._t(c.reshape(n * n, -1)))
        self.one = torch.zeros(n, d.N, dtype=torch.float64, device=dev)
        self.one[torch.arange(n, device=dev), self.orb] = 1.0
        w = np.zeros((n, n))
        for x, (a, ma) in enumerate(st):
            for y, (b, mb) in enumerate(st):
                if ma == mb:
                    w[x, y] = self._reduce(d.j[a], d.j[b], ma)
        self.w1 = d._t(w)
        self.delta = d._t(np.array([[a[1] == b[1] for b in st] for a in st], float))
        i, j = np.triu_indices(n, 1)
        self.up = d._t(i * n + j)
        self.upi, self.upj = d._t(i), d._t(j)

    def _reduce(self, J1, J2, M):
        """<J1 M|T_0|J2 M> / <J1||T||J2>, everything doubled"""
        return _clebsch(J2, M, self.rank, 0, J1, M) / math.sqrt(J1 + 1)

    def _coupled(self, J1, J2):
        w = self.d._t(np.array([[self._reduce(2 * J1, 2 * J2, 2 * M) if M == K else 0.0 for K in range(-J2, J2 + 1)]
                                for M in range(-J1, J1 + 1)], float))
        return (self.C[J1] @ w @ self.C[J2].T).reshape([self.n] * 4), float((w * w).sum())

    def _spread(self, X):
        o = self.orb
        return X[o][:, o][:, :, o][:, :, :, o]

    def _gather(self, X):
        for dim in range(4):
            X = torch.tensordot(X, self.one, ([0], [0]))
        return X

    def scalar(self, G):
        V = torch.zeros([self.n] * 4, dtype=torch.float64, device=self.d.dev)
        for J in range(self.d.nJ):
            V += (self.C[J] @ self.C[J].T).reshape(V.shape) * self._spread(G[2][J])
        return G[1][self.orb][:, self.orb] * self.delta, V

    def tensor(self, f, blocks):
        V = torch.zeros([self.n] * 4, dtype=torch.float64, device=self.d.dev)
        for (J1, J2), X in blocks.items():
            V += self._coupled(J1, J2)[0] * self._spread(X)
        return f[self.orb][:, self.orb] * self.w1, V

    def reduced(self, T, pairs):
        norm = self.one.T @ (self.w1 ** 2) @ self.one
        f = self.one.T @ (T[0] * self.w1) @ self.one / torch.where(norm > 0, norm, 1.0)
        out = {}
        for J1, J2 in pairs:
            k, w2 = self._coupled(J1, J2)
            out[J1, J2] = self._gather(T[1] * k) / w2 if w2 > 0 else torch.zeros([self.d.N] * 4, dtype=torch.float64)
        return f, out

    def commutator(self, A, B):
        n, occ = self.n, self.occ
        (fa, va), (fb, vb) = A, B
        nn = occ[:, None] - occ[None, :]
        f = fa @ fb - fb @ fa
        f = f + torch.einsum("ab,biaj->ij", nn * fa, vb) - torch.einsum("ab,biaj->ij", nn * fb, va)
        m = lambda X: X.reshape(n * n, n * n)  # noqa: E731
        a, b = (m(X)[self.up][:, self.up] for X in (va, vb))
        oi, oj = occ[self.upi], occ[self.upj]
        full, V = [], torch.zeros(n * n, n * n, dtype=torch.float64, device=f.device)
        low = (self.up % n) * n + self.up // n
        for q in ((1 - oi) * (1 - oj), oi * oj):
            at = torch.nonzero(q).reshape(-1)
            x = a[:, at] @ b[at] - b[:, at] @ a[at]
            y = torch.zeros_like(V)
            for r, sr in ((self.up, 1.0), (low, -1.0)):
                for c, sc in ((self.up, 1.0), (low, -1.0)):
                    y[r[:, None], c[None, :]] = sr * sc * x
            full.append(y.reshape([n] * 4))
        f = f + torch.einsum("c,cicj->ij", occ, full[0]) + torch.einsum("c,cicj->ij", 1 - occ, full[1])
        V = full[0] - full[1]
        for g, X, sg in ((fa, vb, 1.0), (fb, va, -1.0)):
            left = torch.tensordot(g, X, 1)
            V += sg * (left - left.transpose(0, 1))
            right = torch.tensordot(X, g, ([3], [0]))
            V -= sg * (right - right.transpose(2, 3))
        at = torch.nonzero(nn.reshape(-1)).reshape(-1)
        pick = lambda X, p: m(X.permute(*p))  # noqa: E731
        x = (pick(va, (1, 3, 0, 2))[:, at] * nn.reshape(-1)[at]) @ pick(vb, (2, 0, 1, 3))[at]
        x = x.reshape([n] * 4).permute(0, 2, 1, 3)  # [i, j, k, l] = sum (na - nb) A_aibk B_bjal
        x = x - x.transpose(0, 1)
        return f, V + x - x.transpose(2, 3)


def _exact_tensor(case, d, h, t):
    """BCH of a tensor stream, through the m-scheme."""
    dev, N, rank = d.dev, d.N, case["rank"]
    H = d.normal_order(d.op(h))
    G = tuple(0.5 * x for x in d.generator("white", H))
    f = torch.zeros(N, N, dtype=torch.float64, device=dev)
    parts, k, at = ((d.hol, d.hol), (d.par, d.par), (d.par, d.hol)), 1, []
    for r, c in parts:
        R, C = (d._t(np.ascontiguousarray(x.T).reshape(-1)) for x in np.meshgrid(r, c, indexing="ij"))
        f[R, C] = t[k:k + len(R)]
        at.append((R, C))
        k += len(R)
    sgn = d._t(np.where((abs(d.j[:, None] - d.j) // 2) % 2 == 0, 1.0, -1.0))
    h_, p_ = d._t(d.hol), d._t(d.par)
    f[h_[:, None], p_] = (f * sgn)[p_[:, None], h_].T
    blocks, where = {}, []
    for J1, J2, T, P in _tensor_blocks(2 * d.nJ - 2, rank):
        k1, k2 = (J1 // 2, T, P), (J2 // 2, T, P ^ (case["dpar"] // 2))
        if k1 not in d.blocks or k2 not in d.blocks:
            continue
        X = blocks.setdefault((k1[0], k2[0]), torch.zeros([N] * 4, dtype=torch.float64, device=dev))
        for r, c in TENSOR_PARTS:
            R, C = d.blocks[k1][r], d.blocks[k2][c]
            i, j = (x.T.reshape(-1) for x in np.meshgrid(np.arange(len(R)), np.arange(len(C)), indexing="ij"))
            if not len(i):
                continue
            (a, b), (x, y) = R[i].T, C[j].T
            s1, s2 = (np.where(u == v, 2 ** 0.5, 1.0) for u, v in ((a, b), (x, y)))
            q1, q2 = (np.where(((d.j[u] + d.j[v]) // 2 - J // 2) % 2 == 0, -1.0, 1.0) for u, v, J in ((a, b, J1), (x, y, J2)))
            val, fac = t[k:k + len(i)], d._t(s1 * s2)
            k += len(i)
            where.append(((k1[0], k2[0]), tuple(d._t(z) for z in (a, b, x, y)), 1.0 / fac))
            for u, v, s in ((b, a, q1), (a, b, 1.0)):
                for w, z, s_ in ((y, x, q2), (x, y, 1.0)):
                    X[tuple(d._t(e) for e in (u, v, w, z))] = val * fac * d._t(s * s_ * np.ones(len(i)))
    flip = {}
    for (J1, J2), X in blocks.items():  # the halves with J1 > J2, by hermiticity
        flip[J1, J2] = X
        if J1 != J2:
            flip[J2, J1] = (-1.0) ** (J1 - J2) * X.permute(2, 3, 0, 1)
    m = _MScheme(d, rank)
    Gm, Tm = m.scalar(G), m.tensor(f, flip)
    out, ad, coef, n = Tm, Tm, 1.0, 0
    while n < 29:
        ad, n = m.commutator(Gm, ad), n + 1
        coef /= n
        out = tuple(x + coef * y for x, y in zip(out, ad))
        fr, bl = m.reduced(ad, list(blocks))
        size = float((fr ** 2).sum() + 0.25 * sum((x ** 2).sum() for x in bl.values())) ** 0.5
        if size * coef < 1e-6:
            break
    fr, bl = m.reduced(out, list(blocks))
    res = [torch.zeros(1, dtype=torch.float64, device=dev)] + [fr[R, C] for R, C in at]
    res += [bl[key][idx] * inv for key, idx, inv in where]
    return {"n": None, "t": torch.cat(res).cpu()}


def exact(case, seed):
    op, emax, gpu = case["op"], case["emax"], torch.cuda.is_available()
    # dense 64-bit values take seconds up to emax 4 on a GPU (one commutator or series: emax 6), and emax 2 or 3 without
    largest = {"batch": 0, "ode": 6, "bch": 6, "hf": 6}.get(op, 4) if gpu else {"batch": 0, "tensor": 2}.get(op, 3)
    if emax > largest or case.get("prec", "fp64") != "fp64":
        return None
    torch.set_default_dtype(torch.float64)
    try:
        orb, con = _orbits(case)
        basis = Basis.from_orbits(orb, con)  # only to draw the same inputs
        scale = basis.vec_from_full(0.0, np.zeros((basis.nsp, basis.nsp)),
                                    [np.outer(basis.pauli_mask(b), basis.pauli_mask(b)).astype(float) for b in basis.blocks])
        d, x = _Dense(orb, con), _inputs(case, seed, basis, scale)
        h = torch.from_numpy(x["h"]).to(d.dev)
        if op == "tensor":
            return _exact_tensor(case, d, h, torch.from_numpy(x["t"]).to(d.dev))
        if op == "hf":
            D, e, H = d.hartree_fock(d.op(h))
            O = d.normal_order(d.rotate(d.op(torch.from_numpy(x["o"]).to(d.dev)), D))
            return {"D": D.cpu(), "e": float(e), "h": d.vec(H).cpu(), "o": d.vec(O).cpu()}
        if op == "gradient":
            h.requires_grad_()
            e0 = d.flow(d.normal_order(d.op(h)), case["gen"], case["ds"], case["steps"])[0][-1]
            e0.backward()
            return {"e0": e0.detach().cpu(), "grad": h.grad.cpu()}
        H = d.normal_order(d.op(h))
        if op == "ode":
            return d.vec(d.commutator(d.generator(case["gen"], H), H)).cpu()
        if op == "bch":
            G = tuple(0.5 * y for y in d.generator("white", H))
            O, _ = d.bch(G, d.op(torch.from_numpy(x["o"]).to(d.dev)))
            return {"n": None, "o": d.vec(O).cpu()}
        e0, H, G = d.flow(H, case["gen"], case["ds"], case["steps"])
        return {"steps": None, "e0": float(e0[-1]), "h": d.vec(H).cpu(), "omega": d.vec(G).cpu()}
    finally:
        torch.set_default_dtype(torch.float32)
