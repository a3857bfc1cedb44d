"""Measured cases of the two-site DMRG path: effective-Hamiltonian matvecs, Lanczos ground states, batches
of independent problems, the drop-in call on host tensors and a whole DMRG run.

A case is a dict of plain values:

  call       "matvec" (a plan applied to a device vector), "lanczos" (ground state on a plan),
             "batch" / "batch_lanczos" (independent problems in one batched plan),
             "apply" (apply_local_hamiltonian on host tensors), "dmrg" (a whole run from a random state)
  model      "hubbard", "xxz" or "molecular"; the batches mix Hubbard and XXZ chains
  nsites     chain length (molecular: orbitals); chi: dimension of both outer bonds (dmrg: max_vdim)
  bond       how the outer bonds' quantum numbers lie:
             "random"  as construct_random_mps draws them, blocks N(0,1): the synthetic problem of bench.py
             "sweep"   a normal distribution around the filling with a width of one particle, which is what
                       the bonds of a converged state look like (few, large, ragged sectors); the
                       environments are those of a random state with these bonds, so that the effective
                       Hamiltonian is symmetric as in a sweep
  form       "grouped" (the default form of a plan) or "pair" (the form for many small sectors)
  structure  seed of the quantum numbers; the entries come from the seed that prepare() is given

The split-FP32 form is left out: it is slower than the FP64 forms at every size, and kept as an option.
"""

import ctypes
import math
from collections import Counter

import numpy as np
import torch

import chemtensor_amd as ct
import chemtensor_amd.compat as compat

OUT, IN = ct.AXIS_OUT, ct.AXIS_IN
FORMS = {"grouped": ct.GROUPED_FP64, "pair": ct.PAIR_FP64}
LANCZOS_STEPS = 20        # per ground state, the default of chemtensor.dmrg
DMRG_SWEEPS = 3


# ---------------------------------------------------------------------------------------------------
# the cases

def listed():
    def c(name, call, model, nsites, chi, bond="random", form="grouped", structure=2024, count=1):
        return dict(name=name, call=call, model=model, nsites=nsites, chi=chi, bond=bond, form=form, structure=structure, count=count)

    return [
        # a small two-site problem (the ends of a chain, a first sweep with few states): latency and launches
        c("matvec_small", "matvec", "hubbard", 16, 32),
        # the headline benchmark: the centre bond of a Hubbard chain with scattered quantum numbers
        c("matvec_headline", "matvec", "hubbard", 32, 512, form="pair"),
        # ordinary and large centre bonds of a converged state, Hubbard (two conserved numbers, many sectors)
        c("matvec_hubbard_512", "matvec", "hubbard", 16, 512, bond="sweep"),
        c("matvec_hubbard_2000", "matvec", "hubbard", 16, 2000, bond="sweep"),
        # one conserved number, few and large sectors, an odd bond dimension
        c("matvec_xxz_515", "matvec", "xxz", 24, 515, bond="sweep"),
        # quantum chemistry: MPO bonds of hundreds, the contraction is bound by the matrix cores
        c("matvec_molecular", "matvec", "molecular", 20, 512),
        # a bond's eigenproblem inside a sweep, on either form
        c("lanczos_headline", "lanczos", "hubbard", 32, 512, form="pair"),
        c("lanczos_hubbard_512", "lanczos", "hubbard", 16, 512, bond="sweep"),
        # many independent chains in one launch per stage (chi from 64 to 1024), and their eigenproblems
        # as the serving loop solves them
        c("batch_64", "batch", "mixed", 64, 1024, count=64),
        c("batch_lanczos_16", "batch_lanczos", "mixed", 64, 256, bond="sweep", count=16),
        # the drop-in call on host tensors, everything included
        c("apply_hubbard_256", "apply", "hubbard", 16, 256, bond="sweep"),
        # a whole run as chemtensor.dmrg does it
        c("dmrg_hubbard_8", "dmrg", "hubbard", 8, 128),
    ]


def draw(rng):
    """One more case of the listed ranges."""
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["matvec", "matvec", "matvec", "pair", "molecular", "lanczos", "lanczos_pair", "batch", "batch_lanczos", "apply", "dmrg"])
    model = rng.choice(["hubbard", "xxz"])
    bond = rng.choice(["random", "sweep", "sweep"])
    c = dict(call="matvec", model=model, nsites=2 * rng.randint(8, 16), chi=logint(24, 1600), bond=bond, form="grouped",
             structure=rng.randrange(1 << 20), count=1)
    if kind in ("matvec", "lanczos", "apply"):
        c["call"] = kind
        if kind != "matvec":
            c["chi"] = logint(24, 800)
        if kind == "lanczos":
            c["bond"] = "sweep"
    elif kind in ("pair", "lanczos_pair"):
        # the form for scattered quantum numbers
        c.update(call="matvec" if kind == "pair" else "lanczos", model="hubbard", nsites=2 * rng.randint(12, 24), bond="random", form="pair",
                 chi=logint(64, 600))
    elif kind == "molecular":
        c.update(model="molecular", nsites=2 * rng.randint(3, 9), bond="random", chi=logint(48, 512))
    elif kind == "batch":
        c.update(call=kind, model="mixed", nsites=64, bond="random", chi=logint(128, 1000), count=rng.randint(4, 48))
    elif kind == "batch_lanczos":
        c.update(call=kind, model="mixed", nsites=64, bond="sweep", chi=logint(48, 250), count=rng.randint(2, 14))
    else:
        hub = model == "hubbard"
        c.update(call=kind, nsites=rng.randint(5, 8) if hub else rng.randint(8, 14), bond="random", chi=logint(12, 120))
    if c["call"] != "dmrg" and c["bond"] == "sweep" and c["model"] == "xxz":
        c["nsites"] = 2 * rng.randint(11, 16)     # 2^(half chain) states have to reach chi
    return c


# ---------------------------------------------------------------------------------------------------
# quantum numbers and operands

def mpo_of(model, nsites, structure):
    if model == "hubbard":
        return ct.MPO.hubbard(nsites, 1.0, 4.0, 0.0)
    if model == "xxz":
        return ct.MPO.xxz(nsites, 1.0, 0.5, 0.0)
    return ct.MPO.spin_molecular(*ct.molecular_coefficients(nsites, structure))


def sector_of(model, nsites):
    return 0 if model == "xxz" else ct.encode_pair(nsites, 0)


class Site:
    """A site tensor of an MPO, as the entry points take it."""

    def __init__(self, mpo, i):
        self.mpo, self.ptr = mpo, ctypes.cast(ctypes.pointer(mpo.s.a[i]), ctypes.c_void_p)


def sweep_bond(model, sites, chi, rng):
    """Quantum numbers of a bond `sites` sites from the left end, as a converged state has them: up to chi
    states, normally distributed around the filling with a width of about one particle per species."""
    if model == "hubbard":
        ways = {(u, d): math.comb(sites, u) * math.comb(sites, d) for u in range(sites + 1) for d in range(sites + 1)}
        weight = {k: math.exp(-((k[0] - sites / 2) ** 2 + (k[1] - sites / 2) ** 2) / 2.14) for k in ways}
        number = {k: ct.encode_pair(k[0] + k[1], k[0] - k[1]) for k in ways}
    else:
        ways = {(u,): math.comb(sites, u) for u in range(sites + 1)}
        weight = {k: math.exp(-((k[0] - sites / 2) ** 2) / 2.14) for k in ways}
        number = {k: 2 * k[0] - sites for k in ways}
    total = sum(weight.values())
    count = {}
    for k in sorted(ways):
        n = chi * weight[k] / total * math.exp(0.15 * rng.standard_normal())
        count[k] = min(ways[k], int(n + rng.random()))
    # the whole of chi, as far as the chain has so many states: one more (fewer) in each sector by turns,
    # from the middle outwards
    order = sorted(ways, key=lambda k: (-weight[k], k))
    rest = min(chi, sum(ways.values())) - sum(count.values())
    while rest != 0:
        before = rest
        for k in order[:max(1, len(order) // 2)]:
            if rest > 0 and count[k] < ways[k]:
                count[k] += 1
                rest -= 1
            elif rest < 0 and count[k] > 1:
                count[k] -= 1
                rest += 1
        if rest == before:
            break
    q = np.array([number[k] for k in sorted(ways) for _ in range(count[k])], dtype=np.int32)
    return q[rng.permutation(q.size)]


def layout(dims, dirs, qnums):
    """Flat position in the dense tensor of each stored entry, in the library's packed order: blocks whose
    signed quantum numbers add up to zero, row-major over the sorted distinct numbers of each axis."""
    at = [{int(q): np.nonzero(qn == q)[0] for q in np.unique(qn)} for qn in qnums]
    strides = [int(np.prod(dims[i + 1:], dtype=np.int64)) for i in range(len(dims))]
    found = []

    def walk(ax, rest, where):
        if ax == len(dims) - 1:
            last = at[ax].get(-rest * int(dirs[ax]))
            if last is not None:
                found.append((where[..., None] + last * strides[ax]).reshape(-1))
            return
        for q in at[ax]:
            walk(ax + 1, rest + int(dirs[ax]) * q, where[..., None] + at[ax][q] * strides[ax])

    walk(0, 0, np.zeros((), dtype=np.int64))
    return np.concatenate(found) if found else np.zeros(0, dtype=np.int64)


def mask_of(qa, qp, qb, device):
    """1 where a site tensor [a, p, b] may have entries."""
    a, p, b = (torch.as_tensor(np.asarray(q, dtype=np.int64), device=device) for q in (qa, qp, qb))
    return (a[:, None, None] + p[None, :, None] == b[None, None, :]).to(torch.float64)


def environments(model, nsites, mpo, left_bonds, right_bonds, seed):
    """Dense left and right environments [a, m, x] and [b, n, c] of the centre pair for a random state."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    op = compat.MPO(mpo)
    qs = mpo.qsite

    def site(qa, qb):
        m = mask_of(qa, qs, qb, dev)
        a = torch.randn(m.shape, generator=gen, device=dev, dtype=torch.float64) * m
        return a / torch.clamp(m.sum((0, 1), keepdim=True).sqrt(), min=1)

    i = nsites // 2 - 1
    left = torch.ones((1, 1, 1), device=dev, dtype=torch.float64)
    for k in range(i):
        a, w = site(left_bonds[k], left_bonds[k + 1]), torch.as_tensor(op.site(k), device=dev)
        t = torch.tensordot(left, a, dims=([2], [0]))                      # a m q x'
        t = torch.tensordot(t, w, dims=([1, 2], [0, 1]))                   # a x' p m'
        left = torch.tensordot(a, t, dims=([0, 1], [0, 2])).permute(0, 2, 1)
    right = torch.ones((1, 1, 1), device=dev, dtype=torch.float64)
    for k in range(nsites - 1, i + 1, -1):
        j = k - i - 2
        a, w = site(right_bonds[j], right_bonds[j + 1]), torch.as_tensor(op.site(k), device=dev)
        # the same scale from the right: a row's entries, not a column's
        a = a / torch.clamp((a * a).sum((1, 2), keepdim=True).sqrt(), min=1e-3)
        t = torch.tensordot(a, right, dims=([2], [0]))                     # b p n' c'
        t = torch.tensordot(t, w, dims=([1, 2], [2, 3]))                   # b c' n q
        right = torch.tensordot(t, a, dims=([1, 3], [2, 1]))
    return left.contiguous(), right.contiguous()


def bonds_of(model, nsites, chi, structure):
    """Quantum numbers of the bonds left of the centre pair (from the end inwards) and right of it (outwards)."""
    rng = np.random.default_rng(structure)
    i = nsites // 2 - 1
    total = sector_of(model, nsites)
    left = [np.zeros(1, dtype=np.int32)] + [sweep_bond(model, k, chi, rng) for k in range(1, i + 1)]
    right = [np.zeros(1, dtype=np.int32)] + [sweep_bond(model, k, chi, rng) for k in range(1, i + 1)]
    return left, [(total - q).astype(np.int32) for q in right][::-1]


def problem(case, seed):
    """theta, h2, left, right of the two-site problem at the centre of the chain, as host tensors."""
    model, nsites, chi = case["model"], case["nsites"], case["chi"]
    rng = np.random.default_rng([int(seed), 17])
    if case["bond"] == "random":
        if model == "molecular":
            t = ct.generate_matvec_problem_mpo(mpo_of(model, nsites, case["structure"]), sector_of(model, nsites), chi, case["structure"])
        else:
            t = ct.generate_matvec_problem(model, nsites, chi, case["structure"])
        for k in (0, 2, 3):
            t[k].deserialize(rng.standard_normal(t[k].nelem()))
        return t
    mpo = mpo_of(model, nsites, case["structure"])
    left_bonds, right_bonds = bonds_of(model, nsites, chi, case["structure"])
    i = nsites // 2 - 1
    h2 = ct.mpo_merge_tensor_pair(Site(mpo, i), Site(mpo, i + 1))
    ql, qr, qs = left_bonds[i], right_bonds[0], mpo.qsite
    qw = h2.meta()[2]
    zero = np.zeros(1, dtype=np.int32)
    theta = ct.HostTensor.zeros([ql.size, len(qw[1]), qr.size], [OUT, OUT, IN], [ql, qw[1], qr])
    left = ct.HostTensor.zeros([1, ql.size, len(qw[0]), ql.size], [OUT, IN, IN, OUT], [zero, ql, qw[0], ql])
    right = ct.HostTensor.zeros([qr.size, len(qw[3]), qr.size, 1], [OUT, OUT, IN, IN], [qr, qw[3], qr, zero])
    el, er = environments(model, nsites, mpo, left_bonds, right_bonds, seed)
    for t, dense in ((left, el), (right, er)):
        at = torch.as_tensor(layout(*t.meta()), device=dense.device)
        t.deserialize(dense.reshape(-1)[at].cpu().numpy())
    v = rng.standard_normal(theta.nelem())
    theta.deserialize(v / np.linalg.norm(v))
    return theta, h2, left, right


def members(case):
    """The problems of a batch: Hubbard and XXZ chains of 16 to 64 sites, bond dimensions up to chi."""
    rng = np.random.default_rng(case["structure"])
    out = []
    for k in range(case["count"]):
        model = ["xxz", "hubbard"][int(rng.integers(2))]
        if case["bond"] == "random":
            nsites = int(rng.integers(16, case["nsites"] + 1)) // 2 * 2
            chi = max(16, case["chi"] >> int(rng.integers(5)))      # 64 .. 1024 for the listed batch
        else:
            nsites = 16 if model == "hubbard" else 20
            chi = int(rng.integers(32, max(33, case["chi"]) + 1))
        out.append(dict(case, model=model, nsites=nsites, chi=chi, structure=case["structure"] + 1000 * k))
    return out


# ---------------------------------------------------------------------------------------------------
# preparation and passes

class Vector:
    """A torch tensor on the GPU as the plans take it."""

    def __init__(self, t):
        self.t, self.ptr = t, ctypes.c_void_p(t.data_ptr())


class Seen:
    """A device array of the library, for torch to look at without a copy (it keeps the array alive)."""

    def __init__(self, a):
        self.a = a
        self.__cuda_array_interface__ = {"shape": (a.n,), "typestr": "<f8", "data": (int(a.ptr.value), False), "version": 2}


def seen(a):
    return torch.as_tensor(Seen(a), device="cuda")


def on_gpu(v):
    return torch.as_tensor(v).to("cuda")


def prepare(case, seed):
    s = dict(case)
    if case["call"] == "dmrg":
        s["mpo"] = compat.MPO(mpo_of(case["model"], case["nsites"], case["structure"]))
        s["seed"] = int(seed)
        return s
    if case["call"] in ("batch", "batch_lanczos"):
        probs = [problem(m, int(seed) + 7919 * k) for k, m in enumerate(members(case))]
        s["plan"] = ct.MatvecBatch(probs)
        s["x"] = Vector(on_gpu(np.concatenate([p[0].serialize() for p in probs])))
    else:
        p = problem(case, seed)
        if case["call"] == "apply":
            s["problem"] = p
            return s
        s["plan"] = ct.MatvecPlan(*p, mode=FORMS[case["form"]])
        s["x"] = Vector(on_gpu(p[0].serialize()))
    s["y"] = Vector(torch.zeros_like(s["x"].t))
    torch.cuda.synchronize()
    s["plan"].synchronize()
    return s


def run(s):
    call = s["call"]
    if call in ("matvec", "batch"):
        s["plan"].apply(s["x"], s["y"])
        return s["y"].t
    if call == "lanczos":
        energy, u = s["plan"].lanczos(s["x"], LANCZOS_STEPS)
        return {"energy": energy, "state": seen(u)}
    if call == "batch_lanczos":
        energy, status, u = s["plan"].lanczos(s["x"], LANCZOS_STEPS)
        return {"energy": energy, "status": status, "state": seen(u)}
    if call == "apply":
        return ct.apply_local_hamiltonian(*s["problem"]).serialize()
    psi, energies, entropy = compat.dmrg(s["mpo"], num_sweeps=DMRG_SWEEPS, maxiter_lanczos=LANCZOS_STEPS, tol_split=1e-10,
                                         max_vdim=s["chi"], qnum_sector=sector_of(s["model"], s["nsites"]) if s["model"] == "hubbard" else s["nsites"] % 2,
                                         rng_seed=s["seed"])
    return {"energies": np.array(energies), "entropy": np.array(entropy), "state": psi.to_statevector()}


# ---------------------------------------------------------------------------------------------------
# the same in plain torch, dense, in 64 bits

class Dense:
    """The effective Hamiltonian of host tensors as dense tensors on the GPU."""

    def __init__(self, p):
        self.at = on_gpu(layout(*p[0].meta()))
        self.theta, self.w, self.l, self.r = (self.dense(t) for t in p)

    @staticmethod
    def dense(t):
        meta = t.meta()
        d = torch.zeros(int(np.prod(meta[0], dtype=np.int64)), dtype=torch.float64, device="cuda")
        d[on_gpu(layout(*meta))] = on_gpu(t.serialize())
        return d.reshape(meta[0])

    def apply(self, v):
        """The packed vector of L^T (W (theta R)) for the packed vector v."""
        th = torch.zeros_like(self.theta).reshape(-1)
        th[self.at] = v
        th = th.reshape(self.theta.shape)
        a, m, x = self.l.shape[1:]
        left = self.l[0].reshape(a * m, x).t().contiguous()                # x (a m)
        q, pp, n = self.w.shape[1:]
        w = self.w.reshape(m * q, pp * n)
        y = torch.empty((x, q, self.r.shape[2]), dtype=torch.float64, device="cuda")
        step = max(1, int(4e9 / (8.0 * a * max(m * q, pp * n))))
        for c0 in range(0, self.r.shape[2], step):
            r = self.r[:, :, c0:c0 + step, 0]
            c = r.shape[2]
            t = (th.reshape(a * pp, -1) @ r.reshape(r.shape[0], n * c)).reshape(a, pp, n, c)
            t = w @ t.permute(1, 2, 0, 3).reshape(pp * n, a * c)           # (m q) (a c)
            t = t.reshape(m, q, a, c).permute(2, 0, 1, 3).reshape(a * m, q * c)
            y[:, :, c0:c0 + step] = (left @ t).reshape(x, q, c)
        return y.reshape(-1)[self.at]


def ground_state(apply, v, steps):
    """Lanczos without re-orthogonalisation from v: the lowest Ritz value."""
    v = v / v.norm()
    n, alpha, beta, basis = v.numel(), [], [], [v]
    for j in range(steps):
        w = apply(basis[j])
        alpha.append(float(w @ basis[j]))
        if j == steps - 1:
            break
        w = w - alpha[j] * basis[j] - (beta[j - 1] * basis[j - 1] if j else 0.0)
        beta.append(float(w.norm()))
        if beta[j] < 100 * n * 2.220446049250313e-16:
            break
        basis.append(w / beta[j])
    k = len(alpha)
    lam, z = np.linalg.eigh(np.diag(alpha) + np.diag(beta[:k - 1], 1) + np.diag(beta[:k - 1], -1))
    return float(lam[0])


def exact(case, seed):
    call = case["call"]
    if call == "dmrg":
        return None
    if call in ("batch", "batch_lanczos"):
        parts = [problem(m, int(seed) + 7919 * k) for k, m in enumerate(members(case))]
    else:
        parts = [problem(case, seed)]
    got = []
    for p in parts:
        d = Dense(p)
        v = on_gpu(p[0].serialize())
        if "lanczos" in call:
            got.append(ground_state(d.apply, v, LANCZOS_STEPS))
        else:
            got.append(d.apply(v))
        del d
    if call in ("matvec", "batch"):
        return torch.cat(got)
    if call == "apply":
        return got[0].cpu().numpy()
    # the sign of an eigenvector is free: its value says nothing against the library's
    if call == "lanczos":
        return {"energy": got[0], "state": None}
    return {"energy": np.array(got), "status": np.zeros(len(got), dtype=np.int32), "state": None}


# ---------------------------------------------------------------------------------------------------
# what a pass cannot do without

def counts(q):
    return Counter(int(v) for v in q)


def matvec_work(ql, qr, h2):
    """Bytes and flops of one effective-Hamiltonian matvec from the quantum numbers of its bonds and the merged
    operator: theta, h2 and both environments read once and the result written once; 2 m n k of every block
    product of theta R and L^T T, and two flops for each entry of T and each operator entry that is not zero
    and acts on it."""
    dims, _, (qm, qs, _, qn) = h2.meta()
    A, P, B, M, N = (counts(q) for q in (ql, qs, qr, qm, qn))
    # the operator's entries that are not zero, by the charge that they carry
    at = layout(*h2.meta())[h2.serialize() != 0] // (dims[2] * dims[3])
    nonzero = Counter((qm[at // dims[1]].astype(np.int64) + qs[at % dims[1]]).tolist())
    right = {}
    for b in B:
        for n in N:
            if b + n in B:
                right.setdefault(b, []).append((n, b + n))
    theta = sum(A[a] * P[p] * B[a + p] for a in A for p in P if a + p in B)
    envs = sum(B[b] * N[n] * B[c] for b in right for n, c in right[b]) + sum(A[a] * M[m] * A[a + m] for a in A for m in M if a + m in A)
    w = h2.nelem()
    f1 = sum(A[a] * P[p] * B[a + p] * sum(N[n] * B[c] for n, c in right.get(a + p, ())) for a in A for p in P if a + p in B)
    f2 = sum(A[a] * B[c] * nonzero.get(c - a, 0) for a in A for c in B)
    f3 = sum(A[x] * P[q] * B[x + q] * A[a] * M[x - a] for a in A for x in A if x - a in M for q in P if x + q in B)
    return {"bytes": 8.0 * (2 * theta + envs + w), "flops": 2.0 * (f1 + f2 + f3), "theta": theta}


def one_work(case):
    model, nsites, chi = case["model"], case["nsites"], case["chi"]
    if case["bond"] == "random":
        if model == "molecular":
            t = ct.generate_matvec_problem_mpo(mpo_of(model, nsites, case["structure"]), sector_of(model, nsites), chi, case["structure"])
        else:
            t = ct.generate_matvec_problem(model, nsites, chi, case["structure"])
        qt = t[0].meta()[2]
        return matvec_work(qt[0], qt[2], t[1])
    i = nsites // 2 - 1
    left, right = bonds_of(model, nsites, chi, case["structure"])
    mpo = mpo_of(model, nsites, case["structure"])
    return matvec_work(left[i], right[0], ct.mpo_merge_tensor_pair(Site(mpo, i), Site(mpo, i + 1)))


def work(case):
    if case["call"] == "dmrg":
        # both directions of every sweep, LANCZOS_STEPS matvecs at each bond of a state of this size; the
        # run itself reads little and returns the state
        d = 4 if case["model"] == "hubbard" else 2
        total = {"bytes": 0.0, "flops": 0.0}
        n = case["nsites"]
        for i in range(n - 1):
            chi = min(case["chi"], d ** (i + 1), d ** (n - 1 - i))
            sites = max(2, min(i + 1, n - 1 - i, 12))
            inner = dict(case, bond="sweep", chi=chi, nsites=2 * sites + 2)
            w = one_work(inner)
            total["flops"] += DMRG_SWEEPS * 2 * LANCZOS_STEPS * w["flops"]
            total["bytes"] += 2 * 8.0 * w["theta"]
        return total
    each = [one_work(m) for m in (members(case) if case["call"] in ("batch", "batch_lanczos") else [case])]
    total = {k: float(sum(w[k] for w in each)) for k in ("bytes", "flops")}
    if "lanczos" in case["call"]:
        total["flops"] *= LANCZOS_STEPS
        # the operands once (they stay in cache), the basis written and read once for the Ritz vector
        total["bytes"] += sum(8.0 * w["theta"] * 2 * LANCZOS_STEPS for w in each)
    return total
