"""The work that programs built on this library have it do, as cases that can be timed.

A DMRG++ run calls the library in a few ways, and each has its cases here:

* the superblock matvec y = H x on a handle that lives for one sweep step (an external Lanczos,
  the plugin's caller), in the three precisions, from the smallest chains to the largest cylinder;
* one step of a sweep: the handle of a new superblock from host blocks, a short Lanczos solve
  from the transformed wave function, and the handle's end;
* the Davidson solver (refinement of mixed-precision states, learned preconditioner runs);
* a Krylov time step of several complex target vectors;
* the wave-function transformation's batched GEMMs between two steps;
* the learned preconditioner: inference over a whole superblock vector, and training steps.

Superblocks are drawn with the structure of the models this repository runs (Heisenberg chain and
ladder: groups by 2Sz; Hubbard chain, ladder and cylinder: groups by N and 2Sz), with group sizes
from a Gaussian histogram of the kept states, so patches come in every size from 1 up and are hardly
ever a multiple of a tile. Operator blocks are dense with spectral norms of order one, as the
truncated operators of a block have.
"""
from __future__ import annotations

import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

import dmrgpp_amd as dm
from dmrgpp_amd.problem import KronProblem

# ---- superblocks ----------------------------------------------------------------------------


def _histogram(total, weights):
    """total states spread over the groups by weight, at least one each, exactly total."""
    w = {q: v for q, v in weights.items() if v * total / sum(weights.values()) >= 0.3}
    s = sum(w.values())
    got = {q: max(1, int(v / s * total)) for q, v in w.items()}
    big = max(got, key=lambda q: (got[q], q))
    got[big] += total - sum(got.values())
    return got


def _groups(family, m, width):
    """Group sizes of a block of m kept states times one site, by quantum number."""
    if family == "spin":  # q = (2Sz, 0); the site doubles the block
        return _histogram(2 * m, {(q, 0): math.exp(-q * q / (2 * width * width))
                                  for q in range(-40, 41, 2)})
    return _histogram(4 * m, {(dn, s): math.exp(-(dn * dn + s * s) / (2 * width * width))
                              for dn in range(-16, 17) for s in range(-16, 17)
                              if (dn + s) % 2 == 0})


# Link operators of one bond across the cut: what the left operator does to the quantum numbers
# (the right one does the opposite), and which earlier one it is the adjoint of.
_LINKS = {"spin": [((2, 0), None), ((-2, 0), 0), ((0, 0), None)],
          "hubbard": [((1, 1), None), ((-1, -1), 0), ((1, -1), None), ((-1, 1), 2)]}


def _structure(case):
    """Patch sizes and the terms (I, J, k, kind) of a case's superblock, from its sizes alone:
    kind 0: H_L times identity, 1: identity times H_R, 2: a link term."""
    left = _groups(case["family"], case["m"], case["width"])
    right = _groups(case["family"], case["m"], case["width"] * 1.06)
    qs = [q for q in sorted(left) if (-q[0], -q[1]) in right]
    L = [left[q] for q in qs]
    R = [right[(-q[0], -q[1])] for q in qs]
    at = {q: i for i, q in enumerate(qs)}
    terms = [(i, i, 0, 0) for i in range(len(qs))] + [(i, i, 1, 1) for i in range(len(qs))]
    links = _LINKS[case["family"]]
    for b in range(case["bonds"]):
        for l, (d, _) in enumerate(links):
            for q, j in at.items():
                i = at.get((q[0] + d[0], q[1] + d[1]))
                if i is not None:
                    terms.append((i, j, 2 + b * len(links) + l, 2))
    return L, R, 2 + case["bonds"] * len(links), terms


def _problem(case, seed):
    """The superblock with values from the seed: a symmetric H."""
    L, R, nC, terms = _structure(case)
    nl = len(_LINKS[case["family"]])
    eyes, jobs, blocks = {}, [], {}

    def new(rows, cols, sym):
        a = np.empty((rows, cols), order="F")
        jobs.append((len(jobs), a, sym))
        return a

    def eye(n):
        if n not in eyes:
            eyes[n] = np.asfortranarray(np.eye(n))
        return eyes[n]

    copies = []
    for i, j, k, kind in terms:
        if kind == 0:
            blocks[(i, j, k)] = (new(L[i], L[i], True), eye(R[i]))
        elif kind == 1:
            blocks[(i, j, k)] = (eye(L[i]), new(R[i], R[i], True))
        else:
            l = (k - 2) % nl
            adj = _LINKS[case["family"]][l][1]
            if adj is None:
                sym = i == j
                blocks[(i, j, k)] = (new(L[i], L[j], sym), new(R[i], R[j], sym))
            else:  # the adjoint of an earlier link of the same bond
                a, b = blocks[(j, i, k - l + adj)]
                c = np.empty((L[i], L[j]), order="F"), np.empty((R[i], R[j]), order="F")
                blocks[(i, j, k)] = c
                copies += [(c[0], a), (c[1], b)]

    def fill(job):
        n, a, sym = job
        rng = np.random.Generator(np.random.SFC64([seed, n]))
        v = a.reshape(-1, order="F")  # a view: the block is Fortran ordered
        rng.random(out=v)
        v -= 0.5
        v *= 2.0 / math.sqrt(max(a.shape))
        if sym:
            a += a.T.copy()

    def turn(c):
        c[0][...] = c[1].T

    with ThreadPoolExecutor(8) as ex:
        list(ex.map(fill, jobs))
        list(ex.map(turn, copies))
    return KronProblem(L=np.array(L), R=np.array(R), nC=nC, blocks=blocks,
                       name="%s-m%d" % (case["family"], case["m"]))


def _cost(case):
    """(n, flops of one matvec, bytes of its non-identity factors in FP64)."""
    L, R, _, terms = _structure(case)
    flops = nbytes = 0
    for i, j, _, kind in terms:
        if kind == 0:
            flops += 2 * R[i] * L[i] * L[i]
            nbytes += 8 * L[i] * L[i]
        elif kind == 1:
            flops += 2 * R[i] * R[i] * L[i]
            nbytes += 8 * R[i] * R[i]
        else:
            flops += min(2 * R[i] * R[j] * L[j] + 2 * R[i] * L[j] * L[i],
                         2 * R[j] * L[j] * L[i] + 2 * R[i] * R[j] * L[i])
            nbytes += 8 * (L[i] * L[j] + R[i] * R[j])
    return sum(a * b for a, b in zip(L, R)), flops, nbytes


class _Vec:
    """A torch tensor on the GPU as the library's calls take device vectors (by address)."""

    def __init__(self, t):
        self.t, self.ptr, self.size = t, t.data_ptr(), t.numel()


def _uniform(n, seed, lo=-1.0, hi=1.0, dtype=torch.float64):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.empty(n, dtype=dtype, device="cuda").uniform_(lo, hi, generator=g)


def _normal(n, seed, dtype=torch.float32):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.empty(n, dtype=dtype, device="cuda").normal_(generator=g)


class _Exact:
    """H in 64 bits by plain products, one term at a time, on the GPU."""

    def __init__(self, prob):
        self.off = [int(o) for o in prob.offsets]
        self.L, self.R = [int(v) for v in prob.L], [int(v) for v in prob.R]
        self.n = prob.n
        self.terms, seen = [], {}

        def up(a):  # column major: the transpose is contiguous
            if id(a) not in seen:
                seen[id(a)] = torch.from_numpy(a.T).cuda().t()
            return seen[id(a)]

        for (i, j, k), (a, b) in prob.blocks.items():
            self.terms.append((i, j, up(a) if k != 1 else None, up(b) if k != 0 else None))

    def __call__(self, x):
        y = torch.zeros_like(x)
        for i, j, a, b in self.terms:
            v = x[self.off[j]:self.off[j + 1]].view(self.L[j], self.R[j])
            if a is not None:
                v = a @ v
            if b is not None:
                v = v @ b.t()
            y[self.off[i]:self.off[i + 1]].view(self.L[i], self.R[i]).add_(v)
        return y


# ---- one matvec -----------------------------------------------------------------------------


def _matvec_prepare(case, seed):
    op = dm.BatchedGemm(_problem(case, seed), case["precision"])
    return {"op": op, "x": _Vec(_uniform(op.n, seed)),
            "y": _Vec(torch.empty(op.n, dtype=torch.float64, device="cuda"))}


def _matvec_run(s):
    # The caller uses y at once (the plugin's matrixVector returns it), so it waits for it.
    s["op"].apply_Htarget(s["x"], s["y"])
    s["op"].sync()
    return s["y"].t


def _matvec_work(case):
    n, flops, nbytes = _cost(case)
    return {"bytes": (nbytes if case["precision"] == "fp64" else nbytes / 2) + 16 * n,
            "flops": flops}


def _matvec_exact(case, seed):
    h = _Exact(_problem(case, seed))
    return h(_uniform(h.n, seed))


# ---- one step of a sweep: new handle, short Lanczos from the transformed wave function --------

_WARM_STEPS = 12  # solves started from the previous step's state take 5 to 16 steps


def _step_prepare(case, seed):
    prob = _problem(case, seed)
    return {"prob": prob, "init": _Vec(_uniform(prob.n, seed)),
            "z": _Vec(torch.empty(prob.n, dtype=torch.float64, device="cuda"))}


def _step_run(s):
    op = dm.BatchedGemm(s["prob"], "fp64")
    r = op.lanczos_ground(s["init"], s["z"], max_steps=_WARM_STEPS)
    op.close()
    return {"energy": r["energy"], "steps": r["steps"], "z": s["z"].t}


def _step_work(case):
    n, flops, nbytes = _cost(case)
    # The blocks once, and per step the recurrence's four vector passes; then z.
    return {"bytes": nbytes + 8 * n * (4 * _WARM_STEPS + 2), "flops": _WARM_STEPS * flops}


def _lanczos(h, v, m):
    """Basis (full reorthogonalization) and tridiagonal matrix of m steps."""
    V, a, b = [v / v.norm()], [], []
    for j in range(m):
        w = h(V[j])
        a.append(float(V[j] @ w))
        for _ in range(2):
            for u in V:
                w = w - (u @ w) * u
        b.append(float(w.norm()))
        V.append(w / b[-1])
    return V[:m], np.diag(a) + np.diag(b[:m - 1], 1) + np.diag(b[:m - 1], -1)


def _step_exact(case, seed):
    h = _Exact(_problem(case, seed))
    V, T = _lanczos(h, _uniform(h.n, seed), _WARM_STEPS)
    w, s = np.linalg.eigh(T)
    c = s[:, 0] * (1.0 if s[:, 0].sum() > 0 else -1.0)  # the library's sign of the Ritz vector
    return {"energy": float(w[0]), "steps": None, "z": sum(float(x) * u for x, u in zip(c, V))}


# ---- Davidson -------------------------------------------------------------------------------

_DAVIDSON_MATVECS = 24


def _davidson_prepare(case, seed):
    s = _matvec_prepare(dict(case, precision="fp64"), seed)
    return s


def _davidson_run(s):
    r = s["op"].davidson_ground(s["x"], s["y"], precond="diag", max_basis=12,
                                max_matvecs=_DAVIDSON_MATVECS)
    return {"energy": r["energy"], "residual": r["residual"], "z": s["y"].t}


def _davidson_work(case):
    n, flops, nbytes = _cost(case)
    # Per iteration V (8 columns on average) is read by the Ritz pass, the projection, the
    # update and the Rayleigh quotient, and W by the Ritz pass.
    return {"bytes": _DAVIDSON_MATVECS * (nbytes + 8 * n * 42),
            "flops": _DAVIDSON_MATVECS * flops}


# ---- Krylov time step -----------------------------------------------------------------------

_DT = 0.05


def _krylov_prepare(case, seed):
    op = dm.BatchedGemm(_problem(case, seed), "fp64")
    nv = case["targets"]
    phi = _uniform(2 * nv * op.n, seed).view(nv, 2 * op.n)
    phi /= phi.norm(dim=1, keepdim=True)
    return {"op": op, "nv": nv, "precision": case["precision"], "phi": _Vec(phi.reshape(-1)),
            "out": _Vec(torch.empty(2 * nv * op.n, dtype=torch.float64, device="cuda"))}


def _krylov_run(s):
    s["op"].krylov_evolve(s["phi"], s["out"], s["nv"], [_DT], stop="expm", tolerance=1e-12,
                          precision=s["precision"])
    return s["out"].t


def _krylov_work(case):
    n, flops, nbytes = _cost(case)
    steps = 9  # the Krylov dimension that a step of this length needs
    # Per step the factors once, and the recurrence's passes over two real columns per target.
    return {"bytes": steps * (nbytes + case["targets"] * 2 * 8 * n * 6),
            "flops": steps * 2 * case["targets"] * flops}


def _krylov_exact(case, seed):
    if _cost(case)[1] * case["targets"] > 3e12:
        return None  # too long
    h = _Exact(_problem(case, seed))
    nv, n = case["targets"], h.n
    phi = _uniform(2 * nv * n, seed).view(nv, 2 * n)
    phi = phi / phi.norm(dim=1, keepdim=True)
    out = torch.empty(nv, n, 2, dtype=torch.float64, device="cuda")
    for t in range(nv):
        for part in range(2):  # exp(-i H t) is linear and H real: the two parts apart
            v = phi[t].view(n, 2)[:, part].contiguous()
            V, T = _lanczos(h, v, min(n, 24))
            w, s = np.linalg.eigh(T)
            c = float(v.norm()) * (s @ (np.exp(-1j * w * _DT) * s[0]))
            re = sum(float(x.real) * u for x, u in zip(c, V))
            im = sum(float(x.imag) * u for x, u in zip(c, V))
            if part == 0:
                out[t, :, 0], out[t, :, 1] = re, im
            else:
                out[t, :, 0] -= im
                out[t, :, 1] += re
    return out.reshape(-1)


# ---- wave-function transformation: Y = V_E X V_L per sub-block, in two batched GEMMs ----------


def _wft_shapes(case):
    """(s, k) per chain: V_E is s x k, X is k rows of an s x s patch, V_L is s x k."""
    kept = _groups(case["family"], case["m"] // 2, case["width"])
    full = _groups(case["family"], case["m"], case["width"])
    shapes = []
    for q in sorted(full):
        for d in ((1, 0), (-1, 0)) if case["family"] == "spin" else ((0, 0), (1, 1), (1, -1), (2, 0)):
            k = kept.get((q[0] + d[0] - 1, q[1] + d[1]))
            if k:
                shapes.append((full[q], k))
    return shapes


def _wft_prepare(case, seed):
    shapes = _wft_shapes(case)
    P = _uniform(sum(s * k for s, k in shapes), seed)
    Q = _uniform(sum(s * k for s, k in shapes), seed + 1)
    X = _uniform(sum(s * s for s, _ in shapes), seed + 2)
    W = torch.empty(sum(k * k for _, k in shapes), dtype=torch.float64, device="cuda")
    Y = torch.empty(sum(s * k for s, k in shapes), dtype=torch.float64, device="cuda")
    first, second, p, x, w = [], [], 0, 0, 0
    for s, k in shapes:
        r = (s - k) // 2  # the sub-block's first row in its patch
        ptr = [t.data_ptr() + 8 * o for t, o in ((P, p), (X, x + max(r, 0)), (Q, p), (W, w), (Y, p))]
        kk = min(s, k)  # rows of the sub-block
        first.append((kk, k, s, s, s, kk, [(ptr[1], ptr[2], ptr[3])]))     # W = X Q
        second.append((s, k, kk, s, kk, s, [(ptr[0], ptr[3], ptr[4])]))    # Y = P W
        p, x, w = p + s * k, x + s * s, w + k * k
    return {"first": first, "second": second, "keep": (P, Q, X, W), "y": Y}


def _wft_run(s):
    dm.gemm_vbatch("N", "N", s["first"])
    dm.gemm_vbatch("N", "N", s["second"])
    return s["y"]


def _wft_work(case):
    sh = [(s, k, min(s, k)) for s, k in _wft_shapes(case)]
    return {"bytes": 8 * sum(s * kk + s * k + s * kk + s * k for s, k, kk in sh),
            "flops": sum(2 * kk * k * s + 2 * s * k * kk for s, k, kk in sh)}


def _wft_exact(case, seed):
    shapes = _wft_shapes(case)
    P = _uniform(sum(s * k for s, k in shapes), seed)
    Q = _uniform(sum(s * k for s, k in shapes), seed + 1)
    X = _uniform(sum(s * s for s, _ in shapes), seed + 2)
    out, p, x = [], 0, 0
    for s, k in shapes:
        r, kk = max((s - k) // 2, 0), min(s, k)
        xs = X[x:x + s * s].view(s, s).t()[r:r + kk]          # column major
        y = P[p:p + s * k].view(k, s).t()[:, :kk] @ (xs @ Q[p:p + s * k].view(k, s).t())
        out.append(y.t().reshape(-1))
        p, x = p + s * k, x + s * s
    return torch.cat(out)


# ---- learned preconditioner -----------------------------------------------------------------

_OFF = {"W1": (0, 256), "b1": (256, 320), "W2": (320, 4416), "b2": (4416, 4480),
        "W3": (4480, 4544), "b3": (4544, 4545)}


def _mlp_params(seed):
    """Parameters of a trained network's size: Glorot weights, small biases."""
    rng = np.random.default_rng(seed)
    p = np.zeros(dm.MLP_PARAMS, dtype=np.float32)
    for name, scale in (("W1", 0.3), ("b1", 0.1), ("W2", 0.2), ("b2", 0.1), ("W3", 0.2),
                        ("b3", 0.1)):
        lo, hi = _OFF[name]
        p[lo:hi] = rng.uniform(-scale, scale, hi - lo)
    return p


def _features(count, seed):
    """(D - theta)/s_D, r/rms(r), u/rms(u) and Olsen's correction, clipped as the solver does."""
    return _normal(count * dm.MLP_FEATURES, seed).clamp_(-4.0, 4.0)


def _targets(x):
    f = x.view(-1, dm.MLP_FEATURES)
    return (torch.tanh(f[:, 1]) * 0.5 - 0.3 * f[:, 3] + 0.1 * f[:, 0] * f[:, 2]).contiguous()


def _mlp_forward64(p, x):
    q = {k: p[lo:hi] for k, (lo, hi) in _OFF.items()}
    h = torch.tanh(x @ q["W1"].view(64, 4).t() + q["b1"])
    h = torch.tanh(h @ q["W2"].view(64, 64).t() + q["b2"])
    return h @ q["W3"] + q["b3"]


def _mlpf_prepare(case, seed):
    net = dm.Mlp(seed=seed, capacity=1)
    net.set_params(_mlp_params(seed))
    return {"net": net, "count": case["count"], "x": _Vec(_features(case["count"], seed)),
            "y": _Vec(torch.empty(case["count"], dtype=torch.float32, device="cuda"))}


def _mlpf_run(s):
    if dm.lib().dmk_mlp_forward(s["net"].handle, s["x"].ptr, s["count"], s["y"].ptr) != 0:
        raise RuntimeError("dmk_mlp_forward failed")
    return s["y"].t


def _mlpf_work(case):
    return {"bytes": 4 * 5 * case["count"], "flops": 2.0 * 64 * (4 + 64 + 1) * case["count"]}


def _mlpf_exact(case, seed):
    p = torch.from_numpy(_mlp_params(seed)).double().cuda()
    x = _features(case["count"], seed).double().view(-1, 4)
    return torch.cat([_mlp_forward64(p, c) for c in x.split(1 << 18)])


_TRAIN_ITERS, _TRAIN_LR = 32, 2e-3


def _mlpt_prepare(case, seed):
    net = dm.Mlp(seed=seed, capacity=case["samples"])
    net.set_params(_mlp_params(seed))
    x = _features(case["samples"], seed)
    net.add_samples(x.cpu().numpy(), _targets(x).cpu().numpy())
    return {"net": net, "batch": case["batch"]}


def _mlpt_run(s):
    # The next steps of a training that goes on over its samples.
    last, _ = s["net"].train(_TRAIN_ITERS, batch=s["batch"], lr=_TRAIN_LR)
    return {"loss": last, "params": s["net"].params()}


def _mlpt_work(case):
    seen = _TRAIN_ITERS * case["batch"] + case["samples"]  # the whole set's loss afterwards
    return {"bytes": 4 * 5 * seen + _TRAIN_ITERS * 4 * 7 * dm.MLP_PARAMS,
            "flops": 6.0 * 64 * (4 + 64 + 1) * _TRAIN_ITERS * case["batch"]
            + 2.0 * 64 * 69 * case["samples"]}


def _mlpt_exact(case, seed):
    p = torch.from_numpy(_mlp_params(seed)).double().cuda().requires_grad_(True)
    x = _features(case["samples"], seed)
    t = _targets(x).double()
    x = x.double().view(-1, 4)
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    b1, b2 = float(np.float32(0.9)), float(np.float32(0.999))
    lr, at, loss = float(np.float32(_TRAIN_LR)), 0, None
    for i in range(1, _TRAIN_ITERS + 1):
        if at + case["batch"] > case["samples"]:
            at = 0
        loss = ((_mlp_forward64(p, x[at:at + case["batch"]]) - t[at:at + case["batch"]]) ** 2).mean()
        (g,) = torch.autograd.grad(loss, p)
        with torch.no_grad():
            m.mul_(b1).add_(g, alpha=1 - b1)
            v.mul_(b2).add_(g * g, alpha=1 - b2)
            p -= lr * (m / (1 - b1 ** i)) / ((v / (1 - b2 ** i)).sqrt() + 1e-8)
        at += case["batch"]
    return {"loss": float(loss), "params": p.detach()}


# ---- the cases --------------------------------------------------------------------------------

_KINDS = {
    "matvec": (_matvec_prepare, _matvec_run, _matvec_work, _matvec_exact),
    "sweep_step": (_step_prepare, _step_run, _step_work, _step_exact),
    "davidson": (_davidson_prepare, _davidson_run, _davidson_work, None),
    "krylov": (_krylov_prepare, _krylov_run, _krylov_work, _krylov_exact),
    "wft": (_wft_prepare, _wft_run, _wft_work, _wft_exact),
    "mlp_forward": (_mlpf_prepare, _mlpf_run, _mlpf_work, _mlpf_exact),
    "mlp_train": (_mlpt_prepare, _mlpt_run, _mlpt_work, _mlpt_exact),
}


def _kron(name, kind, family, m, width, bonds, **more):
    return dict({"name": name, "kind": kind, "family": family, "m": m, "width": width,
                 "bonds": bonds}, **more)


def listed():
    return [
        # The smallest: the Heisenberg chain at m = 128, whose matvecs are latency.
        _kron("chain_m128_fp64", "matvec", "spin", 128, 2.2, 1, precision="fp64"),
        # The precision study's Hubbard chain at m = 1024: 36 patches, one bond.
        _kron("hubbard_chain_m1024_fp32", "matvec", "hubbard", 1024, 1.35, 1, precision="fp32"),
        # The Heisenberg ladder at m = 2048 (the benchmark's size) in the three precisions.
        _kron("ladder_m2048_fp64", "matvec", "spin", 2048, 3.2, 2, precision="fp64"),
        _kron("ladder_m2048_fp32", "matvec", "spin", 2048, 3.2, 2, precision="fp32"),
        _kron("ladder_m2048_bf16x3", "matvec", "spin", 2048, 3.2, 2, precision="bf16x3"),
        # The largest matvec: a Hubbard 4-leg cylinder, four bonds across the cut.
        _kron("cylinder_m3072_fp32", "matvec", "hubbard", 3072, 1.9, 4, precision="fp32"),
        # One step of a finite sweep of the ladder at half the largest number of states.
        _kron("sweep_step_m1024", "sweep_step", "spin", 1024, 3.1, 2),
        # Davidson with the diagonal correction on the Hubbard chain's superblock.
        _kron("davidson_m1024", "davidson", "hubbard", 1024, 1.35, 1),
        # Time evolution of the Hubbard ladder, four complex targets in one launch.
        _kron("krylov_m2048", "krylov", "hubbard", 2048, 1.83, 2, targets=4, precision="fp64"),
        # The wave-function transformation between two steps of the m = 2048 ladder.
        dict(name="wft_m2048", kind="wft", family="spin", m=2048, width=3.2),
        # The learned preconditioner over the ladder's superblock vector.
        dict(name="mlp_forward_ladder", kind="mlp_forward", count=2858152),
        # Its training, with the batch the training program uses.
        dict(name="mlp_train_b8192", kind="mlp_train", samples=1 << 18, batch=8192),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec"] * 6 + ["sweep_step", "davidson", "krylov", "wft", "mlp_forward",
                                        "mlp_train"])
    if kind == "mlp_forward":
        return dict(kind=kind, count=_log_uniform(rng, 20000, 2858152))
    if kind == "mlp_train":
        return dict(kind=kind, samples=_log_uniform(rng, 1 << 15, 1 << 18),
                    batch=_log_uniform(rng, 1000, 16384))
    family = rng.choice(["spin", "hubbard"])
    spread = rng.uniform(0.85, 1.15)
    width = round(spread * (3.2 if family == "spin" else 1.7), 3)
    if kind == "wft":
        return dict(kind=kind, family=family, m=_log_uniform(rng, 128, 2048), width=width)
    if kind == "matvec":
        m = _log_uniform(rng, 96, 4096 if family == "spin" else 2600)
        return dict(kind=kind, family=family, m=m, width=width, bonds=rng.randint(1, 4 if m < 2000 else 2),
                    precision=rng.choice(["fp64", "fp32", "bf16x3"]))
    if kind == "krylov":
        return dict(kind=kind, family=family, m=_log_uniform(rng, 128, 1400), width=width,
                    bonds=rng.randint(1, 2), targets=rng.randint(1, 4),
                    precision="fp64")
    return dict(kind=kind, family=family, m=_log_uniform(rng, 96, 1400), width=width,
                bonds=rng.randint(1, 2))


def prepare(case, seed):
    s = _KINDS[case["kind"]][0](case, seed)
    s["kind"] = case["kind"]
    torch.cuda.synchronize()  # the library's streams do not wait for torch's
    return s


def run(state):
    return _KINDS[state["kind"]][1](state)


def work(case):
    return _KINDS[case["kind"]][2](case)


def exact(case, seed):
    f = _KINDS[case["kind"]][3]
    return f(case, seed) if f else None
