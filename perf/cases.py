"""Workloads of the CP-ALS engine, timed through its public entry points.

A case is a dict of plain values; ``prepare`` makes what a program holds before the call
(the tensor on the GPU, the starting CPD, the plan), ``run`` is one pass, ``work`` the bytes
and operations the pass cannot do without, ``exact`` the same outputs in 64 bits by plain
torch / numpy.  ``draw`` gives further cases of the ranges the listed ones stand for.

Kinds:
    als      dense normal-equation ALS: ``als_optimize`` on a tensor (entry "call": the plan
             is made and released inside the call) or ``ALSPlan.set_cpd / run / get_cpd`` on a
             plan that the program keeps (entry "plan")
    batch    ``BatchALS`` over many small order-3 tensors
    sampled  ``ALSPlan.run_sampled`` with ``LevScoreSampled``
    mlp      forward and backward of the warm-start network
"""
import math

import numpy as np
import torch

import __graft_entry__

DEV = "cuda:0"


def _engine():
    return __graft_entry__.load_package()


def _dims(case):
    return tuple(int(d) for d in case["dims"].split("x"))


def _size(case):
    return math.prod(_dims(case))


# ------------------------------------------------------------------------ cases
def _als(name, dims, rank, sweeps, entry, check="none", elt=8, prec="fp64", noise=1e-2):
    return {"name": name, "kind": "als", "dims": "x".join(map(str, dims)), "rank": rank, "sweeps": sweeps,
            "entry": entry, "check": check, "elt": elt, "prec": prec, "noise": noise}


def listed():
    return [
        # One call on a small tensor (the CPU-sized workload's 64^3, rank 10): many short
        # launches, and the plan's set-up and release belong to the call.
        _als("call_64cubed_r10", (64, 64, 64), 10, 20, "call", noise=1e-3),
        # The headline workload: 512^3 FP64, rank 64, the fit after every sweep.
        _als("fit_512cubed_r64", (512, 512, 512), 64, 10, "plan", check="fit"),
        # A tensor as measured data has it: no mode a multiple of anything, a middling rank.
        _als("odd_301x257x199_r37", (301, 257, 199), 37, 8, "plan", check="fit"),
        # Order 4 at a low rank: little arithmetic per tensor element.
        _als("order4_96x88x80x72_r16", (96, 88, 80, 72), 16, 8, "plan", check="fit"),
        # Order 5 with odd modes: long Khatri-Rao products, small sides; one call.
        _als("call_order5_r24", (23, 21, 20, 19, 18), 24, 10, "call"),
        # Rank close to the mode sizes: the R x R solves weigh as much as the products.
        _als("rank150_200cubed", (200, 200, 200), 150, 5, "plan"),
        # The precision workload: a 10 GB order-4 FP32 tensor at rank 128 in BF16x3.
        _als("bf16x3_224x4_r128", (224, 224, 224, 224), 128, 2, "plan", elt=4, prec="bf16x3", noise=1e-3),
        # FP32 arithmetic on an FP32 tensor whose modes fit no tile.
        _als("fp32_150x130x110x90_r48", (150, 130, 110, 90), 48, 4, "plan", elt=4, prec="fp32", noise=1e-3),
        # The warm-start workload's tensor (200^3, FP32-stored, FP64 arithmetic), one call.
        _als("call_f32_200cubed_r16", (200, 200, 200), 16, 20, "call", elt=4),
        # Many small problems of mixed sizes and ranks, run together.
        {"name": "batch_1024", "kind": "batch", "count": 1024, "lo": 8, "hi": 64, "rlo": 4, "rhi": 24, "sweeps": 10},
        # Leverage-score-sampled ALS with the default (QR) solve.
        {"name": "sampled_256cubed_r32", "kind": "sampled", "dims": "256x256x256", "rank": 32, "samples": 1024,
         "sweeps": 2, "normal": False},
        # The warm-start network: one batch forward and backward.
        {"name": "mlp_200_256_256_200_b256", "kind": "mlp", "width": 200, "hidden": 256, "batch": 256},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _modes(rng, order, elements, multiple=1):
    """`order` mode sizes within a factor of about two of each other, near `elements` in all."""
    mean = elements ** (1.0 / order)
    return tuple(max(6, int(round(mean * math.exp(rng.uniform(-0.35, 0.35)) / multiple)) * multiple)
                 for _ in range(order))


def draw(rng):
    kind = rng.choice(["call", "call", "plan3", "plan3", "odd3", "odd4", "rank", "fp32", "bf16x3", "f32", "batch",
                       "sampled", "mlp"])
    if kind == "call":      # small and middling tensors through als_optimize
        order = rng.choice([3, 3, 4, 5])
        dims = _modes(rng, order, _log_int(rng, 20000, 6000000))
        c = _als("", dims, _log_int(rng, 3, min(40, min(dims))), 10, "call")
    elif kind == "plan3":   # order 3, modes that are multiples of 8 or of 32
        dims = _modes(rng, 3, _log_int(rng, 1000000, 90000000), rng.choice([8, 32]))
        c = _als("", dims, _log_int(rng, 8, 64), 5, "plan", check="fit")
    elif kind == "odd3":    # order 3, any modes
        dims = _modes(rng, 3, _log_int(rng, 1000000, 50000000))
        c = _als("", dims, _log_int(rng, 8, 64), 5, "plan", check=rng.choice(["fit", "none"]))
    elif kind == "odd4":    # order 4, any modes
        dims = _modes(rng, 4, _log_int(rng, 500000, 50000000))
        c = _als("", dims, _log_int(rng, 4, min(48, min(dims))), 5, "plan", check="fit")
    elif kind == "rank":    # ranks above 64
        dims = _modes(rng, 3, _log_int(rng, 4000000, 30000000), rng.choice([1, 8]))
        c = _als("", dims, rng.randint(65, max(66, min(190, (2 * min(dims)) // 3))), 3, "plan")
    elif kind in ("fp32", "bf16x3"):
        order = rng.choice([3, 4])
        dims = _modes(rng, order, _log_int(rng, 4000000, 200000000), rng.choice([1, 32 if order == 4 else 64]))
        c = _als("", dims, _log_int(rng, 8, 64), 2, "plan", elt=4, prec=kind, noise=1e-3)
    elif kind == "f32":
        dims = _modes(rng, 3, _log_int(rng, 1000000, 16000000), rng.choice([1, 8]))
        c = _als("", dims, _log_int(rng, 8, 24), 10, "call", elt=4)
    elif kind == "batch":
        c = {"kind": "batch", "count": _log_int(rng, 64, 1024), "lo": 8, "hi": rng.randint(24, 64), "rlo": 4,
             "rhi": rng.randint(8, 24), "sweeps": 10}
    elif kind == "sampled":
        d = _modes(rng, 3, _log_int(rng, 500000, 16000000))
        rank = _log_int(rng, 8, 48)
        c = {"kind": "sampled", "dims": "x".join(map(str, d)), "rank": rank,
             "samples": _log_int(rng, 8 * rank, 2048), "sweeps": 2, "normal": rng.random() < 0.5}
    else:
        c = {"kind": "mlp", "width": rng.randint(60, 256), "hidden": rng.randint(64, 512),
             "batch": _log_int(rng, 16, 512)}
    c.pop("name", None)
    return c


# ------------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) % (1 << 62))
    return g


def _krp(mats):
    """Row-wise Khatri-Rao product, the first matrix's index slowest."""
    out = mats[0]
    for m in mats[1:]:
        out = (out[:, None, :] * m[None, :, :]).reshape(-1, m.shape[1])
    return out


def _split(dims):
    return max(1, len(dims) // 2)


def _als_inputs(case, seed):
    """(tensor, starting factors): a sum of `rank` outer products of N(0,1) factor columns plus
    Gaussian noise, column-major (mode 1 fastest), and N(0,1) starting factors with unit columns."""
    dims, rank, g = _dims(case), case["rank"], _gen(seed)
    dt = torch.float32 if case.get("elt", 8) == 4 else torch.float64
    true = [torch.randn(d, rank, generator=g, device=DEV, dtype=dt) for d in dims]
    s = _split(dims)
    left = _krp([true[m] for m in reversed(range(s))])
    right = _krp([true[m] for m in reversed(range(s, len(dims)))])
    T = right @ left.T                                       # row = right multi-index, column = left one
    step = max(1, (1 << 26) // T.shape[1])
    for r in range(0, T.shape[0], step):
        rows = T[r:r + step]
        rows.add_(torch.randn(rows.shape, generator=g, device=DEV, dtype=dt), alpha=case.get("noise", 1e-2))
    T = T.reshape(tuple(reversed(dims))).permute(*reversed(range(len(dims))))
    start = []
    for d in dims:
        f = torch.randn(d, rank, generator=g, device=DEV, dtype=torch.float64)
        start.append(f / f.norm(dim=0))
    return T, start


def _host_cpd(E, start):
    return E.CPD([f.cpu().numpy() for f in start], np.ones(start[0].shape[1]))


def _norm(T):
    flat = T.permute(*reversed(range(T.dim()))).reshape(-1)
    return math.sqrt(sum(float((x.double() @ x.double()).item()) for x in flat.split(1 << 28)))


def _batch_inputs(case, seed):
    """(dims, rank, tensor (numpy, column-major), starting factors) per problem.  The sizes are
    the case's; the values come from the seed."""
    sizes = np.random.default_rng([case["count"], case["lo"], case["hi"], case["rhi"]])
    g = _gen(seed)
    out = []
    n = case["count"]
    dims = sizes.integers(case["lo"], case["hi"] + 1, (n, 3))
    ranks = np.minimum(sizes.integers(case["rlo"], case["rhi"] + 1, n), dims.min(axis=1))
    nf = int((dims.sum(axis=1) * ranks).sum())
    nt = int(dims.prod(axis=1).sum())
    true = torch.randn(nf, generator=g, device=DEV, dtype=torch.float64)
    start = torch.randn(nf, generator=g, device=DEV, dtype=torch.float64).cpu().numpy()
    flat = torch.randn(nt, generator=g, device=DEV, dtype=torch.float64).mul_(1e-3)
    fo = to = 0
    where = []
    for d, r in zip(dims.tolist(), ranks.tolist()):
        fs = []
        at = fo
        for k in d:
            fs.append(true[at:at + k * r].view(k, r))
            at += k * r
        I, J, K = d
        flat[to:to + I * J * K] += ((fs[2][:, None, :] * fs[1][None]).reshape(J * K, r) @ fs[0].T).reshape(-1)
        where.append((d, r, fo, to))
        fo, to = at, to + I * J * K
    flat = flat.cpu().numpy()
    for d, r, f0, t0 in where:
        T = flat[t0:t0 + d[0] * d[1] * d[2]].reshape(d, order="F")
        fs = []
        for k in d:
            f = start[f0:f0 + k * r].reshape(k, r)
            fs.append(f / np.linalg.norm(f, axis=0))
            f0 += k * r
        out.append((tuple(d), r, T, fs))
    return out


def _mlp_widths(case):
    return [case["width"], case["hidden"], case["hidden"], case["width"]]


def _mlp_inputs(case, seed):
    """(parameters W_0 | b_0 | ..., X, targets, mask) in FP32."""
    g, w, b = _gen(seed), _mlp_widths(case), case["batch"]
    par = []
    for i, o in zip(w[:-1], w[1:]):
        par.append((torch.randn(i * o, generator=g, device=DEV) * math.sqrt(2.0 / i)).cpu().numpy())
        par.append((torch.randn(o, generator=g, device=DEV) * 0.1).cpu().numpy())
    X = torch.randn(b, w[0], generator=g, device=DEV).cpu().numpy()
    Y = torch.randn(b, w[-1], generator=g, device=DEV).cpu().numpy()
    mask = (torch.rand(b, w[-1], generator=g, device=DEV) < 0.9).float().cpu().numpy()
    return np.concatenate(par), X, Y, mask


# ----------------------------------------------------------------- prepare / run
def prepare(case, seed):
    E = _engine()
    kind = case["kind"]
    if kind == "als":
        T, start = _als_inputs(case, seed)
        st = {"case": case, "E": E, "T": T, "cp": _host_cpd(E, start)}
        if case["check"] == "fit":
            st["norm"] = _norm(T)
        if case["entry"] == "plan":
            st["plan"] = E.ALSPlan(T, case["rank"], prec=case["prec"])
        return st
    if kind == "batch":
        probs = _batch_inputs(case, seed)
        bt = E.BatchALS([p[2] for p in probs], [p[1] for p in probs])
        cps = [E.CPD(p[3], np.ones(p[1])) for p in probs]
        bt.set_cpd(cps)
        bt.tune(2)      # a program tunes once and runs the batch many times
        return {"case": case, "E": E, "batch": bt, "cps": cps}
    if kind == "sampled":
        T, start = _als_inputs(case, seed)
        return {"case": case, "E": E, "T": T, "cp": _host_cpd(E, start), "plan": E.ALSPlan(T, case["rank"]),
                "seed": int(seed)}
    par, X, Y, mask = _mlp_inputs(case, seed)
    net = E.MLP(_mlp_widths(case), batch_cap=case["batch"], seed=1)
    net.set_params(par)
    return {"case": case, "net": net, "X": X, "Y": Y, "mask": mask}


def _cpd_out(cp, dtype=np.float64):
    return {"factors": [f.astype(dtype, copy=False) for f in cp.factors], "lam": cp.lam.astype(dtype, copy=False)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "als":
        E = state["E"]
        if case["check"] == "fit":
            # tolerance 0: the fit is evaluated after every sweep and never stops the run
            check = E.FitCheck(0.0, case["sweeps"], state["norm"])
        else:
            check = E.NoCheck(case["sweeps"])
        if case["entry"] == "call":
            return _cpd_out(E.als_optimize(state["T"], state["cp"], check=check))
        plan = state["plan"]
        plan.set_cpd(state["cp"])
        info = plan.run(check)
        # the reduced-precision forms carry FP32's accuracy at most: their CPD is kept in FP32
        out = _cpd_out(plan.get_cpd(), np.float64 if case["prec"] == "fp64" else np.float32)
        if case["check"] == "fit":
            out["fits"] = info["fits"]
        return out
    if kind == "batch":
        bt = state["batch"]
        bt.set_cpd(state["cps"])
        fits, _ = bt.run(case["sweeps"])
        cps = bt.get_cpd()
        return {"factors": np.concatenate([f.ravel(order="F") for cp in cps for f in cp.factors]),
                "lam": np.concatenate([cp.lam for cp in cps]), "fits": fits}
    if kind == "sampled":
        E, plan = state["E"], state["plan"]
        plan.set_cpd(state["cp"])
        plan.run_sampled(E.LevScoreSampled(case["samples"]), E.NoCheck(case["sweeps"]), normal=case["normal"],
                         rng=state["seed"])
        return _cpd_out(plan.get_cpd())
    net = state["net"]
    Yp = net.forward(state["X"])
    grads, loss = net.gradients(state["X"], state["Y"], state["mask"])
    return {"forward": Yp, "grads": grads, "loss": loss}


# ------------------------------------------------------------------------- work
def work(case):
    kind = case["kind"]
    if kind == "als":
        dims, R, n, N = _dims(case), case["rank"], case["sweeps"], len(_dims(case))
        size = _size(case)
        # the tensor read once; an ALS sweep contracts it with at least N / (N - 1) factors
        # (one contraction of the whole tensor serves at most N - 1 mode updates)
        flops = n * (2.0 * size * R * N / (N - 1) + sum(4.0 * d * R * R + R ** 3 / 3.0 for d in dims))
        return {"bytes": float(size * case["elt"] + 16 * sum(dims) * R), "flops": flops}
    if kind == "batch":
        sizes = np.random.default_rng([case["count"], case["lo"], case["hi"], case["rhi"]])
        dims = sizes.integers(case["lo"], case["hi"] + 1, (case["count"], 3))
        ranks = np.minimum(sizes.integers(case["rlo"], case["rhi"] + 1, case["count"]), dims.min(axis=1))
        el = dims.prod(axis=1).astype(float)
        d1 = dims.sum(axis=1)
        return {"bytes": float(8 * el.sum() + 16 * (d1 * ranks).sum()),
                "flops": float(case["sweeps"] * (3.0 * el * ranks + 4.0 * d1 * ranks ** 2 + ranks ** 3.0).sum())}
    if kind == "sampled":
        dims, R, ns, n = _dims(case), case["rank"], case["samples"], case["sweeps"]
        per = [8.0 * ns * d + 16.0 * d * R for d in dims]
        fl = [4.0 * ns * R * R + 4.0 * ns * d * R for d in dims]
        return {"bytes": float(n * sum(per)), "flops": float(n * sum(fl))}
    w, b = _mlp_widths(case), case["batch"]
    p = sum(i * o for i, o in zip(w[:-1], w[1:]))
    return {"bytes": float(4 * (2 * p + sum(w) + b * (w[0] + 3 * w[-1]))), "flops": float(8.0 * b * p)}


# ------------------------------------------------------------------------ exact
def _mttkrp(T2, dims, s, fac, n):
    """M_n in 64 bits; T2 = the tensor as (right multi-index) x (left multi-index)."""
    N = len(dims)
    left = _krp([fac[m] for m in reversed(range(s))])
    right = _krp([fac[m] for m in reversed(range(s, N))])
    if n >= s:
        P = torch.cat([x.double() @ left for x in T2.split(max(1, (1 << 28) // T2.shape[1]))])
        modes = list(range(s, N))
    else:
        P, at = torch.zeros(T2.shape[1], left.shape[1], device=DEV, dtype=torch.float64), 0
        for x in T2.split(max(1, (1 << 28) // T2.shape[1])):
            P += x.double().T @ right[at:at + x.shape[0]]
            at += x.shape[0]
        modes = list(range(s))
    P = P.reshape([dims[m] for m in reversed(modes)] + [-1])
    order = list(reversed(modes))
    while len(order) > 1:                   # contract the other modes of the side, one at a time
        k = 0 if order[0] != n else 1
        f = fac[order[k]].reshape([-1 if q == k else 1 for q in range(len(order))] + [P.shape[-1]])
        P = (P * f).sum(dim=k)
        del order[k]
    return P


def _fit(norm, M, A, lam, grams):
    had = grams[0].clone()
    for G in grams[1:]:
        had = had * G
    inner = float((M * A * lam).sum())
    square = float(lam @ had @ lam)
    return 1.0 - math.sqrt(abs(norm * norm + square - 2.0 * abs(inner))) / norm


def _exact_als(case, seed):
    T, fac = _als_inputs(case, seed)
    dims, N = _dims(case), len(_dims(case))
    s = _split(dims)
    T2 = T.permute(*reversed(range(N))).reshape(math.prod(dims[s:]), math.prod(dims[:s]))
    norm = _norm(T)
    grams = [f.T @ f for f in fac]
    lam, fits = None, []
    for _ in range(case["sweeps"]):
        for n in range(N):
            V = torch.ones_like(grams[0])
            for m in range(N):
                if m != n:
                    V = V * grams[m]
            M = _mttkrp(T2, dims, s, fac, n)
            X = torch.linalg.solve(V, M.T).T
            lam = X.norm(dim=0)
            fac[n] = X / lam
            grams[n] = fac[n].T @ fac[n]
        if case["check"] == "fit":
            fits.append(_fit(norm, M, fac[-1], lam, grams))
    out = {"factors": [f.cpu().numpy() for f in fac], "lam": lam.cpu().numpy()}
    if case["check"] == "fit":
        out["fits"] = np.array(fits)
    return out


def _exact_batch(case, seed):
    fs, lams, fits = [], [], []
    for dims, _, T, fac in _batch_inputs(case, seed):
        T = np.ascontiguousarray(T)
        unf = [np.ascontiguousarray(np.moveaxis(T, n, 0).reshape(dims[n], -1)) for n in range(3)]
        fac = [f.copy() for f in fac]
        grams = [f.T @ f for f in fac]
        for _ in range(case["sweeps"]):
            for n in range(3):
                a, b = [m for m in range(3) if m != n]
                krp = (fac[a][:, None, :] * fac[b][None]).reshape(-1, fac[a].shape[1])
                M = unf[n] @ krp
                X = np.linalg.solve(grams[a] * grams[b], M.T).T
                lam = np.linalg.norm(X, axis=0)
                fac[n] = X / lam
                grams[n] = fac[n].T @ fac[n]
        norm = np.linalg.norm(T)
        square = lam @ (grams[0] * grams[1] * grams[2]) @ lam
        inner = float((M * fac[2] * lam).sum())
        fits.append(1.0 - math.sqrt(abs(norm * norm + square - 2.0 * abs(inner))) / norm)
        fs += [f.ravel(order="F") for f in fac]
        lams.append(lam)
    return {"factors": np.concatenate(fs), "lam": np.concatenate(lams), "fits": np.array(fits)}


def _exact_sampled(case, seed):
    T, fac = _als_inputs(case, seed)
    fac = [f.cpu().numpy() for f in fac]
    T = T.cpu().numpy()
    rng = np.random.default_rng(int(seed))

    def scores(f):
        q = np.linalg.qr(f)[0]
        return (q * q).sum(axis=1) / min(f.shape)

    def drawn(n):
        cols = []
        for m in range(3):
            if m != n:
                p = np.abs(weights[m])
                cols.append(rng.choice(len(p), size=case["samples"], replace=True, p=p / p.sum()))
        return cols

    weights = [scores(f) for f in fac]
    for n in range(3):
        drawn(n)                            # the draws of the set-up, made again before each solve
    lam = None
    for _ in range(case["sweeps"]):
        for n in range(3):
            cols = drawn(n)
            others = [m for m in range(3) if m != n]
            K = fac[others[0]][cols[0]] * fac[others[1]][cols[1]]
            Ts = np.moveaxis(T, n, 2)[cols[0], cols[1]]
            X = (np.linalg.solve(K.T @ K, K.T @ Ts) if case["normal"] else np.linalg.lstsq(K, Ts, rcond=None)[0]).T
            lam = np.linalg.norm(X, axis=0)
            fac[n] = X / lam
            weights[n] = scores(fac[n])
    return {"factors": fac, "lam": lam}


def _exact_mlp(case, seed):
    par, X, Y, mask = (torch.from_numpy(a).double() for a in _mlp_inputs(case, seed))
    par.requires_grad_(True)
    w, at, x = _mlp_widths(case), 0, X
    for k, (i, o) in enumerate(zip(w[:-1], w[1:])):
        W = par[at:at + i * o].view(i, o)
        x = x @ W + par[at + i * o:at + i * o + o]
        at += i * o + o
        if k + 2 < len(w):
            x = torch.relu(x)
    loss = 0.5 * (mask * (x - Y) ** 2).sum() / case["batch"]
    loss.backward()
    return {"forward": x.detach().numpy(), "grads": par.grad.numpy(), "loss": float(loss.detach())}


def exact(case, seed):
    return {"als": _exact_als, "batch": _exact_batch, "sampled": _exact_sampled, "mlp": _exact_mlp}[case["kind"]](
        case, seed)
