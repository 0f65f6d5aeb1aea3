"""The measured cases of the particle-to-particle path: what a user of the
library has it do, through the public entry points of `flowvpm_amd`.

  functor   UJ_hip on a host particle matrix (upload, sort, U/J, download):
            the pfield.UJ call of a program that keeps its particles on the
            host.
  resident  Field.uj_direct on particles that live on the GPU, and the
            download of what it computed.
  step      one resident rungekutta3 step, and the download of the state.
  list      a planned FMM direct list served to U/J and then to E_str.
  listcall  one direct list handed over with its particles (p2p_ranges), as
            an FMM code does that rebuilds its tree each step.
  adjoint   Field.uj_adjoint of a loss on U, or on U and J.

Fields are the repository's own workloads (rings, the random cloud, the jet
column), perturbed by the seed.  F32C evaluates pairs in FP32 and its results
are handed on as float32; FP64 results are handed on as float64.  Rows are
those of the 46-double particle record: X 0-2, Gamma 3-5, sigma 6, U 9-11,
J 15-23 (J[3 b + a] = du_a/dx_b), SFS 39-41.
"""
import math

import numpy as np
import torch

from __graft_entry__ import load_package

vpm = load_package()

FLOP_PER_PAIR = {"gaussianerf": 88, "winckelmans": 97, "gaussian": 86, "singular": 79}
ESTR_FLOP = 48          # per E_str pair
ADJOINT_FLOP = 170      # per adjoint pair, loss on U and J (88 for a loss on U)


def listed():
    return [
        # one vortex ring of the reference's test: the smallest call, all latency
        dict(name="functor_ring_100", kind="functor", field="ring", n=100, kernel="gaussianerf", precision="f32c"),
        # a small unsteady wake kept on the host, U/J and E_str per call; ragged size
        dict(name="functor_cloud_3001", kind="functor", field="cloud", n=3001, kernel="gaussianerf",
             precision="f32c", sfs=True),
        # a ring of 8,000 particles stepped on the GPU: sorts, four U/J, relaxation
        dict(name="step_ring_8000", kind="step", field="ring", n=8000, kernel="gaussianerf", precision="f32c",
             les=False),
        # the leapfrog rings with dynamic SFS and core spreading, one step
        dict(name="step_leapfrog_65536", kind="step", field="leapfrog", n=65536, kernel="gaussianerf",
             precision="f32c", les=True),
        # another kernel, odd size, every pair in its full form
        dict(name="uj_cloud_winckelmans_30011", kind="resident", field="cloud", n=30011, kernel="winckelmans",
             precision="f32c"),
        # the ordinary dense cloud: a third of the pairs near
        dict(name="uj_cloud_65536", kind="resident", field="cloud", n=65536, kernel="gaussianerf",
             precision="f32c"),
        # the reference's FP64 arithmetic
        dict(name="uj_leapfrog_f64_16384", kind="resident", field="leapfrog", n=16384, kernel="gaussianerf",
             precision="f64", sfs=True),
        # the tuned FP64 form, odd size
        dict(name="uj_jet_f64far_100003", kind="resident", field="jet", n=100003, kernel="gaussianerf",
             precision="f64far"),
        # the largest: the jet column of 2^20 particles
        dict(name="uj_jet_1048576", kind="resident", field="jet", n=1 << 20, kernel="gaussianerf",
             precision="f32c"),
        # the backward of a U/J evaluation
        dict(name="adjoint_cloud_32768", kind="adjoint", field="cloud", n=32768, kernel="gaussianerf",
             precision="f32c", jbar=True),
        # FMM near field on 16-particle leaves, planned once per tree
        dict(name="list_jet_262144_leaf16", kind="list", field="jet", n=262144, kernel="gaussianerf",
             precision="f32c", leaf=16),
        # FMM near field of one call, ragged 50-particle leaves
        dict(name="listcall_jet_50021_leaf50", kind="listcall", field="jet", n=50021, kernel="gaussianerf",
             precision="f32c", leaf=50),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["functor", "resident", "resident", "resident", "step", "list", "listcall", "adjoint"])
    kernel = rng.choice(["gaussianerf", "gaussianerf", "gaussianerf", "winckelmans", "gaussian"])
    if kind == "functor":
        field = rng.choice(["ring", "cloud", "jet"])
        return dict(kind=kind, field=field, n=_log(rng, 60, 20000), kernel=kernel, precision="f32c",
                    sfs=rng.random() < 0.5)
    if kind == "resident":
        precision = rng.choice(["f32c", "f32c", "f32c", "f64", "f64far"])
        n = _log(rng, 2000, {"f32c": 400000, "f64": 40000, "f64far": 130000}[precision])
        return dict(kind=kind, field=rng.choice(["cloud", "jet", "leapfrog"]), n=n, kernel=kernel,
                    precision=precision, sfs=rng.random() < 0.3)
    if kind == "step":
        les = rng.random() < 0.5
        return dict(kind=kind, field=rng.choice(["ring", "leapfrog"]), n=_log(rng, 1000, 100000),
                    kernel="gaussianerf", precision="f32c", les=les)
    if kind == "adjoint":
        return dict(kind=kind, field=rng.choice(["cloud", "jet"]), n=_log(rng, 1000, 60000), kernel=kernel,
                    precision="f32c", jbar=rng.random() < 0.5)
    return dict(kind=kind, field=rng.choice(["cloud", "jet"]), n=_log(rng, 5000, 200000), kernel=kernel,
                precision="f32c", leaf=rng.choice([8, 11, 16, 27, 50, 64]))


def _field(case, seed):
    """The case's particle matrix, perturbed by the seed."""
    n, W = case["n"], vpm.workloads
    rng = np.random.default_rng([seed, n])
    if case["field"] == "cloud":
        return W.random_cloud(n, seed=seed)
    if case["field"] == "jet":
        return W.jet_column(n, seed=seed)
    if case["field"] == "ring":
        P = W.ring_cfg0() if n == 8000 else W.ring_test(Nphi=n, Rcross=min(0.15, 12 * math.pi / n))
    else:
        P = W.leapfrog_cfg2(Nphi=-(-n // 128))[:n].copy()
    step = P[:, 6].min() / 3
    P[:, 0:3] += rng.uniform(-0.1 * step, 0.1 * step, (n, 3))
    P[:, 3:6] *= 1.0 + 0.05 * rng.normal(size=(n, 1))
    return P


def _handed_on(case, a):
    return a.astype(np.float32) if case["precision"] == "f32c" else a.copy()


def prepare(case, seed):
    P = _field(case, seed)
    n = P.shape[0]
    kind = case["kind"]
    if kind == "functor":
        return dict(case=case, P=P)
    if kind in ("list", "listcall"):
        P = vpm.workloads.morton_order(P)
        pairs = vpm.workloads.leaf_direct_list(P, leaf=case["leaf"])
        if kind == "listcall":
            return dict(case=case, P=P, pairs=pairs)
    out = np.zeros((n, vpm.NFIELDS))
    if kind == "step":
        les = case["les"]
        pf = vpm.ParticleField(n, kernel=case["kernel"], precision=case["precision"],
                               SFS=vpm.SFS_Cd_twolevel_nobackscatter if les else vpm.noSFS,
                               viscous=vpm.CoreSpreading(1e-6, float(P[:, 6].min())) if les else vpm.Inviscid())
        vpm.add_particles(pf, P)
        vpm.pfield_upload(pf)
        return dict(case=case, pf=pf, out=out)
    f = vpm.Field(n)
    f.set_particles(P)
    state = dict(case=case, f=f, out=out)
    if kind == "list":
        state["plan"] = f.plan_ranges(*pairs)
    elif kind == "adjoint":
        w, W = vpm.workloads.adjoint_weights(n, seed=seed + 1)
        state["w"], state["W"] = w, W if case["jbar"] else np.zeros((n, 9))
    return state


def run(state):
    case = state["case"]
    kind, kernel, prec = case["kind"], case["kernel"], case["precision"]
    if kind == "functor":
        P, sfs = state["P"], case.get("sfs", False)
        vpm.UJ_hip(P, kernel=kernel, precision=prec, reset_sfs=sfs, sfs=sfs)
        outs = [P[:, 9:12], P[:, 15:24]] + ([P[:, 39:42]] if sfs else [])
    elif kind == "resident":
        f, out, sfs = state["f"], state["out"], case.get("sfs", False)
        f.uj_direct(kernel, prec, reset=True, reset_sfs=sfs, sfs=sfs)
        f.get_particles(out, rows=(9, 24))
        if sfs:
            f.get_particles(out, rows=(39, 42))
        outs = [out[:, 9:12], out[:, 15:24]] + ([out[:, 39:42]] if sfs else [])
    elif kind == "step":
        pf, out = state["pf"], state["out"]
        vpm.rungekutta3(pf, _dt(case), relax=not case["les"], resident=True)
        pf.device_field().get_particles(out, rows=(0, 7))
        outs = [out[:, 0:3], out[:, 3:6], out[:, 6]]
    elif kind == "list":
        # U and J, then SFS, accumulate onto the field, as the entry points say
        f, out = state["f"], state["out"]
        state["plan"].p2p(kernel, prec)
        state["plan"].estr(kernel, prec)
        f.get_particles(out, rows=(9, 42))
        outs = [out[:, 9:12], out[:, 15:24], out[:, 39:42]]
    elif kind == "listcall":
        P = state["P"]
        vpm.p2p_ranges(P, *state["pairs"], kernel=kernel, precision=prec)
        outs = [P[:, 9:12], P[:, 15:24]]
    else:
        outs = state["f"].uj_adjoint(state["w"], state["W"], kernel, prec)
    return [_handed_on(case, a) for a in outs]


def _dt(case):
    # small enough that a state stays well behaved over thousands of steps
    return 1e-4 if case["n"] < 20000 else 1e-3


_list_pairs = {}


def _particle_pairs(case):
    """Particle pairs of a case's direct list."""
    key = (case["field"], case["n"], case["leaf"])
    if key not in _list_pairs:
        tb, te, sb, se = vpm.workloads.leaf_direct_list(vpm.workloads.morton_order(_field(case, 0)),
                                                        leaf=case["leaf"])
        _list_pairs[key] = float(((te - tb) * (se - sb)).sum())
    return _list_pairs[key]


def work(case):
    """Bytes: each particle's source rows read and result rows written once.
    Flops: the reference's expressions, 88 per Gaussian-erf U/J pair etc."""
    n, kind = case["n"], case["kind"]
    uj, es = FLOP_PER_PAIR[case["kernel"]], ESTR_FLOP
    pairs = _particle_pairs(case) if "leaf" in case else float(n) * n
    if kind == "step":      # three stages, and the relaxation's evaluation or four E_str passes and the test filter
        flops = (4 * uj + (4 * es if case["les"] else 0)) * pairs
        nbytes = 8.0 * n * 4 * (7 + 12 + 9)
    elif kind == "adjoint":
        flops = (ADJOINT_FLOP if case["jbar"] else 88) * pairs
        nbytes = 8.0 * n * (7 + 12 + 7)
    else:
        sfs = case.get("sfs", False) or kind == "list"
        flops = (uj + (es if sfs else 0)) * pairs
        nbytes = 8.0 * n * (7 + 12 + (15 if sfs else 0))
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------------- FP64 values
# The same sums in plain torch, in 64 bits, a block of targets at a time.

_DEV = "cuda" if torch.cuda.is_available() else "cpu"
_EXACT_PAIRS = 1.3e10       # larger cases have no FP64 value


def _g_and_qdg(kernel, q):
    """g(q) and q g'(q) of a regularization kernel."""
    if kernel == "gaussianerf":
        a = math.sqrt(2 / math.pi) * q * torch.exp(-0.5 * q * q)
        return torch.erf(q / math.sqrt(2)) - a, a * q * q
    if kernel == "gaussian":
        q3 = q ** 3
        return -torch.expm1(-q3), 3 * q3 * torch.exp(-q3)
    t = q * q
    return q ** 3 * (t + 2.5) / (t + 1) ** 2.5, 7.5 * q ** 3 / (t + 1) ** 3.5


def _zeta(kernel, q):
    if kernel == "gaussianerf":
        return torch.exp(-0.5 * q * q) / (2 * math.pi) ** 1.5
    if kernel == "gaussian":
        return 3 / (4 * math.pi) * torch.exp(-q ** 3)
    return 7.5 / (4 * math.pi) / (q * q + 1) ** 3.5


def _pairs_uj(d, G, S, kernel):
    """Weights of each pair with separation d[..., 3]: c (crss), aux, aux2."""
    r2 = (d * d).sum(-1)
    zero = r2 == 0
    r2 = torch.where(zero, torch.ones_like(r2), r2)
    r = torch.sqrt(r2)
    g, qdg = _g_and_qdg(kernel, r / S)
    g = torch.where(zero, torch.zeros_like(g), g)
    qdg = torch.where(zero, torch.zeros_like(qdg), qdg)
    w = -1 / (4 * math.pi) / (r2 * r)
    c = w[..., None] * torch.linalg.cross(d, G.expand_as(d))
    return g[..., None] * c, ((qdg - 3 * g) / r2)[..., None] * c, g * w


def _eps(W):
    """The epsilon term of J from W = sum g w Gamma."""
    z = torch.zeros_like(W[:, 0])
    return torch.stack([z, -W[:, 2], W[:, 1], W[:, 2], z, -W[:, 0], -W[:, 1], W[:, 0], z], 1)


def _uj_block(X, G, S, xt, kernel):
    d = xt[:, None, :] - X[None]
    u, ac, w = _pairs_uj(d, G[None], S[None], kernel)
    W = w @ G
    J = torch.stack([(ac * d[..., b:b + 1]).sum(1) for b in range(3)], 1).reshape(-1, 9)
    return u.sum(1), J + _eps(W)


def _blocks(n, per=3.0e6):
    m = max(1, int(per / n))
    return [slice(i, min(i + m, n)) for i in range(0, n, m)]


def _uj(X, G, S, kernel):
    got = [_uj_block(X, G, S, X[b], kernel) for b in _blocks(X.shape[0])]
    return torch.cat([u for u, _ in got]), torch.cat([j for _, j in got])


def _estr(X, G, S, J, kernel):
    q3 = (J.reshape(-1, 3, 3) * G[:, None, :]).sum(-1)          # J^T Gamma: sum_c J[3 a + c] Gamma_c
    out = []
    for b in _blocks(X.shape[0]):
        z = _zeta(kernel, torch.linalg.norm(X[b][:, None, :] - X[None], dim=-1) / S) / S ** 3
        A = z @ G
        out.append((J[b].reshape(-1, 3, 3) * A[:, None, :]).sum(-1) - z @ q3)
    return torch.cat(out)


def _list_pair_blocks(X, pairs):
    """(targets, sources) of a direct list's particle pairs, a block at a time."""
    tb, te, sb, se = (torch.from_numpy(np.ascontiguousarray(a)).to(X.device) for a in pairs)
    cnt = (te - tb) * (se - sb)
    ends = torch.cumsum(cnt, 0)
    lo = 0
    while lo < cnt.numel():
        hi = int(torch.searchsorted(ends, (ends[lo] - cnt[lo]) + 2_000_000, right=True))
        hi = max(hi, lo + 1)
        k = torch.repeat_interleave(torch.arange(lo, hi, device=X.device), cnt[lo:hi])
        at = torch.arange(k.numel(), device=X.device) - (ends[k] - cnt[k] - (ends[lo] - cnt[lo]))
        ns = (se - sb)[k]
        yield tb[k] + at // ns, sb[k] + at % ns
        lo = hi


def _list_uj(X, G, S, pairs, kernel):
    U, J, W = (torch.zeros(X.shape[0], k, dtype=X.dtype, device=X.device) for k in (3, 9, 3))
    for i, j in _list_pair_blocks(X, pairs):
        d = X[i] - X[j]
        u, ac, w = _pairs_uj(d, G[j], S[j], kernel)
        U.index_add_(0, i, u)
        W.index_add_(0, i, w[:, None] * G[j])
        J.index_add_(0, i, torch.cat([ac * d[:, b:b + 1] for b in range(3)], 1))
    return U, J + _eps(W)


def _list_estr(X, G, S, J, pairs, kernel):
    q3 = (J.reshape(-1, 3, 3) * G[:, None, :]).sum(-1)
    A, B = torch.zeros_like(X), torch.zeros_like(X)
    for i, j in _list_pair_blocks(X, pairs):
        z = (_zeta(kernel, torch.linalg.norm(X[i] - X[j], dim=-1) / S[j]) / S[j] ** 3)[:, None]
        A.index_add_(0, i, z * G[j])
        B.index_add_(0, i, z * q3[j])
    return (J.reshape(-1, 3, 3) * A[:, None, :]).sum(-1) - B


def _rk3(X, G, S, dt, kernel):
    """rungekutta3 of ReformulatedVPM(0, 1/5) without SFS, then Pedrizzetti
    relaxation with factor 0.3."""
    f, g = 0.0, 0.2
    MX, MG, MS = torch.zeros_like(X), torch.zeros_like(G), torch.zeros_like(S)
    for a, b in ((0.0, 1 / 3), (-5 / 9, 15 / 16), (-153 / 128, 8 / 15)):
        U, J = _uj(X, G, S, kernel)
        MX = a * MX + dt * U
        st = (J.reshape(-1, 3, 3) * G[:, None, :]).sum(-1)
        m4 = (f + g) / (1 + 3 * f) * (st * G).sum(-1) / (G * G).sum(-1)
        MG = a * MG + dt * (st - 3 * m4[:, None] * G)
        MS = a * MS - dt * S * m4
        X, G, S = X + b * MX, G + b * MG, S + b * MS
    J = _uj(X, G, S, kernel)[1]
    w = torch.stack([J[:, 5] - J[:, 7], J[:, 6] - J[:, 2], J[:, 1] - J[:, 3]], 1)
    nw, ng = torch.linalg.norm(w, dim=1, keepdim=True), torch.linalg.norm(G, dim=1, keepdim=True)
    return X, 0.7 * G + 0.3 * ng * w / nw, S


def exact(case, seed):
    kind, kernel, n = case["kind"], case["kernel"], case["n"]
    if "leaf" not in case and float(n) * n > _EXACT_PAIRS:
        return None
    if kind == "step" and (case["les"] or float(n) * n > _EXACT_PAIRS / 4):
        return None
    if kind == "adjoint" and float(n) * n > _EXACT_PAIRS / 4:
        return None
    P = _field(case, seed)
    if "leaf" in case:
        P = vpm.workloads.morton_order(P)
    T = torch.from_numpy(P[:, 0:7].copy()).to(_DEV)
    X, G, S = T[:, 0:3].contiguous(), T[:, 3:6].contiguous(), T[:, 6].contiguous()
    if kind == "step":
        outs = _rk3(X, G, S, _dt(case), kernel)
    elif kind == "adjoint":
        w, W = vpm.workloads.adjoint_weights(n, seed=seed + 1)
        w, W = torch.from_numpy(w).to(_DEV), torch.from_numpy(W if case["jbar"] else np.zeros((n, 9))).to(_DEV)
        for t in (X, G, S):
            t.requires_grad_(True)
        for b in _blocks(n, 1.0e6):
            U, J = _uj_block(X, G, S, X[b], kernel)
            ((U * w[b]).sum() + (J * W[b]).sum()).backward()
        outs = X.grad, G.grad, S.grad
    elif "leaf" in case:
        pairs = vpm.workloads.leaf_direct_list(P, leaf=case["leaf"])
        U, J = _list_uj(X, G, S, pairs, kernel)
        outs = (U, J, _list_estr(X, G, S, J, pairs, kernel)) if kind == "list" else (U, J)
    else:
        U, J = _uj(X, G, S, kernel)
        outs = (U, J, _estr(X, G, S, J, kernel)) if case.get("sfs", False) else (U, J)
    return [o.detach().cpu().numpy() for o in outs]
