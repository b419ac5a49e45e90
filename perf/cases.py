"""Performance cases of the P2P near-field library: the work a user's program has it do.

Every case goes through a public entry point of ``stkfmm_amd`` as a program calls it.  The kinds:

* ``host``       ``evaluate_kernel`` on host arrays (the drop-in for STKFMM::evaluateKernel);
* ``leafblocks`` ``ker_eval`` over a sequence of target-leaf x source-leaf blocks of different sizes
                 (the drop-in for pvfmm's Ker_t calls);
* ``device``     ``p2p_device`` on resident tensors;
* ``instances``  one plan of many independent self-interaction sums, points ordered by the plan;
* ``ulist``      the U-list of an adaptive octree, one plan per layer;
* ``surfaces``   the S2M, X, W and L2T lists of the same tree around order-p surfaces;
* ``wall``       ``wall_device``, the no-slip image system;
* ``autograd``   a differentiable direct sum, forward and backward.

Inputs follow the distributions of ``stkfmm_amd.workloads`` (uniform points, Gaussian and log-normal
clusters, normal forces) and are drawn from the case's seed.  The outputs start at zero in every pass,
as a program that wants the sum alone has them; ``exact`` states the same sums in plain float64 torch.
"""
import math

import numpy as np
import torch

import stkfmm_amd as S
from stkfmm_amd import autograd as A

K, PP, U, P = S.KERNEL, S.PPKERNEL, S.UKER, S.PREC
DEV = "cuda"

# floating-point operations of one pair (FMA = 2), from the pair formulas; adjoints count the one
# pass that gives all three gradients
FLOPS = {U.LAPLACE_P: 12, U.LAPLACE_DIPOLEP: 19, U.LAPLACE_PGRAD: 20, U.LAPLACE_DIPOLEPGRAD: 31,
         U.LAPLACE_PGRADGRAD: 39, U.STOKES_VEL: 29, U.STOKES_PVEL: 35, U.STOKES_DOUBLEPVEL: 45,
         U.STOKES_REGVEL: 35, U.RPY_U: 40, U.RPY_ULAPU: 56, U.STK_ULAPU: 45, U.STOKES_PVEL_FUSED: 72,
         U.STOKES_PVELGRAD: 119, U.STOKES_DOUBLEPVELGRAD: 106, U.STOKES_PVELLAPLACIAN: 60,
         U.STOKES_DOUBLELAPLACIAN: 71, U.STOKES_TRACTION: 57, U.LAPLACE_QUADPGRADGRAD: 124}
ADJOINT_FLOPS = {U.LAPLACE_PGRAD: 50, U.STOKES_VEL: 62, U.STOKES_REGVEL: 75, U.STOKES_PVEL: 75, U.RPY_ULAPU: 100}
# source and its image against one target
WALL_FLOPS = {K.Stokes: 90, K.RPY: 170}


def listed():
    return [
        # the smallest call: a script or a test that checks a few hundred points, on host arrays
        dict(name="host_lapgrad_1k", kind="host", kernel=int(K.LapPGrad), p2p=int(PP.SLS2T), ns=1000, nt=1000,
             prec=0),
        # pvfmm's near-field loop with its Ker_t entries replaced: 24 leaf blocks, no two alike
        dict(name="leafblocks_pvel", kind="leafblocks", uker=int(U.STOKES_PVEL), blocks=24, shape=1, nt_lo=150,
             nt_hi=1000, ns_lo=1000, ns_hi=9000),
        # a small differentiable sum inside an optimisation loop (odd sizes, mixed precision)
        dict(name="autograd_stokes_mixed_3k", kind="autograd", uker=int(U.STOKES_VEL), ns=3001, nt=2503, prec=1),
        # the reference's direct sum at the size the benchmark runs it
        dict(name="device_lapgrad_8k", kind="device", kernel=int(K.LapPGrad), p2p=int(PP.SLS2T), ns=8192, nt=8192,
             prec=0),
        # an ordinary large direct sum of a double layer, ragged
        dict(name="device_pvel_dl_40k", kind="device", kernel=int(K.PVel), p2p=int(PP.DLS2T), ns=40009, nt=30011,
             prec=0),
        # many independent suspensions at once (sizes of the benchmark's instances)
        dict(name="instances_stokes_mixed", kind="instances", uker=int(U.STOKES_VEL), instances=128, shape=5,
             n_lo=1024, n_hi=32768, prec=1),
        # the headline: near field of a million-point Stokes evaluation, both layers, mixed precision
        dict(name="ulist_pvel_mixed_1m", kind="ulist", ukers=str(int(U.STOKES_PVEL_FUSED)), points="clusters",
             n=1000000, cap=1000, prec=1),
        # a log-normal suspension of spheres, double precision
        dict(name="ulist_rpy_fp64", kind="ulist", ukers=str(int(U.RPY_ULAPU)), points="lognormal", n=524288,
             cap=1000, prec=0),
        # velocity gradients of both layers, 16 outputs, double precision
        dict(name="ulist_pvelgrad_fp64", kind="ulist",
             ukers="%d,%d" % (U.STOKES_PVELGRAD, U.STOKES_DOUBLEPVELGRAD), points="clusters", n=262144, cap=500,
             prec=0),
        # the rest of the tree's near field: sources to surfaces and surfaces to targets
        dict(name="surfaces_pvel_mixed", kind="surfaces", kernel=int(K.PVel), points="clusters", n=262144, cap=500,
             p=8, shape=3, prec=1),
        # Stokes flow above a no-slip wall at the benchmark's size
        dict(name="wall_stokes_64k", kind="wall", kernel=int(K.Stokes), ns=65536, nt=65536),
        # gradients at the benchmark's size, double precision
        dict(name="autograd_pvel_fp64_64k", kind="autograd", uker=int(U.STOKES_PVEL), ns=65536, nt=65536, prec=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "leafblocks", "device", "device", "instances", "ulist", "ulist", "surfaces", "wall",
                       "autograd", "autograd"])
    direct = [(K.LapPGrad, PP.SLS2T), (K.LapPGrad, PP.DLS2T), (K.LapPGradGrad, PP.SLS2T), (K.Stokes, PP.SLS2T),
              (K.RPY, PP.SLS2T), (K.StokesRegVel, PP.SLS2T), (K.PVel, PP.SLS2T), (K.PVel, PP.DLS2T),
              (K.PVelGrad, PP.SLS2T), (K.Traction, PP.SLS2T)]
    if kind == "host":
        k, p = rng.choice(direct)
        return dict(kind=kind, kernel=int(k), p2p=int(p), ns=_log(rng, 200, 20000), nt=_log(rng, 200, 20000),
                    prec=rng.choice([0, 0, 1]))
    if kind == "leafblocks":
        uk = rng.choice([U.LAPLACE_PGRAD, U.STOKES_VEL, U.STOKES_PVEL, U.STOKES_DOUBLEPVEL, U.RPY_ULAPU])
        hi = _log(rng, 200, 2000)
        return dict(kind=kind, uker=int(uk), blocks=rng.randint(6, 32), shape=rng.randint(0, 1 << 20),
                    nt_lo=hi // 8, nt_hi=hi, ns_lo=hi, ns_hi=9 * hi)
    if kind == "device":
        k, p = rng.choice(direct)
        return dict(kind=kind, kernel=int(k), p2p=int(p), ns=_log(rng, 300, 50000), nt=_log(rng, 300, 50000),
                    prec=rng.choice([0, 1]))
    if kind == "instances":
        lo = _log(rng, 200, 3000)
        return dict(kind=kind, uker=int(rng.choice([U.STOKES_VEL, U.LAPLACE_PGRAD])), instances=rng.randint(16, 96),
                    shape=rng.randint(0, 1 << 20), n_lo=lo, n_hi=8 * lo, prec=rng.choice([0, 1]))
    if kind == "ulist":
        ukers = rng.choice([(U.STOKES_PVEL_FUSED,), (U.RPY_ULAPU,), (U.LAPLACE_PGRAD, U.LAPLACE_DIPOLEPGRAD),
                            (U.STOKES_VEL,), (U.STOKES_PVELGRAD, U.STOKES_DOUBLEPVELGRAD), (U.STOKES_TRACTION,),
                            (U.STOKES_PVELLAPLACIAN, U.STOKES_DOUBLELAPLACIAN), (U.LAPLACE_QUADPGRADGRAD,)])
        return dict(kind=kind, ukers=",".join(str(int(u)) for u in ukers), points=rng.choice(["clusters", "lognormal"]),
                    n=_log(rng, 30000, 300000), cap=_log(rng, 200, 1000), prec=rng.choice([0, 1]))
    if kind == "surfaces":
        return dict(kind=kind, kernel=int(rng.choice([K.PVel, K.LapPGrad, K.Stokes])), points="clusters",
                    n=_log(rng, 30000, 300000), cap=_log(rng, 200, 1000), p=rng.choice([6, 8, 10]),
                    shape=rng.randint(0, 1 << 20), prec=rng.choice([0, 1]))
    if kind == "wall":
        return dict(kind=kind, kernel=int(rng.choice([K.Stokes, K.RPY])), ns=_log(rng, 1000, 45000),
                    nt=_log(rng, 1000, 45000))
    return dict(kind=kind, uker=int(rng.choice([U.STOKES_VEL, U.STOKES_PVEL, U.LAPLACE_PGRAD, U.RPY_ULAPU,
                                                U.STOKES_REGVEL])),
                ns=_log(rng, 500, 50000), nt=_log(rng, 500, 50000), prec=rng.choice([0, 1]))


# ---- inputs ---------------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _uniform(g, n, k=3):
    return torch.rand((n, k), generator=g, dtype=torch.float64, device=DEV)


def _values(g, uker, n):
    """Source values of a micro-kernel: charges, forces, dipoles and stresses N(0,1); TrD 0; sphere radii and
    regularisation lengths U[1e-4, 5e-4]."""
    ks, _ = S.uker_dims(uker)
    v = torch.randn((n, ks), generator=g, dtype=torch.float64, device=DEV)
    if uker in (U.STOKES_PVEL, U.STOKES_PVEL_FUSED, U.STOKES_PVELGRAD, U.STOKES_PVELLAPLACIAN, U.STOKES_TRACTION):
        v[:, 3] = 0.0
    if uker in (U.RPY_U, U.RPY_ULAPU, U.STOKES_REGVEL):
        v[:, 3] = 1e-4 + 4e-4 * torch.rand(n, generator=g, dtype=torch.float64, device=DEV)
    return v


def _cloud(points, n, seed):
    """Points of a tree, as stkfmm_amd.workloads distributes them, on the host."""
    r = np.random.default_rng(seed)
    if points == "clusters":  # half uniform, half in 16 Gaussian clusters
        c = r.random((16, 3))
        x = np.concatenate([r.random((n // 2, 3)), c[np.arange(n - n // 2) % 16] + r.normal(0.0, 0.01, (n - n // 2, 3))])
    else:                     # 64 log-normal clusters
        c, radii, which = r.random((64, 3)), np.exp(r.uniform(math.log(1e-3), math.log(5e-2), 64)), np.arange(n) % 64
        v = r.normal(size=(n, 3))
        v /= np.linalg.norm(v, axis=1, keepdims=True)
        x = c[which] + (radii[which] * r.lognormal(0.0, 0.5, n))[:, None] * v
    return x - np.floor(x)


def _sizes(case, lo, hi, n, stream):
    r = np.random.default_rng([case["shape"], stream])
    return np.floor(np.exp(r.uniform(math.log(lo), math.log(hi), n))).astype(np.int64)


def _tree(case, seed):
    # the number of surfaces follows from the points: those of a surface case are its own (`shape`), and
    # its densities the seed's
    x = _cloud(case["points"], case["n"], case.get("shape", seed))
    t = S.Tree(x, case["cap"])
    return t, torch.from_numpy(np.ascontiguousarray(x[t.perm])).to(DEV)


def _surface_ukers(kernel):
    return S.get_s2m_uker(kernel), S.get_s2l_uker(kernel), S.get_m2t_uker(kernel), S.get_uker(kernel, PP.L2T)


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    st = dict(case=case)
    if kind in ("host", "device"):
        uk = S.get_uker(case["kernel"], case["p2p"])
        sc, tc, sv = _uniform(g, case["ns"]), _uniform(g, case["nt"]), _values(g, uk, case["ns"])
        st.update(uk=uk, sc=sc, sv=sv, tc=tc)
        if kind == "host":
            st.update(sc=sc.cpu().numpy(), sv=sv.cpu().numpy(), tc=tc.cpu().numpy())
    elif kind == "leafblocks":
        nt = _sizes(case, case["nt_lo"], case["nt_hi"], case["blocks"], 0)
        ns = _sizes(case, case["ns_lo"], case["ns_hi"], case["blocks"], 1)
        uk = U(case["uker"])
        sc, tc, sv = (t.cpu().numpy() for t in (_uniform(g, int(ns.sum())), _uniform(g, int(nt.sum())),
                                                _values(g, uk, int(ns.sum()))))
        st.update(uk=uk, sc=sc, sv=sv, tc=tc, sb=np.concatenate([[0], np.cumsum(ns)]),
                  tb=np.concatenate([[0], np.cumsum(nt)]))
    elif kind == "instances":
        n = _sizes(case, case["n_lo"], case["n_hi"], case["instances"], 0)
        off = np.concatenate([[0], np.cumsum(n)])
        uk, tot = U(case["uker"]), int(off[-1])
        plan = S.Plan(uk, P(case["prec"]), tot, tot, off[:-1], off[1:], None, np.arange(len(n) + 1), off[:-1], off[1:],
                      tune=dict(sort_points=1))
        st.update(uk=uk, off=off, sc=_uniform(g, tot), sv=_values(g, uk, tot), plan=plan)
    elif kind == "ulist":
        t, x = _tree(case, seed)
        ukers = [U(int(u)) for u in case["ukers"].split(",")]
        st.update(tree=t, x=x, ukers=ukers, sv=[_values(g, u, t.n) for u in ukers],
                  plans=[S.Plan.from_tree(t, u, P(case["prec"]), tune="auto") for u in ukers])
    elif kind == "surfaces":
        t, x = _tree(case, seed)
        pr = P(case["prec"])
        s2m, s2l, m2t, l2t = _surface_ukers(case["kernel"])
        up, down = S.LeafSurfaces(t, case["p"], S.RAD_OUTER), S.LeafSurfaces(t, case["p"], S.RAD_OUTER)
        nodes = S.NodeSurfaces(t, case["p"], S.RAD_INNER)
        st.update(tree=t, x=x, up=up, down=down, nodes=nodes, v_s2m=_values(g, s2m, t.n), v_s2l=_values(g, s2l, t.n),
                  v_m2t=_values(g, m2t, t.n_nodes * nodes.count), v_l2t=_values(g, l2t, t.n_leaves * down.count),
                  s2m=up.to_surface_plan(s2m, pr, tune="auto"), x_list=nodes.x_plan(s2l, pr, tune="auto"),
                  w_list=nodes.w_plan(m2t, pr, tune="auto"), l2t=down.from_surface_plan(l2t, pr, tune="auto"))
    elif kind == "wall":
        sc, tc = _uniform(g, case["ns"]), _uniform(g, case["nt"])
        sc[:, 2] *= 0.5
        tc[:, 2] *= 0.5
        st.update(sc=sc, tc=tc, sv=_values(g, U.STOKES_VEL if case["kernel"] == K.Stokes else U.RPY_ULAPU, case["ns"]))
    else:
        uk = U(case["uker"])
        sc, tc, sv = _uniform(g, case["ns"]), _uniform(g, case["nt"]), _values(g, uk, case["ns"])
        w = torch.randn((case["nt"], S.uker_dims(uk)[1]), generator=g, dtype=torch.float64, device=DEV)
        st.update(uk=uk, sc=sc.requires_grad_(), sv=sv.requires_grad_(), tc=tc.requires_grad_(), w=w)
    return st


# ---- one pass -------------------------------------------------------------------------------------

def _zeros(n, k):
    return torch.zeros((n, k), dtype=torch.float64, device=DEV)


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "host":
        out = np.zeros((case["nt"], S.uker_dims(st["uk"])[1]))
        return S.evaluate_kernel(case["kernel"], 0, case["p2p"], st["sc"], st["sv"], st["tc"], out, P(case["prec"]))
    if kind == "leafblocks":
        out = np.zeros((st["tc"].shape[0], S.uker_dims(st["uk"])[1]))
        for s0, s1, t0, t1 in zip(st["sb"][:-1], st["sb"][1:], st["tb"][:-1], st["tb"][1:]):
            S.ker_eval(st["uk"], st["sc"][s0:s1], st["sv"][s0:s1], st["tc"][t0:t1], out[t0:t1])
        return out
    if kind == "device":
        out = _zeros(case["nt"], S.uker_dims(st["uk"])[1])
        return S.p2p_device(case["kernel"], case["p2p"], st["sc"], st["sv"], st["tc"], out, P(case["prec"]))
    if kind == "instances":
        out = _zeros(st["sc"].shape[0], st["plan"].kt)
        return st["plan"].execute(st["sc"], st["sv"], st["sc"], out)
    if kind == "ulist":
        out = _zeros(st["tree"].n, st["plans"][0].kt)
        for u, plan, sv in zip(st["ukers"], st["plans"], st["sv"]):
            if u == U.STOKES_PVEL_FUSED:
                plan.execute(st["x"], sv[:, :4], st["x"], out, src_value2=sv[:, 4:])
            else:
                plan.execute(st["x"], sv, st["x"], out)
        return out
    if kind == "surfaces":
        t = st["tree"]
        check = _zeros(t.n_leaves * st["up"].count, st["s2m"].kt)
        local = _zeros(t.n_nodes * st["nodes"].count, st["x_list"].kt)
        trg = _zeros(t.n, st["l2t"].kt)
        st["s2m"].execute(st["x"], st["v_s2m"], st["up"].coord, check)
        st["x_list"].execute(st["x"], st["v_s2l"], st["nodes"].coord, local)
        st["w_list"].execute(st["nodes"].coord, st["v_m2t"], st["x"], trg)
        st["l2t"].execute(st["down"].coord, st["v_l2t"], st["x"], trg)
        return [check, local, trg]
    if kind == "wall":
        out = _zeros(case["nt"], 3 if case["kernel"] == K.Stokes else 6)
        return S.wall_device(case["kernel"], st["sc"], st["sv"], st["tc"], out)
    u = A.p2p(st["uk"], st["sc"], st["sv"], st["tc"], precision=P(case["prec"]))
    return [u.detach(), *torch.autograd.grad(u, (st["sc"], st["sv"], st["tc"]), st["w"])]


# ---- work -----------------------------------------------------------------------------------------

def _io(uker, ns, nt):
    ks, kt = S.uker_dims(uker)
    return 8.0 * (ns * (3 + ks) + nt * (3 + kt))


def work(case):
    kind = case["kind"]
    if kind in ("host", "device"):
        uk = S.get_uker(case["kernel"], case["p2p"])
        return dict(bytes=_io(uk, case["ns"], case["nt"]), flops=_flops(uk) * case["ns"] * case["nt"])
    if kind == "leafblocks":
        uk = U(case["uker"])
        nt = _sizes(case, case["nt_lo"], case["nt_hi"], case["blocks"], 0)
        ns = _sizes(case, case["ns_lo"], case["ns_hi"], case["blocks"], 1)
        return dict(bytes=_io(uk, int(ns.sum()), int(nt.sum())), flops=_flops(uk) * float((ns * nt).sum()))
    if kind == "instances":
        n = _sizes(case, case["n_lo"], case["n_hi"], case["instances"], 0)
        uk = U(case["uker"])
        return dict(bytes=_io(uk, int(n.sum()), 0) + 8.0 * int(n.sum()) * S.uker_dims(uk)[1],
                    flops=_flops(uk) * float((n * n).sum()))
    if kind == "ulist":
        t = S.Tree(_cloud(case["points"], case["n"], 1), case["cap"])  # the seed moves the pairs by a few per cent
        ukers = [U(int(u)) for u in case["ukers"].split(",")]
        return dict(bytes=8.0 * t.n * (3 + sum(S.uker_dims(u)[0] for u in ukers) + S.uker_dims(ukers[0])[1]),
                    flops=sum(_flops(u) for u in ukers) * t.pairs)
    if kind == "surfaces":
        t = S.Tree(_cloud(case["points"], case["n"], case["shape"]), case["cap"])
        s2m, s2l, m2t, l2t = _surface_ukers(case["kernel"])
        m = S.surface_count(case["p"])
        leaf = t.leaf_end - t.leaf_begin
        w = float(np.dot(np.diff(t.w_ptr).astype(float), leaf)) * m
        return dict(bytes=_io(s2m, t.n, t.n_leaves * m) + _io(s2l, t.n, t.n_nodes * m) + _io(m2t, t.n_nodes * m, t.n)
                    + _io(l2t, t.n_leaves * m, t.n),
                    flops=(_flops(s2m) + _flops(l2t)) * t.n * m + (_flops(s2l) + _flops(m2t)) * w)
    if kind == "wall":
        k = 3 if case["kernel"] == K.Stokes else 4
        return dict(bytes=8.0 * (case["ns"] * (3 + k) + case["nt"] * (3 + (3 if k == 3 else 6))),
                    flops=float(WALL_FLOPS[K(case["kernel"])]) * case["ns"] * case["nt"])
    uk = U(case["uker"])
    ks, kt = S.uker_dims(uk)
    return dict(bytes=8.0 * (case["ns"] * 2 * (3 + ks) + case["nt"] * (6 + 2 * kt)),
                flops=float(_flops(uk) + ADJOINT_FLOPS[uk]) * case["ns"] * case["nt"])


def _flops(uker):
    return float(FLOPS[U(int(uker))])


# ---- the same sums in plain float64 torch -----------------------------------------------------------

def _dot(a, b):
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]


def _pair(uker, r, f):
    """Outputs of one micro-kernel for displacements r = (x, y, z) and source values f (lists of tensors that
    broadcast to [targets, sources]), with its scale factor left out."""
    r2 = _dot(r, r)
    if uker == U.STOKES_REGVEL:
        e2 = f[3] * f[3]
        s = torch.rsqrt(r2 + e2)
        s3, fr = s * s * s, _dot(f, r)
        return [((r2 + 2 * e2) * f[i] + r[i] * fr) * s3 for i in range(3)]
    s = torch.where(r2 > 0, torch.rsqrt(torch.where(r2 > 0, r2, torch.ones_like(r2))), torch.zeros_like(r2))
    s3 = s * s * s
    s5 = s3 * s * s
    if uker == U.LAPLACE_P:
        return [f[0] * s]
    if uker == U.LAPLACE_DIPOLEP:
        return [_dot(f, r) * s3]
    if uker == U.LAPLACE_PGRAD:
        return [f[0] * s] + [-f[0] * s3 * r[i] for i in range(3)]
    if uker == U.LAPLACE_DIPOLEPGRAD:
        c = _dot(f, r)
        return [c * s3] + [f[i] * s3 - 3 * c * r[i] * s5 for i in range(3)]
    if uker == U.LAPLACE_PGRADGRAD:
        h = [f[0] * (3 * r[i] * r[j] * s5 - (s3 if i == j else 0.0)) for i in range(3) for j in range(i, 3)]
        return [f[0] * s] + [-f[0] * s3 * r[i] for i in range(3)] + h
    if uker in (U.STOKES_VEL, U.STOKES_PVEL, U.RPY_U, U.RPY_ULAPU, U.STK_ULAPU, U.STOKES_PVELGRAD,
                U.STOKES_PVELLAPLACIAN, U.STOKES_TRACTION):
        c = _dot(f, r)
        if uker == U.STOKES_VEL:
            return [f[i] * s + r[i] * c * s3 for i in range(3)]
        if uker in (U.RPY_U, U.RPY_ULAPU, U.STK_ULAPU):
            q = [f[i] * s3 - 3 * c * r[i] * s5 for i in range(3)]
            b = 0.0 if uker == U.STK_ULAPU else f[3] * f[3] / 3
            u = [f[i] * s + r[i] * c * s3 + b * q[i] for i in range(3)]
            return u if uker == U.RPY_U else u + [2 * q[i] for i in range(3)]
        a = c - f[3]
        if uker == U.STOKES_TRACTION:
            return [r[i] * r[j] * a * s5 + (f[3] * s3 / 3 if i == j else 0.0) for i in range(3) for j in range(3)]
        pu = [2 * c * s3] + [f[i] * s + r[i] * a * s3 for i in range(3)]
        if uker == U.STOKES_PVEL:
            return pu
        gp = [2 * (f[i] * s3 - 3 * r[i] * c * s5) for i in range(3)]
        if uker == U.STOKES_PVELLAPLACIAN:
            return pu + gp
        return pu + gp + [(s3 * a if i == j else 0.0) - 3 * r[i] * r[j] * a * s5 + (r[i] * f[j] - r[j] * f[i]) * s3
                          for i in range(3) for j in range(3)]
    s7 = s5 * s * s
    sym = [f[0] + f[0], f[1] + f[3], f[2] + f[6], f[4] + f[4], f[5] + f[7], f[8] + f[8]]
    c = [sym[0] * r[0] + sym[1] * r[1] + sym[2] * r[2], sym[1] * r[0] + sym[3] * r[1] + sym[4] * r[2],
         sym[2] * r[0] + sym[4] * r[1] + sym[5] * r[2]]
    q, tr = 0.5 * _dot(c, r), f[0] + f[4] + f[8]
    if uker == U.LAPLACE_QUADPGRADGRAD:
        s9 = s7 * s * s
        h = []
        for k, (i, j) in enumerate([(0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2)]):
            v = (35 * q * s9 - 5 * tr * s7) * r[i] * r[j] - 5 * (r[j] * c[i] + r[i] * c[j]) * s7 + sym[k] * s5
            h.append(3 * (v + tr * s5 - 5 * q * s7) if i == j else 3 * v)
        return [3 * q * s5 - tr * s3] + [-3 * (5 * r[i] * q * s7 - (c[i] + r[i] * tr) * s5) for i in range(3)] + h
    pu = [2 * (tr * s3 - 3 * q * s5)] + [-3 * r[i] * q * s5 for i in range(3)]
    if uker == U.STOKES_DOUBLEPVEL:
        return pu
    gp = [6 * (5 * r[i] * q * s7 - (c[i] + r[i] * tr) * s5) for i in range(3)]
    if uker == U.STOKES_DOUBLELAPLACIAN:
        return pu + gp
    if uker == U.STOKES_DOUBLEPVELGRAD:
        return pu + gp + [15 * q * r[i] * r[j] * s7 - 3 * r[i] * c[j] * s5 - (3 * q * s5 if i == j else 0.0)
                          for i in range(3) for j in range(3)]
    raise ValueError("no formula for %r" % (uker,))


def _scale(uker):
    if uker in (U.LAPLACE_P, U.LAPLACE_DIPOLEP, U.LAPLACE_PGRAD, U.LAPLACE_DIPOLEPGRAD, U.LAPLACE_PGRADGRAD,
                U.LAPLACE_QUADPGRADGRAD):
        return 1 / (4 * math.pi)
    return -3 / (4 * math.pi) if uker == U.STOKES_TRACTION else 1 / (8 * math.pi)


def _sum(uker, sc, sv, tc, elems=1 << 25):
    """[targets, outputs] of a direct sum."""
    if uker == U.STOKES_PVEL_FUSED:
        return _sum(U.STOKES_PVEL, sc, sv[:, :4], tc) + _sum(U.STOKES_DOUBLEPVEL, sc, sv[:, 4:], tc)
    f = [sv[None, :, k] for k in range(sv.shape[1])]
    x = [sc[None, :, d] for d in range(3)]
    step = max(1, elems // max(1, sc.shape[0]))
    got = []
    for b in range(0, tc.shape[0], step):
        o = _pair(uker, [tc[b:b + step, d, None] - x[d] for d in range(3)], f)
        got.append(torch.stack([v.sum(1) for v in o], 1))
        del o
    return torch.cat(got) * _scale(uker)


def _lists(uker, sc, sv, tc, gb, ge, ptr, rb, re, out):
    """The sums of a work list, added to out."""
    for k in range(len(gb)):
        rows = [(int(rb[r]), int(re[r])) for r in range(int(ptr[k]), int(ptr[k + 1])) if re[r] > rb[r]]
        if rows and ge[k] > gb[k]:
            out[gb[k]:ge[k]] += _sum(uker, torch.cat([sc[b:e] for b, e in rows]), torch.cat([sv[b:e] for b, e in rows]),
                                     tc[gb[k]:ge[k]])


def _wall(kernel, sc, sv, tc):
    """StkWallFMM's image system as its constituent sums."""
    img = sc * torch.tensor([1.0, 1.0, -1.0], dtype=torch.float64, device=sc.device)
    both = torch.cat([sc, img])
    z, f, x3 = sc[:, 2], sv, tc[:, 2]
    nil = torch.zeros_like(z)
    pair = lambda a, b: torch.cat([a, b])  # noqa: E731
    col = lambda a, b: torch.cat([a, b])[:, None]  # noqa: E731
    horiz = torch.stack([f[:, 0], f[:, 1], nil], 1)
    dip = torch.stack([-z * f[:, 0], -z * f[:, 1], z * f[:, 2]], 1)
    if kernel == K.Stokes:
        u = _sum(U.STOKES_VEL, both, pair(horiz, -horiz), tc)
        l1 = _sum(U.LAPLACE_PGRAD, both, col(-0.5 * f[:, 2], 0.5 * f[:, 2]), tc)
        l1 = l1 + _sum(U.LAPLACE_DIPOLEPGRAD, img, dip, tc)
        l2 = _sum(U.LAPLACE_PGRAD, both, col(f[:, 2] * z, -f[:, 2] * z), tc)
        u = u + 0.5 * l2[:, 1:4] + x3[:, None] * l1[:, 1:4]
        u[:, 2] -= l1[:, 0]
        return u
    b = f[:, 3]
    rp = _sum(U.RPY_ULAPU, both, pair(torch.cat([horiz, b[:, None]], 1), torch.cat([-horiz, b[:, None]], 1)), tc)
    sd = _sum(U.LAPLACE_PGRADGRAD, both, col(-0.5 * f[:, 2], 0.5 * f[:, 2]), tc)
    # the Hessian of a dipole potential, through the quadrupole-free third derivative of 1/r
    sd = sd + _dipole_gradgrad(img, dip, tc)
    sz = _sum(U.LAPLACE_PGRAD, both, col(0.5 * z * f[:, 2], -0.5 * z * f[:, 2]), tc)
    dz = torch.stack([nil, nil, b * b * f[:, 2] / 6], 1)
    sz = sz + _sum(U.LAPLACE_DIPOLEPGRAD, both, pair(dz, dz), tc)
    q0 = 2 * b * b * f[:, 2] / 6
    quad = torch.stack([q0, nil, nil, nil, q0, nil, 2 * b * b * f[:, 0] / 6, 2 * b * b * f[:, 1] / 6, nil], 1)
    q = _sum(U.LAPLACE_QUADPGRADGRAD, img, quad, tc)
    u = rp.clone()
    u[:, :3] += sz[:, 1:4] + x3[:, None] * (sd[:, 1:4] + q[:, 1:4])
    u[:, 2] -= sd[:, 0] + q[:, 0]
    for i, k in ((3, 6), (4, 8), (5, 9)):
        u[:, i] += 2 * (sd[:, k] + q[:, k])
    return u


def _dipole_gradgrad(sc, sv, tc, elems=1 << 25):
    """[p, grad(3), Hessian xx, xy, xz, yy, yz, zz] of dipoles."""
    got = []
    for b in range(0, tc.shape[0], max(1, elems // sc.shape[0])):
        t = tc[b:b + max(1, elems // sc.shape[0])]
        r = [t[:, d, None] - sc[None, :, d] for d in range(3)]
        f = [sv[None, :, d] for d in range(3)]
        r2 = _dot(r, r)
        s = torch.where(r2 > 0, torch.rsqrt(r2), torch.zeros_like(r2))
        s3, c = s * s * s, _dot(f, r)
        s5 = s3 * s * s
        s7 = s5 * s * s
        o = [c * s3] + [f[i] * s3 - 3 * c * r[i] * s5 for i in range(3)]
        o += [15 * c * r[i] * r[j] * s7 - 3 * (r[i] * f[j] + r[j] * f[i] + (c if i == j else 0.0)) * s5
              for i in range(3) for j in range(i, 3)]
        got.append(torch.stack([v.sum(1) for v in o], 1))
    return torch.cat(got) / (4 * math.pi)


def _autograd(uker, sc, sv, tc, w, elems=1 << 22):
    """u and the gradients of sum(w u) with respect to sc, sv and tc, block by block."""
    sc, sv = sc.detach().requires_grad_(), sv.detach().requires_grad_()
    step = max(1, elems // sc.shape[0])
    us, gt = [], []
    gc, gv = torch.zeros_like(sc), torch.zeros_like(sv)
    for b in range(0, tc.shape[0], step):
        t = tc[b:b + step].detach().requires_grad_()
        u = _sum(uker, sc, sv, t, 1 << 30)
        c, v, x = torch.autograd.grad(u, (sc, sv, t), w[b:b + step])
        us.append(u.detach())
        gt.append(x)
        gc += c
        gv += v
    return [torch.cat(us), gc, gv, torch.cat(gt)]


def exact(case, seed):
    st = prepare(case, seed)
    kind = case["kind"]
    if kind == "host":
        sc, sv, tc = (torch.from_numpy(st[k]).to(DEV) for k in ("sc", "sv", "tc"))
        return _sum(st["uk"], sc, sv, tc).cpu().numpy()
    if kind == "leafblocks":
        sc, sv, tc = (torch.from_numpy(st[k]).to(DEV) for k in ("sc", "sv", "tc"))
        return torch.cat([_sum(st["uk"], sc[a:b], sv[a:b], tc[c:d]) for a, b, c, d in
                          zip(st["sb"][:-1], st["sb"][1:], st["tb"][:-1], st["tb"][1:])]).cpu().numpy()
    if kind == "device":
        return _sum(st["uk"], st["sc"], st["sv"], st["tc"])
    if kind == "instances":
        return torch.cat([_sum(st["uk"], st["sc"][a:b], st["sv"][a:b], st["sc"][a:b])
                          for a, b in zip(st["off"][:-1], st["off"][1:])])
    if kind == "ulist":
        t = st["tree"]
        out = _zeros(t.n, st["plans"][0].kt)
        for u, sv in zip(st["ukers"], st["sv"]):
            _lists(u, st["x"], sv, st["x"], t.leaf_begin, t.leaf_end, t.ulist_ptr, t.rng_begin, t.rng_end, out)
        return out
    if kind == "surfaces":
        t, m = st["tree"], st["up"].count
        s2m, s2l, m2t, l2t = _surface_ukers(case["kernel"])
        check, local, trg = (_zeros(n, S.uker_dims(u)[1]) for n, u in
                             ((t.n_leaves * m, s2m), (t.n_nodes * m, s2l), (t.n, l2t)))
        lb, nb = np.arange(t.n_leaves) * m, np.arange(t.n_nodes) * m
        one = np.arange(t.n_leaves + 1)
        _lists(s2m, st["x"], st["v_s2m"], st["up"].coord, lb, lb + m, one, t.leaf_begin, t.leaf_end, check)
        _lists(s2l, st["x"], st["v_s2l"], st["nodes"].coord, nb, nb + m, t.x_ptr, t.leaf_begin[t.x_leaf],
               t.leaf_end[t.x_leaf], local)
        _lists(m2t, st["nodes"].coord, st["v_m2t"], st["x"], t.leaf_begin, t.leaf_end, t.w_ptr, t.w_node * m,
               t.w_node * m + m, trg)
        _lists(l2t, st["down"].coord, st["v_l2t"], st["x"], t.leaf_begin, t.leaf_end, one, lb, lb + m, trg)
        return [check, local, trg]
    if kind == "wall":
        return _wall(K(case["kernel"]), st["sc"], st["sv"], st["tc"])
    return _autograd(st["uk"], st["sc"], st["sv"], st["tc"], st["w"])
