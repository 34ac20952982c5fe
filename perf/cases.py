"""The work that programs have this library do, as measurable cases: value iteration (one solve,
repeated sweeps, batches, gradients), point-based value iteration (solves, backups of a kept
solver, batches, gradients, dense beliefs), and running policies (value and action, belief
updates). Sizes are those of nova_amd/synth.py, bench.py and the tests, or smaller and ragged
ones between.

A case is a dict of plain values. prepare(case, seed) makes what a program holds before the
call, run(state) makes one pass through the public entry points and returns its whole outputs,
work(case) says what bytes and operations a pass cannot do without, tolerance(case) how far two
correct implementations may lie apart, exact(case, seed) the outputs in 64 bits.

A program that calls one model again and again keeps the model and its solver, and brings new
values, alphas or beliefs to each call: those kinds (vi_run, pbvi_run, pbvi_dense, update) share
one model per case, drawn from the case's sizes, and take the call's inputs from the seed. The
others build their models from the seed.
"""
import ctypes as ct
import math
import zlib

import numpy as np
import torch

from nova_amd import _abi, mdp_vi, pomdp_pbvi, synth
from nova_amd.autograd import BellmanFixedPoint, PBVIBeliefValue
from nova_amd.mdp import MDP
from nova_amd.pomdp import POMDP

FAST, EXACT, DENSE_BF16, DENSE_FP32 = 0, 1, 2, 3


def listed():
    return [
        # a grid-world sized MDP solved from scratch: a call of a planner that replans often
        dict(name="vi_solve_900", kind="vi_solve", n=900, m=5, ns=5, horizon=50, ragged=True),
        # bench.py's headline workload: 200 sweeps of a large MDP from a given V
        dict(name="vi_run_1m", kind="vi_run", n=1_000_000, m=8, ns=16, sweeps=200, ragged=False),
        # 64 uneven MDPs solved together (bench.py's batch of MDPs)
        dict(name="vi_batch_64", kind="vi_batch", count=64, nmin=500, nmax=8000, horizon=50),
        # V* and its gradient in R and T (forward and backward of the differentiable solve)
        dict(name="vi_grad_200k", kind="vi_grad", n=200_000, m=8, ns=16, ragged=False),
        # nova's own CPU benchmark instance, solved with nova's rounding
        dict(name="pbvi_solve_64", kind="pbvi_solve", mode=EXACT, n=64, m=4, z=8, ns=4, r=128,
             rz=8, horizon=100, ragged=False),
        # the large sparse-belief workload of bench.py: one backup of every belief
        dict(name="pbvi_run_20k", kind="pbvi_run", mode=FAST, n=20_000, m=16, z=32, ns=8, r=4096,
             rz=64, iterations=1, ragged=False),
        # a policy's objective and its gradient in R (recorded forward run, backward replay), in
        # the arithmetic whose choices are reproducible
        dict(name="pbvi_grad_5k", kind="pbvi_grad", n=5000, m=8, z=16, ns=8, r=1024, rz=32,
             horizon=30, ragged=False),
        # dense beliefs on the matrix cores: one backup
        dict(name="pbvi_dense_bf16", kind="pbvi_dense", mode=DENSE_BF16, n=20_000, m=8, z=16,
             ns=8, r=2048),
        # 16 uneven POMDPs solved together (bench.py's batch, its first replanning steps)
        dict(name="pbvi_batch_16", kind="pbvi_batch", count=16, nmin=500, nmax=8000, rmin=256,
             rmax=2048, horizon=4),
        # a policy server: the action of a few beliefs, exactly as nova computes it
        dict(name="policy_serve_4", kind="policy", precision=0, n=5000, r=1024, k=4),
        # a simulator's step: the values of many beliefs at single precision
        dict(name="policy_16k_fp32", kind="policy", precision=1, n=20_000, r=4096, k=16_384),
        # the same simulator's belief updates
        dict(name="update_16k", kind="update", n=20_000, m=16, z=32, ns=8, k=16_384,
             ragged=False),
    ]


def _logint(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["vi_solve", "vi_run", "vi_batch", "vi_grad", "pbvi_solve", "pbvi_run",
                       "pbvi_grad", "pbvi_dense", "pbvi_batch", "policy", "policy", "update"])
    c = dict(kind=kind)
    ragged = rng.random() < 0.4
    if kind == "vi_solve":
        # tens to tens of thousands of states
        c.update(n=_logint(rng, 30, 30_000), m=rng.randint(2, 16), ns=rng.randint(2, 16),
                 horizon=rng.randint(10, 100), ragged=ragged)
    elif kind == "vi_run":
        # from cache-resident models to the largest
        c.update(n=_logint(rng, 2000, 1_000_000), m=rng.randint(2, 8), ns=rng.randint(3, 16),
                 sweeps=rng.randint(10, 200), ragged=ragged)
    elif kind == "vi_batch":
        c.update(count=rng.randint(3, 64), nmin=rng.randint(50, 500), nmax=rng.randint(600, 8000),
                 horizon=rng.randint(10, 50))
    elif kind == "vi_grad":
        c.update(n=_logint(rng, 500, 200_000), m=rng.randint(2, 8), ns=rng.randint(3, 16),
                 ragged=ragged)
    elif kind == "pbvi_solve":
        # nova's small domains: few states, supports from a handful of states to nearly all
        n = _logint(rng, 8, 300)
        c.update(mode=EXACT, n=n, m=rng.randint(2, 8), z=rng.randint(2, 17),
                 ns=rng.randint(2, min(8, n)), r=_logint(rng, 15, 200),
                 rz=rng.randint(2, min(n, 30)), horizon=rng.randint(10, 50), ragged=ragged)
    elif kind == "pbvi_run":
        if rng.random() < 0.6:
            c.update(mode=FAST, n=_logint(rng, 500, 20_000), m=rng.randint(2, 16),
                     z=rng.randint(2, 32), ns=rng.randint(2, 8), r=_logint(rng, 100, 4096),
                     rz=rng.randint(4, 64), iterations=1, ragged=ragged)
        else:
            c.update(mode=EXACT, n=_logint(rng, 500, 5000), m=rng.randint(2, 8),
                     z=rng.randint(2, 16), ns=rng.randint(2, 8), r=_logint(rng, 100, 1024),
                     rz=rng.randint(4, 32), iterations=rng.randint(1, 5), ragged=ragged)
    elif kind == "pbvi_grad":
        c.update(n=_logint(rng, 300, 5000), m=rng.randint(2, 8), z=rng.randint(2, 16),
                 ns=rng.randint(2, 8), r=_logint(rng, 60, 1024), rz=rng.randint(4, 32),
                 horizon=rng.randint(3, 30), ragged=ragged)
    elif kind == "pbvi_dense":
        mode = rng.choice([DENSE_BF16, DENSE_FP32])
        c.update(mode=mode, n=_logint(rng, 300, 20_000 if mode == DENSE_BF16 else 8000),
                 m=rng.randint(2, 8), z=rng.randint(2, 16), ns=rng.randint(2, 8),
                 r=_logint(rng, 100, 2048 if mode == DENSE_BF16 else 1024))
    elif kind == "pbvi_batch":
        c.update(count=rng.randint(2, 16), nmin=rng.randint(100, 500),
                 nmax=rng.randint(600, 8000), rmin=rng.randint(50, 250),
                 rmax=rng.randint(300, 2048), horizon=rng.randint(1, 4))
    elif kind == "policy":
        # one belief of a server to a simulator's thousands
        precision = rng.choice([0, 0, 1, 2])
        n, r = _logint(rng, 50, 20_000), _logint(rng, 20, 4096)
        k = _logint(rng, 1, 16_384)
        if precision == 0:      # exact: a smaller call, as its arithmetic costs more
            k = min(k, max(1, int(1.0e11 / (n * r))))
        c.update(precision=precision, n=n, r=r, k=k)
    else:
        c.update(n=_logint(rng, 100, 20_000), m=rng.randint(2, 16), z=rng.randint(2, 32),
                 ns=rng.randint(2, 8), k=_logint(rng, 1, 16_384), ragged=ragged)
    return c


# ---- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _dirichlet(shape, g):
    """Rows of Dirichlet(1) weights: normalised Exp(1), float32."""
    x = torch.empty(shape, dtype=torch.float32, device="cuda").exponential_(generator=g)
    return x / x.sum(dim=-1, keepdim=True, dtype=torch.float64).to(torch.float32)


def _transitions(n, m, ns, ragged, g):
    """S (int32) and T (float32) on the GPU, n x m x ns; ragged: lists of 1 to ns successors,
    ended by -1, their probabilities still summing to 1."""
    S = torch.randint(0, n, (n, m, ns), generator=g, device="cuda", dtype=torch.int32)
    if not ragged:
        return S, _dirichlet((n, m, ns), g)
    length = torch.randint(1, ns + 1, (n, m, 1), generator=g, device="cuda")
    past = torch.arange(ns, device="cuda").view(1, 1, ns) >= length
    T = torch.empty((n, m, ns), device="cuda").exponential_(generator=g).masked_fill_(past, 0.0)
    T /= T.sum(dim=2, keepdim=True)
    return S.masked_fill_(past, -1), T


def _rewards(n, m, g):
    return torch.rand((n, m), generator=g, device="cuda") * 2 - 1


def _supports(n, r, rz, g):
    """r supports of rz distinct states, ascending: one state from each of rz equal ranges."""
    lo = torch.arange(rz, device="cuda", dtype=torch.int64) * n // rz
    hi = torch.arange(1, rz + 1, device="cuda", dtype=torch.int64) * n // rz
    u = torch.rand((r, rz), generator=g, device="cuda", dtype=torch.float64)
    return (lo + (u * (hi - lo)).long()).to(torch.int32)


def _pomdp_arrays(c, seed, dense=False):
    """The model as numpy arrays, as POMDP.from_arrays takes them, with GammaInitial."""
    g = _gen(seed)
    S, T = _transitions(c["n"], c["m"], c["ns"], c.get("ragged", False), g)
    O = _dirichlet((c["m"], c["n"], c["z"]), g)
    R = _rewards(c["n"], c["m"], g)
    r, n = c["r"], c["n"]
    if dense:
        Z = torch.arange(n, dtype=torch.int32).repeat(r, 1)
        B = _dirichlet((r, n), g)
    else:
        Z = _supports(n, r, c["rz"], g)
        B = _dirichlet((r, c["rz"]), g)
    gamma = np.float32(0.95)
    R = R.cpu().numpy()
    g0 = np.float32(R.min() / (1.0 - float(gamma)))
    return dict(S=S.cpu().numpy(), T=T.cpu().numpy(), O=O.cpu().numpy(), R=R, Z=Z.cpu().numpy(),
                B=B.cpu().numpy(), gamma=gamma, horizon=c.get("horizon", 1),
                Gamma0=np.full((r, n), g0, np.float32))


def _gamma0(c, seed):
    """Alphas of a running solver: around Rmin / (1 - gamma), each with its own spread."""
    x = torch.rand((c["r"], c["n"]), generator=_gen(seed), device="cuda")
    return x.mul_(2.0).sub_(21.0)


def _shape_seed(c):
    return zlib.crc32(repr(sorted((k, v) for k, v in c.items() if k != "name")).encode()) >> 1


_kept = {}


def _keep(c, make):
    """The model and solver that a program keeps between its calls: one case's at a time."""
    key = repr(sorted((k, v) for k, v in c.items() if k != "name"))
    if key not in _kept:
        _kept.clear()
        _kept[key] = make()
    return _kept[key]


class _DeviceArray:
    """A float array of the library's, for torch to look at where it lies."""

    def __init__(self, pointer, shape, typestr):
        address = ct.cast(pointer, ct.c_void_p).value
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, version=2,
                                             data=(address, False))


def _device_view(pointer, shape, typestr="<f4"):
    return torch.as_tensor(_DeviceArray(pointer, shape, typestr), device="cuda")


def _with_mode(mode, call):
    old = pomdp_pbvi.set_mode(mode)
    try:
        return call()
    finally:
        pomdp_pbvi.set_mode(old)


def _mdp(c, seed):
    g = _gen(seed)
    S, T = _transitions(c["n"], c["m"], c["ns"], c["ragged"], g)
    R = _rewards(c["n"], c["m"], g)
    return S, T, R


def _mdp_on_device(c, seed, horizon):
    S, T, R = (x.cpu().numpy() for x in _mdp(c, seed))
    mdp = MDP.from_arrays(S, T, R, gamma=0.99, horizon=horizon)
    mdp.initialize_gpu()
    return mdp


def _batch_sizes(c):
    """The sizes of a batch's instances, drawn as synth.py draws them but from the case alone."""
    g = np.random.Generator(np.random.PCG64(_shape_seed(c)))

    def log(lo, hi):
        return int(round(math.exp(g.uniform(math.log(lo), math.log(hi)))))

    sizes = []
    for _ in range(c["count"]):
        x = dict(n=log(c["nmin"], c["nmax"]), m=int(g.integers(4, 17)), ns=int(g.choice([4, 8])))
        if "rmin" in c:
            x.update(r=log(c["rmin"], c["rmax"]), z=int(g.integers(4, 33)), rz=16)
        sizes.append(x)
    return sizes


def _batch_pomdps(c, seed):
    return [synth.pomdp_arrays(gamma=0.95, horizon=c["horizon"], seed=int(seed) * 1024 + k, **x)
            for k, x in enumerate(_batch_sizes(c))]


def _batch_mdps(c, seed):
    return [synth.mdp_arrays(gamma=0.95, horizon=c["horizon"], seed=int(seed) * 1024 + k, **x)
            for k, x in enumerate(_batch_sizes(c))]


def _policy_inputs(c, seed):
    g = _gen(seed)
    G = torch.rand((c["r"], c["n"]), generator=g, device="cuda").mul_(6.0).sub_(3.0)
    pi = torch.randint(0, 16, (c["r"],), generator=g, device="cuda", dtype=torch.int32)
    return G, pi, _dirichlet((c["k"], c["n"]), g)


def _update_inputs(c, seed):
    g = _gen(seed)
    B = _dirichlet((c["k"], c["n"]), g)
    a = torch.randint(0, c["m"], (c["k"],), generator=g, device="cuda", dtype=torch.int32)
    o = torch.randint(0, c["z"], (c["k"],), generator=g, device="cuda", dtype=torch.int32)
    return B, a.cpu().numpy(), o.cpu().numpy()


def prepare(case, seed):
    c, kind = case, case["kind"]
    s = dict(case=case)
    if kind == "vi_solve":
        s["mdp"] = _mdp_on_device(c, seed, c["horizon"])
        s["V0"] = np.zeros(c["n"], np.float32)
    elif kind == "vi_run":
        def make():
            mdp = _mdp_on_device(c, _shape_seed(c), c["sweeps"])
            return mdp, mdp_vi.MDPValueIterationGPU(mdp, Vinitial=np.zeros(c["n"], np.float32))
        s["mdp"], s["solver"] = _keep(c, make)
        s["V0"] = torch.rand(c["n"], generator=_gen(seed), device="cuda").mul_(40.0).sub_(20.0)
    elif kind == "vi_batch":
        s["mdps"] = []
        for w in _batch_mdps(c, seed):
            mdp = MDP.from_arrays(w["S"], w["T"], w["R"], gamma=w["gamma"], horizon=c["horizon"])
            mdp.initialize_gpu()
            s["mdps"].append(mdp)
        s["solvers"] = [mdp_vi.MDPValueIterationGPU(x, Vinitial=np.zeros(x.n, np.float32))
                        for x in s["mdps"]]
    elif kind == "vi_grad":
        S, T, R = _mdp(c, seed)
        s.update(S=S, T=T.requires_grad_(True), R=R.requires_grad_(True),
                 g=torch.full((c["n"],), 1.0 / c["n"], device="cuda"))
    elif kind == "pbvi_solve":
        s["P"] = _pomdp_arrays(c, seed)
        s["pomdp"] = POMDP.from_dict(s["P"])
        s["pomdp"].initialize_gpu()
    elif kind in ("pbvi_run", "pbvi_dense"):
        def make():
            P = _pomdp_arrays(c, _shape_seed(c), dense=kind == "pbvi_dense")
            p = POMDP.from_dict(P)
            p.initialize_gpu()
            return p, _with_mode(c["mode"], lambda: pomdp_pbvi.POMDPPBVIGPU(
                p, GammaInitial=P["Gamma0"]))
        s["pomdp"], s["solver"] = _keep(c, make)
        s["Gamma0"] = _gamma0(c, seed)
    elif kind == "pbvi_grad":
        s["P"] = _pomdp_arrays(c, _shape_seed(c))
        s["R"] = _rewards(c["n"], c["m"], _gen(seed)).requires_grad_(True)
    elif kind == "pbvi_batch":
        batch = _batch_pomdps(c, seed)
        s["pomdps"] = [POMDP.from_dict(P) for P in batch]
        for p in s["pomdps"]:
            p.initialize_gpu()
        s["solvers"] = _with_mode(FAST, lambda: [
            pomdp_pbvi.POMDPPBVIGPU(p, GammaInitial=P["Gamma0"])
            for p, P in zip(s["pomdps"], batch)])
    elif kind == "policy":
        s["Gamma"], s["pi"], s["B"] = _policy_inputs(c, seed)
        s["V"] = torch.empty(c["k"], dtype=torch.float32, device="cuda")
        s["action"] = torch.empty(c["k"], dtype=torch.int32, device="cuda")
        s["alpha"] = torch.empty(c["k"], dtype=torch.int32, device="cuda")
        s["lib"] = _abi.load()
        torch.cuda.synchronize()
    else:
        def make():
            p = POMDP.from_dict(_pomdp_arrays(dict(c, r=1, rz=1), _shape_seed(c)))
            p.initialize_gpu()
            return p
        s["pomdp"] = _keep(c, make)
        s["B"], s["a"], s["o"] = _update_inputs(c, seed)
    return s


# ---- one pass

def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "vi_solve":
        policy = mdp_vi.MDPValueIterationGPU(s["mdp"], Vinitial=s["V0"]).solve()
        return dict(V=policy.V_array(), pi=policy.pi_array())
    if kind == "vi_run":
        s["solver"].run(c["sweeps"], d_V0=s["V0"].data_ptr())
        V, pi = s["solver"].device_values()
        return dict(V=V, pi=pi)
    if kind == "vi_batch":
        res, _ = mdp_vi.batch_execute(s["solvers"])
        return dict(V=np.concatenate([v for v, _ in res]),
                    pi=np.concatenate([p for _, p in res]))
    if kind == "vi_grad":
        V = BellmanFixedPoint.apply(s["R"], s["T"], s["S"], 0.99)
        dR, dT = torch.autograd.grad(V, (s["R"], s["T"]), s["g"])
        return dict(V=V.detach(), dR=dR, dT=dT)
    if kind == "pbvi_solve":
        policy = _with_mode(c["mode"], lambda: pomdp_pbvi.POMDPPBVIGPU(
            s["pomdp"], GammaInitial=s["P"]["Gamma0"]).solve())
        return dict(Gamma=policy.Gamma_array(), pi=policy.pi_array())
    if kind in ("pbvi_run", "pbvi_dense"):
        # a backup of given alphas by a kept solver: they go where its next update reads
        x = s["solver"]
        shape = (c["r"], c["n"])
        x.currentHorizon = 0
        _device_view(x.d_Gamma, shape).copy_(s["Gamma0"])
        iterations = c.get("iterations", 1)
        x.run(iterations)
        G = x.d_Gamma if iterations % 2 == 0 else x.d_GammaPrime
        return dict(Gamma=_device_view(G, shape), pi=_device_view(x.d_pi, (c["r"],), "<i4"))
    if kind == "pbvi_grad":
        def both():
            L = PBVIBeliefValue.apply(s["R"], s["P"])
            return L, torch.autograd.grad(L, s["R"])[0]
        L, dR = _with_mode(EXACT, both)
        return dict(L=L.detach(), dR=dR)
    if kind == "pbvi_batch":
        res, _ = _with_mode(FAST, lambda: pomdp_pbvi.batch_execute(s["solvers"]))
        return dict(Gamma=np.concatenate([g.ravel() for g, _ in res]),
                    pi=np.concatenate([p for _, p in res]))
    if kind == "policy":
        rc = s["lib"].nova_amd_alpha_vectors_value_and_action_gpu(
            c["n"], c["r"], s["Gamma"].data_ptr(), s["pi"].data_ptr(), c["k"],
            s["B"].data_ptr(), c["precision"], s["V"].data_ptr(), s["action"].data_ptr(),
            s["alpha"].data_ptr())
        if rc != 0:
            raise RuntimeError("value and action failed with code %d" % rc)
        return dict(V=s["V"], action=s["action"], alpha=s["alpha"])
    Bp, status = s["pomdp"].belief_update_batch(s["B"], s["a"], s["o"])
    return dict(Bp=Bp, status=status)


# ---- what a pass cannot do without

def _pbvi_work(n, m, z, ns, r, rz, iterations):
    """The cheaper of scoring every (successor of a support state, observation) pair against
    every alpha, and of projecting every alpha first and scoring the supports; then the winners."""
    direct = 2.0 * r * m * z * r * rz * ns
    projected = 2.0 * r * m * z * (n * ns + r * rz)
    flops = iterations * (min(direct, projected) + 2.0 * r * z * n)
    model = 8.0 * n * m * ns + 4.0 * m * n * z + 4.0 * n * m + 8.0 * r * rz
    return dict(bytes=model + 8.0 * r * n + 4.0 * r, flops=flops)


def work(case):
    c, kind = case, case["kind"]
    if kind in ("vi_solve", "vi_run"):
        sweeps = c.get("horizon", c.get("sweeps"))
        n, m, ns = c["n"], c["m"], c["ns"]
        # a model past the caches is read by every sweep; a smaller one once
        per = 8.0 * n * m * ns + 4.0 * n * m
        times = sweeps if per > 256e6 else 1
        return dict(bytes=times * (per + 12.0 * n), flops=2.0 * sweeps * n * m * ns)
    if kind == "vi_batch":
        sizes = _batch_sizes(c)
        rows = sum(x["n"] * x["m"] for x in sizes)
        entries = sum(x["n"] * x["m"] * x["ns"] for x in sizes)
        return dict(bytes=8.0 * entries + 4.0 * rows + 12.0 * sum(x["n"] for x in sizes),
                    flops=2.0 * c["horizon"] * entries)
    if kind == "vi_grad":
        n, m, ns = c["n"], c["m"], c["ns"]
        sweeps = 16     # as many as the solve needs at gamma = 0.99 and a residual of 1e-6
        return dict(bytes=sweeps * (8.0 * n * m * ns + 4.0 * n * m) + 4.0 * n * m * (ns + 1)
                    + 12.0 * n * ns, flops=2.0 * sweeps * n * m * ns + 2.0 * sweeps * n * ns)
    if kind in ("pbvi_solve", "pbvi_run"):
        return _pbvi_work(c["n"], c["m"], c["z"], c["ns"], c["r"], c["rz"],
                          c.get("iterations", c.get("horizon")))
    if kind == "pbvi_grad":
        w = _pbvi_work(c["n"], c["m"], c["z"], c["ns"], c["r"], c["rz"], c["horizon"])
        w["flops"] += c["horizon"] * 2.0 * c["r"] * c["n"] * (c["ns"] + c["z"] + 1)
        return w
    if kind == "pbvi_dense":
        n, m, z, r = c["n"], c["m"], c["z"], c["r"]
        return dict(bytes=4.0 * (3 * r * n + m * n * z), flops=2.0 * m * z * r * r * n)
    if kind == "pbvi_batch":
        each = [_pbvi_work(x["n"], x["m"], x["z"], x["ns"], x["r"], x["rz"], c["horizon"])
                for x in _batch_sizes(c)]
        return dict(bytes=sum(w["bytes"] for w in each), flops=sum(w["flops"] for w in each))
    n, k = c["n"], c["k"]
    if kind == "policy":
        return dict(bytes=4.0 * (n * c["r"] + n * k + c["r"] + 3 * k), flops=2.0 * n * c["r"] * k)
    # the predecessor lists once per action, O once per (action, observation) met, b and b'
    lists = 8.0 * n * c["ns"] * min(c["m"], k) + 4.0 * n * min(c["m"] * c["z"], k)
    return dict(bytes=lists + 8.0 * n * k, flops=(2.0 * c["ns"] + 3.0) * n * k)


def tolerance(case):
    kind = case["kind"]
    if kind in ("vi_solve", "vi_run", "vi_batch", "update"):
        return "exact"          # nova's order of operations, bit for bit
    if kind == "pbvi_solve" or (kind == "pbvi_run" and case["mode"] == EXACT):
        return "exact"
    if kind == "policy":
        if case["precision"] == 0:
            return "exact"
        # sums of n products: 2e-6 from 64 bits at single precision, 8e-4 from operands rounded
        # to bf16; near-ties may choose another alpha
        return {"rel": 8e-6, "differ": 2e-2} if case["precision"] == 1 else \
            {"rel": 2e-3, "differ": 5e-2}
    if kind == "vi_grad":
        # the solve stops at a residual of 1e-6; a near-tied action moves the gradient
        return {"rel": 1e-3}
    if kind == "pbvi_grad":
        return {"rel": 1e-5}    # single-precision sums over recorded choices
    if kind == "pbvi_dense":
        # near-ties decided by the operands' rounding (bf16: the alphas are 9e-3 from those of
        # 64 bits) or the sums' (single precision)
        return {"rel": 2e-2, "differ": 0.1} if case["mode"] == DENSE_BF16 else \
            {"rel": 1e-3, "differ": 2e-2}
    # single-precision scores: near-ties may choose another alpha, whose row then differs
    return {"rel": 1e-3, "differ": 1e-2}


# ---- the same in 64 bits

def _sweep64(S, T, R, gamma, V):
    """One Bellman sweep; S with -1 entries (whose T is 0)."""
    n, m, ns = S.shape
    Q = R.double()
    step = max(1, 20_000_000 // (n * m))
    for i in range(0, ns, step):
        idx = S[:, :, i:i + step].clamp(min=0).long()
        t = T[:, :, i:i + step].double() * (S[:, :, i:i + step] >= 0)
        Q = Q + gamma * (t * V[idx]).sum(dim=2)
    return Q.max(dim=1)


def _vi64(S, T, R, gamma, V, sweeps):
    gamma = float(np.float32(gamma))
    for _ in range(sweeps):
        V, _ = _sweep64(S, T, R, gamma, V)
    return V


def _fixed_point64(S, T, R, gamma):
    """V*, its greedy policy and the policy's rows (successors, probabilities)."""
    gamma = float(np.float32(gamma))
    n = S.shape[0]
    V = torch.zeros(n, dtype=torch.float64, device="cuda")
    rows = torch.arange(n, device="cuda")
    for _ in range(40):
        V, pi = _sweep64(S, T, R, gamma, V)
        Sp = S[rows, pi].clamp(min=0).long()
        Tp = T[rows, pi].double() * (S[rows, pi] >= 0)
        Rp = R[rows, pi].double()
        for _ in range(100):
            V = Rp + gamma * (Tp * V[Sp]).sum(dim=1)
    return V, pi, Sp, Tp


def _pbvi64(P, G, iterations, dense):
    """PBVI backups in 64 bits by projecting the alphas: (Gamma, pi)."""
    S, T, O, R, B = (torch.as_tensor(P[k], device="cuda") for k in "STORB")
    n, m, ns = S.shape
    z, (r, rz) = O.shape[2], P["Z"].shape
    gamma = float(np.float32(P["gamma"]))
    Z = torch.as_tensor(P["Z"], device="cuda").long()
    if dense:
        W = B.double()
    else:
        W = torch.sparse_coo_tensor(
            torch.stack([torch.arange(r, device="cuda").repeat_interleave(rz), Z.reshape(-1)]),
            B.double().reshape(-1), (r, n)).to_sparse_csr()
    G = torch.as_tensor(G, device="cuda").double()
    rows = torch.arange(r, device="cuda")
    for _ in range(iterations):
        best = torch.full((r,), -math.inf, dtype=torch.float64, device="cuda")
        act = torch.zeros(r, dtype=torch.int64, device="cuda")
        chosen = torch.zeros((r, z), dtype=torch.int64, device="cuda")
        for a in range(m):
            t = T[:, a].double() * (S[:, a] >= 0)
            sp = S[:, a].clamp(min=0).long()
            # b T_a, r x n: the mass that each belief moves to each successor state
            M = torch.zeros((r, n), dtype=torch.float64, device="cuda")
            Wd = W if dense else W.to_dense()
            for i in range(ns):
                M.index_add_(1, sp[:, i], Wd * t[:, i])
            val = Wd @ R[:, a].double()
            js = torch.empty((r, z), dtype=torch.int64, device="cuda")
            for o in range(z):
                sc, j = ((M * O[a, :, o].double()) @ G.T).max(dim=1)
                val = val + gamma * sc
                js[:, o] = j
            better = val > best
            best = torch.where(better, val, best)
            act = torch.where(better, torch.full_like(act, a), act)
            chosen[better] = js[better]
        out = torch.empty((r, n), dtype=torch.float64, device="cuda")
        for a in range(m):
            mine = rows[act == a]
            for lo in range(0, mine.numel(), 256):
                i = mine[lo:lo + 256]
                h = torch.zeros((i.numel(), n), dtype=torch.float64, device="cuda")
                for o in range(z):
                    h += O[a, :, o].double() * G[chosen[i, o]]
                acc = R[:, a].double().expand(i.numel(), n).clone()
                for q in range(ns):
                    t = T[:, a, q].double() * (S[:, a, q] >= 0)
                    acc += gamma * t * h[:, S[:, a, q].clamp(min=0).long()]
                out[i] = acc
        G = out
    return G, act


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "vi_solve":
        V = torch.zeros(c["n"], dtype=torch.float64, device="cuda")
        return dict(V=_vi64(*_mdp(c, seed), 0.99, V, c["horizon"]), pi=None)
    if kind == "vi_run":
        V0 = torch.rand(c["n"], generator=_gen(seed), device="cuda").mul_(40.0).sub_(20.0)
        return dict(V=_vi64(*_mdp(c, _shape_seed(c)), 0.99, V0.double(), c["sweeps"]), pi=None)
    if kind == "vi_batch":
        out = []
        for w in _batch_mdps(c, seed):
            S, T, R = (torch.as_tensor(w[k], device="cuda") for k in "STR")
            V = torch.zeros(S.shape[0], dtype=torch.float64, device="cuda")
            out.append(_vi64(S, T, R, w["gamma"], V, c["horizon"]))
        return dict(V=torch.cat(out), pi=None)
    if kind == "vi_grad":
        S, T, R = _mdp(c, seed)
        n = c["n"]
        gamma = float(np.float32(0.99))
        V, pi, Sp, Tp = _fixed_point64(S, T, R, 0.99)
        rho = torch.full((n,), 1.0 / n, device="cuda").double()
        lam = rho.clone()
        for _ in range(3000):
            lam = rho + gamma * torch.zeros_like(lam).index_add_(
                0, Sp.reshape(-1), (Tp * lam[:, None]).reshape(-1))
        rows = torch.arange(n, device="cuda")
        dR = torch.zeros((n, c["m"]), dtype=torch.float64, device="cuda")
        dR[rows, pi] = lam
        dT = torch.zeros((n, c["m"], c["ns"]), dtype=torch.float64, device="cuda")
        dT[rows, pi] = gamma * lam[:, None] * V[Sp] * (S[rows, pi] >= 0)
        return dict(V=V, dR=dR, dT=dT)
    if kind == "policy":
        G, _, B = _policy_inputs(c, seed)
        Gt = G.double().T.contiguous()
        V = torch.cat([(b.double() @ Gt).max(dim=1).values for b in B.split(2048)])
        return dict(V=V, action=None, alpha=None)
    if kind == "update":
        B, a, o = _update_inputs(c, seed)
        P = _pomdp_arrays(dict(c, r=1, rz=1), _shape_seed(c))
        S, T, O = (torch.as_tensor(P[k], device="cuda") for k in "STO")
        out = torch.zeros((c["k"], c["n"]), dtype=torch.float64, device="cuda")
        act = torch.as_tensor(a, device="cuda").long()
        obs = torch.as_tensor(o, device="cuda").long()
        for x in range(c["m"]):
            for q in (act == x).nonzero().reshape(-1).split(512):
                bp = torch.zeros((q.numel(), c["n"]), dtype=torch.float64, device="cuda")
                for i in range(c["ns"]):
                    t = T[:, x, i].double() * (S[:, x, i] >= 0)
                    bp.index_add_(1, S[:, x, i].clamp(min=0).long(), B[q].double() * t)
                bp *= O[x].double().T[obs[q]]
                out[q] = bp / bp.sum(dim=1, keepdim=True)
        return dict(Bp=out, status=None)
    if kind == "pbvi_run" and c["mode"] == FAST or kind == "pbvi_dense":
        if 2.0 * c["m"] * c["z"] * c["r"] ** 2 * c["n"] > 4e14:
            return None         # minutes in 64 bits
        dense = kind == "pbvi_dense"
        P = _pomdp_arrays(c, _shape_seed(c), dense=dense)
        G, _ = _pbvi64(P, _gamma0(c, seed), 1, dense)
        return dict(Gamma=G, pi=None)
    # many backups in a row: which of two near-tied alphas is taken early steers the later ones
    return None
