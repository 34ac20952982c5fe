"""Gradient of the PBVI objective L = sum_b max_alpha alpha . b with respect to R by argmax
replay: against FP64 central finite differences of the oracle's FP64 PBVI (free argmaxes) on a
small instance, and at n = 5000, m = 8, z = 16, ns = 8, r = 1024, rz = 32, 30 iterations against
an FP64 replay of the same recorded choices computed here with numpy/scipy."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

from nova_amd import synth
from nova_amd.autograd import PBVIBeliefValue, pbvi_objective, pbvi_replay_grad

pytestmark = pytest.mark.gpu


def oracle_L(oracle, P, R, H):
    Q = dict(P)
    Q["R"] = R
    G, _ = oracle.pbvi_run(Q, horizon=H, dtype=np.float64)
    Z, B = P["Z"], P["B"]
    L = 0.0
    for i in range(Z.shape[0]):
        k = Z[i] >= 0
        L += np.max(G[:, Z[i][k]] @ B[i][k].astype(np.float64))
    return L


def test_replay_vs_finite_differences(oracle):
    P = synth.pomdp_arrays(n=30, m=3, z=4, ns=4, r=20, rz=5, seed=61, gamma=0.9, horizon=8)
    R = torch.from_numpy(P["R"]).cuda().requires_grad_(True)
    L = PBVIBeliefValue.apply(R, P)
    L.backward()
    g = R.grad.cpu().numpy()
    L64 = oracle_L(oracle, P, P["R"], 8)
    assert abs(float(L.detach()) - L64) <= 1e-4 * max(1.0, abs(L64))
    rng = np.random.default_rng(0)
    h = 1e-3
    errs = []
    for c in range(64):
        s, a = int(rng.integers(30)), int(rng.integers(3))
        Rp, Rm = P["R"].astype(np.float64).copy(), P["R"].astype(np.float64).copy()
        Rp[s, a] += h
        Rm[s, a] -= h
        # the FP64 oracle runs on float32 model arrays: perturb in float32 and use the
        # actual step
        Rp32, Rm32 = Rp.astype(np.float32), Rm.astype(np.float32)
        step = float(Rp32[s, a]) - float(Rm32[s, a])
        fd = (oracle_L(oracle, P, Rp32, 8) - oracle_L(oracle, P, Rm32, 8)) / step
        errs.append(abs(fd - g[s, a]) / max(1e-6, abs(fd), abs(g[s, a])))
    print("PBVI replay vs FD: max relative error %.3g" % max(errs))
    assert np.median(errs) < 1e-3
    assert np.mean(np.array(errs) < 1e-3) >= 0.95   # kinks (argmax changes) may cross a few


def numpy_replay(P, recJ, recA, arg):
    """FP64 replay of recorded choices (the same mathematics as the device kernels)."""
    S, T, O, Z, B = P["S"], P["T"], P["O"], P["Z"], P["B"]
    n, m, ns = S.shape
    z = O.shape[2]
    r, rz = Z.shape
    H = recA.shape[0]
    g = float(P["gamma"])
    Pa = []
    for a in range(m):
        rows = np.repeat(np.arange(n), ns)
        cols = S[:, a, :].ravel()
        vals = T[:, a, :].ravel().astype(np.float64)
        ok = cols >= 0
        Pa.append(sp.csr_matrix((vals[ok], (rows[ok], cols[ok])), shape=(n, n)))
    mu = np.zeros((r, n))
    for i in range(r):
        k = Z[i] >= 0
        np.add.at(mu[arg[i]], Z[i][k], B[i][k].astype(np.float64))
    dR = np.zeros((n, m))
    for t in range(H - 1, -1, -1):
        A, J = recA[t], recJ[t]
        u = np.zeros((r, n))
        for a in range(m):
            idx = np.nonzero(A == a)[0]
            if idx.size:
                dR[:, a] += mu[idx].sum(axis=0)
                u[idx] = (Pa[a].T @ mu[idx].T).T
        new = np.zeros((r, n))
        live = np.nonzero(A >= 0)[0]
        for o in range(z):
            vals = g * O[A[live], :, o].astype(np.float64) * u[live]
            np.add.at(new, J[live, o], vals)
        kept = np.nonzero(A < 0)[0]
        new[kept] += mu[kept]
        mu = new
    return dR


def test_replay_full_size_vs_fp64_replay():
    P = synth.workload("pbvi_diff_n5000")
    res = pbvi_objective(P, P["R"])
    dR = pbvi_replay_grad(res).cpu().numpy()
    H, r, z = res["horizon"], P["Z"].shape[0], P["O"].shape[2]
    recJ = res["recJ"].cpu().numpy().reshape(H, r, z)
    recA = res["recA"].cpu().numpy().reshape(H, r)
    ref = numpy_replay(P, recJ, recA, res["arg"].cpu().numpy())
    err = np.max(np.abs(dR - ref)) / np.max(np.abs(ref))
    print("PBVI replay n=5000: max |dR - dR_fp64| / max|dR_fp64| = %.3g" % err)
    assert err <= 1e-4


@pytest.mark.parametrize("n,r,ns", [(36_864, 256, 2), (36_865, 256, 2),    # mu fits LDS, or not
                                    (36_864, 3, 2), (300, 255, 5), (300, 256, 5), (1, 256, 1)])
def test_replay_at_the_limits_of_the_predecessor_gather(n, r, ns):
    """mu in LDS (at least 256 alphas of at most 36,864 states) and mu gathered from L2, with one
    state that has a long predecessor list and rows that end early, against the FP64 replay."""
    P = synth.pomdp_arrays(n=n, m=3, z=2, ns=ns, r=r, rz=min(n, 4), seed=n + r, gamma=0.9,
                           horizon=3)
    P["S"] = P["S"].copy()
    P["S"][: n // 2, 0, 0] = 0
    P["S"][n // 2:, 1, -1] = -1
    res = pbvi_objective(P, P["R"])
    dR = pbvi_replay_grad(res).cpu().numpy()
    z = P["O"].shape[2]
    ref = numpy_replay(P, res["recJ"].cpu().numpy().reshape(3, r, z),
                       res["recA"].cpu().numpy().reshape(3, r), res["arg"].cpu().numpy())
    assert np.max(np.abs(dR - ref)) <= 1e-4 * np.max(np.abs(ref))


def test_replay_of_few_alphas_spreads_over_the_states():
    """A step of a replay of 8 alphas of 100,000 states (26 MB of lists and rows) takes well below
    half a millisecond; with one workgroup per alpha it takes more than one."""
    import time
    times = {}
    for horizon in (4, 44):
        P = synth.pomdp_arrays(n=100_000, m=4, z=4, ns=8, r=8, rz=8, seed=1, gamma=0.95,
                               horizon=horizon)
        res = pbvi_objective(P, P["R"])
        best = np.inf
        for _ in range(5):
            torch.cuda.synchronize()
            t = time.perf_counter()
            pbvi_replay_grad(res)
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t)
        times[horizon] = best
    step = (times[44] - times[4]) / 40
    print("replay step, r = 8, n = 100,000: %.0f us" % (step * 1e6))
    assert step <= 5e-4
