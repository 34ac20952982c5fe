"""Executing alpha-vector policies over many beliefs on the GPU, through the C ABI, against the
oracle: nova_amd_alpha_vectors_value_and_action_gpu (pomdp_alpha_vectors.cpp:52-79 per belief)
and nova_amd_belief_update_batch_gpu (pomdp_model_cpu.cpp:89-137 per triple).

exact value/action and the belief update: bit for bit against the oracle's float twin.
Calls of at most 1.25 Mi (belief, alpha) pairs (exact ones of short rows: 576 Ki; bf16: at most 64
beliefs) run on the vector ALUs, one wave per 16 alphas; the sizes below lie on both sides.
fp32: the chosen alpha is the FP64 maximiser except at near-ties (its FP64
      value within 1e-5 * max(1, |V|) of the maximum) and V within 1e-5 relative.
bf16: reported (alpha disagreement rate, value error against FP64); the value
      of the chosen alpha stays within 1e-2 * max |V| of the FP64 maximum.
"""
import ctypes as ct

import numpy as np
import pytest

from conftest import bits
from nova_amd import synth
from nova_amd.pomdp import POMDP
from nova_amd.pomdp_alpha_vectors import POMDPAlphaVectors

pytestmark = pytest.mark.gpu


def policy(G, pi):
    import ctypes as ct
    from nova_amd import _abi
    p = POMDPAlphaVectors()
    r, n = G.shape
    lib = _abi.load()
    assert lib.pomdp_alpha_vectors_initialize(ct.byref(p), n, int(pi.max()) + 1, r) == 0
    np.ctypeslib.as_array(p.Gamma, (r * n,))[:] = G.reshape(-1)
    np.ctypeslib.as_array(p.pi, (r,))[:] = pi
    return p


def instance(k, n, r, seed, m=5):
    rng = np.random.default_rng(seed)
    G = rng.uniform(-3, 3, (r, n)).astype(np.float32)
    pi = rng.integers(0, m, r).astype(np.uint32)
    B = rng.exponential(size=(k, n))
    B[rng.random((k, n)) < 0.5] = 0.0          # sparse-ish dense rows
    B = (B / np.maximum(B.sum(axis=1, keepdims=True), 1e-30)).astype(np.float32)
    return G, pi, B


SHAPES = [(1, 1, 1), (70, 33, 65), (300, 257, 130), (1000, 600, 500)]


@pytest.mark.parametrize("k,n,r", SHAPES)
def test_exact_bitwise_vs_oracle(oracle, k, n, r):
    G, pi, B = instance(k, n, r, seed=k + n + r)
    # duplicated alphas: the first of equal maxima must win
    if r > 3:
        G[r // 2] = G[1]
        G[r - 1] = G[1]
    p = policy(G, pi)
    V, act, j = p.value_and_action_batch(B, "exact", return_alpha=True)
    V, act, j = V.cpu().numpy(), act.cpu().numpy(), j.cpu().numpy()
    for i in range(k):
        vo, ao, jo = oracle.alpha_value(G, pi, B[i])
        assert bits(np.float32(vo)) == bits(V[i]) and ao == act[i] and jo == j[i], i
    print("exact value/action: k=%d n=%d r=%d bit-identical" % (k, n, r), flush=True)


@pytest.mark.parametrize("k,n,r,offset", [
    (1, 1, 1, 0), (4, 16, 16, 0), (5, 17, 17, 0), (3, 255, 15, 0), (9, 256, 33, 0),
    (2, 260, 64, 1), (7, 513, 100, 0), (1030, 36, 130, 0), (2049, 130, 66, 3), (600, 20, 2200, 0),
])
def test_exact_few_beliefs_bitwise(oracle, k, n, r, offset):
    """The one-wave tiles of calls with few (belief, alpha) pairs: one and two beliefs per lane,
    rows aligned to 16 bytes or not (n odd, or arrays offset by some floats), partial tiles."""
    import torch
    from nova_amd import _abi
    G, pi, B = instance(k, n, r, seed=7 * k + n + r)
    if r > 3:
        G[r - 1] = G[1]
    if n > 2:
        G[0, 1] = np.inf          # (an infinity times a zero belief entry is a NaN, never chosen)
    Gt = torch.zeros(r * n + offset, device="cuda")
    Bt = torch.zeros(k * n + offset, device="cuda")
    Gt[offset:] = torch.from_numpy(G).reshape(-1)
    Bt[offset:] = torch.from_numpy(B).reshape(-1)
    pt = torch.from_numpy(pi.astype(np.int32)).cuda()
    V = torch.empty(k, device="cuda")
    a = torch.empty(k, dtype=torch.int32, device="cuda")
    j = torch.empty(k, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    lib = _abi.load()
    for entry, extra in ((lib.nova_amd_alpha_vectors_value_and_action_gpu, [0]),
                         (lib.nova_amd_alpha_vectors_value_and_action_noalloc_gpu, [])):
        V.zero_()
        torch.cuda.synchronize()
        assert entry(n, r, Gt.data_ptr() + 4 * offset, pt.data_ptr(), k,
                     Bt.data_ptr() + 4 * offset, *extra, V.data_ptr(), a.data_ptr(),
                     j.data_ptr()) == 0
        Vh, ah, jh = V.cpu().numpy(), a.cpu().numpy(), j.cpu().numpy()
        for i in range(0, k, max(1, k // 60)):
            vo, ao, jo = oracle.alpha_value(G, pi, B[i])
            assert bits(np.float32(vo)) == bits(Vh[i]) and ao == ah[i] and jo == jh[i], i


@pytest.mark.parametrize("k,n,r,offset", [
    (1300, 97, 1100, 0), (1300, 257, 1100, 1), (2600, 32, 600, 0),     # above 1.25 Mi pairs
    (1024, 64, 641, 0), (1024, 65, 641, 0),      # short rows above 576 Ki pairs, and one state more
    (1023, 64, 641, 0), (41_000, 7, 16, 0), (41_000, 7, 17, 0),        # too few in one direction
    (8191, 20, 70, 0), (8192, 20, 70, 0), (8192, 65, 70, 0),           # either merge
])
def test_exact_square_tiles_and_few_beliefs_at_their_limits(oracle, k, n, r, offset):
    """Both sides of the rules between the 64 x 64 tiles and the one-wave tiles, with rows of one
    step of 32 states and of several, full and ragged, through both entries."""
    test_exact_few_beliefs_bitwise(oracle, k, n, r, offset)


def test_exact_calls_of_many_beliefs_and_few_alphas_keep_their_time():
    """1,000,000 (belief, alpha) pairs of 50 states cost no more than 1,320,000: the call must not
    spend its time in a wave per belief that merges two partials."""
    import time
    import torch
    from nova_amd import _abi

    def best_of(k, r, runs=60):
        g = torch.Generator(device="cuda")
        g.manual_seed(k)
        G = torch.rand((r, 50), generator=g, device="cuda")
        B = torch.rand((k, 50), generator=g, device="cuda")
        pi = torch.zeros(r, dtype=torch.int32, device="cuda")
        V = torch.empty(k, device="cuda")
        a = torch.empty(k, dtype=torch.int32, device="cuda")
        times = []
        for _ in range(runs):
            torch.cuda.synchronize()
            t = time.perf_counter()
            assert _abi.load().nova_amd_alpha_vectors_value_and_action_gpu(
                50, r, G.data_ptr(), pi.data_ptr(), k, B.data_ptr(), 0, V.data_ptr(),
                a.data_ptr(), None) == 0
            times.append(time.perf_counter() - t)
        return min(times)

    fewer, more = best_of(50_000, 20), best_of(40_000, 33)
    print("exact value/action: 1.00 M pairs %.1f us, 1.32 M %.1f us" % (fewer * 1e6, more * 1e6))
    assert fewer <= 1.35 * more


@pytest.mark.parametrize("extra", [4, 5])        # rows aligned to 16 bytes, or not
def test_few_beliefs_rows_past_4_gb(extra):
    """A belief and an alpha of more than 2^30 states: values at both ends of the rows, so that an
    offset that wraps at 4 GB reads others. The few terms are sums of small integers: exact."""
    import torch
    from nova_amd import _abi
    n = 2 ** 30 + extra
    B, G = torch.zeros(n, device="cuda"), torch.zeros(n, device="cuda")
    at = [0, 1, 2, 3, 4, 255, 256, 2 ** 30 - 1, 2 ** 30, 2 ** 30 + 1, n - 1]
    for x, s in enumerate(at):
        B[s] = x + 1
        G[s] = 2 * x + 1
    pi = torch.full((1,), 3, dtype=torch.int32, device="cuda")
    V = torch.zeros(1, device="cuda")
    a = torch.zeros(1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    assert _abi.load().nova_amd_alpha_vectors_value_and_action_gpu(
        n, 1, G.data_ptr(), pi.data_ptr(), 1, B.data_ptr(), 0, V.data_ptr(), a.data_ptr(),
        None) == 0
    assert float(V) == sum((x + 1) * (2 * x + 1) for x in range(len(at))) and int(a) == 3


def test_exact_no_alpha_above_sentinel():
    """Every value at or below -1e10: V = -1e10, action 0 and alpha -1 (the reference leaves
    Vb and a at their initial values). Exact and fp32 only: in bf16 the sentinel itself rounds
    to -9.9992e9, so alphas holding it count as ordinary values."""
    G = np.full((5, 4), -1e10, np.float32)
    pi = np.array([3, 1, 2, 4, 1], np.uint32)
    B = np.array([[1, 0, 0, 0], [0.25, 0.25, 0.25, 0.25]], np.float32)
    p = policy(G, pi)
    for prec in ("exact", "fp32"):
        V, act, j = p.value_and_action_batch(B, prec, return_alpha=True)
        assert np.all(V.cpu().numpy() == np.float32(-1e10)), prec
        assert np.all(act.cpu().numpy() == 0) and np.all(j.cpu().numpy() == -1), prec


# the last two on the matrix cores, the others below their 1.25 Mi pairs
@pytest.mark.parametrize("k,n,r", SHAPES[1:] + [(2100, 257, 700), (4096, 2000, 1024)])
def test_fp32_matrix_cores_vs_fp64(k, n, r):
    G, pi, B = instance(k, n, r, seed=3 * k + r)
    p = policy(G, pi)
    V, act, j = p.value_and_action_batch(B, "fp32", return_alpha=True)
    V, act, j = V.cpu().numpy(), act.cpu().numpy(), j.cpu().numpy()
    C = B.astype(np.float64) @ G.astype(np.float64).T
    best = C.max(axis=1)
    scale = np.maximum(1.0, np.abs(best))
    chosen = C[np.arange(k), j]
    assert np.all(best - chosen <= 1e-5 * scale)
    assert np.all(np.abs(V - best) <= 1e-5 * scale)
    assert np.array_equal(act, pi[j])
    differ = int((j != C.argmax(axis=1)).sum())
    print("fp32: k=%d n=%d r=%d, %d of %d alpha choices differ from FP64 (near-ties)"
          % (k, n, r, differ, k), flush=True)


@pytest.mark.parametrize("k,n,r", [(1000, 600, 500), (4096, 2000, 1024)])
def test_bf16_matrix_cores_reported(k, n, r):
    G, pi, B = instance(k, n, r, seed=5 * k + r)
    p = policy(G, pi)
    V, act, j = p.value_and_action_batch(B, "bf16", return_alpha=True)
    V, act, j = V.cpu().numpy(), act.cpu().numpy(), j.cpu().numpy()
    C = B.astype(np.float64) @ G.astype(np.float64).T
    best = C.max(axis=1)
    chosen = C[np.arange(k), j]
    vmax = np.max(np.abs(best))
    rate = float(np.mean(j != C.argmax(axis=1)))
    err = float(np.max(best - chosen)) / vmax
    print("bf16: k=%d n=%d r=%d, alpha disagreement %.3g, value loss of the chosen alpha "
          "%.3g of max|V|, |V - V_fp64| %.3g" % (k, n, r, rate, err,
                                                 np.max(np.abs(V - best)) / vmax), flush=True)
    assert err <= 1e-2 and np.array_equal(act, pi[j])


@pytest.mark.parametrize("k,n,r", [(1, 1, 1), (5, 17, 16), (9, 257, 33), (64, 130, 300),
                                   (300, 40, 4000)])
@pytest.mark.parametrize("prec", ["fp32", "bf16"])
def test_few_beliefs_fp32_and_bf16(k, n, r, prec):
    """Calls of few beliefs on the vector ALUs: V within the accumulation error of n fp32 sums
    (n * 2^-24 * max sum |b||alpha|) of the FP64 maximum over the operands as the mode rounds
    them, and the chosen alpha's value too."""
    G, pi, B = instance(k, n, r, seed=13 * k + n + r)
    p = policy(G, pi)
    V, act, j = p.value_and_action_batch(B, prec, return_alpha=True)
    V, act, j = V.cpu().numpy(), act.cpu().numpy(), j.cpu().numpy()
    if prec == "bf16":
        G, B = bf16_round(G), bf16_round(B)
    C = B.astype(np.float64) @ G.astype(np.float64).T
    bound = (n + 1) * 2.0 ** -24 * (np.abs(B).astype(np.float64) @ np.abs(G).T).max(axis=1) + 1e-30
    assert np.all(np.abs(V - C.max(axis=1)) <= bound)
    assert np.all(C.max(axis=1) - C[np.arange(k), j] <= 2 * bound)
    assert np.array_equal(act, pi[j])


@pytest.mark.parametrize("n,r", [(100, 600), (1000, 600), (4999, 1200), (20000, 600)])
def test_bf16_few_beliefs_are_as_precise_as_the_matrix_cores(n, r):
    """bf16 calls of at most 64 beliefs and calls of more: the rms error of the sums against FP64
    (over the rounded operands) is no larger on the vector ALUs."""
    import torch
    k = 256
    G, pi, B = instance(k, n, r, seed=n + r)
    p = policy(G, pi)
    best = (bf16_round(B).astype(np.float64) @ bf16_round(G).astype(np.float64).T).max(axis=1)
    gemm = p.value_and_action_batch(B, "bf16")[0].cpu().numpy()
    few = torch.cat([p.value_and_action_batch(B[q:q + 64], "bf16")[0]
                     for q in range(0, k, 64)]).cpu().numpy()
    rms = [float(np.sqrt(np.mean((x - best) ** 2) / np.mean(best ** 2))) for x in (few, gemm)]
    print("bf16 sums, n=%d: few %.3g, GEMM %.3g" % (n, *rms))
    assert rms[0] <= rms[1]


# more than 1.25 Mi (belief, alpha) pairs: the split GEMM
@pytest.mark.parametrize("k,n,r", [(1300, 1, 1100), (1025, 64, 1300), (5200, 130, 257),
                                   (700, 1000, 2000)])
def test_fp32_split_vs_fp64(k, n, r):
    """fp32 as three bf16 parts: V within n fp32 roundings of the FP64 maximum, over operands of
    mixed signs and magnitudes (2^-100 and 2^60 among them)."""
    rng = np.random.default_rng(k + n)
    G = rng.standard_normal((r, n)).astype(np.float32) * \
        np.float32(2.0) ** rng.integers(-12, 13, (r, n)).astype(np.float32)
    B = rng.standard_normal((k, n)).astype(np.float32)
    B[rng.random((k, n)) < 0.3] = 0.0
    G[0, 0], B[1, 0] = 2.0 ** -100, 2.0 ** 60
    pi = rng.integers(0, 5, r).astype(np.uint32)
    V, act, j = policy(G, pi).value_and_action_batch(B, "fp32", return_alpha=True)
    V, act, j = V.cpu().numpy(), act.cpu().numpy(), j.cpu().numpy()
    C = B.astype(np.float64) @ G.astype(np.float64).T
    bound = (n + 1) * 2.0 ** -24 * (np.abs(B).astype(np.float64) @ np.abs(G).T).max(axis=1)
    assert np.all(np.abs(V - C.max(axis=1)) <= bound)
    assert np.all(C.max(axis=1) - C[np.arange(k), j] <= 2 * bound)
    assert np.array_equal(act, pi[j])


@pytest.mark.parametrize("odd", [np.inf, -np.inf, np.nan, 3.4e38, 1e-36, 1e-40])
def test_fp32_operands_without_bf16_parts(odd):
    """One operand value that has no exact bf16 parts: the call is left to the fp32 matrix
    instructions, and gives what they give (an infinity wins, a NaN never does)."""
    k, n, r = 1400, 70, 1000
    G, pi, B = instance(k, n, r, seed=3)
    B[:, 5] = 0.0
    B[7, 5] = 0.5
    G[11, 5] = odd
    with np.errstate(invalid="ignore"):
        C = B.astype(np.float64) @ G.astype(np.float64).T
    C[np.isnan(C)] = -np.inf
    V, act, j = policy(G, pi).value_and_action_batch(B, "fp32", return_alpha=True)
    V, j = V.cpu().numpy().astype(np.float64), j.cpu().numpy()
    best = C.max(axis=1)
    fine = np.isfinite(best)
    assert np.allclose(V[fine], best[fine], rtol=1e-5, atol=1e-5)
    assert np.array_equal(V[~fine], best[~fine])
    assert np.all(j[~fine] == 11)


@pytest.mark.parametrize("k,n,r", [(1400, 513, 1000), (1024, 600, 1300), (700, 1000, 2000)])
def test_fp32_fallback_vs_fp64(k, n, r):
    """The fp32 matrix instructions, which take the calls whose operands have no bf16 parts, over rows
    of many steps, full and ragged: V within n fp32 roundings of the FP64 maximum."""
    G, pi, B = instance(k, n, r, seed=k + n)
    B[0, 0] = 1e-36
    V, act, j = policy(G, pi).value_and_action_batch(B, "fp32", return_alpha=True)
    V, act, j = V.cpu().numpy(), act.cpu().numpy(), j.cpu().numpy()
    C = B.astype(np.float64) @ G.astype(np.float64).T
    bound = (n + 1) * 2.0 ** -24 * (np.abs(B).astype(np.float64) @ np.abs(G).T).max(axis=1)
    assert np.all(np.abs(V - C.max(axis=1)) <= bound)
    assert np.all(C.max(axis=1) - C[np.arange(k), j] <= 2 * bound)
    assert np.array_equal(act, pi[j])


@pytest.mark.parametrize("x,y", [(1.998 * 2.0 ** 63, 1.9985 * 2.0 ** 63),    # just below the range
                                 (1.998 * 2.0 ** 120, 1.998 * 2.0 ** 40),    # infinite
                                 (2.0 ** 62, 1.75 * 2.0 ** 62)])             # one within the split's
def test_fp32_large_operands(x, y):
    """Operands whose bf16 parts are finite but whose parts' products are not: the value is the
    fp32 product's (finite where that is, +infinity otherwise)."""
    k, n, r = 1400, 70, 1000
    G, pi, B = instance(k, n, r, seed=4)
    B[:, 5] = 0.0
    G[:, 5] = 0.0
    B[7, 5], G[11, 5] = x, y
    V, act, j = policy(G, pi).value_and_action_batch(B, "fp32", return_alpha=True)
    V, j = V.cpu().numpy().astype(np.float64), j.cpu().numpy()
    with np.errstate(over="ignore"):
        want = float(np.float32(B[7, 5]) * np.float32(G[11, 5]))
    assert j[7] == 11 and act.cpu().numpy()[7] == pi[11]
    assert V[7] == want or abs(V[7] - want) <= 2.0 ** -23 * want
    rest = np.delete(np.arange(k), 7)
    C = B.astype(np.float64)[rest] @ G.astype(np.float64).T
    assert np.all(np.abs(V[rest] - C.max(axis=1)) <= 1e-5 * np.maximum(1.0, np.abs(C.max(axis=1))))


@pytest.mark.parametrize("nonzeros", [4, 16, 64])
def test_fp32_split_is_no_less_precise_on_sparse_beliefs(nonzeros):
    """Beliefs of a few nonzeros among 1,000 states: the split GEMM's rms error against FP64 is at
    most that of one FMA per product in order (the calls of few beliefs, whose sums are those of
    the fp32 matrix instruction bit for bit)."""
    import torch
    k, n, r = 4096, 1000, 512
    rng = np.random.default_rng(nonzeros)
    G = rng.uniform(-3, 3, (r, n)).astype(np.float32)
    pi = rng.integers(0, 5, r).astype(np.uint32)
    B = np.zeros((k, n))
    at = rng.random((k, n)).argsort(axis=1)[:, :nonzeros]
    np.put_along_axis(B, at, rng.exponential(size=(k, nonzeros)), axis=1)
    B = (B / B.sum(axis=1, keepdims=True)).astype(np.float32)
    best = (B.astype(np.float64) @ G.astype(np.float64).T).max(axis=1)
    p = policy(G, pi)
    V = p.value_and_action_batch(B, "fp32")[0].cpu().numpy()
    chain = torch.cat([p.value_and_action_batch(B[q:q + 2048], "fp32")[0]
                       for q in range(0, k, 2048)]).cpu().numpy()       # 1 Mi pairs each
    rms = [float(np.sqrt(np.mean(((x - best) / best) ** 2))) for x in (V, chain)]
    print("sparse beliefs, %d nonzeros: split %.3g, one FMA per product %.3g" % (nonzeros, *rms))
    assert rms[0] <= rms[1]


def test_fp32_call_with_a_tiny_entry_skips_the_split_gemm():
    """A belief entry below 2^-100 leaves the call to the fp32 instructions, without the split
    GEMM's work first: the fp32 GEMM takes about 1.7 times the split one, both together 2.7."""
    import time
    import torch
    from nova_amd import _abi
    k, n, r = 8192, 4096, 4096
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    G = torch.rand((r, n), generator=g, device="cuda").mul_(6).sub_(3)
    B = torch.rand((k, n), generator=g, device="cuda").add_(0.1)
    pi = torch.zeros(r, dtype=torch.int32, device="cuda")
    V = torch.empty(k, device="cuda")
    a = torch.empty(k, dtype=torch.int32, device="cuda")

    def best_of(runs):
        times = []
        for _ in range(runs):
            torch.cuda.synchronize()
            t = time.perf_counter()
            assert _abi.load().nova_amd_alpha_vectors_value_and_action_gpu(
                n, r, G.data_ptr(), pi.data_ptr(), k, B.data_ptr(), 1, V.data_ptr(),
                a.data_ptr(), None) == 0
            times.append(time.perf_counter() - t)
        return min(times)

    tame = best_of(8)
    B[k - 1, n - 1] = 1e-35
    wild = best_of(8)
    print("fp32 value/action: %.0f us, with a tiny entry %.0f us" % (tame * 1e6, wild * 1e6))
    assert wild <= 2.2 * tame


def test_large_fp32_against_exact_sample():
    """At n = 20,000 and r = 4,096 (the dense PBVI size) with k = 8,192 beliefs: fp32 against
    exact on the first 256 beliefs (same choice or a near-tie)."""
    k, n, r = 8192, 20000, 4096
    G, pi, B = instance(k, n, r, seed=99)
    p = policy(G, pi)
    V, act, j = p.value_and_action_batch(B, "fp32", return_alpha=True)
    Ve, acte, je = p.value_and_action_batch(B[:256], "exact", return_alpha=True)
    V, j = V.cpu().numpy()[:256], j.cpu().numpy()[:256]
    Ve, je = Ve.cpu().numpy(), je.cpu().numpy()
    scale = np.maximum(1.0, np.abs(Ve))
    assert np.all(np.abs(V - Ve) <= 1e-5 * scale)
    print("large: %d of 256 sampled choices differ between fp32 and exact"
          % int((j != je).sum()), flush=True)


@pytest.mark.parametrize("n,m,z,ns,k", [(40, 3, 4, 5, 200), (700, 4, 6, 9, 300)])
def test_belief_update_batch_bitwise(oracle, n, m, z, ns, k):
    P = synth.pomdp_arrays(n=n, m=m, z=z, ns=ns, r=4, rz=3, seed=n + k)
    # a ragged successor list and an observation impossible under one action
    P["S"] = P["S"].copy()
    P["S"][0, 0, 2] = -1
    P["O"] = P["O"].copy()
    P["O"][1, :, 0] = 0.0
    rng = np.random.default_rng(k)
    B = rng.exponential(size=(k, n))
    B[rng.random((k, n)) < 0.7] = 0.0
    B[:, 0] += 1e-3
    B = (B / B.sum(axis=1, keepdims=True)).astype(np.float32)
    a = rng.integers(0, m, k).astype(np.uint32)
    o = rng.integers(0, z, k).astype(np.uint32)
    a[:5], o[:5] = 1, 0                       # impossible observations
    a[5] = m                                  # an action out of range
    p = POMDP.from_dict(P)
    p.initialize_gpu()
    Bp, status = p.belief_update_batch(B, a, o)
    Bp, status = Bp.cpu().numpy(), status.cpu().numpy()
    assert status[5] == 1
    for i in range(k):
        if i == 5:
            continue
        rc, bp = oracle.belief_update(P, B[i], int(a[i]), int(o[i]))
        assert status[i] == rc, i
        assert np.array_equal(bits(Bp[i]), bits(bp)), i
    assert np.all(status[:5] == 10)
    print("belief update batch: n=%d k=%d bit-identical (%d impossible observations)"
          % (n, k, int((status == 10).sum())), flush=True)


@pytest.mark.parametrize("n,m,z,ns,k", [(1, 2, 3, 1, 4100), (130, 3, 5, 4, 4101),
                                        (257, 40, 2, 9, 4200), (8192, 2, 3, 3, 33),
                                        (8200, 3, 2, 4, 70),
                                        (2, 1, 2, 1, 2_100_000)])     # more tiles than a grid's y
def test_belief_update_tiles_equal_single_triples(oracle, n, m, z, ns, k):
    """Batches that go through tiles of 32 triples (many triples, or n from 8,192 on) against the
    oracle on a sample and against calls below those sizes on every triple: ragged and skewed
    successor lists, uneven actions, impossible observations, actions and observations out of
    range (their rows are left as they were)."""
    import torch
    from nova_amd import _abi
    P = synth.pomdp_arrays(n=n, m=m, z=z, ns=min(ns, n), r=2, rz=1, seed=n + k)
    rng = np.random.default_rng(k)
    S = P["S"].copy()
    if n > 2:
        S[rng.random(S.shape[:2]) < 0.2, -1] = -1
    S[: n // 2, 0, 0] = 0                      # one state with a long predecessor list
    P["S"] = S
    P["O"] = P["O"].copy()
    P["O"][0, :, 0] = 0.0
    p = POMDP.from_dict(P)
    p.initialize_gpu()
    B = rng.exponential(size=(k, n)).astype(np.float32)
    B /= B.sum(axis=1, keepdims=True)
    a = np.minimum(rng.geometric(0.5, k) - 1, m - 1).astype(np.int32)
    o = rng.integers(0, z, k).astype(np.int32)
    a[3], o[4] = m, z
    lib = _abi.load()
    Bt, at, ot = (torch.from_numpy(x).cuda() for x in (B, a, o))

    def call(lo, hi):
        out = torch.full((hi - lo, n), -7.0, device="cuda")
        st = torch.empty(hi - lo, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        assert lib.nova_amd_belief_update_batch_gpu(
            ct.byref(p), hi - lo, Bt[lo:hi].data_ptr(), at[lo:hi].data_ptr(),
            ot[lo:hi].data_ptr(), out.data_ptr(), st.data_ptr()) == 0
        return out.cpu().numpy(), st.cpu().numpy()

    got, status = call(0, k)
    assert status[3] == 1 and status[4] == 1 and np.all(got[3:5] == -7.0)
    if n < 8192:
        step = 4000              # (below the tiles' 4,096)
        parts = [call(lo, min(lo + step, k)) for lo in range(0, k, step)]
        assert np.array_equal(bits(got), bits(np.concatenate([x for x, _ in parts])))
        assert np.array_equal(status, np.concatenate([x for _, x in parts]))
    for i in [i for i in range(0, k, max(1, k // 40)) if i not in (3, 4)]:
        rc, bp = oracle.belief_update(P, B[i], int(a[i]), int(o[i]))
        assert status[i] == rc and np.array_equal(bits(got[i]), bits(bp)), i


@pytest.mark.parametrize("n,k", [(1_000_000, 1),      # one tile of 128 MB
                                 (200_000, 70),       # chunks of five tiles, the last one of three
                                 (1_048_576, 40), (1_048_577, 3)])   # the largest, and no tiles
def test_belief_update_of_large_models_takes_bounded_memory(oracle, n, k):
    """The workspace of an update stays within 128 MiB and the triples' own 24 bytes (beside the
    predecessor lists), and is given back with the model; results equal the oracle's."""
    import torch
    from nova_amd import _abi
    m, z, ns = 2, 2, 2
    P = synth.pomdp_arrays(n=n, m=m, z=z, ns=ns, r=2, rz=1, seed=n + k)
    P["S"] = P["S"].copy()
    P["S"][:100, 0, 0] = 0
    p = POMDP.from_dict(P)
    p.initialize_gpu()
    rng = np.random.default_rng(k)
    B = rng.exponential(size=(k, n)).astype(np.float32)
    B /= B.sum(axis=1, keepdims=True)
    a = rng.integers(0, m, k).astype(np.int32)
    o = rng.integers(0, z, k).astype(np.int32)
    Bt, at, ot = (torch.from_numpy(x).cuda() for x in (B, a, o))
    out = torch.empty((k, n), device="cuda")
    st = torch.empty(k, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    assert _abi.load().nova_amd_belief_update_batch_gpu(
        ct.byref(p), k, Bt.data_ptr(), at.data_ptr(), ot.data_ptr(), out.data_ptr(),
        st.data_ptr()) == 0
    lists = 4 * (m * (n + 1) + 2 * n * m * ns + m * z * n)
    slack = 32 << 20                 # (the driver hands out whole blocks; kernels are loaded)
    assert before - torch.cuda.mem_get_info()[0] <= lists + (128 << 20) + 24 * k + slack
    got, status = out.cpu().numpy(), st.cpu().numpy()
    for i in range(0, k, max(1, k // 8)):
        rc, bp = oracle.belief_update(P, B[i], int(a[i]), int(o[i]))
        assert status[i] == rc and np.array_equal(bits(got[i]), bits(bp)), i
    free = torch.cuda.mem_get_info()[0]
    model = 4 * (2 * n * m * ns + n * m + m * n * z)
    p.uninitialize_gpu()
    assert torch.cuda.mem_get_info()[0] - free >= lists + model - slack


def bf16_round(x):
    """float32 -> nearest bfloat16 (ties to even), returned as float32."""
    u = np.asarray(x, np.float32).view(np.uint32).astype(np.uint64)
    u = ((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16
    return u.astype(np.uint32).view(np.float32)


@pytest.mark.parametrize("k,n,r", [(1, 1, 1), (70, 33, 65), (300, 257, 130), (513, 100, 300),
                                   (1000, 600, 500)])
def test_bf16_blocked_kernel_equals_legacy(monkeypatch, k, n, r):
    """The k-blocked direct-to-LDS bf16 GEMM and the row-major register-staged one round the
    same operands and accumulate the k-steps in the same order: V, action and alpha are
    bit-identical (ragged k, n and r; 1 to 10 column tiles)."""
    G, pi, B = instance(k, n, r, seed=11 * k + n)
    p = policy(G, pi)
    monkeypatch.delenv("NOVA_AMD_DENSE_KERNEL", raising=False)
    V, act, j = (x.cpu().numpy() for x in p.value_and_action_batch(B, "bf16", return_alpha=True))
    monkeypatch.setenv("NOVA_AMD_DENSE_KERNEL", "legacy")
    Vl, actl, jl = (x.cpu().numpy() for x in p.value_and_action_batch(B, "bf16",
                                                                      return_alpha=True))
    monkeypatch.delenv("NOVA_AMD_DENSE_KERNEL")
    assert np.array_equal(bits(V), bits(Vl)) and np.array_equal(act, actl)
    assert np.array_equal(j, jl)
    # against FP64 on the bf16-rounded operands: only fp32 accumulation error remains
    C = bf16_round(B).astype(np.float64) @ bf16_round(G).astype(np.float64).T
    mag = np.abs(bf16_round(B)).astype(np.float64) @ np.abs(bf16_round(G)).astype(np.float64).T
    tol = 1e-6 * n * mag.max(axis=1) + 1e-30
    assert np.all(np.abs(V - C[np.arange(k), j]) <= tol)
    assert np.all(C.max(axis=1) - C[np.arange(k), j] <= 2 * tol)
    print("bf16 blocked == legacy: k=%d n=%d r=%d" % (k, n, r), flush=True)


def test_belief_update_batch_long_lists_and_global_belief(oracle):
    """n = 30,000 (past the LDS copy of b: b is read from global memory) and successors skewed
    onto states 0-63, whose block then holds more predecessor entries than a wave's product
    scratch (several sub-ranges per block): bit for bit against the oracle's float twin."""
    n, m, z, ns, k = 30000, 2, 3, 4, 12
    P = synth.pomdp_arrays(n=n, m=m, z=z, ns=ns, r=2, rz=2, seed=77)
    P["S"] = P["S"].copy()
    rng = np.random.default_rng(77)
    hot = rng.random((n, m)) < 0.2                  # about 24,000 entries onto states 0-63
    P["S"][:, :, 0] = np.where(hot, rng.integers(0, 64, (n, m)), P["S"][:, :, 0])
    B = rng.exponential(size=(k, n)).astype(np.float32)
    B = (B / B.sum(axis=1, keepdims=True)).astype(np.float32)
    a = rng.integers(0, m, k).astype(np.uint32)
    o = rng.integers(0, z, k).astype(np.uint32)
    p = POMDP.from_dict(P)
    p.initialize_gpu()
    Bp, status = p.belief_update_batch(B, a, o)
    Bp, status = Bp.cpu().numpy(), status.cpu().numpy()
    for i in range(k):
        rc, bp = oracle.belief_update(P, B[i], int(a[i]), int(o[i]))
        assert status[i] == rc and np.array_equal(bits(Bp[i]), bits(bp)), i
    print("belief update batch: n=30000, skewed lists, bit-identical", flush=True)


@pytest.mark.parametrize("n,m,z,ns,k", [(65536, 2, 3, 4, 6), (65537, 2, 3, 4, 6),
                                        (8, 4097, 2, 2, 40)],
                         ids=["n65536_16bit_lists", "n65537_32bit_lists", "m4097_unordered"])
def test_belief_update_batch_index_width_and_order_bounds(oracle, n, m, z, ns, k):
    """The boundaries of the batched belief update's internal forms, bit for bit against the
    oracle's float twin: predecessor lists with 16-bit indices (n <= 65,536) and 32-bit ones
    (n = 65,537), and triples run in call order instead of grouped by action (m > 4,096)."""
    P = synth.pomdp_arrays(n=n, m=m, z=z, ns=ns, r=2, rz=2, seed=n + m)
    rng = np.random.default_rng(n + m)
    B = rng.exponential(size=(k, n)).astype(np.float32)
    B = (B / B.sum(axis=1, keepdims=True)).astype(np.float32)
    a = rng.integers(0, m, k).astype(np.uint32)
    o = rng.integers(0, z, k).astype(np.uint32)
    a[0] = m - 1                                  # the last action and state indices in use
    p = POMDP.from_dict(P)
    p.initialize_gpu()
    Bp, status = p.belief_update_batch(B, a, o)
    Bp, status = Bp.cpu().numpy(), status.cpu().numpy()
    for i in range(k):
        rc, bp = oracle.belief_update(P, B[i], int(a[i]), int(o[i]))
        assert status[i] == rc and np.array_equal(bits(Bp[i]), bits(bp)), i
    print("belief update batch: n=%d m=%d bit-identical" % (n, m), flush=True)
