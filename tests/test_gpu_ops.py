"""GPU parity of the op-level entry points against the CPU oracle, through the C ABI.
Integer/byte results and everything routing depends on are compared bit for bit."""
import time

import numpy as np
import pytest
import torch

from ferrite_amd import synth
from ferrite_amd.backend import InvalidArg, ShapeMismatch

pytestmark = pytest.mark.gpu


def dev(hip, a, dtype=None):
    return hip.upload(np.asarray(a), dtype)


def host(hip, t):
    hip.sync()
    return t.cpu().numpy()


def replay_us(hip, call, copies=50):
    """Time of one of `copies` calls in a captured graph, best of five replays."""
    call()
    hip.begin_capture()
    for _ in range(copies):
        call()
    trace = hip.end_capture()
    hip.begin_verify(trace)
    times = []
    for _ in range(5):
        hip.sync()
        t0 = time.perf_counter()
        hip.begin_verify(trace)
        hip.sync()
        times.append(time.perf_counter() - t0)
    hip.graph_destroy(trace)
    return min(times) / copies * 1e6


# ---- matmul: the reference's sequential-k chain, bit for bit ----
def test_matmul_matches_manual(hip):  # golden.rs:14-27
    x, w = dev(hip, np.array([[1, 2], [3, 4]], np.float32)), dev(hip, np.array([[5, 6], [7, 8]], np.float32))
    out = torch.zeros(2, 2, device=hip.device)
    hip.matmul(x, w, None, out)
    assert host(hip, out).tolist() == [[17, 23], [39, 53]]
    hip.matmul(x, w, dev(hip, np.array([0.5, -0.5], np.float32)), out)
    assert host(hip, out).tolist() == [[17.5, 22.5], [39.5, 52.5]]


@pytest.mark.parametrize("n,k,o", [(5, 300, 70), (32, 4096, 128), (3, 37, 5), (1, 64, 1), (130, 256, 16), (7, 7168, 256)])
def test_matmul_bit_exact_vs_oracle(hip, oracle, n, k, o):
    rng = np.random.default_rng(n * 1000 + k)
    x = rng.normal(0, 1, (n, k)).astype(np.float32)
    w = rng.normal(0, 0.02, (o, k)).astype(np.float32)
    b = rng.normal(0, 1, o).astype(np.float32)
    out = torch.empty(n, o, device=hip.device)
    hip.matmul(dev(hip, x), dev(hip, w), None, out)
    assert np.array_equal(host(hip, out), oracle.matmul(x, w))
    hip.matmul(dev(hip, x), dev(hip, w), dev(hip, b), out)
    assert np.array_equal(host(hip, out), oracle.matmul(x, w, b))


# tile edges (16 rows, 16 outputs, 64 outputs a block); k remainders of the 16-wide steps, of the 64-wide chunks and of the
# rounds of three (matrix cores) and four chunks; rows that are only 4-byte aligned; values whose products are denormal or -0.
# The kernel each row is there for is asserted: the one-chain-per-lane kernel up to 512 tiles of 16 x 16, the matrix-core one
# beyond, and for up to four rows beyond 1024 tiles the one without padding rows.
def _chain_kernel(n, k, o):
    tiles = -(-n // 16) * -(-o // 16)
    if k % 4 or n * o < 1024:
        return "simple"
    return "rows" if n <= 4 and tiles > 1024 else "mfma" if tiles > 512 else "valu"


VALU_SHAPES = [(1, 4, 1024), (15, 12, 80), (16, 16, 64), (17, 20, 65), (33, 52, 32), (64, 64, 16), (31, 68, 129), (100, 132, 128),
               (3, 128, 400), (20, 192, 90), (40, 260, 33), (9, 324, 130)]
MFMA_SHAPES = [(n, k, o) for n, o in ((520, 272), (17, 8200), (3, 8300)) for k in (4, 8, 12, 16, 60, 64, 72, 128)] + \
              [(1030, 100, 272), (257, 260, 1041), (100, 132, 3072), (7, 736, 9000), (513, 192, 260), (520, 204, 270), (530, 328, 272)]
ROWS_SHAPES = [(1, 4, 16400), (2, 60, 16385), (3, 64, 16449), (4, 68, 20000), (4, 132, 16447), (1, 1000, 17000)]


@pytest.mark.parametrize("n,k,o,kernel", [s + ("valu",) for s in VALU_SHAPES] + [s + ("mfma",) for s in MFMA_SHAPES] +
                         [s + ("rows",) for s in ROWS_SHAPES] + [(33, 52, 31, "simple"), (17, 50, 70, "simple")])
def test_matmul_tiles_bit_exact_vs_oracle(hip, oracle, n, k, o, kernel):
    assert _chain_kernel(n, k, o) == kernel
    rng = np.random.default_rng(n * 1000 + k)
    x = rng.normal(0, 1, (n, k)).astype(np.float32)
    w = rng.normal(0, 0.02, (o, k)).astype(np.float32)
    x[0], w[0] = x[0] * np.float32(1e-30), w[0] * np.float32(1e-10)   # denormal products and sums
    x[n // 2, ::3] = -0.0
    w[o // 2, ::2] = 0.0
    xbuf = torch.empty(n * k + 1, device=hip.device)
    xd = xbuf[1:].view(n, k)
    xd.copy_(torch.from_numpy(x))
    out = torch.full((n, o), -1.0, device=hip.device)
    hip.matmul(xd, dev(hip, w), None, out)
    assert np.array_equal(host(hip, out), oracle.matmul(x, w))


@pytest.mark.parametrize("n,k,o,kernel", [(40, 100, 48, "valu"), (40, 324, 48, "valu"), (530, 100, 272, "mfma"), (530, 328, 272, "mfma"),
                                          (4, 100, 16400, "rows"), (33, 52, 31, "simple")])
def test_matmul_nan_and_infinity_vs_oracle(hip, oracle, n, k, o, kernel):
    """Infinities (also against zero weights and against each other), NaN and products that overflow stay in their row or
    output and come out as the chain has them."""
    assert _chain_kernel(n, k, o) == kernel
    rng = np.random.default_rng(n + k)
    x = rng.normal(0, 1, (n, k)).astype(np.float32)
    w = rng.normal(0, 1, (o, k)).astype(np.float32)
    x[0, k - 1], x[1, 3], x[n - 1, 0], x[2, 5], x[2, 6] = np.inf, np.nan, -np.inf, 3e38, -3e38
    w[3, 0], w[5, 7], w[o - 1, k - 1], w[7] = 0.0, np.nan, np.inf, 1e30
    out = torch.empty(n, o, device=hip.device)
    hip.matmul(dev(hip, x), dev(hip, w), None, out)
    ref = oracle.matmul(x, w)
    assert np.isnan(ref).any() and np.isinf(ref).any() and np.isfinite(ref).any()
    assert np.array_equal(host(hip, out), ref, equal_nan=True)


def test_matmul_of_few_rows_is_not_padded_to_sixteen(hip):
    """Against very many outputs four rows take half the time of twelve; in tiles of 16 rows they took as long."""
    w = torch.randn(131072, 64, device=hip.device)
    took = {}
    for n in (4, 12):
        x, out = torch.randn(n, 64, device=hip.device), torch.empty(n, 131072, device=hip.device)
        took[n] = replay_us(hip, lambda: hip.matmul(x, w, None, out))
    print(took)
    assert took[4] < 0.75 * took[12], took


def test_matmul_shape_errors(hip):
    z = lambda *s: torch.zeros(*s, device=hip.device)
    with pytest.raises(ShapeMismatch):
        hip.matmul(z(2, 3), z(2, 4), None, z(2, 2))
    with pytest.raises(InvalidArg):
        hip.matmul(z(2, 3), z(4, 3), None, z(2, 2))


# ---- the sum of squares behind rmsnorm: the serial chain's bits whichever part of it is walked in parallel ----
def _sumsq_rows(dim, rng):
    rows = [rng.normal(0, s, dim) for s in (1.0, 1e-3, 1e4, 1e-18, 1e-23, 1e17)]
    rows += [np.sqrt(rng.integers(0, 1 << b, dim) * 2.0 ** -b) for b in (1, 3, 6, 10)]
    rows += [rng.integers(-4, 5, dim) * 0.5, rng.integers(0, 64, dim) / 8.0,           # squares of few bits: exact ties
             np.full(dim, 1.0), np.full(dim, 0.1), np.full(dim, 3.0 * 2.0 ** -12), np.zeros(dim)]
    rows += [np.exp(np.linspace(-20, 20, dim)), np.exp(np.linspace(20, -20, dim))]       # a binade every few values / one
    spike = rng.normal(0, 1, dim)
    spike[dim // 2], spike[dim // 3] = 4096.0, 64.0
    rows += [np.exp(np.linspace(np.log(1e-18), np.log(1e-14), dim)), np.exp(np.linspace(np.log(1e-14), np.log(1e-18), dim)),
             rng.normal(0, 2.0 ** -53, dim), rng.normal(0, 2.0 ** -75, dim)]   # sums around 2^-100, where walking begins; denormals
    late = np.zeros(dim)
    late[-3:] = [1e-30, 1e-12, 3.0]
    rng_ties = 2.0 ** rng.integers(-13, 1, dim)                                           # halves of the running sum's ulp
    rng_ties[0] = 4096.0
    rows += [spike, late, rng_ties, -np.abs(rng.normal(0, 1, dim))]
    return np.stack(rows).astype(np.float32)


@pytest.mark.parametrize("dim", [4, 60, 64, 256, 260, 1000, 4096, 5120, 7168, 8192, 12296])
def test_rmsnorm_sum_of_squares_is_the_serial_chain(hip, oracle, dim):
    rng = np.random.default_rng(dim)
    x = _sumsq_rows(dim, rng)
    x = np.concatenate([x, x * np.float32(1.3), rng.normal(0, 1, (40, dim)).astype(np.float32)])
    w = rng.normal(1, 0.1, dim).astype(np.float32)
    out = torch.empty(x.shape, device=hip.device)
    hip.rmsnorm(dev(hip, x), dev(hip, w), 1e-6, out)
    assert np.array_equal(host(hip, out), oracle.rmsnorm(x, w, 1e-6))
    # without eps the smallest sums show as well
    hip.rmsnorm(dev(hip, x), dev(hip, w), 0.0, out)
    assert np.array_equal(host(hip, out), oracle.rmsnorm(x, w, 0.0), equal_nan=True)
    # more rows than the four-waves-per-row kernel takes
    many = np.tile(x, (1100 // len(x) + 1, 1))
    out = torch.empty(many.shape, device=hip.device)
    for eps in (1e-6, 0.0):
        hip.rmsnorm(dev(hip, many), dev(hip, w), eps, out)
        assert np.array_equal(host(hip, out)[:len(x)], oracle.rmsnorm(x, w, eps), equal_nan=True)
    bad = x[:3].copy()
    bad[0, dim // 2], bad[1, dim - 1], bad[2, 0] = np.inf, np.nan, 3e38
    out = torch.empty(bad.shape, device=hip.device)
    hip.rmsnorm(dev(hip, bad), dev(hip, w), 1e-6, out)
    assert np.array_equal(host(hip, out), oracle.rmsnorm(bad, w, 1e-6), equal_nan=True)


def _narrow(x, keep):
    """f32 values rounded to `keep` mantissa bits (7: bf16)."""
    drop = 23 - keep
    u = x.view(np.uint32).astype(np.uint64)
    u = (u + (1 << (drop - 1)) - 1 + ((u >> drop) & 1)) >> drop << drop
    return u.astype(np.uint32).view(np.float32)


def _value_kinds(rows, dim):
    """What a residual stream may hold: squares of narrow values make ties of the running sum, zeros leave it as it is."""
    x = np.random.default_rng(dim).normal(0, 1, (rows, dim)).astype(np.float32)
    sparse = x * (np.random.default_rng(dim + 1).random((rows, dim)) < 0.1)
    return dict(normal=x, bf16=_narrow(x, 7), bf16_small=_narrow(x * np.float32(0.037), 7), fp16=_narrow(x, 10), fp8=_narrow(x, 3),
                zeros=np.zeros_like(x), sparse=sparse.astype(np.float32))


@pytest.mark.parametrize("dim", [256, 1028, 4096, 7168])
def test_rmsnorm_of_narrow_values_is_the_serial_chain(hip, oracle, dim):
    w = np.random.default_rng(3).normal(1, 0.1, dim).astype(np.float32)
    for kind, x in _value_kinds(40, dim).items():
        out = torch.empty(x.shape, device=hip.device)
        hip.rmsnorm(dev(hip, x), dev(hip, w), 1e-6, out)
        assert np.array_equal(host(hip, out), oracle.rmsnorm(x, w, 1e-6)), kind


@pytest.mark.parametrize("dim", [4096, 7168])
def test_rmsnorm_takes_no_longer_for_narrow_values(hip, dim):
    """Rows of bf16 values or of zeros go the same parallel way as any others.  (Walked value by value they took three
    to seven times as long; 2 leaves room for the parity scan and for the clock.)"""
    w = torch.ones(dim, device=hip.device)
    took = {}
    for kind, x in _value_kinds(192, dim).items():
        x, out = dev(hip, x), torch.empty(192, dim, device=hip.device)
        took[kind] = replay_us(hip, lambda: hip.rmsnorm(x, w, 1e-6, out))
    print({k: round(v, 1) for k, v in took.items()})
    assert max(took.values()) < 2.0 * took["normal"], took


# ---- swiglu ----
def test_swiglu_bit_exact_vs_oracle(hip, oracle):  # golden.rs:44-55 values included
    rng = np.random.default_rng(1)
    gu = rng.normal(0, 4, (17, 2 * 96)).astype(np.float32)
    gu[0, :4] = [2., 20., -200., 95.]
    gu[0, 96:100] = [3., 1., 50., -50.]
    out = torch.empty(17, 96, device=hip.device)
    hip.swiglu_limited(dev(hip, gu), 10.0, out)
    assert np.array_equal(host(hip, out), oracle.swiglu_limited(gu, 10.0))
    with pytest.raises(InvalidArg):
        hip.swiglu_limited(dev(hip, gu[:, :191]), 10.0, out)


# ---- routing ----
def route(hip, logits, bias, k, scale, ng=1, tg=1):
    n = logits.shape[0]
    probs = torch.empty(n, k, device=hip.device)
    ids = torch.empty(n, k, device=hip.device)
    ids32 = torch.empty(n, k, dtype=torch.int32, device=hip.device)
    hip.moe_route(dev(hip, logits.astype(np.float32)), dev(hip, bias.astype(np.float32)), k, scale, probs, ids, ng, tg, ids32)
    p, i, i32 = host(hip, probs), host(hip, ids), host(hip, ids32)
    assert np.array_equal(i.astype(np.int32), i32)
    return p, i


def test_moe_route_noaux_tc(hip):  # golden.rs:189-210
    p, i = route(hip, np.array([[1.0, 2.0, 0.5]]), np.array([0.0, 0.0, 0.5]), 2, 1.0)
    assert i.tolist() == [[2.0, 1.0]]
    s = lambda v: 1.0 / (1.0 + np.exp(-v))
    assert abs(p[0, 0] - s(0.5) / (s(2.0) + s(0.5))) < 1e-5 and abs(p[0, 1] - s(2.0) / (s(2.0) + s(0.5))) < 1e-5


def test_moe_route_ramp_fixture(hip, oracle):  # gpu_smoke.rs:139-155: ids exact, probs 1e-5 (here: exact)
    n, e, k = 2, 288, 8
    logits = (np.arange(n * e, dtype=np.float32) * np.float32(0.017) - np.float32(2.0)).reshape(n, e)
    bias = (np.arange(e) % 11).astype(np.float32) * np.float32(0.01)
    p, i = route(hip, logits, bias, k, 2.5)
    po, io = oracle.moe_route(logits, bias, k, 2.5)
    assert np.array_equal(i, io) and np.array_equal(p, po)


@pytest.mark.parametrize("n,e,k,ng,tg", [(8, 16, 4, 4, 2), (32, 128, 8, 8, 4), (33, 256, 8, 8, 4), (64, 128, 8, 1, 1),
                                         (5, 288, 8, 1, 1), (4, 64, 6, 4, 3), (16, 512, 32, 16, 8), (3, 8, 8, 1, 1)])
def test_moe_route_bit_exact_vs_oracle(hip, oracle, n, e, k, ng, tg):
    rng = np.random.default_rng(e + n)
    logits = rng.normal(0, 1.7, (n, e)).astype(np.float32)
    bias = rng.normal(0, 0.01, e).astype(np.float32)
    p, i = route(hip, logits, bias, k, 2.5, ng, tg)
    po, io = oracle.moe_route(logits, bias, k, 2.5, ng, tg)
    assert np.array_equal(i, io)
    assert np.array_equal(p, po)


def test_moe_route_ties_lower_index_first(hip, oracle):  # cpu.rs:560
    logits = np.zeros((2, 128), np.float32)
    bias = np.zeros(128, np.float32)
    bias[[5, 70, 9]] = 0.25
    for ng, tg in [(1, 1), (8, 4)]:
        p, i = route(hip, logits, bias, 8, 1.0, ng, tg)
        po, io = oracle.moe_route(logits, bias, 8, 1.0, ng, tg)
        assert np.array_equal(i, io) and np.array_equal(p, po)
    assert route(hip, logits, bias, 8, 1.0)[1][0].tolist() == [5, 9, 70, 0, 1, 2, 3, 4]


@pytest.mark.parametrize("e,k,ng,tg", [(512, 32, 8, 4), (160, 8, 8, 4), (96, 6, 8, 3), (64, 8, 64, 16), (128, 8, 2, 1), (256, 8, 2, 1),
                                       (32, 8, 8, 4), (16, 16, 1, 1), (300, 7, 1, 1), (48, 4, 16, 2), (32, 32, 1, 1), (31, 6, 1, 1),
                                       (33, 32, 1, 1), (8, 2, 4, 2), (24, 5, 8, 4)])
def test_moe_route_groups_and_thresholds_vs_oracle(hip, oracle, e, k, ng, tg):
    """Groups that are aligned runs of 1 to 64 lanes, groups that are not, more than 64 experts a group; scores on a coarse grid,
    so that many tie at the selection's threshold, in and across the 64-expert slots; infinite biases; both sides of the line
    between ranking and the threshold (32 experts)."""
    rng = np.random.default_rng(e * 37 + ng)
    logits = (np.round(rng.normal(0, 1.5, (24, e)) * 2) / 2).astype(np.float32)
    logits[3] = 0.25
    logits[5, : e // 2] = -300.0
    bias = (rng.integers(0, 3, e) * 0.125).astype(np.float32)
    bias[[1, e // 2]] = -np.inf
    bias[e - 1] = np.inf
    p, i = route(hip, logits, bias, k, 2.5, ng, tg)
    po, io = oracle.moe_route(logits, bias, k, 2.5, ng, tg)
    assert np.array_equal(i, io) and np.array_equal(p, po)


@pytest.mark.parametrize("experts,topk,shared", [(16, 4, 128), (64, 32, 0), (100, 6, 128), (288, 8, 128)])
def test_layer_tables_of_a_single_token(hip, oracle, experts, topk, shared):
    """One token's tables come from the wave that routed it (one or several blocks of 64 experts): equal to the permutation's,
    also where NaN scores leave slots empty, and the units are one row each."""
    from ferrite_amd import synth
    from ferrite_amd.backend import MODE_MFMA_FP8
    cfg = synth.MoeConfig(1, 256, experts, topk, 128, shared, 1, 1)
    inp = synth.make_inputs(cfg, seed=experts)
    for nan_from in (experts, topk // 2):
        inp.router_bias[nan_from:] = np.nan
        layer = hip.load_moe_layer(inp)
        x = torch.from_numpy(inp.x).to(hip.device)
        out = torch.empty_like(x)
        for _ in range(2):   # the second call finds the counters as the first left them
            hip.moe_layer_dev_mxfp4(layer, x, out, MODE_MFMA_FP8)
        hip.sync()
        v = {k: t.cpu().numpy() for k, t in hip.workspace_view(layer, 1, MODE_MFMA_FP8).items()}
        po, io = oracle.moe_route(v["logits"], inp.router_bias, topk, cfg.routed_scaling, 1, 1, nan_policy=1)
        assert np.array_equal(v["ids"], io.astype(np.int32)) and np.array_equal(v["probs"], po)
        t = oracle.moe_permute(v["ids"], experts)
        for key in ("counts", "starts", "perm_map", "gather_src", "active"):
            assert np.array_equal(v[key], t[key]), key
        assert int(v["n_active"][0]) == t["n_active"] == min(topk, nan_from)
        assert np.isfinite(out.cpu().numpy()).all()


def test_moe_route_extreme_logits(hip, oracle):
    logits = np.array([[-200, -100, -88.5, -30, 0, 30, 88.5, 100, 200, 1e-30, -1e-30, 17.3, -17.3, 5, -5, 0.1]], np.float32)
    p, i = route(hip, logits, np.zeros(16, np.float32), 8, 2.5)
    po, io = oracle.moe_route(logits, np.zeros(16, np.float32), 8, 2.5)
    assert np.array_equal(i, io) and np.array_equal(p, po)


def test_moe_route_nan_scores(hip, oracle):
    """NaN logits: never selected; slots that no finite score can fill get id -1 and weight 0, as the reference's
    device router leaves them (kernels/cuda/ferrite_kernels.cu:1233-1270).  Bit-equal to the oracle's statement of
    that policy, grouped and ungrouped, and through the fused layer: such slots contribute nothing."""
    rng = np.random.default_rng(11)
    logits = rng.normal(0, 1.5, (8, 64)).astype(np.float32)
    bias = rng.normal(0, 0.01, 64).astype(np.float32)
    logits[0, 5] = np.nan
    logits[1, :] = np.nan
    logits[2, :61] = np.nan
    logits[3, 16:32] = np.nan
    logits[4, ::2] = np.nan
    for ng, tg in ((1, 1), (4, 2)):
        p, i = route(hip, logits, bias, 6, 2.5, ng, tg)
        po, io = oracle.moe_route(logits, bias, 6, 2.5, ng, tg, nan_policy=1)
        assert np.array_equal(i, io), (ng, tg)
        assert np.array_equal(p, po), (ng, tg)
    assert i[1].tolist() == [-1] * 6 and p[1].tolist() == [0.0] * 6


def test_layer_with_nan_activations_keeps_other_tokens_intact(hip, oracle):
    """A token whose activations are NaN routes nowhere (ids -1, no row in the permutation); every other token's row
    is bit-identical to a run without it, in both the fused-head and the separate-launch path."""
    from ferrite_amd import synth
    from ferrite_amd.backend import MODE_MFMA_FP8
    for n in (24, 300):
        cfg = synth.MoeConfig(n, 256, 16, 4, 128, 128, 4, 2)
        inp = synth.make_inputs(cfg, seed=n)
        layer = hip.load_moe_layer(inp)
        x = torch.from_numpy(inp.x).to(hip.device)
        out = torch.empty_like(x)
        hip.moe_layer_dev_mxfp4(layer, x, out, MODE_MFMA_FP8)
        hip.sync()
        clean = out.cpu().numpy()
        x[7, :] = float("nan")
        hip.moe_layer_dev_mxfp4(layer, x, out, MODE_MFMA_FP8)
        hip.sync()
        got = out.cpu().numpy()
        v = hip.workspace_view(layer, n, MODE_MFMA_FP8)
        assert v["ids"][7].cpu().tolist() == [-1] * 4
        assert v["perm_map"].view(n, 4)[7].cpu().tolist() == [-1] * 4
        keep = np.arange(n) != 7
        assert np.array_equal(got[keep], clean[keep])
        # (row 7 itself holds whatever the shared expert makes of the quantised row: the reference's e4m3 encoder
        # saturates non-finite values to +-448, quant.rs:98-124, so it need not be NaN)


def test_moe_route_shape_errors(hip):
    z = lambda *s: torch.zeros(*s, device=hip.device)
    with pytest.raises(InvalidArg):
        hip.moe_route(z(2, 8), z(7), 2, 1.0, z(2, 2), z(2, 2))
    with pytest.raises(InvalidArg):
        hip.moe_route(z(2, 8), z(8), 2, 1.0, z(2, 3), z(2, 2))
    with pytest.raises(InvalidArg):
        hip.moe_route(z(2, 8), z(8), 2, 1.0, z(2, 2), z(2, 2), 3, 2)   # E % n_group


# ---- permutation ----
def permute(hip, ids, e):
    t = hip.moe_permute(dev(hip, ids.astype(np.int32)), e)
    hip.sync()
    return {k: v.cpu().numpy() for k, v in t.items()}


def test_moe_permute_reference_vector(hip, oracle):  # chain_dev.rs:25042-25061 routing table, as it stands there
    """The reference's vector lists an expert twice inside a token (5,1,5 and 9,1,9); its order is
    [1,3,7] [5] [0,2,4] [6,8] for experts 1, 2, 5, 9 with counts 3, 1, 3, 2."""
    ids = np.array([[5, 1, 5], [1, 5, 2], [9, 1, 9]])
    t = permute(hip, ids, 12)
    assert t["gather_src"].tolist() == [1, 3, 7, 5, 0, 2, 4, 6, 8]
    assert t["counts"].tolist() == [0, 3, 1, 0, 0, 3, 0, 0, 0, 2, 0, 0]
    assert t["active"][:4].tolist() == [1, 2, 5, 9] and int(t["n_active"][0]) == 4
    o = oracle.moe_permute(ids, 12)
    for key in ("counts", "starts", "perm_map", "gather_src", "active"):
        assert np.array_equal(t[key], o[key]), key
    t = permute(hip, np.array([[5, 1, 7], [1, 5, 2], [9, 1, 3]]), 12)
    assert t["gather_src"].tolist() == [1, 3, 7, 5, 8, 0, 4, 2, 6]
    assert t["counts"].tolist() == [0, 3, 1, 1, 0, 2, 0, 1, 0, 1, 0, 0]


@pytest.mark.parametrize("n,k,e", [(40, 6, 5), (700, 8, 16), (3000, 4, 3)])
def test_moe_permute_repeated_experts_in_a_token(hip, oracle, n, k, e):
    """ids drawn with replacement: many tokens repeat an expert; also beyond the single-block path."""
    rng = np.random.default_rng(n)
    ids = rng.integers(0, e, (n, k)).astype(np.int32)
    t = permute(hip, ids, e)
    o = oracle.moe_permute(ids, e)
    for key in ("counts", "starts", "perm_map", "gather_src", "active"):
        assert np.array_equal(t[key], o[key]), key
    assert np.array_equal(t["gather_src"], np.argsort(ids.ravel(), kind="stable"))


@pytest.mark.parametrize("n,k,e", [(1, 1, 1), (7, 3, 5), (32, 8, 128), (192, 8, 128), (1000, 8, 256), (1024, 8, 128),
                                   (1025, 8, 128), (4096, 8, 128), (8192, 8, 256), (3000, 4, 16)])
def test_moe_permute_memcmp_vs_oracle(hip, oracle, n, k, e):
    rng = np.random.default_rng(n + e)
    pop = rng.dirichlet(np.full(e, 0.3))  # skewed expert popularity
    ids = np.stack([rng.choice(e, size=k, replace=False, p=pop) for _ in range(n)]).astype(np.int32)
    t = permute(hip, ids, e)
    o = oracle.moe_permute(ids, e)
    for key in ("counts", "starts", "perm_map", "gather_src", "active"):
        assert np.array_equal(t[key], o[key]), key
    assert int(t["n_active"][0]) == o["n_active"]
    assert np.array_equal(t["gather_src"], np.argsort(ids.ravel(), kind="stable"))


@pytest.mark.parametrize("m,e,needs", [(513, 512, False), (577, 512, True), (640, 479, False), (640, 480, True),
                                       (1024, 307, False), (1024, 308, True), (1025, 1, True)])
def test_moe_permute_without_scratch(hip, oracle, m, e, needs):
    """One block does the permutation, and no scratch is asked for, while masks, prefixes, counts and starts take 60 KiB:
    12 bytes an expert and 64 assignments + 8 an expert + 4; at most 1024 assignments."""
    assert needs == (m > 1024 or e * (12 * ((m + 63) // 64) + 8) + 4 > 60 * 1024)
    ids = dev(hip, np.random.default_rng(m + e).integers(0, e, (m, 1)).astype(np.int32))
    t = {k: torch.zeros(c, dtype=torch.int32, device=hip.device) for k, c in
         (("counts", e), ("starts", e + 1), ("perm_map", m), ("gather_src", m), ("active", e), ("n_active", 1))}
    rc = hip.lib.ferrite_moe_permute(ids.data_ptr(), m, 1, e, *(v.data_ptr() for v in t.values()), None, 0,
                                     torch.cuda.current_stream(hip.device).cuda_stream)
    torch.cuda.synchronize()
    assert rc == (3 if needs else 0)   # FERRITE_ERR_WORKSPACE, FERRITE_OK
    if not needs:
        o = oracle.moe_permute(ids.cpu().numpy(), e)
        for key in ("counts", "starts", "perm_map", "gather_src", "active"):
            assert np.array_equal(t[key].cpu().numpy(), o[key]), key


def test_moe_permute_out_of_range_ids_drop_out(hip, oracle):  # dsv41_route.cu:253-261,300-303
    ids = np.array([[0, 7], [-1, 0], [2, 1]], np.int32)
    t = permute(hip, ids, 4)
    o = oracle.moe_permute(ids, 4)
    for key in ("counts", "starts", "perm_map", "gather_src"):
        assert np.array_equal(t[key], o[key]), key


# ---- formats ----
def test_mxfp4_dequant_bit_exact(hip, oracle):
    rng = np.random.default_rng(3)
    w = rng.integers(0, 256, (96, 128), dtype=np.uint8)
    s = rng.integers(100, 140, (96, 8), dtype=np.uint8)
    got = host(hip, hip.mxfp4_dequant(dev(hip, w), dev(hip, s)))
    assert np.array_equal(got.view(np.uint32), oracle.dequant_fp4_row32(w, s).view(np.uint32))


def test_mxfp4_dequant_all_codes_and_layout(hip):  # quant.rs:459-478 nibble order, every code
    w = np.zeros((1, 16), np.uint8)
    w[0, 0] = 0b1001_0111                       # element 0 = code 7 (6.0), element 1 = code 9 (-0.5)
    w[0, 8:16] = (np.arange(0, 16, 2) | (np.arange(1, 16, 2) << 4)).astype(np.uint8)
    got = host(hip, hip.mxfp4_dequant(dev(hip, w), dev(hip, np.array([[128]], np.uint8))))[0]
    assert got[0] == 12.0 and got[1] == -1.0
    assert got[16:].tolist() == [0, 1, 2, 3, 4, 6, 8, 12, 0, -1, -2, -3, -4, -6, -8, -12]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_act_quant_bit_exact_vs_oracle(hip, oracle, dtype):
    rng = np.random.default_rng(4)
    x = (rng.normal(0, 1, (64, 256)) * np.repeat(10.0 ** rng.uniform(-4, 4, (64, 8)), 32, axis=1)).astype(np.float32)
    x[3, 32:64] = 0.0
    x[5, 0:32] = np.linspace(7.3 / 512, 8.1 / 512, 32) * 1.0   # the subnormal clamp rule after scaling by 2^0.. region
    x[5, 0] = 448.0
    xt = torch.from_numpy(x).to(dtype)
    xr = xt.to(torch.float32).numpy()
    q, s = hip.act_quant_fp8(xt.to(hip.device))
    qo, so = oracle.act_quant_fp8(xr, 32, True)
    assert np.array_equal(host(hip, q).ravel(), qo)
    sbytes = host(hip, s).ravel()
    assert np.array_equal(np.exp2(sbytes.astype(np.float64) - 127), so.astype(np.float64))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_act_quant_two_terms_bit_exact_vs_oracle(hip, oracle, dtype):
    """Both terms of the two-term quantiser: codes and scales equal the oracle's, which is the reference's
    quantiser applied to x and then to what it leaves over."""
    rng = np.random.default_rng(6)
    x = (rng.normal(0, 1, (48, 512)) * np.repeat(10.0 ** rng.uniform(-4, 4, (48, 16)), 32, axis=1)).astype(np.float32)
    x[2, 64:96] = 0.0
    x[4, 0:32] = np.linspace(7.3 / 512, 8.1 / 512, 32)
    x[4, 0] = 448.0
    x[6, 32:64] = 2.0 ** -120          # scales at the smallest normal
    xt = torch.from_numpy(x).to(dtype)
    xr = xt.to(torch.float32).numpy()
    q1, s1, q2, s2 = (host(hip, t).ravel() for t in hip.act_quant_fp8_x2(xt.to(hip.device)))
    o1, t1, o2, t2 = oracle.act_quant_fp8_x2(xr)
    assert np.array_equal(q1, o1) and np.array_equal(q2, o2)
    assert np.array_equal(np.exp2(s1.astype(np.float64) - 127), t1.astype(np.float64))
    assert np.array_equal(np.exp2(s2.astype(np.float64) - 127), t2.astype(np.float64))
    # the first term is the one-term quantiser's output
    q, s = hip.act_quant_fp8(xt.to(hip.device))
    assert np.array_equal(host(hip, q).ravel(), q1) and np.array_equal(host(hip, s).ravel(), s1)


def test_act_quant_blocks_with_nan_and_scale_edges(hip, oracle):
    """NaN (either sign) in a block takes the general encoder, its neighbours the finite one; magnitudes on either side of
    every step of the power-of-two scale (448 * 2^e)."""
    rng = np.random.default_rng(9)
    x = rng.normal(0, 1, (40, 64)).astype(np.float32)
    x[:40, 32] = (448.0 * 2.0 ** np.arange(-20, 20)).astype(np.float32)
    x[1::3, 32] = np.nextafter(x[1::3, 32], np.float32(np.inf))
    x[2::3, 32] = np.nextafter(x[2::3, 32], np.float32(0))
    x[4, 3], x[7, 31], x[9, 0:32:5] = np.nan, -np.nan, np.nan
    q1, s1, q2, s2 = (host(hip, t).ravel() for t in hip.act_quant_fp8_x2(torch.from_numpy(x).to(hip.device)))
    o1, t1, o2, t2 = oracle.act_quant_fp8_x2(x)
    nan_blocks = np.isnan(x.reshape(-1, 32)).any(1)
    assert nan_blocks.sum() == 3
    assert np.array_equal(q1, o1) and np.array_equal(np.exp2(s1.astype(np.float64) - 127), t1.astype(np.float64))
    assert np.array_equal(q2.reshape(-1, 32)[~nan_blocks], o2.reshape(-1, 32)[~nan_blocks])
    assert np.array_equal(np.exp2(s2.astype(np.float64) - 127)[~nan_blocks], t2.astype(np.float64)[~nan_blocks])


def test_act_quant_at_the_top_of_the_f32_range(hip, oracle):
    """Block maxima from the last code below 2^128 to FLT_MAX.  From 248 * 2^120 on the code is 256 and code times scale is
    infinite in f32: the second term is then made from what an infinite product leaves over.  Its scale is infinite, as the
    oracle's, and its codes, which stand for nothing then, are all +-448."""
    amax = np.concatenate([np.array([0x7f000000, 0x7f600000, 0x7f600001, 0x7f700000, 0x7f77ffff, 0x7f780000, 0x7f780001, 0x7f7c0000,
                                     0x7f7fffff], np.uint32).view(np.float32), np.array([3.4e38, 3.3e38, 3.2e38], np.float32)])
    rng = np.random.default_rng(13)
    x = (rng.uniform(-1, 1, (2 * len(amax), 32)) * 2.0 ** rng.integers(90, 127, (2 * len(amax), 1))).astype(np.float32)
    x[: len(amax), 7], x[len(amax):, 30] = amax, -amax
    q1, s1, q2, s2 = (host(hip, t).ravel() for t in hip.act_quant_fp8_x2(torch.from_numpy(x).to(hip.device)))
    o1, t1, o2, t2 = oracle.act_quant_fp8_x2(x)
    assert np.array_equal(q1, o1) and np.array_equal(np.exp2(s1.astype(np.float64) - 127), t1.astype(np.float64))
    over = np.tile(amax >= np.float32(248.0 * 2.0 ** 120), 2)
    assert over.sum() == 12 and np.array_equal(np.isinf(t2), over)
    assert (s2[over] == 255).all() and np.array_equal(np.exp2(s2[~over].astype(np.float64) - 127), t2[~over].astype(np.float64))
    assert np.array_equal(q2.reshape(-1, 32)[~over], o2.reshape(-1, 32)[~over])
    assert ((q2.reshape(-1, 32)[over] & 0x7f) == 0x7e).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_mxfp4_quant_ties_and_special_values_vs_oracle(hip, oracle, dtype):
    """Values one ulp around every tie and code of the e2m1 grid at several block scales, signed zeros, quotients that
    underflow, and blocks with NaN or infinities (which take the general encoder): codes and scales as the oracle's."""
    rng = np.random.default_rng(12)
    grid = np.array([0, .25, .5, .75, 1, 1.25, 1.5, 1.75, 2, 2.5, 3, 3.5, 4, 5, 6], np.float32)
    near = np.concatenate([grid, np.nextafter(grid, np.float32(9)), np.nextafter(grid, np.float32(0))])
    near = np.concatenate([near, -near, np.array([-0.0, 1e-45, -1e-45], np.float32)])
    x = rng.choice(near, (96, 256)).astype(np.float32)
    x[:, ::32] = 6.0
    x *= np.repeat(2.0 ** rng.choice([-100.0, -20.0, 0.0, 3.0, 90.0], (96, 8)), 32, axis=1).astype(np.float32)
    x[90, :32] = 0.0
    x[91, 32:64], x[91, 32] = -1e-30, 3e38
    x[92, 5], x[93, 40], x[94, 64:96] = np.inf, -np.inf, np.inf
    xt = torch.from_numpy(x).to(dtype)
    codes, scales = hip.mxfp4_quant(xt.to(hip.device))
    want, s = oracle.act_quant_fp4(xt.float().numpy())
    assert np.array_equal(host(hip, codes).ravel(), want)
    finite = np.isfinite(s)
    assert (~finite).sum() == 3
    assert np.array_equal(np.exp2(host(hip, scales).ravel().astype(np.float64)[finite] - 127), s.astype(np.float64)[finite])
    assert (host(hip, scales).ravel()[~finite] == 255).all()


@pytest.mark.parametrize("hidden,inter,shared,experts", [(1152, 1408, 256, 3), (2048, 640, 0, 2)])
def test_pack_of_uneven_reductions_is_a_pure_permutation(hip, oracle, hidden, inter, shared, experts):
    """9, 11, 16 and 5 k steps: whole and cut chunks of a block, padded scale groups, whole-layer and per-expert packing."""
    inp = synth.make_inputs(synth.MoeConfig(4, hidden, experts, 2, inter, shared, 1, 1), seed=hidden)
    layer = hip.load_moe_layer(inp)
    whole = layer.packed.clone()
    for e in range(experts):
        pair = lambda m: (hip.upload(getattr(inp, m + "_w")[e]), hip.upload(getattr(inp, m + "_s")[e]))
        hip.pack_expert(layer, e, pair("gate"), pair("up"), pair("down"))
        for which, m in enumerate(("gate", "up", "down")):
            got = host(hip, hip.packed_dequant(layer, e, which))
            assert np.array_equal(got, oracle.dequant_fp4_row32(getattr(inp, m + "_w")[e], getattr(inp, m + "_s")[e])), (e, which)
    hip.sync()
    assert torch.equal(layer.packed, whole)


def test_pack_is_a_pure_permutation(hip, oracle):
    """dequant(packed) == dequant(checkpoint layout) for every matrix of several experts, bit for bit."""
    cfg = synth.MoeConfig(4, 256, 3, 2, 128, 256, 1, 1)
    inp = synth.make_inputs(cfg, seed=5)
    layer = hip.load_moe_layer(inp)
    for e in range(cfg.n_experts + 1):
        for which, (wn, sn) in enumerate([("gate", "gate"), ("up", "up"), ("down", "down")]):
            if e < cfg.n_experts:
                w, s = getattr(inp, f"{wn}_w")[e], getattr(inp, f"{sn}_s")[e]
            else:
                w, s = getattr(inp, f"sh_{wn}_w")[0], getattr(inp, f"sh_{sn}_s")[0]
            got = host(hip, hip.packed_dequant(layer, e, which))
            assert np.array_equal(got, oracle.dequant_fp4_row32(w, s)), (e, which)


# ---- the steps before and after the layer ----
@pytest.mark.parametrize("n,dim", [(1, 4), (11, 4096), (3, 517), (5, 7168), (2, 9000), (3, 520), (7, 1028), (1500, 256)])
def test_rmsnorm_bit_exact_vs_oracle(hip, oracle, n, dim):  # gpu_smoke.rs:56-70 shape [11, 4096] included
    rng = np.random.default_rng(n * 1000 + dim)
    x = (rng.standard_normal((n, dim)) * rng.uniform(1e-3, 30, (n, 1))).astype(np.float32)
    w = rng.uniform(0.5, 1.5, dim).astype(np.float32)
    if dim == 4:
        x[0] = [1., 2., 3., 4.]                       # golden.rs:30-42
    out = torch.empty(n, dim, device=hip.device)
    hip.rmsnorm(torch.from_numpy(x).to(hip.device), torch.from_numpy(w).to(hip.device), 1e-5, out)
    hip.sync()
    assert np.array_equal(out.cpu().numpy(), oracle.rmsnorm(x, w, 1e-5))


def test_rmsnorm_sequential_sum_and_errors(hip, oracle):
    from ferrite_amd.backend import InvalidArg
    row = np.full((1, 4097), 2.0 ** -13, np.float32)   # the left-to-right f32 sum drops every small square
    row[0, 0] = 1.0
    w = np.ones(4097, np.float32)
    out = torch.empty(1, 4097, device=hip.device)
    hip.rmsnorm(torch.from_numpy(row).to(hip.device), torch.from_numpy(w).to(hip.device), 0.0, out)
    hip.sync()
    assert np.array_equal(out.cpu().numpy(), oracle.rmsnorm(row, w, 0.0))
    with pytest.raises(InvalidArg):
        hip.rmsnorm(torch.zeros(2, 8, device=hip.device), torch.zeros(7, device=hip.device), 1e-5,
                    torch.zeros(2, 8, device=hip.device))


@pytest.mark.parametrize("s,nh,h", [(2, 4, 64), (32, 4, 4096), (5, 2, 12), (3, 8, 7168)])
def test_hc_post_bit_exact_vs_oracle(hip, oracle, s, nh, h):  # gpu_smoke.rs:308-348 shape (2, 4, 64) included
    rng = np.random.default_rng(s * 100 + nh)
    x = rng.standard_normal((s, h)).astype(np.float32)
    res = rng.standard_normal((s, nh, h)).astype(np.float32)
    post = rng.uniform(0, 2, (s, nh)).astype(np.float32)
    comb = rng.uniform(0, 1, (s, nh, nh)).astype(np.float32)
    if (s, nh, h) == (2, 4, 64):
        x = ((np.arange(s * h) * 7 % 31) * 0.03).astype(np.float32).reshape(s, h)
        res = ((np.arange(s * nh * h) * 13 % 47) * 0.02 - 0.5).astype(np.float32).reshape(s, nh, h)
    d = lambda a: torch.from_numpy(a).to(hip.device)
    out = hip.hc_post(d(x), d(res), d(post), d(comb))
    hip.sync()
    assert np.array_equal(out.cpu().numpy(), oracle.hc_post(x, res, post, comb))


def test_ops_in_a_capture_of_the_programs_own(hip):
    """torch.cuda.graph around calls that need no workspace: every replay gives what the eager calls give."""
    g = torch.Generator().manual_seed(5)
    x, w = (torch.randn(r, 256, generator=g).cuda() for r in (8, 48))
    norm, logits = torch.empty_like(x), torch.empty(8, 48, device="cuda")

    def calls():
        hip.rmsnorm(x, w[0], 1e-6, norm)
        hip.matmul(norm, w, None, logits)
        codes, scales = hip.mxfp4_quant(norm)
        return [norm, logits, codes, scales, hip.mxfp4_dequant(codes, scales), *hip.act_quant_fp8(norm),
                *hip.act_quant_fp8_x2(norm)]

    calls()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = calls()
    for _ in range(3):
        x.copy_(torch.randn(8, 256, generator=g))
        graph.replay()
        got = [t.clone() for t in captured]
        for a, b in zip(got, calls()):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
        torch.cuda.synchronize()


def test_hc_post_shape_errors(hip):
    from ferrite_amd.backend import Declined, ShapeMismatch
    z = lambda *sh: torch.zeros(*sh, device=hip.device)
    with pytest.raises(ShapeMismatch):
        hip.hc_post(z(2, 8), z(2, 4, 8), z(2, 3), z(2, 4, 4))
    with pytest.raises(Declined):
        hip.hc_post(z(2, 8), z(2, 9, 8), z(2, 9), z(2, 9, 9))     # more than 8 flows
