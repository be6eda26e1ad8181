"""The work that a user of this framework has it do, as cases that can be timed and compared.

Every case goes through the public entry points of ferrite_amd.backend: the MoE FFN layer alone, the rmsnorm -> layer ->
hc_post block, a captured decode step of several layers, the layer at sizes that the matrix-core modes decline, the ops
that an engine calls one by one, and the ingest of an unquantised checkpoint.  Sizes are those of synth.CONFIGS (decode
at 32 and 192 tokens, a 4096-token prefill chunk, 8192 skewed tokens of a larger model) and generic ones between and
beside them.

Fields of a case: kind; n tokens; hidden, experts, topk, inter, shared (intermediate size of the shared expert, 0 = none),
n_group, topk_group; mode (fp8 = one e4m3 term per activation, fp8x2 = two); dtype of x and of the output; zipf (> 0: expert
popularity skewed by the correction bias); layers of a step / experts of an ingest; hc (hyper-connection streams, 0 = none).
"""
import ctypes
import functools
import math

import torch

from ferrite_amd import backend, synth

MODES = {"fp8": backend.MODE_MFMA_FP8, "fp8x2": backend.MODE_MFMA_FP8_X2}
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
EPS = 1e-6


def _case(name, kind, n, hidden, experts, topk, inter, shared, n_group=1, topk_group=1, mode="fp8x2", dtype="bf16", zipf=0.0, layers=1,
          hc=0):
    c = dict(kind=kind, n=n, hidden=hidden, experts=experts, topk=topk, inter=inter, shared=shared, n_group=n_group,
             topk_group=topk_group, mode=mode, dtype=dtype, zipf=zipf, layers=layers, hc=hc)
    return dict(c, name=name) if name else c


def listed():
    flash = (4096, 128, 8, 1536, 1536, 8, 4)   # the decode / prefill shape of synth.CONFIGS: H, E, k, I, shared, groups
    return [
        # the smallest configuration (synth c0), one eager call: latency, launches and the host path
        _case("layer_tiny_8", "layer", 8, 256, 16, 4, 128, 128, 4, 2, mode="fp8", dtype="f32"),
        # a single user's decode: four layers of the captured step, each with its own weights, one token
        _case("step_1", "step", 1, *flash, dtype="f32", layers=4),
        # decode at 32 tokens (c1), one eager layer call in the bf16-class activation format
        _case("layer_32", "layer", 32, *flash),
        # an odd decode batch through the whole FFN half of a decoder layer, in the one-term serving format
        _case("block_57", "block", 57, *flash, mode="fp8", dtype="f32", hc=4),
        # decode with multi-token prediction (c4, 64 x 3 tokens): three layers of the captured step
        _case("step_192", "step", 192, *flash, dtype="f32", layers=3),
        # decode batches and prompts mixed in one call, ragged: between the decode and the prefill sizes
        _case("layer_509", "layer", 509, *flash),
        # a prefill chunk in the bf16-class format with the hyper-connection update behind it
        _case("block_2047", "block", 2047, *flash, dtype="f32", hc=4),
        # the prefill chunk of c2 in the one-term serving format
        _case("layer_4096", "layer", 4096, *flash, mode="fp8"),
        # the largest prefill (c3): a bigger model, 256 experts, popularity skewed
        _case("layer_8192_skew", "layer", 8192, 7168, 256, 8, 2048, 2048, 8, 4, mode="fp8", zipf=1.1),
        # a model whose sizes are no multiples of 128: the call falls back to f32 activations
        _case("fallback_27", "layer", 27, 2080, 32, 6, 736, 736, dtype="f32"),
        # an engine that calls the ops one by one: norm, router, routing, permutation, the shared expert in f32, hc_post
        _case("ops_100", "ops", 100, *flash, dtype="f32", hc=4),
        # loading an unquantised checkpoint: bf16 experts to MXFP4 and into the packed layout
        _case("ingest_4", "ingest", 1, 4096, 4, 1, 1536, 0, layers=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        c = _draw(rng)
        # no dearer than the largest listed case: expert FLOPs (twice with two terms) and weight bytes
        terms = 2 if c["mode"] == "fp8x2" and c["kind"] != "ingest" else 1
        if work(c)["flops"] * terms <= 6.5e12 and c["experts"] * c["hidden"] * c["inter"] <= 256 * 7168 * 2048:
            return c


def _draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "block", "block", "step", "fallback", "ops", "ingest"])
    hidden = rng.choice([2048, 2560, 4096, 5120, 7168])
    inter = rng.choice([512, 768, 1024, 1408, 1536, 2048])
    experts = rng.choice([32, 64, 96, 128, 160, 256])
    topk = rng.choice([4, 6, 8])
    n_group, topk_group = rng.choice([(1, 1), (8, 4), (4, 2)])
    shared = rng.choice([inter, inter, 0])
    mode = rng.choice(["fp8", "fp8x2"])
    if kind == "layer":
        return _case(None, "layer", _log(rng, 1, 8192), hidden, experts, topk, inter, shared, n_group, topk_group, mode,
                     rng.choice(["bf16", "f32"]), rng.choice([0.0, 0.0, 1.1]))
    if kind == "block":
        return _case(None, "block", _log(rng, 1, 4096), hidden, experts, topk, inter, shared, n_group, topk_group, mode, "f32",
                     hc=rng.choice([2, 4]))
    if kind == "step":
        return _case(None, "step", _log(rng, 1, 256), hidden, min(experts, 128), topk, inter, shared, n_group, topk_group, mode, "f32",
                     layers=rng.randint(2, 4))
    if kind == "fallback":
        return _case(None, "layer", _log(rng, 1, 64), 32 * rng.choice([45, 65, 90]), min(experts, 64), topk,
                     32 * rng.choice([15, 23, 33]), rng.choice([736, 0]), 1, 1, mode, "f32")
    if kind == "ops":
        return _case(None, "ops", _log(rng, 1, 256), hidden, experts, topk, inter, inter, n_group, topk_group, mode, "f32",
                     hc=rng.choice([2, 4]))
    k = rng.randint(1, 8)
    return _case(None, "ingest", 1, hidden, k, 1, inter, 0, dtype=rng.choice(["bf16", "f32"]), layers=k)


@functools.lru_cache(maxsize=None)
def _hip():
    return backend.HipBackend()   # one per program: the library handle and its stream


def _config(c):
    return synth.MoeConfig(c["n"], c["hidden"], c["experts"], c["topk"], c["inter"], c["shared"], c["n_group"], c["topk_group"],
                           act_bf16=c["dtype"] == "bf16", bias_zipf=c["zipf"])


def _tensors(hip, c, g):
    """A layer's weights in the checkpoint layout: MXFP4 codes and scales made on the device."""
    cfg = _config(c)
    E, H, I, S = cfg.n_experts, cfg.hidden, cfg.inter, cfg.shared_inter
    dev = hip.device

    def codes(*shape):
        return torch.randint(0, 256, shape, dtype=torch.uint8, device=dev, generator=g)

    def scales(*shape):
        return torch.randint(119, 121, shape, dtype=torch.uint8, device=dev, generator=g)

    t = dict(router_w=torch.randn(E, H, device=dev, generator=g) * 0.02)
    if cfg.bias_zipf > 0:
        t["router_bias"] = hip.upload(synth.zipf_bias(int(torch.randint(0, 1 << 30, (1,), device=dev, generator=g)), E, cfg.bias_zipf))
    else:
        t["router_bias"] = torch.randn(E, device=dev, generator=g) * 0.01
    for key in ("gate", "up"):
        t[key + "_w"], t[key + "_s"] = codes(E, I, H // 2), scales(E, I, H // 32)
        if S:
            t["sh_" + key + "_w"], t["sh_" + key + "_s"] = codes(1, S, H // 2), scales(1, S, H // 32)
    t["down_w"], t["down_s"] = codes(E, H, I // 2), scales(E, H, I // 32)
    if S:
        t["sh_down_w"], t["sh_down_s"] = codes(1, H, S // 2), scales(1, H, S // 32)
    return t


def _layer(hip, c, g):
    """The layer as a loader leaves it: packed where the matrix-core modes take the shape, in the checkpoint layout
    where they do not."""
    cfg, t, dev = _config(c), _tensors(hip, c, g), hip.device
    layer = backend.MoeLayer(cfg, t, None)
    nbytes = hip.lib.ferrite_moe_packed_bytes(ctypes.byref(layer.shape))
    if nbytes == 0:
        return layer
    layer.packed = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    torch.cuda.synchronize()
    rc = hip.lib.ferrite_moe_pack_weights(ctypes.byref(layer.shape), ctypes.byref(layer.weights), layer.packed.data_ptr(),
                                          hip.stream.cuda_stream)
    if rc:
        raise RuntimeError("pack_weights: %d" % rc)
    hip.sync()
    keep = {k: t[k] for k in ("router_w", "router_bias")}
    packed, layer = layer.packed, backend.MoeLayer(cfg, keep, None)
    layer.packed = packed
    return layer


class _State:
    """What the program keeps between calls; a captured graph is destroyed with it."""

    def __init__(self, hip, case):
        self.hip, self.case, self.mode, self.trace = hip, case, MODES[case["mode"]], None

    def __del__(self):
        if self.trace is not None:
            self.hip.graph_destroy(self.trace)


def _streams(c, g, dev, s):
    n, H, nh = c["n"], c["hidden"], c["hc"]
    s.norm_w = torch.rand(H, device=dev, generator=g) + 0.5
    s.residual = torch.randn(n, nh, H, device=dev, generator=g)
    s.post = torch.rand(n, nh, device=dev, generator=g) * 2.0
    s.comb = torch.softmax(torch.randn(n, nh, nh, device=dev, generator=g), dim=-1).contiguous()


def _step(s):
    for layer, x, norm_w, out in zip(s.layers, s.x, s.norm_ws, s.out):
        s.hip.moe_block_mxfp4(layer, x, norm_w, EPS, None, None, None, out, s.mode, workspace=s.ws)


def prepare(case, seed):
    hip = _hip()
    dev = hip.device
    g = torch.Generator(device=dev).manual_seed(seed)
    s = _State(hip, case)
    n, H, kind = case["n"], case["hidden"], case["kind"]
    dt = DTYPES[case["dtype"]]
    if kind == "ingest":
        I, E = case["inter"], case["layers"]
        s.layer = backend.MoeLayer(_config(case), {}, None)
        s.layer.packed = torch.zeros(hip.lib.ferrite_moe_packed_bytes(ctypes.byref(s.layer.shape)), dtype=torch.uint8, device=dev)
        mk = lambda rows, cols: (torch.randn(rows, cols, device=dev, generator=g) * 0.02).to(dt)
        s.experts = [(mk(I, H), mk(I, H), mk(H, I)) for _ in range(E)]
        return s
    s.x = torch.randn(n, H, device=dev, generator=g).to(dt)
    if kind == "ops":
        E, I, k = case["experts"], case["inter"], case["topk"]
        mk = lambda *shape: torch.randn(*shape, device=dev, generator=g) * 0.02
        s.router_w, s.bias, s.gate_up_w, s.down_w = mk(E, H), mk(E) * 0.5, mk(2 * I, H), mk(H, I)
        _streams(case, g, dev, s)
        new = lambda *shape: torch.empty(*shape, device=dev)
        s.h, s.logits, s.probs, s.ids = new(n, H), new(n, E), new(n, k), new(n, k)
        s.ids_i32 = torch.empty(n, k, dtype=torch.int32, device=dev)
        s.gate_up, s.act, s.ffn = new(n, 2 * I), new(n, I), new(n, H)
        return s
    if kind == "step":
        s.layers = [_layer(hip, case, g) for _ in range(case["layers"])]
        s.norm_ws = [torch.rand(H, device=dev, generator=g) + 0.5 for _ in s.layers]
        # every layer reads a stream of its own (what the attention in front of it leaves): an input that followed from
        # the layer before would turn a rounding difference into another choice of experts
        s.x = torch.randn(case["layers"], n, H, device=dev, generator=g)
        s.out = torch.empty_like(s.x)
        s.ws = hip.block_workspace(s.layers[0], n, s.mode)
        _step(s)
        hip.sync()
        hip.begin_capture()
        _step(s)
        s.trace = hip.end_capture()
        return s
    s.layer = _layer(hip, case, g)
    if kind == "block":
        _streams(case, g, dev, s)
        s.out = torch.empty(n, case["hc"], H, device=dev)
        s.ws = hip.block_workspace(s.layer, n, s.mode)
    else:
        s.out = torch.empty(n, H, dtype=dt, device=dev)
        s.ws = hip.workspace(s.layer, n, s.mode)
    return s


def run(s):
    hip, c, kind = s.hip, s.case, s.case["kind"]
    if kind == "layer":
        hip.moe_layer_dev_mxfp4(s.layer, s.x, s.out, s.mode, s.ws)
        return s.out
    if kind == "block":
        hip.moe_block_mxfp4(s.layer, s.x, s.norm_w, EPS, s.residual, s.post, s.comb, s.out, s.mode, workspace=s.ws)
        return s.out
    if kind == "step":
        hip.begin_verify(s.trace)   # replays the captured step
        return s.out
    if kind == "ops":
        hip.rmsnorm(s.x, s.norm_w, EPS, s.h)
        hip.matmul(s.h, s.router_w, None, s.logits)
        hip.moe_route(s.logits, s.bias, c["topk"], 2.5, s.probs, s.ids, c["n_group"], c["topk_group"], s.ids_i32)
        tables = hip.moe_permute(s.ids_i32, c["experts"])
        hip.matmul(s.h, s.gate_up_w, None, s.gate_up)
        hip.swiglu_limited(s.gate_up, 10.0, s.act)
        hip.matmul(s.act, s.down_w, None, s.ffn)
        out = hip.hc_post(s.ffn, s.residual, s.post, s.comb)
        return [out, s.logits, s.probs, s.ids_i32, tables]
    for e, mats in enumerate(s.experts):
        gate, up, down = (hip.mxfp4_quant(m) for m in mats)
        hip.pack_expert(s.layer, e, gate, up, down)
    return s.layer.packed


def work(case):
    n, H, E, k, I, S = (case[f] for f in ("n", "hidden", "experts", "topk", "inter", "shared"))
    kind, size = case["kind"], 2 if case["dtype"] == "bf16" else 4
    mxfp4 = 0.5 + 1.0 / 32
    if kind == "ingest":
        return {"bytes": case["layers"] * 3 * H * I * (size + mxfp4), "flops": 0}
    if kind == "ops":
        nh = case["hc"]
        bytes_ = 4 * (n * H + E * H + 3 * H * I + n * nh * H * 2 + n * E) + 8 * n * k * 4
        return {"bytes": bytes_, "flops": 2 * n * H * (E + 3 * I)}
    hit = E * (1.0 - (1.0 - k / E) ** n)   # experts that at least one token picks
    weights = (hit * I + S) * 3 * H * mxfp4 + E * H * 4
    tokens = n * H * size * 2
    if kind == "block":
        tokens = n * H * 4 * (1 + 2 * case["hc"])
    if kind == "step":
        return {"bytes": case["layers"] * (weights + tokens), "flops": case["layers"] * 2 * n * H * (3 * (k * I + S) + E)}
    return {"bytes": weights + tokens, "flops": 2 * n * H * (3 * (k * I + S) + E)}


def tolerance(case):
    # the ops and the ingest are bit-exact restatements of the reference's arithmetic
    if case["kind"] in ("ops", "ingest"):
        return "exact"
    # four times what the layer shows against the same arithmetic with its sums in 64 bits (max: of single values)
    if any(case[f] % 128 for f in ("hidden", "inter", "shared")):
        return {"rel": 2e-6, "max": 8e-6}   # f32 activations throughout: 2.1e-7, 8.9e-7
    decode = case["n"] * case["topk"] < 16 * case["experts"]   # expert outputs in f32; in bf16 for larger batches
    if case["mode"] == "fp8x2" and case["dtype"] == "f32" and decode:
        return {"rel": 4e-4, "max": 3e-3}   # 8.1e-5, 7.0e-4
    if case["mode"] == "fp8x2":
        return {"rel": 1e-2, "max": 6e-2}   # bf16 outputs or expert outputs: 2.6e-3, 1.5e-2
    return {"rel": 1e-2, "max": 1.5e-1}     # an e4m3 code of three mantissa bits that falls to its neighbour: 2.6e-3, 3.5e-2


def _values(codes, scales):
    """MXFP4 codes (low nibble = even column) and e8m0 scales of one matrix as 64-bit values."""
    mags = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]
    table = torch.tensor(mags + [-m for m in mags], dtype=torch.float64, device=codes.device)
    v = torch.stack([table[(codes & 15).long()], table[(codes >> 4).long()]], dim=-1).reshape(codes.shape[0], -1, 32)
    return (v * torch.exp2(scales.double() - 127.0).unsqueeze(-1)).reshape(codes.shape[0], -1)


def _swiglu64(gate, up, limit):
    gate, up = gate.clamp(max=limit), up.clamp(-limit, limit)
    return gate * torch.sigmoid(gate) * up


def _norm64(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _route64(logits, bias, topk, n_group, topk_group, scaling):
    sig = torch.sigmoid(logits)
    choice = sig + bias.double()
    if n_group > 1 and topk_group < n_group:
        groups = choice.reshape(choice.shape[0], n_group, -1)
        score = groups.topk(min(2, groups.shape[-1]), -1).values.sum(-1)
        keep = torch.zeros_like(score).scatter_(1, score.topk(topk_group, -1).indices, 1.0) > 0
        choice = torch.where(keep.unsqueeze(-1), groups, -math.inf).reshape(choice.shape)
    ids = choice.topk(topk, -1).indices
    w = sig.gather(1, ids)
    return ids, w / (w.sum(-1, keepdim=True) + 2.0 ** -23) * scaling


def _ffn64(cfg, t, x):
    """The layer on x [n, H] with nothing quantised but its weights."""
    ids, w = _route64(x @ t["router_w"].double().T, t["router_bias"], cfg.topk, cfg.n_group, cfg.topk_group, cfg.routed_scaling)

    def expert(prefix, e, rows):
        gate, up, down = (_values(t[prefix + m + "_w"][e], t[prefix + m + "_s"][e]) for m in ("gate", "up", "down"))
        return _swiglu64(rows @ gate.T, rows @ up.T, cfg.swiglu_limit) @ down.T

    out = expert("sh_", 0, x) if cfg.shared_inter else torch.zeros_like(x)
    for e in range(cfg.n_experts):
        tok, slot = (ids == e).nonzero(as_tuple=True)
        if len(tok):
            out.index_add_(0, tok, expert("", e, x[tok]) * w[tok, slot].unsqueeze(-1))
    return out


def _hc_post64(x, s):
    return s.post.double().unsqueeze(-1) * x.unsqueeze(1) + s.comb.double().transpose(1, 2) @ s.residual.double()


def exact(case, seed):
    """What run() returns, in 64 bits.  The engine's ids and tables and an ingest's bytes are whole numbers: none here."""
    kind, n, H = case["kind"], case["n"], case["hidden"]
    if kind == "ingest":
        return None
    hip = _hip()
    g = torch.Generator(device=hip.device).manual_seed(seed)
    if kind == "ops":
        s = prepare(case, seed)
        h = _norm64(s.x.double(), s.norm_w)
        logits = h @ s.router_w.double().T
        probs = _route64(logits, s.bias, case["topk"], case["n_group"], case["topk_group"], 2.5)[1]
        gate, up = (h @ s.gate_up_w.double().T).chunk(2, -1)
        out = _hc_post64(_swiglu64(gate, up, 10.0) @ s.down_w.double().T, s)
        return [out, logits, probs, None, None]
    x = torch.randn(n, H, device=hip.device, generator=g).to(DTYPES[case["dtype"]]).double()
    if kind == "step":
        weights = [_tensors(hip, case, g) for _ in range(case["layers"])]
        norm_ws = [torch.rand(H, device=hip.device, generator=g) + 0.5 for _ in weights]
        xs = torch.randn(case["layers"], n, H, device=hip.device, generator=g)
        return torch.stack([_ffn64(_config(case), t, _norm64(xl.double(), w)) for t, w, xl in zip(weights, norm_ws, xs)])
    t = _tensors(hip, case, g)
    if kind == "layer":
        return _ffn64(_config(case), t, x)
    s = _State(hip, case)
    _streams(case, g, hip.device, s)
    return _hc_post64(_ffn64(_config(case), t, _norm64(x, s.norm_w)), s)
