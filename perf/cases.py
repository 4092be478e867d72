"""The work a program has this library do, as cases that can be timed and checked.

A case is one call (or one token's calls down a stack of layers) through the
public entry points: `Layer.forward` / `Layer.forward_residual` on device
tensors, the host drop-in `qwen3_ffn`, and `Matrix.mat_mat`.  Shapes are those
of the repository's workload table (tie_amd.synth.CONFIGS): Qwen3-MoE 30B-A3B
and 235B-A22B, LFM2-8B-A1B, and the dense matrices around the block.

Weights are random GGUF blocks at the size of a trained layer's (about
N(0, 0.02)), made on the GPU from the seed: super-block scales
|N(0, s)| in f16, Q4_K sub-block scales and minimums over their 6 bits, Q6_K
sub-block scales over all of int8 (as quantisers emit them), codes uniform.
"""
import types

import torch

import tie_amd

F32, Q4_K, Q6_K, BF16 = tie_amd.F32, tie_amd.Q4_K, tie_amd.Q6_K, tie_amd.BF16
TYPES = {"f32": F32, "q4k": Q4_K, "q6k": Q6_K, "bf16": BF16}
PATHS = {"auto": tie_amd.PATH_AUTO, "exact": tie_amd.PATH_EXACT, "mfma": tie_amd.PATH_MFMA}
WEIGHT_BYTES = {"f32": 4.0, "q4k": 144 / 256, "q6k": 210 / 256, "bf16": 2.0}

SHAPES = {
    "30b": dict(d=2048, F=768, E=128, k=8, routing=0),
    "235b": dict(d=4096, F=1536, E=128, k=8, routing=0),
    "lfm2": dict(d=2048, F=1792, E=32, k=4, routing=1),
}
EPS = 1e-6
# up to here TIE_HIP_PATH_AUTO runs the block in TIE's own fp32 arithmetic
EXACT_TOKENS = 14


def moe(shape, T, gu="q4k", down="q6k", **kw):
    return dict(dict(kind="moe", shape=shape, T=T, gu=gu, down=down, layers=1, residual=False, topk=False,
                     zipf=False, host=False), **kw)


def dense(rows, inn, wtype, T, path="auto"):
    return dict(kind="dense", rows=rows, inn=inn, wtype=wtype, T=T, path=path)


def listed():
    return [
        # TIE's own call: one decoded token through one layer's FFN half, host
        # buffers in and out, the weights uploaded at the first call
        dict(moe("30b", 1, host=True, residual=True, topk=True), name="host_decode_30b"),
        # one decoded token down a stack of layers on the device (weights of
        # 8 layers, so that no call finds its experts in a cache)
        dict(moe("30b", 1, layers=8, residual=True), name="decode_30b_8_layers"),
        # a small decode batch, sigmoid routing: still in TIE's fp32 order
        dict(moe("lfm2", 8, topk=True), name="batch_lfm2_t8"),
        # the headline decode batch
        dict(moe("30b", 32), name="batch_30b_t32"),
        # an odd batch between decode and prefill, whole FFN half
        dict(moe("30b", 101, residual=True), name="batch_30b_t101_ffn"),
        # a prompt of ordinary length
        dict(moe("30b", 500), name="prefill_30b_t500"),
        # a long prompt's chunk
        dict(moe("30b", 2048), name="prefill_30b_t2048"),
        # the large model's chunk: the largest of the list
        dict(moe("235b", 1024), name="prefill_235b_t1024"),
        # unquantised experts, unevenly loaded
        dict(moe("30b", 512, gu="bf16", down="bf16", zipf=True), name="prefill_bf16_zipf_t512"),
        # the LM head of one decoded token
        dict(dense(151936, 2048, "q6k", 1), name="lm_head_q6k_t1"),
        # a query projection of a decode batch, in TIE's fp32 order
        dict(dense(4096, 2048, "q4k", 32), name="dense_q4k_t32"),
        # the same projection of a prompt, matrix cores asked for
        dict(dense(4096, 2048, "q4k", 509, path="mfma"), name="dense_q4k_t509_mfma"),
    ]


def _spread(rng, lo, hi):
    """A whole number spread over [lo, hi] in its logarithm."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    if rng.random() < 0.25:
        wtype = rng.choice(["q4k", "q4k", "q6k", "q6k", "bf16", "f32"])
        path = "mfma" if wtype in ("q4k", "q6k") and rng.random() < 0.5 else "auto"
        unit = 256 if path == "mfma" else 64
        rows = unit * _spread(rng, 512 // unit, 8192 // unit)
        inn = 256 * _spread(rng, 4, 24)
        most = (32 << 30) if path == "mfma" else (1 << 30)  # multiply-adds of one call
        return dense(rows, inn, wtype, _spread(rng, 1, max(1, min(2048 if path == "mfma" else 256, most // (rows * inn)))), path)
    shape = rng.choice(["30b", "30b", "30b", "lfm2", "235b"])
    gu, down = rng.choice([("q4k", "q6k"), ("q4k", "q6k"), ("q4k", "q4k"), ("q6k", "q6k"), ("bf16", "bf16")])
    if shape == "235b":
        gu, down = "q4k", rng.choice(["q4k", "q6k"])
    T = _spread(rng, 1, 1000 if shape == "235b" else 2048)
    if gu == "bf16":
        T = min(T, 700)
    return moe(shape, T, gu, down, layers=8 if T == 1 else 1, residual=rng.random() < 0.4, topk=rng.random() < 0.3,
               zipf=shape != "lfm2" and rng.random() < 0.25)


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, std, *shape):
    return torch.randn(*shape, generator=g, device="cuda") * std


def _tensor(g, wtype, n_mat, rows, inn, std):
    """[n_mat][rows][inn] weights of about N(0, std) in GGUF layout, as bytes on the GPU."""
    if wtype == "f32":
        return _normal(g, std, n_mat * rows, inn).view(torch.uint8).reshape(-1)
    if wtype == "bf16":
        return torch.cat([_normal(g, std, rows, inn).bfloat16().view(torch.uint8).reshape(-1) for _ in range(n_mat)])
    n, size = n_mat * rows * (inn // 256), 144 if wtype == "q4k" else 210
    b = torch.empty(n * size, dtype=torch.uint8, device="cuda")
    whole = n * size // 8
    b[: whole * 8].view(torch.int64).random_(-(1 << 63), None, generator=g)
    b[whole * 8:] = 0
    b = b.view(n, size)

    def scales(s):
        return _normal(g, s, n).abs_().half().view(torch.uint8).view(n, 2)

    if wtype == "q4k":
        # codes 0..15 about 7.5 times scales 0..63, minus minimums 0..63
        b[:, 0:2] = scales(std / 350)
        b[:, 2:4] = scales(std / 50)
    else:
        # codes -32..31 times scales -128..127
        b[:, 208:210] = scales(std / 1350)
    return b.view(-1)


def _weights(case, seed):
    s = SHAPES[case["shape"]]
    d, F, E = s["d"], s["F"], s["E"]
    g = _gen(seed)
    w = dict(router=_normal(g, 0.02, E, d), gate=_tensor(g, case["gu"], E, F, d, 0.02),
             up=_tensor(g, case["gu"], E, F, d, 0.02), down=_tensor(g, case["down"], E, d, F, 0.02), bias=None,
             pbias=_normal(g, 0.05, E) if s["routing"] else None, norm=1.0 + _normal(g, 0.1, d))
    if case["zipf"]:  # a few experts wanted by most tokens
        rank = torch.randperm(E, generator=g, device="cuda").double() + 1.0
        w["bias"] = rank.pow(-1.2).float()
    return w


def _input(case, seed):
    d = SHAPES[case["shape"]]["d"]
    # a normalised activation, or (before the norm) a hidden state
    return _normal(_gen(seed + 1), 2.0 if case["residual"] else 1.0, case["T"], d)


def _dense_inputs(case, seed):
    g = _gen(seed)
    return _tensor(g, case["wtype"], 1, case["rows"], case["inn"], 0.02), _normal(g, 1.0, case["T"], case["inn"])


# the host program's model: mapped once, valid and unchanged while the
# process lives, as the drop-in asks
_MAPPED = {}


def _mapped(case):
    key = (case["shape"], case["gu"], case["down"])
    if key not in _MAPPED:
        s = SHAPES[case["shape"]]
        w = {k: v.cpu().numpy() if v is not None else None for k, v in _weights(case, 77).items()}
        layer = types.SimpleNamespace(d=s["d"], F=s["F"], E=s["E"], router=w["router"], gate=w["gate"], up=w["up"],
                                      down=w["down"], gate_type=TYPES[case["gu"]], up_type=TYPES[case["gu"]],
                                      down_type=TYPES[case["down"]], bias=None, routing=s["routing"], probs_bias=w["pbias"])
        _MAPPED[key] = (layer, w["norm"])
    return _MAPPED[key]


def prepare(case, seed):
    tie_amd.init(0)
    if case["kind"] == "dense":
        w, x = _dense_inputs(case, seed)
        m = tie_amd.Matrix(w, TYPES[case["wtype"]], case["rows"], case["inn"], on_device=True)
        return dict(case=case, matrix=m, x=x, out=torch.zeros(case["T"], case["rows"], device="cuda"))
    s = SHAPES[case["shape"]]
    if case["host"]:
        layer, norm = _mapped(case)
        x = _input(case, seed).cpu().numpy()
        tie_amd.qwen3_ffn(x, layer, s["k"], norm, EPS)  # the model's upload
        return dict(case=case, layer=layer, norm=norm, x=x, k=s["k"])
    layers, norms = [], []
    for n in range(case["layers"]):
        w = _weights(case, seed * 64 + n)
        layers.append(tie_amd.Layer(s["d"], s["F"], s["E"], w["router"], w["gate"], w["up"], w["down"],
                                    TYPES[case["gu"]], TYPES[case["gu"]], TYPES[case["down"]], bias=w["bias"],
                                    on_device=True, routing=s["routing"], probs_bias=w["pbias"]))
        norms.append(w["norm"])
    T = case["T"]
    st = dict(case=case, layers=layers, norms=norms, x=_input(case, seed), k=s["k"], idx=None, w=None)
    # the hidden state goes down the stack in place; without the residual each
    # layer has its own output
    st["out"] = [torch.zeros(T, s["d"], device="cuda") for _ in range(1 if case["residual"] else case["layers"])]
    if case["topk"]:
        st["idx"] = [torch.zeros(T, s["k"], dtype=torch.int32, device="cuda") for _ in layers]
        st["w"] = [torch.zeros(T, s["k"], device="cuda") for _ in layers]
    return st


def run(state):
    case = state["case"]
    if case["kind"] == "dense":
        state["matrix"].mat_mat(state["x"], case["T"], state["out"], flags=PATHS[case["path"]])
        return state["out"]
    if case["host"]:
        return tie_amd.qwen3_ffn(state["x"], state["layer"], state["k"], state["norm"], EPS)
    T, k, out = case["T"], state["k"], state["out"]
    hidden = state["x"]
    for n, layer in enumerate(state["layers"]):
        idx = state["idx"][n] if state["idx"] else None
        w = state["w"][n] if state["w"] else None
        if case["residual"]:
            layer.forward_residual(hidden, state["norms"][n], EPS, T, k, out[0], idx, w)
            hidden = out[0]
        else:
            layer.forward(state["x"], T, k, out[n], idx, w)
    return dict(out=out, idx=state["idx"], w=state["w"])


# ---------------------------------------------------------------- the least work
def work(case):
    if case["kind"] == "dense":
        rows, inn, T = case["rows"], case["inn"], case["T"]
        return {"bytes": rows * inn * WEIGHT_BYTES[case["wtype"]] + 4.0 * T * (rows + inn), "flops": 2.0 * rows * inn * T}
    s = SHAPES[case["shape"]]
    d, F, E, k, T = s["d"], s["F"], s["E"], s["k"], case["T"]
    used = E * (1.0 - (1.0 - k / E) ** T)  # experts that T tokens' choices reach
    weights = used * d * F * (2 * WEIGHT_BYTES[case["gu"]] + WEIGHT_BYTES[case["down"]])
    return {"bytes": case["layers"] * (weights + 4.0 * E * d + 8.0 * T * d),
            "flops": case["layers"] * (6.0 * T * k * d * F + 2.0 * T * E * d)}


def tolerance(case):
    """Four times the error against 64 bits that was measured: 32-bit sums 1e-7
    to 9e-7, f16 operands with 32-bit sums 3.4e-4 (one product) and 6.2e-4
    (the block), bf16 weights with split activations 4.4e-6."""
    if case["kind"] == "dense":
        return {"rel": 1.4e-3} if case["path"] == "mfma" else {"rel": 4e-6}
    if case["T"] <= EXACT_TOKENS:
        return {"rel": 4e-6}
    return {"rel": 2e-5} if case["gu"] == "bf16" else {"rel": 2.5e-3}


# ---------------------------------------------------------------- 64 bits
def _dequant(buf, wtype, rows, inn):
    """One matrix's weights in float64 (block layouts: gguf.h:100-113)."""
    if wtype == "f32":
        return buf.view(torch.float32).view(rows, inn).double()
    if wtype == "bf16":
        return buf.view(torch.bfloat16).view(rows, inn).double()

    def half(b):
        return b.contiguous().view(torch.float16).double()

    if wtype == "q4k":
        b = buf.view(-1, 144)
        d, dmin, s, q = half(b[:, 0:2]), half(b[:, 2:4]), b[:, 4:16].int(), b[:, 16:].reshape(-1, 4, 32)
        lo, hi, top = s[:, 0:4], s[:, 4:8], s[:, 8:12]
        sc = torch.cat([lo & 63, (top & 15) | (lo >> 6 << 4)], 1).double()
        mn = torch.cat([hi & 63, (top >> 4) | (hi >> 6 << 4)], 1).double()
        codes = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        return ((d * sc)[:, :, None] * codes - (dmin * mn)[:, :, None]).view(rows, inn)
    b = buf.view(-1, 210)
    ql, qh = b[:, 0:128].int().view(-1, 2, 2, 32), b[:, 128:192].int().view(-1, 2, 32)
    sc, d = b[:, 192:208].contiguous().view(torch.int8).double(), half(b[:, 208:210])
    codes = torch.stack([(ql[:, :, i % 2] >> 4 * (i // 2) & 15) | ((qh >> 2 * i & 3) << 4) for i in range(4)], 2)
    return ((codes.reshape(-1, 16, 16) - 32).double() * (d * sc)[:, :, None]).view(rows, inn)


def _silu_nodes():
    """The 8192 nodes of TIE's SiLU table over [-10, 10] (engine.c:204-225,
    297-303): e^-x starts from its bit-pattern estimate, which the polynomial
    does not undo for large |x|, so the table is not the SiLU itself."""
    x = torch.arange(8192, dtype=torch.float64) * (20.0 / 8191.0) - 10.0
    u = (torch.clamp(-x, -88.37626266479492, 88.37626266479492) * 12102203.0 + 1065353216.0).float().int().view(torch.float32).double()
    p = (1.9875691500e-4 * u + 1.3981999507e-3) * u
    p = p * p + (8.3334519073e-3 * p + 4.1665795894e-2) * p
    p = p * p + (1.6666665459e-1 * p + 5.0000001201e-1) * p
    return (x / (1.0 + u + u * p)).cuda()


def _swiglu(g, u, nodes):
    pos = (g + 10.0) * (8191.0 / 20.0)
    i = pos.round().clamp(0, 8190).long()
    return (nodes[i] + (pos - i) * (nodes[i + 1] - nodes[i])) * u


def _block(case, w, x):
    s = SHAPES[case["shape"]]
    d, F, E, k = s["d"], s["F"], s["E"], s["k"]
    logits = x @ w["router"].double().T
    if w["bias"] is not None:
        logits = logits + w["bias"].double()
    if s["routing"]:
        p = torch.sigmoid(logits)
        idx = (p + w["pbias"].double()).topk(k).indices
        gate = p.gather(1, idx)
        gate = gate / (gate.sum(1, keepdim=True) + 1e-6)
    else:
        best = logits.topk(k)
        idx, gate = best.indices, best.values.softmax(1)
    out, nodes = torch.zeros_like(x), _silu_nodes()
    mats = {n: w[n].view(torch.uint8).view(E, -1) for n in ("gate", "up", "down")}
    for e in idx.unique().tolist():
        t, j = (idx == e).nonzero(as_tuple=True)
        h = _swiglu(x[t] @ _dequant(mats["gate"][e], case["gu"], F, d).T, x[t] @ _dequant(mats["up"][e], case["gu"], F, d).T, nodes)
        out.index_add_(0, t, gate[t, j, None] * (h @ _dequant(mats["down"][e], case["down"], d, F).T))
    return out, idx.int(), gate


def exact(case, seed):
    if case["kind"] == "dense":
        w, x = _dense_inputs(case, seed)
        return x.double() @ _dequant(w, case["wtype"], case["rows"], case["inn"]).T
    x = _input(case, seed).double()
    outs, idxs, ws = [], [], []
    for n in range(case["layers"]):
        w = _weights(case, 77 if case["host"] else seed * 64 + n)
        z = x
        if case["residual"]:
            z = x / (x.square().mean(1, keepdim=True) + EPS).sqrt() * w["norm"].double()
        out, idx, gate = _block(case, w, z)
        if case["residual"]:
            x = out = x + out
        outs.append(out)
        idxs.append(idx)
        ws.append(gate)
    if case["host"]:
        return outs[0], idxs[0], ws[0]
    return dict(out=outs[-1:] if case["residual"] else outs, idx=idxs if case["topk"] else None, w=ws if case["topk"] else None)
