"""The work whose speed counts: calls of the MoE layer as an engine makes them, with their inputs, results and limits.

Every case is one of three kinds of program:

* "graph": a decode step. The engine holds several layers, each with its own weights at its own addresses and its own
  activations (attention runs between them), and replays one captured graph of their forwards.
* "eager": a prompt block. One asynchronous ``MoeLayer.forward`` on device buffers.
* "host": the drop-in ``Gpu.moe`` on host bytes: the selected experts of one token, read from a model file.

Weights are N(0, 0.02) in GGUF blocks, activations N(0, 1), routers N(0, 0.02), as everywhere in this repository.
"""
import math
from types import SimpleNamespace

import numpy as np
import torch

from ingot_amd import configs as CF
from ingot_amd import moe as M

FORMATS = {"Q4_K": M.Q4_K, "Q6_K": M.Q6_K, "Q8_0": M.Q8_0, "IQ2_XS": M.IQ2_XS, "IQ3_XXS": M.IQ3_XXS, "IQ4_NL": M.IQ4_NL}
# bits per weight, and the columns a block holds
BITS = {"Q4_K": 4.5, "Q6_K": 6.5625, "Q8_0": 8.5, "IQ2_XS": 2.3125, "IQ3_XXS": 3.0625, "IQ4_NL": 4.5}
SIGMA = 0.02
EXTRA_ROWS = 512

# The layers of the benchmark configurations: a Qwen3-30B-A3B shape, one with 512 narrow experts and a gated shared
# expert, and a GLM shape with sigmoid routing.
QWEN = {"H": 2048, "E": 128, "K": 8, "F": 768, "routing": "softmax", "bias": "", "shared": ""}
WIDE = {"H": 2048, "E": 512, "K": 10, "F": 512, "routing": "softmax", "bias": "", "shared": "Q8_0 gated"}
GLM = {"H": 4096, "E": 128, "K": 8, "F": 1408, "routing": "sigmoid", "bias": "uniform", "shared": "same"}


def _case(name, run, T, layers, gate, down, shape, **more):
    return {"name": name, "run": run, "T": T, "layers": layers, "gate": gate, "down": down, "norm": False, **shape, **more}


def listed():
    return [
        # One user, one token: the latency of a decode step's MoE layers (the norm and the residual fused, as in a trunk).
        _case("decode 1 token Q4_K", "graph", 1, 8, "Q4_K", "Q4_K", QWEN, norm=True),
        # A few users at once.
        _case("decode 8 tokens Q4_K", "graph", 8, 8, "Q4_K", "Q4_K", QWEN, norm=True),
        # A served batch: more pairs than experts, a few rows for each; the Q4_K_M mix keeps the down projections in Q6_K.
        _case("decode 32 tokens Q4_K/Q6_K", "graph", 32, 4, "Q4_K", "Q6_K", QWEN, norm=True),
        # One token, and a speculative draft of four to be verified, on many narrow experts at two bits.
        _case("wide decode 1 token IQ2_XS", "graph", 1, 4, "IQ2_XS", "IQ2_XS", WIDE),
        _case("wide verify 4 tokens IQ2_XS", "graph", 4, 4, "IQ2_XS", "IQ2_XS", WIDE),
        # Sixty-four tokens on wide experts: a few rows for each expert, every weight read.
        _case("glm 64 tokens IQ3_XXS/IQ4_NL", "eager", 64, 1, "IQ3_XXS", "IQ4_NL", GLM),
        # Prompt blocks: the headline's (skewed routing), a long one, one of odd length on many experts, and one on
        # 8-bit weights.
        _case("prefill 512 Q4_K skewed", "eager", 512, 1, "Q4_K", "Q4_K", QWEN, bias="zipf"),
        _case("prefill 4096 Q4_K/Q6_K", "eager", 4096, 1, "Q4_K", "Q6_K", QWEN),
        _case("wide prefill 509 IQ2_XS", "eager", 509, 1, "IQ2_XS", "IQ2_XS", WIDE),
        _case("prefill 333 Q8_0", "eager", 333, 1, "Q8_0", "Q8_0", QWEN),
        # One MoE FFN from a model file's bytes.
        _case("host 1 token Q4_K", "host", 1, 1, "Q4_K", "Q4_K", QWEN, shared="Q8_0 gated"),
    ]


def draw(rng):
    """Any of the three programs; 1 to 4096 tokens, the three shapes or a generic one, every pair of formats."""
    while True:
        T = int(round(math.exp(rng.uniform(0.0, math.log(4096.0)))))
        run = "host" if T == 1 and rng.random() < 0.3 else "graph" if T <= 48 else "eager"
        gate, down = rng.choice([("Q4_K", "Q4_K"), ("Q4_K", "Q6_K"), ("IQ2_XS", "IQ2_XS"), ("IQ3_XXS", "IQ4_NL"), ("Q8_0", "Q8_0")])
        c = dict(rng.choice([QWEN, WIDE, GLM, None, None]) or {
            "H": rng.choice([1024, 2048, 4096]), "E": rng.choice([32, 60, 64, 128, 256]), "K": rng.randint(2, 10),
            "F": 256 * rng.randint(2, 6), "routing": rng.choice(["softmax", "sigmoid"]),
            "bias": "", "shared": rng.choice(["", "same", "Q8_0 gated"])})
        if c["routing"] == "softmax":
            c["bias"] = rng.choice(["", "zipf"])
        if c["F"] % 256 and down != "Q8_0":
            gate, down = "IQ3_XXS", "IQ4_NL"  # whole blocks in a row
        c.update(run=run, T=T, layers=rng.choice([2, 4]) if run == "graph" else 1, gate=gate, down=down,
                 norm=run != "host" and rng.random() < 0.5)
        if run == "host":
            c["shared"] = rng.choice(["", "Q8_0 gated"])
        expert_bytes = c["F"] * c["H"] * (2 * BITS[gate] + BITS[down]) / 8
        if T * c["K"] * c["F"] * c["H"] <= 4096 * 8 * 768 * 2048 and expert_bytes * c["E"] * c["layers"] <= 2.5e9:
            return c


# ---- inputs ----
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _template(rng, fmt, rows, cols):
    """GGUF rows of weights of about SIGMA; an expert is a run of them."""
    return CF.synth_matrix(FORMATS[fmt], int(rng.integers(1 << 62)), 1, rows, cols, SIGMA)


def _plan(case, seed):
    """Everything the weights and inputs are made of, from the seed alone: templates, the experts' places in them, vectors, x."""
    rng = np.random.default_rng([seed, 71])
    H, E, K, F, T = (case[k] for k in "HEKFT")
    n = E if case["run"] != "host" else K
    p = {"mats": {}, "shared": {}}
    for which, fmt, rows, cols in (("gate", case["gate"], F, H), ("up", case["gate"], F, H), ("down", case["down"], H, F)):
        p["mats"][which] = (_template(rng, fmt, rows + EXTRA_ROWS, cols), rng.integers(0, EXTRA_ROWS, n), rows)
    p["router"] = rng.standard_normal((E, H), dtype=np.float32) * np.float32(SIGMA)
    p["bias"] = None
    if case["bias"] == "zipf":
        p["bias"] = np.array([1.5 * math.log((e + 1.0) ** -1.1) for e in range(E)], np.float32)
    elif case["bias"] == "uniform":
        p["bias"] = rng.uniform(-0.1, 0.1, E).astype(np.float32)
    if case["shared"]:
        gf, df = ("Q8_0", "Q8_0") if "Q8_0" in case["shared"] else (case["gate"], case["down"])
        for which, fmt, rows, cols in (("gate", gf, F, H), ("up", gf, F, H), ("down", df, H, F)):
            p["shared"][which] = _template(rng, fmt, rows, cols)
    p["sgvec"] = rng.standard_normal(H, dtype=np.float32) * np.float32(SIGMA) if "gated" in case["shared"] else None
    p["gain"] = 1.0 + rng.standard_normal(H, dtype=np.float32) * np.float32(0.02) if case["norm"] else None
    p["x"] = [_rows(case, p, rng) for _ in range(case["layers"])]
    if case["run"] == "host":
        w = np.exp(rng.standard_normal(K))
        p["weights"] = (w / w.sum()).astype(np.float32)
    return p


def _rows(case, p, rng):
    """T rows of N(0, 1) whose K-th and next router scores lie apart: where they are nearer than 32-bit sums resolve, either
    expert is right, and outputs could not be compared."""
    T, H = case["T"], case["H"]
    x = rng.standard_normal((T + 8 + T // 32, H), dtype=np.float32)
    if case["run"] == "host":
        return x[:T]
    s = _scores(case, p, torch.from_numpy(x).to(_device()).double())[1]
    top = torch.topk(s, min(case["K"] + 1, case["E"]), dim=1).values
    apart = (top[:, case["K"] - 1] - top[:, case["K"]] > 2e-5 if case["K"] < case["E"] else torch.ones(len(x), dtype=torch.bool)).cpu().numpy()
    return np.ascontiguousarray(x[np.argsort(~apart, kind="stable")[:T]])


def _slab(entry):
    t, places, rows = entry
    step = rows * t.stride
    data = np.empty(len(places) * step, np.uint8)
    for e, o in enumerate(places):
        data[e * step:(e + 1) * step] = t.data[o * t.stride:o * t.stride + step]
    return M.Matrix(data, t.cols, rows, len(places), t.kind, t.stride)


def prepare(case, seed):
    p = _plan(case, seed)
    gpu = M.default_gpu()
    mats = [_slab(p["mats"][k]) for k in ("gate", "up", "down")]
    shared = tuple(p["shared"][k] for k in ("gate", "up", "down")) if p["shared"] else None
    if case["run"] == "host":
        vec = p["sgvec"]
        gate = M.Matrix(vec.view(np.uint8), vec.size, 1, 1, M.F32, 4 * vec.size) if shared else None
        return {"case": case, "gpu": gpu, "mats": mats, "shared": shared, "gate": gate, "x": p["x"][0][0], "weights": p["weights"]}
    spec = M.LayerSpec(hidden=case["H"], experts=case["E"], top_k=case["K"], router=p["router"], gate=mats[0], up=mats[1], down=mats[2],
                       routing=M.ROUTE_SIGMOID if case["routing"] == "sigmoid" else M.ROUTE_SOFTMAX, router_bias=p["bias"],
                       shared=shared, shared_gate_vec=p["sgvec"], norm_gain=p["gain"])
    layers = [M.MoeLayer(gpu, spec)]
    layers += [layers[0].clone() for _ in range(case["layers"] - 1)]
    for layer in layers:
        layer.spec = None  # the host bytes are no longer needed
        layer.reserve(case["T"])
    x = [torch.from_numpy(v).cuda() for v in p["x"]]
    out = [torch.zeros_like(v) for v in x]
    state = {"case": case, "gpu": gpu, "layers": layers, "x": x, "out": out,
             "calls": [(layer, SimpleNamespace(ptr=a.data_ptr()), SimpleNamespace(ptr=b.data_ptr())) for layer, a, b in zip(layers, x, out)]}
    torch.cuda.synchronize()
    if case["run"] == "graph":
        gpu.graph_begin()
        _forwards(state)
        state["graph"] = gpu.graph_end()
    return state


def _forwards(state):
    T = state["case"]["T"]
    for layer, x, out in state["calls"]:
        layer.forward(x, T, out)


def run(state):
    kind = state["case"]["run"]
    if kind == "host":
        return state["gpu"].moe(state["mats"], state["shared"], state["gate"], state["x"], state["weights"])
    if kind == "graph":
        state["graph"].launch()
    else:
        _forwards(state)
    return state["out"]


# ---- what a pass cannot do without ----
def _touched(case):
    """Experts that T tokens select, from routing scores of the case's distribution."""
    if case["run"] == "host":
        return case["K"]
    H, E, K, T = (case[k] for k in "HEKT")
    rng = np.random.default_rng(5)
    s = rng.standard_normal((T, E)) * SIGMA * math.sqrt(H)
    if case["routing"] == "sigmoid":
        s = 1.0 / (1.0 + np.exp(-s)) + (rng.uniform(-0.1, 0.1, E) if case["bias"] else 0.0)
    elif case["bias"]:
        s = s + np.array([1.5 * math.log((e + 1.0) ** -1.1) for e in range(E)])
    return len(np.unique(np.argpartition(-s, K - 1, axis=1)[:, :K]))


def work(case):
    H, E, K, F, T = (case[k] for k in "HEKFT")
    expert = F * H * (2 * BITS[case["gate"]] + BITS[case["down"]]) / 8
    shared = 0.0 if not case["shared"] else 3 * F * H * 8.5 / 8 if "Q8_0" in case["shared"] else expert
    vectors = 4 * H * (("gated" in case["shared"]) + case["norm"]) + (4 * E if case["bias"] else 0)
    router = 0 if case["run"] == "host" else 4 * E * H
    one = _touched(case) * expert + shared + router + vectors + 8 * T * H
    flops = 6.0 * T * F * H * (K + bool(case["shared"])) + (2.0 * T * E * H if router else 0)
    return {"bytes": one * case["layers"], "flops": flops * case["layers"]}


def tolerance(case):
    """32-bit sums of 512 to 4096 products, twice over: either form of them is up to 1.3e-6 off 64 bits."""
    return {"rel": 5e-6, "max": 1e-4}


# ---- the same layer in 64 bits ----
def _scores(case, p, x):
    """(normalised x, the scores that experts are selected by, the logits whose softmax or sigmoid weighs them)."""
    dev = x.device
    if p["gain"] is not None:
        x = x * torch.rsqrt(x.square().mean(1, keepdim=True) + 1e-6) * torch.from_numpy(p["gain"]).to(dev).double()
    logits = x @ torch.from_numpy(p["router"]).to(dev).double().T
    bias = torch.from_numpy(p["bias"]).to(dev).double() if p["bias"] is not None else 0.0
    if case["routing"] == "sigmoid":
        return x, torch.sigmoid(logits) + bias, logits
    return x, logits + bias, logits + bias


def _ffn(x, gate, up, down):
    g, u = x @ gate.T, x @ up.T
    return (g * torch.sigmoid(g) * u) @ down.T


def exact(case, seed):
    p = _plan(case, seed)
    dev = _device()
    full = {k: (_values(t, dev), places, rows) for k, (t, places, rows) in p["mats"].items()}
    shared = [_values(p["shared"][k], dev) for k in ("gate", "up", "down")] if p["shared"] else None
    experts = len(full["gate"][1])
    outs = []
    for rows in p["x"]:
        x0 = torch.from_numpy(rows).to(dev).double()
        if case["run"] == "host":
            x, K = x0, case["K"]
            ids = torch.arange(K, device=dev).expand(1, K)
            w = torch.from_numpy(p["weights"]).to(dev).double().expand(1, K)
        else:
            x, s, logits = _scores(case, p, x0)
            ids = torch.topk(s, case["K"], dim=1).indices
            w = torch.gather(logits, 1, ids)
            if case["routing"] == "sigmoid":
                w = torch.sigmoid(w)
                w = w / w.sum(1, keepdim=True)
            else:
                w = torch.softmax(w, 1)
        out = x0.clone() if case["norm"] else torch.zeros_like(x0)
        for e in range(experts):
            t, k = torch.nonzero(ids == e, as_tuple=True)
            if len(t):
                mats = [v[int(places[e]):int(places[e]) + n] for v, places, n in (full[m] for m in ("gate", "up", "down"))]
                out.index_add_(0, t, _ffn(x[t], *mats) * w[t, k][:, None])
        if shared:
            y = _ffn(x, *shared)
            if p["sgvec"] is not None:
                y = y * torch.sigmoid(x @ torch.from_numpy(p["sgvec"]).to(dev).double())[:, None]
            out += y
        outs.append(out)
    return outs[0][0].cpu().numpy() if case["run"] == "host" else outs


# ---- the GGUF formats' values, in 64 bits. The codebooks' entries are packed: 8 values of 2 bits, and 4 of 3 bits. ----
IQ4_VALUES = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]
IQ2_LEVELS = [8, 25, 43, 0]
IQ3_LEVELS = [4, 12, 20, 28, 36, 44, 52, 62]
IQ2_XS_GRID = (
    "0000000200050008000a001100140016001900200022002500280041004400460049005000520055005800610064008000820085"
    "008800910094009900a001010104010601090110011201150118011a012101240140014201450148015101540160016801810184"
    "0190020002020205020802110214022002410244025002550280028a040104040406040904100412041504180421042404400442"
    "04450448045104540456046004810484049005000502050505080511051405200541054405500561058006010604061006260640"
    "064206840800080208050808080a08110814082008250841084408500858088008a008aa0901090409100940098109890a000a20"
    "0a280a960aa010011004100610091010101210151018102110241040104210451048105110541060106a10811084109011001102"
    "11051108111111141120114111441150118011941196120112041206121012401260140014021405140814111414142014411444"
    "1449145014641480150115041510154016001614164918011804181018121840185418861900190519661a511aa9200020022005"
    "2008200a201120142020204120442050208020a021012104211021402148216522002222228022a8240124042410242924402500"
    "2541255225992601261a26a628002808280a28202855288828a2296829902a082a202a822a882a8a400140044006400940104012"
    "40154018402140244040404240454048404a40514054406040654081408440904100410241054108411141144120414141444150"
    "4180418541a242014204421042124229424044004402440544084411441444194420444144444450448044944501450445104524"
    "4540459a4600460a464446504801480448104840484548544862490049114944495049694a045000500250055008501150145020"
    "502850415044505050805101510451105115514051425200524452aa540154045410542154405460548154a15500550855805588"
    "5621566856a158005814584158505899591a594059425a85600160046010604060546062608660a961006224624a629264006416"
    "65106540654565a46801686a69256a066a546a628000800280058008801180148020802a8041804480508080808280a880aa8101"
    "810481068110814081518159820082208280828282a082a8840184048410841284158440846084898500854485a58618866a8800"
    "88088825885a8880888288a889068a228a808a888a968aa890019004901090409056908491009122916492569289940094059444"
    "945094589529959095929641985198a699499a159a60a000a002a008a00aa020a02aa0a0a151a159a1a6a200a202a208a22aa280"
    "a2a0a440a495a665a698a80aa820a822a828a8a0a8a8a904a984a986aa28aa2aaa91aaaa"
)
IQ3_XXS_GRID = (
    "00000200400900b00f01001201902203b03d04104304804a05105505805a06106c07808008208408909009209909b09f0a90af0b"
    "d0c10c70c80ca0d50f810b11f12412f13b13d14114715a16a19d1b41c81cc1ce1e31f120120320820a21121321821a21c2272282"
    "4024224925025228128328828a2912982ba2c02c22d02d92e62f63013053283503543663793853d23e040040240940b410412416"
    "41942244144344544844a45145847347747848048248948f49049249f4a04ad4c14c84cc4f84fc51d52b54355756157c5c15c35c"
    "e5e560160860a61161362863563a6406426506596646666816836886956aa6ba6c96db71872773a74074675276d78c79e7b37db7"
    "f080480f81d81f82b82f87c89089f8a08b08b68c78e59049299349559639789c59c89ca9d8a0aa21a38a40a46a56a6da8ca9aaba"
    "ac2aebb08b13b17b3ab42b59ba8bd4be2c14c24c26c34c51c71c8fcb4cd8cded24d45d6ad9bdc3dd1e03e05e07e08e1ae2ae56e6"
    "0e8aea5eaaec0ecdedbef0f11f21f40f42f54f98"
)


def _grid(text, width, bits, count, levels):
    v = torch.tensor([int(text[i:i + width], 16) for i in range(0, len(text), width)])
    at = (v[:, None] >> (bits * torch.arange(count))) & ((1 << bits) - 1)
    return torch.tensor(levels, dtype=torch.float64)[at]


def _signs(bits7):
    """Eight signs from seven bits: the eighth makes their number even."""
    b = (bits7[..., None] >> torch.arange(7, device=bits7.device)) & 1
    b = torch.cat([b, b.sum(-1, keepdim=True) & 1], -1)
    return 1.0 - 2.0 * b.double()


def _values(m, dev):
    """The [rows, cols] weights of a matrix as torch.float64."""
    fmt = {v: k for k, v in FORMATS.items()}[m.kind]
    rows = m.rows * m.count
    raw = torch.from_numpy(m.data).to(dev).reshape(rows, -1)
    size = {"Q4_K": 144, "Q6_K": 210, "Q8_0": 34, "IQ2_XS": 74, "IQ3_XXS": 98, "IQ4_NL": 18}[fmt]
    b = raw.reshape(-1, size)

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()

    def u16(at, n):
        v = b[:, at:at + 2 * n].reshape(len(b), n, 2).int()
        return v[..., 0] | v[..., 1] << 8

    if fmt == "Q8_0":
        v = half(0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif fmt == "IQ4_NL":
        q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).long()
        v = half(0) * torch.tensor(IQ4_VALUES, dtype=torch.float64, device=dev)[q]
    elif fmt == "Q4_K":
        s = b[:, 4:16].int()
        sc = torch.cat([s[:, :4] & 63, s[:, 8:] & 15 | s[:, :4] >> 6 << 4], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, s[:, 8:] >> 4 | s[:, 4:8] >> 6 << 4], 1).double()
        n = b[:, 16:].reshape(-1, 4, 32)
        q = torch.stack([n & 15, n >> 4], 2).reshape(-1, 8, 32).double()
        v = half(0)[:, :, None] * sc[:, :, None] * q - half(2)[:, :, None] * mn[:, :, None]
    elif fmt == "Q6_K":
        low, high = b[:, :128].reshape(-1, 2, 2, 32).int(), b[:, 128:192].reshape(-1, 2, 1, 32).int()
        low = torch.stack([low & 15, low >> 4], 2).reshape(-1, 2, 4, 32)
        q = low | ((high >> (2 * torch.arange(4, device=dev, dtype=torch.int32)[:, None])) & 3) << 4
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        v = half(208)[:, :, None] * sc[:, :, None] * (q - 32).reshape(-1, 16, 16).double()
    elif fmt == "IQ2_XS":
        q = u16(2, 32).long()
        sc = b[:, 66:74].int()
        sc = torch.stack([sc & 15, sc >> 4], 2).reshape(-1, 16).repeat_interleave(2, 1).double()
        grid = _grid(IQ2_XS_GRID, 4, 2, 8, IQ2_LEVELS).to(dev)[q & 511]
        v = (half(0) * (0.5 + sc) * 0.25)[:, :, None] * grid * _signs(q >> 9)
    else:
        aux = u16(66, 16).long().reshape(-1, 8, 2)
        aux = aux[..., 0] | aux[..., 1] << 16
        grid = _grid(IQ3_XXS_GRID, 3, 3, 4, IQ3_LEVELS).to(dev)[b[:, 2:66].long()].reshape(-1, 8, 4, 8)
        sign = _signs((aux[:, :, None] >> (7 * torch.arange(4, device=dev))) & 127)
        v = (half(0) * (0.5 + (aux >> 28)) * 0.5)[:, :, None, None] * grid * sign
    return v.reshape(rows, m.cols)
