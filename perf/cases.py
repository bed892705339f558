"""Performance cases: the work that programs built on this framework have it do, through its Python entry points.

Six kinds of case, each over the sizes that the repository's configurations, tests and benchmark use or could use:

  linear   the W4A32 Linear as one call (rows are quantised, multiplied, offset): from one row to thousands
  pass     one token's (or a small batch's) W4A32 Linears of several decoder layers and the head, replayed from a HIP graph
  vision   an image through the patch embedding, the Linears of a vision layer and the merger
  decoder  the W4A32 decoder: a prompt alone, or a prompt and then tokens one by one (a step replayed from a HIP graph)
  suripel, lesarax
           the layered decoders in bf16 or f32: a prompt alone, or a prompt and then tokens one by one

Tokens behind a prompt are the program's choice (its own sampler, or a text to be scored) and not the greedy one. Weights are
random in the usual scale (standard deviation 0.02, less where a layer writes to the residual stream: by the square root of twice
the number of layers); norm weights and Linear inputs have channels of unequal size, as trained models do.
"""
import importlib
import math

import torch

pkg = importlib.import_module("mllm-advanced_amd")


def listed():
    wide = {"hidden": 1536, "heads": 12, "kv_heads": 2, "ff": 8960}
    model = {**wide, "layers": 28, "vocab": 151936}
    return [
        # one projection of one token, called on its own: the smallest call there is
        {"name": "linear_one_row", "kind": "linear", "rows": 1, "k": 1536, "n": 1536, "bias": True},
        # the widest projection of the 1.5B shape on a batch of long prompts: the largest call there is
        {"name": "linear_8192_rows", "kind": "linear", "rows": 8192, "k": 1536, "n": 8960, "bias": False},
        # the Linears of one decoded token, and of five sequences decoded together
        {"name": "pass_one_row", "kind": "pass", "rows": 1, **wide, "layers": 8, "vocab": 151936},
        {"name": "pass_five_rows", "kind": "pass", "rows": 5, **wide, "layers": 8, "vocab": 151936},
        # a 448 x 448 image: 1024 patches
        {"name": "vision_448", "kind": "vision", "side": 448, "width": 1280, "ff": 5120, "out": 1536},
        # the 1.5B-shaped W4A32 decoder: the time to the first token of a 512-token prompt; a short question and its answer
        {"name": "decoder_prompt", "kind": "decoder", **model, "head": "w4a32", "prompt": 512, "steps": 0},
        {"name": "decoder_request", "kind": "decoder", **model, "head": "w4a32", "prompt": 131, "steps": 32},
        # the layered decoder: a long prompt on the largest size; a question and its answer on the 1.5B shape; and, in f32, on the
        # smallest size, as a check of a model or a draft model runs
        {"name": "suripel_prompt", "kind": "suripel", "dtype": "bfloat16", "hidden": 3584, "heads": 28, "kv_heads": 4,
         "dim": 128, "ff": 18944, "layers": 28, "vocab": 152064, "window": 1024, "prompt": 2048, "steps": 0},
        {"name": "suripel_request", "kind": "suripel", "dtype": "bfloat16", **model, "dim": 128, "window": 1024,
         "prompt": 200, "steps": 32},
        {"name": "suripel_request_f32", "kind": "suripel", "dtype": "float32", "hidden": 1024, "heads": 8, "kv_heads": 2,
         "dim": 128, "ff": 4096, "layers": 24, "vocab": 65536, "window": 1024, "prompt": 300, "steps": 16},
        # the looped decoder with latent attention and experts: a text of odd length scored (every token's logits), and a
        # question and its answer
        {"name": "lesarax_prompt", "kind": "lesarax", "dtype": "bfloat16", **model, "dim": 128, "window": 1024, "kv_rank": 256,
         "experts": 16, "top": 4, "prompt": 1501, "steps": 0, "scored": True},
        {"name": "lesarax_request", "kind": "lesarax", "dtype": "bfloat16", **model, "dim": 128, "window": 1024, "kv_rank": 256,
         "experts": 16, "top": 4, "prompt": 100, "steps": 32},
    ]


def draw(rng):
    def spread(lo, hi):
        return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))

    kind = rng.choice(["linear", "linear", "pass", "vision", "decoder", "decoder", "suripel", "suripel", "lesarax"])
    if kind == "linear":
        rows, k = spread(1, 8192), 32 * spread(8, 280)
        n = spread(64, min(18944, max(64, 8192 * 1536 * 8960 // (rows * k))))
        return {"kind": kind, "rows": rows, "k": k, "n": n, "bias": rng.random() < 0.5}
    if kind == "vision":
        return {"kind": kind, "side": 28 * rng.randint(4, 20), "width": 64 * rng.randint(12, 20), "ff": 32 * rng.randint(90, 160),
                "out": rng.choice([896, 1536, 3584])}
    heads = 2 * rng.randint(4, 12 if kind != "decoder" else 14)
    kv = rng.choice([g for g in (1, 2, 4) if heads % g == 0])
    if kind == "pass":
        return {"kind": kind, "rows": rng.randint(1, 8), "hidden": 128 * heads, "heads": heads, "kv_heads": kv,
                "ff": 32 * rng.randint(80, 400), "layers": rng.randint(2, 8), "vocab": rng.randint(32000, 152064)}
    steps = rng.choice([0, spread(2, 20)])
    prompt = spread(2, 2048 if steps == 0 else 600)
    c = {"kind": kind, "heads": heads, "kv_heads": kv, "layers": rng.randint(4, 24), "vocab": rng.randint(32000, 152064),
         "prompt": prompt, "steps": steps}
    if kind == "decoder":
        return {**c, "hidden": 32 * rng.randint(2 * heads, 4 * heads), "ff": 32 * rng.randint(80, 320),
                "head": rng.choice(["w4a32", "float16"])}
    dim = rng.choice([64, 96, 128])
    c.update(dim=dim, hidden=rng.randint(heads * dim // 2, heads * dim) + 64, window=spread(64, 2048),
             scored=steps == 0 and rng.random() < 0.3)
    if kind == "suripel":
        f32 = rng.random() < 0.25
        return {**c, "dtype": "float32" if f32 else "bfloat16", "ff": spread(1500, 9000) // (2 if f32 else 1)}
    experts = rng.choice([8, 16, 24])
    return {**c, "dtype": "bfloat16", "kv_rank": rng.choice([128, 192, 256, 512]), "experts": experts, "top": rng.randint(1, 4),
            "ff": spread(1500, 9000)}


# ------------------------------------------------------------------------------------------------ inputs
class Inputs:
    """Random tensors in the order they are asked for, on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, *shape, std=0.02, mean=0.0):
        return torch.randn(shape, generator=self.gen, device="cuda").mul_(std).add_(mean)

    def gain(self, n):
        """Positive factors of unequal size around 1."""
        return torch.exp(self.normal(n, std=0.3))

    def rows(self, m, k):
        return self.normal(m, k, std=1.0) * torch.exp(self.normal(k, std=0.5))

    def ids(self, n, vocab):
        return torch.randint(0, vocab, (n,), generator=self.gen, device="cuda", dtype=torch.int64)

    def bf16(self, *shape, std=0.02, mean=0.0):
        return self.normal(*shape, std=std, mean=mean).to(torch.bfloat16)


def linear_shapes(c):
    """name -> (in, out, has a bias) of a W4A32 decoder layer"""
    W, q, kv, F = c["hidden"], c["heads"] * 128, c["kv_heads"] * 128, c["ff"]
    return {"q": (W, q, True), "k": (W, kv, True), "v": (W, kv, True), "o": (q, W, False), "gate": (W, F, False),
            "up": (W, F, False), "down": (F, W, False)}


def linear_layer(c, inp, make):
    """A layer's Linears, each as make(weights, bias or None)."""
    out = {}
    for name, (k, n, bias) in linear_shapes(c).items():
        w = inp.normal(n, k, std=0.01 / math.sqrt(2 * c["layers"]) if name in ("o", "down") else 0.02)
        out[name] = make(w, inp.normal(n) if bias else None)
    return out


def decoder_head(c, inp, emb, make):
    """The head's rows are the embedding's in another order, so that one next token stands out from the others."""
    w = emb[torch.randperm(c["vocab"], generator=inp.gen, device="cuda")] * 0.02
    return w.half() if c.get("head") == "float16" else make(w, None)


def layered_config(c):
    """The dictionary of config.json."""
    W, H, d, L = c["hidden"], c["heads"], c["dim"], c["layers"]
    layers = []
    if c["kind"] == "suripel":
        last_kv = None
        for i in range(L):
            kind = ("attention", "delta", "retention")[i % 3]
            m = {"heads": H, "dim": d, "vdim": d}
            if kind == "attention":  # every second one reads the keys and values of the one before it
                m.update(kv_heads=c["kv_heads"], conv=4, scale=d ** -0.5, mask={"size": c["window"], "pool": 16})
                if last_kv is None:
                    last_kv = i
                else:
                    m["kv_from"], last_kv = last_kv, None
            elif kind == "delta":
                m.update(kv_heads=H // 2, conv=4)
            else:
                m.update(decay=[1 - 2.0 ** -(5 + 5 * h / H) for h in range(H)], rot={"dims": d, "base": 1e6})
            layers.append({"type": kind, "mixer": m, "mlp": {"kind": "dense", "ff": c["ff"]}})
        return {"architecture": "Suripel", "width": W, "vocab": c["vocab"], "canon": {"taps": 4}, "norm": {"eps": 1e-5},
                "layers": layers}
    # as many layer runs as `layers` says, the middle half of them two passes through a quarter of the layers
    quarter = L // 4
    mlp = {"kind": "moe", "expert": {"ff": c["ff"] // 4, "limit": 7.0}, "router": {"experts": c["experts"], "top": c["top"]}}
    for i in range(L - quarter):
        if i % 4 == 2:
            m = {"heads": H, "kv_heads": c["kv_heads"], "dim": d, "vdim": d, "scale": d ** -0.5, "rot": {"dims": 64, "base": 1e6}}
            layers.append({"type": "attention", "mixer": m, "mlp": mlp})
        else:
            m = {"heads": H, "dim": d, "rot_dim": 64, "vdim": d, "q_rank": W // 2, "kv_rank": c["kv_rank"],
                 "scale": (d + 64) ** -0.5, "mask": {"size": c["window"]}, "rot": {"dims": 64, "base": 1e6}}
            layers.append({"type": "latent_attention", "mixer": m, "mlp": mlp})
    return {"architecture": "Lesarax", "width": W, "vocab": c["vocab"], "norm": {"eps": 1e-5}, "residual_mult": 0.5,
            "loop": {"start": quarter, "stop": 2 * quarter, "times": 2}, "layers": layers}


def layered_shapes(cfg, layer):
    """name -> shape of the matrices of a layer without its experts"""
    W, m, t = cfg["width"], layer["mixer"], layer["type"]
    H, d = m["heads"], m["dim"]
    G = m.get("kv_heads", H)
    s = {}
    if cfg["architecture"] == "Suripel":
        s["mix.q"] = ((G if t == "delta" else H) * d, W)
        if m.get("kv_from") is None:
            s["mix.k"], s["mix.v"] = (G * d, W), ((G if t == "attention" else H) * d, W)
        if t != "attention":
            s["mix.g"] = (H * d, W)
        if t == "delta":
            s["mix.a"], s["mix.b"] = (H, W), (H, W)
        s["mlp.up"], s["mlp.down"] = (layer["mlp"]["ff"], W), (W, layer["mlp"]["ff"])
    else:
        if t == "attention":
            s["mix.q"], s["mix.k"] = (H * d, W), (G * d, W)
        else:
            r, kr, rot = m["q_rank"], m["kv_rank"], m["rot_dim"]
            s.update({"mix.dq": (r, W), "mix.uq": (H * (d + rot), r), "mix.dkv": (kr + rot, W), "mix.uk": (H * d, kr),
                      "mix.uv": (H * d, kr), "mix.g": (H, W)})
        s["mlp.router"] = (layer["mlp"]["router"]["experts"], W)
    s["mix.o"] = (W, H * d)
    return s


def layered_weights(cfg, inp):
    """Tensors under the parameter names of model.safetensors, every value a bf16."""
    W, V, small = cfg["width"], cfg["vocab"], 0.02 / math.sqrt(2 * len(cfg["layers"]))
    suripel = cfg["architecture"] == "Suripel"
    gain = lambda n: inp.gain(n).to(torch.bfloat16)
    w = {"embed": inp.bf16(V, W, std=1.0), "final.norm": gain(W)}
    if suripel:
        w["head"] = (w["embed"][torch.randperm(V, generator=inp.gen, device="cuda")] * 0.02).to(torch.bfloat16)
    else:
        w["loop.in"] = inp.bf16(W, 2 * W, std=(2 * W) ** -0.5)
    for i, layer in enumerate(cfg["layers"]):
        p, m = f"l{i}.", layer["mixer"]
        for name, shape in layered_shapes(cfg, layer).items():
            w[p + name] = inp.bf16(*shape, std=small if name in ("mix.o", "mlp.down") else 0.02)
        w[p + "norm1"], w[p + "norm2"] = gain(W), gain(W)
        if suripel:
            w[p + "canon1"], w[p + "canon2"] = inp.bf16(W, 4, std=0.3), inp.bf16(W, 4, std=0.3)
            w[p + "mlp.act"] = torch.tensor([0.25, 0.5, 0.25, 0.0], device="cuda")
            for n in "qkv":
                if "conv" in m and p + "mix." + n in w:
                    w[p + f"mix.{n}.conv"] = inp.bf16(w[p + "mix." + n].shape[0], m["conv"], std=0.4)
            if layer["type"] == "delta":
                w[p + "mix.A_log"], w[p + "mix.dt_bias"] = inp.bf16(m["heads"]), inp.bf16(m["heads"], mean=-3.0)
                w[p + "mix.norm"] = gain(m["vdim"])
            continue
        w[p + "mix.sink"] = inp.bf16(m["heads"], std=1.0)
        if layer["type"] != "attention":
            w[p + "mix.dq.norm"], w[p + "mix.dkv.norm"] = gain(m["q_rank"]), gain(m["kv_rank"])
        E, F = layer["mlp"]["router"]["experts"], layer["mlp"]["expert"]["ff"]
        gate, up, down = inp.bf16(E, F, W), inp.bf16(E, F, W), inp.bf16(E, W, F, std=small)
        for e in range(E):
            w[f"{p}mlp.e{e}.gate"], w[f"{p}mlp.e{e}.up"], w[f"{p}mlp.e{e}.down"] = gate[e], up[e], down[e]
    return w


# ------------------------------------------------------------------------------------------------ what a program keeps
class Linear:
    """Weights packed once, workspace and output kept."""

    def __init__(self, w, bias, rows):
        self.n, k = w.shape
        self.packed = pkg.quant_pack_rhs(w, bias)
        self.ws = torch.empty(int(pkg.lib().w4a32_workspace_bytes_n(rows, k, self.n)), dtype=torch.uint8, device="cuda")
        self.out = torch.empty((rows, self.n), dtype=torch.float32, device="cuda")

    def __call__(self, x):
        return pkg.matmul_ws(x, self.packed, self.n, ws=self.ws, out=self.out)


def captured(fn):
    fn()
    torch.cuda.current_stream().synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def prepare_linear(c, inp):
    w = inp.normal(c["n"], c["k"])
    linear = Linear(w, inp.normal(c["n"]) if c["bias"] else None, c["rows"])
    x = inp.rows(c["rows"], c["k"])
    return lambda: linear(x)


def pass_groups(c):
    """Linears that share their input go out together."""
    return (("q", "k", "v"), ("o",), ("gate", "up"), ("down",))


def prepare_pass(c, inp):
    shapes, m = linear_shapes(c), c["rows"]
    layers = [linear_layer(c, inp, pkg.quant_pack_rhs) for _ in range(c["layers"])]
    head = pkg.quant_pack_rhs(inp.normal(c["vocab"], c["hidden"]))
    x = {k: inp.rows(m, k) for k in sorted({s[0] for s in shapes.values()})}
    ws = {k: torch.empty(pkg.workspace_bytes(m, k), dtype=torch.uint8, device="cuda") for k in x}

    def work():
        out = []
        for layer in layers:
            for group in pass_groups(c):
                k = shapes[group[0]][0]
                out += pkg.matmul_grouped(x[k], [layer[n] for n in group], [shapes[n][1] for n in group], ws=ws[k])
        return out + pkg.matmul_grouped(x[c["hidden"]], [head], [c["vocab"]], ws=ws[c["hidden"]])

    graph, out = captured(work)

    def one():
        graph.replay()
        return out
    one.kept = (layers, head, x, ws)
    return one


def vision_inputs(c, inp):
    W, F = c["width"], c["ff"]
    image = inp.normal(1, 3, 2, c["side"], c["side"], std=1.0)
    patch = torch.zeros((W, 1184), device="cuda")
    patch[:, :1176] = inp.normal(W, 1176)
    shapes = {"qkv": (W, 3 * W), "proj": (W, W), "fc1": (W, F), "fc2": (F, W), "merge1": (4 * W, 4 * W),
              "merge2": (4 * W, c["out"])}
    return image, patch, {n: (inp.normal(b, a), inp.normal(b)) for n, (a, b) in shapes.items()}


def vision_chain(image_rows, patch, linears):
    p = patch(image_rows)
    f = linears["fc1"](p)
    g = linears["merge1"](p.view(p.shape[0] // 4, -1))
    return {"patches": p, "qkv": linears["qkv"](p), "proj": linears["proj"](p), "fc1": f, "fc2": linears["fc2"](f), "merge1": g,
            "merge2": linears["merge2"](g)}


def prepare_vision(c, inp):
    image, patch, linears = vision_inputs(c, inp)
    m = (c["side"] // 14) ** 2
    patch = Linear(patch, None, m)
    linears = {n: Linear(w, b, m // 4 if n.startswith("merge") else m) for n, (w, b) in linears.items()}
    return lambda: vision_chain(pkg.op_im2col_conv3d(image, (2, 14, 14), (2, 14, 14)), patch, linears)


def prepare_decoder(c, inp):
    W, V, n, steps = c["hidden"], c["vocab"], c["prompt"], c["steps"]
    emb = inp.normal(V, W, std=1.0)
    layers = [{**linear_layer(c, inp, pkg.quant_pack_rhs), "attn_norm": inp.gain(W), "ffn_norm": inp.gain(W)}
              for _ in range(c["layers"])]
    head = decoder_head(c, inp, emb, pkg.quant_pack_rhs)
    dec = pkg.Decoder(W, c["heads"], c["kv_heads"], c["ff"], V, layers, emb, inp.gain(W), head, max_seq=n + steps + 8,
                      max_batch_tokens=n, lm_head_dense=c["head"] == "float16")
    ids = inp.ids(n + steps, V)
    prompt, logits = ids[:n], dec.logits
    if steps == 0:
        return lambda: (logits, dec.prefill(prompt))
    graph, _ = captured(dec.step)

    def request():
        out = torch.empty((steps + 1, V), dtype=torch.float32, device="cuda")
        dec.prefill(prompt)
        out[0] = logits
        for i in range(steps):
            dec.token.copy_(ids[n + i:n + i + 1])
            graph.replay()
            out[i + 1] = logits
        return out
    return request


def prepare_layered(c, inp):
    cfg = layered_config(c)
    n, steps = c["prompt"], c["steps"]
    w = layered_weights(cfg, inp)
    dec = pkg.LayeredDecoder(cfg, w, c["dtype"], max_seq=n + steps + 8, max_batch_tokens=n)
    del w
    state = dec.new_state()
    ids = inp.ids(n + steps + 1, c["vocab"])
    prompt = ids[:n]
    if steps == 0:
        return lambda: dec.forward(state, prompt, 0, want=None if c.get("scored") else [n - 1])
    graph, _ = captured(lambda: dec.step(state))

    def request():
        picks = torch.empty((steps,), dtype=torch.int64, device="cuda")
        first = dec.forward(state, prompt, 0, want=[n - 1])
        for i in range(steps):
            dec.token.copy_(ids[n + i:n + i + 1])
            graph.replay()
            picks[i:i + 1] = dec.token
        return first, picks, dec.forward(state, ids[n + steps:], n + steps, want=[0])
    return request


PREPARE = {"linear": prepare_linear, "pass": prepare_pass, "vision": prepare_vision, "decoder": prepare_decoder,
           "suripel": prepare_layered, "lesarax": prepare_layered}


def prepare(case, seed):
    return PREPARE[case["kind"]](case, Inputs(seed))


def run(state):
    return state()


# ------------------------------------------------------------------------------------------------ sizes and tolerances
def linear_work(m, k, n):
    """Weights with their block scales, activations in, results out."""
    return {"bytes": n * k / 2 + n * k / 16 + 4 * m * (k + n), "flops": 2 * m * k * n}


def summed(works):
    works = list(works)
    return {u: float(sum(w[u] for w in works)) for u in ("bytes", "flops")}


def attended(n, steps, window):
    """(query, key) pairs of a causal window over a prompt and the tokens behind it"""
    total = n + steps
    short = min(total, window)
    return short * (short + 1) / 2 + (total - short) * window


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        return summed([linear_work(c["rows"], c["k"], c["n"])])
    if kind == "pass":
        layer = [linear_work(c["rows"], k, n) for k, n, _ in linear_shapes(c).values()]
        return summed(layer * c["layers"] + [linear_work(c["rows"], c["hidden"], c["vocab"])])
    if kind == "vision":
        m, W, F = (c["side"] // 14) ** 2, c["width"], c["ff"]
        return summed([{"bytes": 4 * 6 * c["side"] ** 2, "flops": 0}, linear_work(m, 1176, W), linear_work(m, W, 3 * W),
                       linear_work(m, W, W), linear_work(m, W, F), linear_work(m, F, W), linear_work(m // 4, 4 * W, 4 * W),
                       linear_work(m // 4, 4 * W, c["out"])])
    n, steps, W, V, L = c["prompt"], c["steps"], c["hidden"], c["vocab"], c["layers"]
    passes = 1 + steps + (steps > 0 and kind != "decoder")  # through the weights
    rows = n if c.get("scored") else passes                 # of logits
    tokens = n + passes - 1
    if kind == "decoder":
        body = L * sum(k * m for k, m, _ in linear_shapes(c).values())
        head = W * V * (2 if c["head"] == "float16" else 0.5625)
        pairs = attended(n, steps, n + steps)
        cache = 8 * c["kv_heads"] * 128 * L
        return {"bytes": passes * (0.5625 * body + head + 4 * V) + cache * tokens + cache * sum(n + i for i in range(steps)),
                "flops": 2 * body * tokens + 2 * W * V * passes + 4 * pairs * c["heads"] * 128 * L}
    cfg, elem = layered_config(c), 2 if c["dtype"] == "bfloat16" else 4
    lp = cfg.get("loop")
    nbytes = flops = 0.0
    for i, layer in enumerate(cfg["layers"]):
        times = lp["times"] if lp and lp["start"] <= i < lp["stop"] else 1
        weights = sum(a * b for a, b in layered_shapes(cfg, layer).values())
        nbytes += elem * weights * passes * times
        flops += 2 * weights * tokens * times
        if "expert" in layer["mlp"]:
            expert, E, top = 3 * W * layer["mlp"]["expert"]["ff"], c["experts"], c["top"]
            nbytes += elem * expert * times * (E * (1 - (1 - top / E) ** n) + top * (passes - 1))
            flops += 2 * expert * top * tokens * times
        m, d = layer["mixer"], c["dim"]
        if layer["type"] in ("attention", "latent_attention"):
            window = m["mask"]["size"] if m.get("mask") else n + passes
            per = 2 * d + (64 if layer["type"] == "latent_attention" else 0)
            flops += 2 * per * c["heads"] * attended(n, passes - 1, window) * times
            kept = c["kv_rank"] + 64 if layer["type"] == "latent_attention" else 2 * d * c["kv_heads"]
            nbytes += elem * kept * times * (n + sum(min(window, n + j) for j in range(passes - 1)))
        else:
            flops += 4 * c["heads"] * d * d * tokens
            nbytes += 4 * c["heads"] * d * d * (1 + 2 * (passes - 1))
    if lp:
        nbytes += elem * 2 * W * W * passes * lp["times"]
        flops += 4 * W * W * tokens * lp["times"]
    written = rows if steps == 0 else 2  # the logits of the steps between stay inside the model
    return {"bytes": nbytes + elem * W * V * passes + 4 * V * written, "flops": flops + 2 * W * V * rows}


def tolerance(case):
    """About four times what these paths were seen to differ by from exact(), or, deep models, from themselves with a prompt
    taken in two portions (other sums in another order). A W4A32 Linear rounds its input rows to 8 bits, so a difference in a
    last bit moves single values by a whole step: up to 3e-4 in one Linear, 7e-4 behind two more, about 1e-2 behind a whole model.
    In bf16 every product's input is rounded (7e-3), and experts can change places (5e-3 of all logits, more in single rows)."""
    kind = case["kind"]
    if kind in ("linear", "pass"):
        return {"rel": 1e-3, "max": 0.02}
    if kind == "vision":
        return {"rel": 3e-3, "max": 0.2}
    if kind == "decoder":
        return {"rel": 0.03, "max": 0.6}
    if case["dtype"] == "float32":
        return {"rel": 5e-6}
    return {"rel": 0.025, "max": 1.0 - 1e-6}


# ------------------------------------------------------------------------------------------------ the same in 64 bits
def quantised_weights(w):
    """The values the 4-bit format keeps of w [N][K]: per 32 the first largest magnitude / -8 as scale, cut to bf16."""
    b = w.view(w.shape[0], -1, 32)
    scale = b.gather(2, b.abs().argmax(2, keepdim=True)) / -8.0
    q = b * torch.where(scale != 0, 1.0 / scale, torch.zeros_like(scale))
    q = torch.clamp(torch.trunc(q.double() + torch.copysign(torch.full_like(q, 0.5).double(), q.double())), -8, 7)
    scale = (scale.contiguous().view(torch.int32) & -65536).view(torch.float32)
    return (q * scale.double()).view(w.shape)


def quantised_rows(x):
    """Rows to 8 bits and back: an asymmetric range that holds 0, halves away from 0."""
    lo, hi = x.amin(1, keepdim=True).clamp(max=0), x.amax(1, keepdim=True).clamp(min=0)
    scale = torch.where(lo == hi, torch.ones_like(lo), 255.0 / (hi - lo))
    zero = torch.where((lo + hi) * scale - 1 > 0, -128 - lo * scale, 127 - hi * scale).clamp(-128, 127).round()
    v = x * scale
    q = torch.clamp(torch.trunc(v + torch.copysign(torch.full_like(v, 0.5), v)) + zero, -128, 127)
    return (q - zero) / scale


class ExactLinear:
    def __init__(self, w, bias=None):
        self.w, self.bias = w, bias  # widened when it is used: a whole model would not fit otherwise

    def __call__(self, x):
        y = quantised_rows(x) @ quantised_weights(self.w).t()
        return y if self.bias is None else y + self.bias.double()


def over_rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def rotated(x, dims, base, pos0=0):
    """x [T][heads][dim]: dimension i turns with i + dims / 2."""
    half = dims // 2
    i = torch.arange(half, device="cuda", dtype=torch.float64)
    a = (pos0 + torch.arange(x.shape[0], device="cuda", dtype=torch.float64))[:, None, None] * base ** (-2.0 * i / dims)
    u, v = x[..., :half], x[..., half:dims]
    return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin(), x[..., dims:]], -1)


def attention(q, k, v, scale, size=None, pool=None, sinks=None):
    """Causal softmax attention of q [T][H][d] on k, v [T][G][..] over the last `size` tokens; with `pool`, also on the mean of
    every block of that many tokens that the window has left behind; with `sinks`, one more term in the denominator."""
    T, H = q.shape[:2]
    rep = H // k.shape[1]
    i = torch.arange(T, device="cuda")[:, None]
    j = torch.arange(T, device="cuda")[None]
    seen = j <= i
    if size is not None:
        seen = seen & (j > i - size)
    if pool:
        nb = T // pool
        means = [t[:nb * pool].view(nb, pool, t.shape[1], t.shape[2]).mean(1) for t in (k, v)]
        k, v = torch.cat([means[0], k]), torch.cat([means[1], v])
        seen = torch.cat([torch.arange(nb, device="cuda")[None] * pool + pool - 1 <= i - size, seen], 1)
    out = torch.empty((T, H, v.shape[2]), dtype=torch.float64, device="cuda")
    for h in range(H):
        s = (q[:, h] @ k[:, h // rep].t()) * scale
        s.masked_fill_(~seen, -math.inf)
        if sinks is not None:
            s = torch.cat([s, sinks[h].double().expand(T, 1)], 1)
        p = torch.softmax(s, 1)
        out[:, h] = p[:, :v.shape[0]] @ v[:, h // rep]
    return out


def exact_decoder(c, inp):
    W, V, n, H, G = c["hidden"], c["vocab"], c["prompt"], c["heads"], c["kv_heads"]
    emb = inp.normal(V, W, std=1.0)
    layers = [{**linear_layer(c, inp, ExactLinear), "attn_norm": inp.gain(W), "ffn_norm": inp.gain(W)}
              for _ in range(c["layers"])]
    head = decoder_head(c, inp, emb, ExactLinear)
    last = inp.gain(W).double()
    ids = inp.ids(n + c["steps"], V)
    h = emb[ids].double()
    for layer in layers:
        x = over_rms(h, 1e-6) * layer["attn_norm"].double()
        q, k, v = (layer[t](x).view(x.shape[0], -1, 128) for t in "qkv")
        a = attention(rotated(q, 128, 1e6), rotated(k, 128, 1e6), v, 128 ** -0.5)
        h = h + layer["o"](a.reshape(x.shape[0], -1))
        x = over_rms(h, 1e-6) * layer["ffn_norm"].double()
        g = layer["gate"](x)
        h = h + layer["down"](g * torch.sigmoid(g) * layer["up"](x))
    x = over_rms(h[n - 1:], 1e-6) * last
    logits = x @ head.double().t() if c["head"] == "float16" else head(x)
    return logits if c["steps"] else (logits[0], None)


def causal_conv(x, w):
    w, taps = w.double(), w.shape[1]
    padded = torch.cat([x.new_zeros((taps - 1, x.shape[1])), x])
    return sum(w[:, j] * padded[j:j + x.shape[0]] for j in range(taps))


def silu(x):
    return x * torch.sigmoid(x)


def suripel_mixer(w, p, layer, h, kv, i):
    m, T = layer["mixer"], h.shape[0]
    H, d = m["heads"], m["dim"]
    of = lambda n: h @ w[p + n].double().t()
    if layer["type"] == "attention":
        conv = lambda n: causal_conv(of(n), w[p + n + ".conv"]).view(T, -1, d)
        if m.get("kv_from") is None:
            kv[i] = conv("k"), conv("v")
        k, v = kv[m.get("kv_from", i)]
        o = attention(conv("q"), k, v, m["scale"], m["mask"]["size"], m["mask"]["pool"])
        return o.reshape(T, -1) @ w[p + "o"].double().t()
    if layer["type"] == "delta":
        q, k, v = (silu(causal_conv(of(n), w[p + n + ".conv"])).view(T, -1, d) for n in "qkv")
        unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)
        q, k = (unit(t).repeat_interleave(H // m["kv_heads"], 1) for t in (q, k))
        q = q * d ** -0.5
        beta = torch.sigmoid(of("b"))
        g = torch.exp(-torch.exp(w[p + "A_log"].double())
                      * torch.nn.functional.softplus(of("a") + w[p + "dt_bias"].double(), threshold=100.0))
        S = torch.zeros((H, d, d), dtype=torch.float64, device="cuda")
        o = torch.empty((T, H, d), dtype=torch.float64, device="cuda")
        for t in range(T):
            S = S * g[t][:, None, None]
            u = beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
            S = S + k[t][:, :, None] * u[:, None]
            o[t] = (S * q[t][:, :, None]).sum(1)
        o = over_rms(o, 1e-5) * w[p + "norm"].double()
    else:
        q, k, v = (of(n).view(T, H, d) for n in "qkv")
        rot = m["rot"]
        q, k = rotated(q, rot["dims"], rot["base"]), rotated(k, rot["dims"], rot["base"]) * d ** -0.5
        back = (torch.arange(T, device="cuda")[:, None] - torch.arange(T, device="cuda")[None]).double()
        o = torch.stack([((q[:, x] @ k[:, x].t()) * torch.where(back >= 0, m["decay"][x] ** back.clamp(min=0), 0.0)) @ v[:, x]
                         for x in range(H)], 1)
        o = over_rms(o, 1e-5)
    return (o.reshape(T, -1) * silu(of("g"))) @ w[p + "o"].double().t()


def exact_suripel(cfg, w, ids, rows):
    def norm(x, name):
        x = x - x.mean(-1, keepdim=True)
        return over_rms(x, 1e-5) * w[name].double()

    x, kv = w["embed"][ids].double(), {}
    for i, layer in enumerate(cfg["layers"]):
        p = f"l{i}."
        h = norm(x, p + "norm1")
        x = x + suripel_mixer(w, p + "mix.", layer, h + causal_conv(h, w[p + "canon1"]), kv, i)
        h = norm(x, p + "norm2")
        z = (h + causal_conv(h, w[p + "canon2"])) @ w[p + "mlp.up"].double().t()
        a, b, c, e = w[p + "mlp.act"].double()
        z = a * over_rms(z, 1e-5) + b * over_rms(z ** 2, 1e-5) + c * over_rms(z ** 3, 1e-5) + e
        x = x + z @ w[p + "mlp.down"].double().t()
    return norm(x[rows], "final.norm") @ w["head"].double().t()


def lesarax_mixer(w, p, layer, h):
    m, T = layer["mixer"], h.shape[0]
    H, d, rot = m["heads"], m["dim"], m["rot"]
    of = lambda n, x: x @ w[p + n].double().t()
    turn = lambda x: rotated(x, rot["dims"], rot["base"])
    if layer["type"] == "attention":  # the values are the keys before rotation
        q, k = of("q", h).view(T, H, d), of("k", h).view(T, -1, d)
        return of("o", attention(turn(q), turn(k), k, m["scale"], sinks=w[p + "sink"]).reshape(T, -1))
    q = of("uq", over_rms(of("dq", h), 1e-5) * w[p + "dq.norm"].double()).view(T, H, -1)
    c = of("dkv", h)
    kr = turn(c[:, None, m["kv_rank"]:])
    c = over_rms(c[:, :m["kv_rank"]], 1e-5) * w[p + "dkv.norm"].double()
    q = torch.cat([q[..., :d], turn(q[..., d:])], -1)
    k = torch.cat([of("uk", c).view(T, H, d), kr.expand(T, H, kr.shape[2])], -1)
    o = attention(q, k, of("uv", c).view(T, H, -1), m["scale"], m["mask"]["size"], sinks=w[p + "sink"])
    return of("o", (o * torch.sigmoid(of("g", h))[..., None]).reshape(T, -1))


def experts(w, p, mlp, h):
    top, chosen = (h @ w[p + "router"].double().t()).topk(mlp["router"]["top"], 1)
    share, limit = torch.softmax(top, 1), mlp["expert"]["limit"]
    out = torch.zeros_like(h)
    for e in range(mlp["router"]["experts"]):
        rows, slot = (chosen == e).nonzero(as_tuple=True)
        if rows.numel():
            x = h[rows]
            g = (x @ w[f"{p}e{e}.gate"].double().t()).clamp(max=limit)
            u = (x @ w[f"{p}e{e}.up"].double().t()).clamp(-limit, limit)
            out[rows] += share[rows, slot, None] * ((g * torch.sigmoid(1.702 * g) * (u + 1)) @ w[f"{p}e{e}.down"].double().t())
    return out


def exact_lesarax(cfg, w, ids, rows):
    norm = lambda x, name: over_rms(x, 1e-5) * w[name].double()
    lp = cfg["loop"]
    x0 = w["embed"][ids].double()
    x = x0
    order = list(range(lp["start"])) + lp["times"] * list(range(lp["start"], lp["stop"]))
    for i in order + list(range(lp["stop"], len(cfg["layers"]))):
        layer, p = cfg["layers"][i], f"l{i}."
        if i == lp["start"] < lp["stop"]:
            x = torch.cat([x, x0], 1) @ w["loop.in"].double().t()
        x = x + cfg["residual_mult"] * lesarax_mixer(w, p + "mix.", layer, norm(x, p + "norm1"))
        x = x + cfg["residual_mult"] * experts(w, p + "mlp.", layer["mlp"], norm(x, p + "norm2"))
    return norm(x[rows], "final.norm") @ w["embed"].double().t()


def exact_layered(c, inp):
    cfg = layered_config(c)
    w = layered_weights(cfg, inp)
    n, steps = c["prompt"], c["steps"]
    ids = inp.ids(n + steps + 1, c["vocab"])
    if steps == 0:
        ids = ids[:n]
    forward = exact_suripel if c["kind"] == "suripel" else exact_lesarax
    want = list(range(n)) if c.get("scored") else [n - 1] if steps == 0 else [n - 1, n + steps]
    logits = forward(cfg, w, ids, torch.tensor(want, device="cuda"))
    return logits if steps == 0 else (logits[:1], None, logits[1:])


def exact(case, seed):
    c, inp = case, Inputs(seed)
    if c["kind"] == "decoder":
        return exact_decoder(c, inp)
    if c["kind"] in ("suripel", "lesarax"):
        return exact_layered(c, inp)
    if c["kind"] == "linear":
        linear = ExactLinear(inp.normal(c["n"], c["k"]), inp.normal(c["n"]) if c["bias"] else None)
        return linear(inp.rows(c["rows"], c["k"]).double())
    if c["kind"] == "pass":
        shapes = linear_shapes(c)
        layers = [linear_layer(c, inp, ExactLinear) for _ in range(c["layers"])]
        head = ExactLinear(inp.normal(c["vocab"], c["hidden"]))
        x = {k: inp.rows(c["rows"], k).double() for k in sorted({s[0] for s in shapes.values()})}
        names = [n for group in pass_groups(c) for n in group]
        return [layer[n](x[shapes[n][0]]) for layer in layers for n in names] + [head(x[c["hidden"]])]
    image, patch, linears = vision_inputs(c, inp)
    g = c["side"] // 14
    cols = image.view(3, 2, g, 14, g, 14).permute(2, 4, 0, 1, 3, 5).reshape(g * g, 1176).double()
    cols = torch.cat([cols, cols.new_zeros((g * g, 8))], 1)
    return vision_chain(cols, ExactLinear(patch), {n: ExactLinear(w, b) for n, (w, b) in linears.items()})
