"""The work by which this engine's speed is judged: prompts, decoding, and whole lives of requests, over the designs and
layer sizes that its benchmark and tests use.

A case is plain values: ``design`` and ``size`` (layer sizes as ``bench.py --designs`` has them; ``scout``: the published
Llama 4 Scout layers, four of the 48; ``tiny``: the tests' smallest model), ``dtype``, ``requests``, ``prompt`` (the mean
length; ``ragged``: lengths from a half to one and a half of it), ``steps`` (decoded tokens per request behind the prompt),
``portion`` (the step's token budget that the engine is made with).  A pass is ``Engine.prefill`` of all prompts,
``Engine.decode_step`` for every further token (teacher-forced, as a replay or a scoring run does it) and ``release``;
its outputs are the float32 logits of every call.

Weights are drawn by checkpoint name from the seed.  A trained router tells a token's experts apart clearly; a random one
does not, and near-ties would make two correct implementations choose differently.  So every router's rows are directions
of their own, a token's embedding says along them which experts are its first and second choice, and the matrices that
write to the residual stream are drawn smaller by the root of their number, as deep models are initialised.
"""
import hashlib
import math
import random

import torch

from jax_llm_examples_amd import Engine, get_architecture
from jax_llm_examples_amd.engine import build_model
from jax_llm_examples_amd.weights.loader import place

DEVICE = "cuda:0"
EPS = 1e-5
SIZES = {
    "tiny": dict(width=64, heads=4, kv=2, ff=256, span=32, dim=16, rot=16, rank=32, vocab=512, experts=4),
    "2k": dict(width=2048, heads=16, kv=8, ff=8192, span=1024, dim=128, rot=64, rank=512, vocab=32000, experts=8),
    "4k": dict(width=4096, heads=32, kv=8, ff=14336, span=4096, dim=128, rot=64, rank=512, vocab=32000, experts=8),
    "scout": dict(width=5120, heads=40, kv=8, ff=16384, span=8192, dim=128, rot=64, rank=512, vocab=202048, experts=16),
}
LAYERS = 4
YARN = {"factor": 4.0, "original": 8192, "fast": 32.0, "slow": 1.0}
FIRST, SECOND, OTHER, ROUTER_NORM = 8.0, 6.0, -6.0, 0.6  # how far a token lies along its experts' directions


def case(name, design, size, dtype="bfloat16", requests=1, prompt=2048, ragged=False, steps=0, portion=2048):
    return {"name": name, "design": design, "size": size, "dtype": dtype, "requests": requests, "prompt": prompt,
            "ragged": ragged, "steps": steps, "portion": portion}


def listed():
    return [
        # the smallest calls: a replay of a few tokens on a tiny float32 model; launches and the host are what it costs
        case("replay tiny fp32", "llama4-moe", "tiny", "float32", requests=3, prompt=40, ragged=True, steps=12, portion=32),
        # one user at a time on Llama 4 Scout's layers: a short question and its answer, bound by reading weights
        case("chat scout b1", "llama4-moe", "scout", prompt=97, steps=24),
        # a small server on the same layers: eight ragged prompts, then decoding together
        case("serve scout b8", "llama4-moe", "scout", requests=8, prompt=384, ragged=True, steps=12),
        # the benchmark's prompt on the same layers
        case("prompt scout 2048", "llama4-moe", "scout"),
        # a long document over two attention chunks on dense layers, in one step
        case("document dense 8191", "llama4-dense", "4k", prompt=8191, portion=8192),
        # the true float32 path: a prompt of ordinary length and some decoding
        case("float32 dense 777", "llama4-dense", "2k", "float32", requests=2, prompt=777, steps=8),
        # attention over a cached latent: the benchmark's prompt, and long contexts decoded together
        case("prompt rovidra 2048", "rovidra", "4k"),
        case("serve rovidra b8", "rovidra", "2k", requests=8, prompt=1100, ragged=True, steps=24),
        # a memory written by the delta rule beside attention with kept tokens: the benchmark's prompt, and many short chats
        case("prompt sudilorn 2048", "sudilorn", "2k"),
        case("serve sudilorn b64", "sudilorn", "2k", requests=64, prompt=80, ragged=True, steps=16),
        # a Mamba-2 memory, window and latent attention, routed experts: a prompt in two portions, and a mixed batch
        case("prompt folivik 3001", "folivik", "4k", prompt=3001),
        case("serve folivik b16", "folivik", "2k", requests=16, prompt=300, ragged=True, steps=24),
    ]


def draw(rng):
    """Any design at the sizes it is listed with or the next one, prompts and batches spread over their logarithms."""
    spread = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    design = rng.choice(["llama4-moe", "llama4-dense", "rovidra", "sudilorn", "folivik"])
    size = rng.choice(["tiny", "scout", "2k"] if design == "llama4-moe" else ["2k", "4k"])
    dtype = "float32" if size == "tiny" or design == "llama4-dense" and size == "2k" and rng.random() < 0.5 else "bfloat16"
    c = case("", design, size, dtype, requests=spread(1, 64), ragged=rng.random() < 0.5,
             steps=rng.choice([0, 0, spread(4, 24)]), portion=rng.choice([32, 48]) if size == "tiny" else 2048)
    if size == "scout":
        c["requests"], c["steps"] = min(c["requests"], 8), min(c["steps"], 12)
    if size == "4k":
        c["steps"] = min(c["steps"], 8)
    if size == "tiny":
        c["requests"] = min(c["requests"], 6)
    # (all prompts together are no longer than the longest listed one of their kind)
    total = {"tiny": 240, "scout": 3072}.get(size, 1600 if dtype == "float32" else 4096)
    c["prompt"] = min(spread(24, total), max(24, total // c["requests"]))
    del c["name"]
    return c


# ------------------------------------------------------------------------------------------------ configurations
def config(c):
    z, size = SIZES[c["size"]], c["size"]
    D, H, ff = z["width"], z["heads"], z["ff"]
    rot = {"base": 500000.0, "dims": z["rot"]}
    head = {"heads": H, "kv_heads": z["kv"], "dim": z["dim"], "vdim": z["dim"], "scale": z["dim"] ** -0.5}
    latent = {"heads": H, "dim": z["dim"], "rot_dim": z["rot"], "vdim": z["dim"], "kv_rank": z["rank"],
              "scale": (z["dim"] + z["rot"]) ** -0.5, "rot": rot}
    if c["design"].startswith("llama4"):
        moe = c["design"] == "llama4-moe"
        nope = moe  # (every fourth layer without rotation, with a temperature: Scout's arrangement)
        scout = {"rope_type": "llama3", "factor": 16.0, "low_freq_factor": 1.0, "high_freq_factor": 1.0,
                 "original_max_position_embeddings": 8192}
        return {"architectures": ["Llama4ForCausalLM"], "num_hidden_layers": LAYERS, "hidden_size": D,
                "num_attention_heads": H, "num_key_value_heads": z["kv"], "head_dim": z["dim"],
                "interleave_moe_layer_step": 1, "moe_layers": list(range(LAYERS)) if moe else [],
                "num_local_experts": z["experts"], "num_experts_per_tok": 1, "intermediate_size": ff // 2,
                "intermediate_size_mlp": ff, "vocab_size": z["vocab"], "rope_theta": 500000.0,
                "rope_scaling": scout if size == "scout" else None,
                "no_rope_layers": [0 if nope and i % 4 == 3 else 1 for i in range(LAYERS)],
                "attention_chunk_size": z["span"], "use_qk_norm": True, "attn_temperature_tuning": nope,
                "floor_scale": 16 if size == "tiny" else 8192, "attn_scale": 0.1, "rms_norm_eps": EPS,
                "tie_word_embeddings": False}
    if c["design"] == "rovidra":  # every second layer reads the latent of the layer before it
        return {"architecture": "Rovidra", "vocab": z["vocab"], "width": D, "embedding": {"scale": D ** 0.5},
                "norm": {"eps": EPS},
                "layers": [{"type": "latent_attention",
                            "mixer": dict(latent, mask={"size": z["span"]}, **({"kv_from": i - 1} if i % 2 else {})),
                            "mlp": {"kind": "dense", "ff": ff}} for i in range(LAYERS)]}
    if c["design"] == "sudilorn":
        pair = {"left": dict(head, mask={"size": z["span"], "keep_first": 8}, rot={"base": 10000.0, "dims": z["rot"]}),
                "right": {"heads": H, "kv_heads": z["kv"], "dim": z["dim"], "vdim": z["dim"], "conv": 4},
                "left_scale": 1.0, "right_scale": 0.7}
        maps = {"heads": H // 2, "kv_heads": z["kv"] // 2, "dim": z["dim"], "vdim": 2 * z["dim"], "conv": 4, "diff": 0.5,
                "scale": z["dim"] ** -0.5, "mask": {"size": z["span"]}, "rot": dict(rot, scaling=YARN)}
        moe = {"kind": "moe", "router": {"experts": 8, "top": 2, "groups": {"count": 4, "keep": 2}},
               "expert": {"ff": ff // 2}}
        return {"architecture": "Sudilorn", "vocab": z["vocab"], "width": D, "norm": {"eps": EPS}, "residual_mult": 0.7,
                "layers": [{"type": "attention" if i % 3 == 2 else "parallel", "mixer": maps if i % 3 == 2 else pair,
                            "mlp": moe} for i in range(LAYERS)]}
    memory = {"heads": D // 32, "vdim": 64, "state": 128, "groups": 8, "conv": 4, "norm_groups": 8}
    kinds = [("mamba2", memory), ("attention", dict(head, mask={"size": z["span"]})), ("mamba2", memory),
             ("latent_attention", dict(latent, q_rank=3 * z["rank"]))]
    moe = {"kind": "moe", "router": {"experts": 8, "top": 2, "identity": 2, "scale": 2.0, "groups": {"count": 5, "keep": 3}},
           "expert": {"ff": ff // 2}, "shared": {"ff": ff // 2}}
    return {"architecture": "Folivik", "vocab": z["vocab"], "width": D, "norm": {"eps": EPS},
            "layers": [{"type": t, "mixer": m, "mlp": moe} for t, m in kinds]}


# ------------------------------------------------------------------------------------------------ weights and tokens
UNIFORM = {"A_log": (-2.0, 1.0), "dt_bias": (-3.0, 0.0), "D": (0.5, 1.5), "shift": (0.0, 1.0), "act": (-1.0, 1.0),
           "ls1": (0.5, 1.5), "ls2": (0.5, 1.5), "r1": (0.2, 1.0), "r2": (0.05, 0.5), "temp": (0.8, 1.2)}
NORMAL = {"b": 0.3, "correction": 0.02, "lq1": 0.3, "lk1": 0.3, "lq2": 0.3, "lk2": 0.3}  # (vectors)


class Weights:
    """The case's checkpoint, drawn tensor by tensor, each by its own name: the engine is filled from it, and the plain
    64-bit model asks it for the same numbers."""

    def __init__(self, c, seed):
        self.c, self.seed, self.z = c, seed, SIZES[c["size"]]
        self.dtype = getattr(torch, c["dtype"])
        self.experts = {"llama4-moe": self.z["experts"], "sudilorn": 8, "folivik": 10}.get(c["design"], 0)
        self._directions = None

    def generator(self, name):
        h = hashlib.sha256(f"{self.seed}:{name}".encode()).digest()
        return torch.Generator(device=DEVICE).manual_seed(int.from_bytes(h[:7], "little"))

    def normal(self, name, shape, std, dtype):
        return torch.randn(shape, generator=self.generator(name), dtype=dtype, device=DEVICE).mul_(std)

    def directions(self):
        """[layers, experts, width]: orthonormal rows, a router's experts."""
        if self._directions is None:
            n = LAYERS * self.experts
            q, _ = torch.linalg.qr(self.normal("directions", (self.z["width"], n), 1.0, torch.float64).cpu())
            self._directions = q.T.reshape(LAYERS, self.experts, -1).float().to(DEVICE)
        return self._directions

    def embedding(self, shape):
        if self.c["design"] == "rovidra":
            return self.normal("embed", shape, self.z["width"] ** -0.5, self.dtype)
        x = self.normal("embed", shape, 1.0, torch.float32)
        if self.experts:
            u = self.directions().reshape(-1, shape[1])
            first = torch.randint(0, self.experts, (shape[0], LAYERS, 1), generator=self.generator("first"), device=DEVICE)
            step = torch.randint(1, self.experts, first.shape, generator=self.generator("second"), device=DEVICE)
            along = torch.full((shape[0], LAYERS, self.experts), OTHER, device=DEVICE)
            if self.c["design"] != "llama4-moe":  # (two experts a token)
                along.scatter_(2, (first + step) % self.experts, SECOND)
            along.scatter_(2, first, FIRST)
            x += (along.reshape(shape[0], -1) - x @ u.T) @ u
        return x.to(self.dtype)

    def __call__(self, name, shape):
        """The stored tensor ``name``, in the type that the engine keeps it in."""
        last = name.split(".")[-1]
        if name in ("embed", "model.embed_tokens.weight"):
            return self.embedding(shape)
        if "router" in name:
            layer = int(name.removeprefix("model.layers.").removeprefix("l").split(".")[0])
            return self.directions()[layer] * ROUTER_NORM
        if last in UNIFORM:
            lo, hi = UNIFORM[last]
            return torch.rand(shape, generator=self.generator(name), device=DEVICE) * (hi - lo) + lo
        if "norm" in name:
            one = 0.0 if self.c["design"] == "sudilorn" and ".mix." not in name else 1.0  # (its norms hold w of 1 + w)
            return self.normal(name, shape, 0.1, torch.float32) + one
        if last in NORMAL and len(shape) == 1:
            return self.normal(name, shape, NORMAL[last], torch.float32)
        fan = shape[1] if name.endswith("_proj") else shape[-1]  # (Llama's stacked experts are stored [expert, in, out])
        out = name.split(".")[-2 if name.endswith("weight") else -1] in ("o", "down", "o_proj", "down_proj")
        return self.normal(name, shape, (2 * LAYERS * fan if out else fan) ** -0.5, self.dtype)


def tokens(c, seed):
    """Prompts, and the tokens decoded behind them: [steps][requests]."""
    rng = random.Random(f"tokens {seed}")
    n, mean, vocab = c["requests"], c["prompt"], SIZES[c["size"]]["vocab"]
    # (every set of lengths has the same sum, so that other inputs are the same work)
    lengths = [mean if not c["ragged"] else max(1, int(round(mean * (0.5 + (i + 0.5) / n)))) for i in range(n)]
    rng.shuffle(lengths)
    prompts = [[rng.randrange(vocab) for _ in range(k)] for k in lengths]
    return prompts, [[rng.randrange(vocab) for _ in range(n)] for _ in range(c["steps"])]


def prepare(c, seed):
    top = config(c)
    arch = get_architecture(top.get("architecture") or top["architectures"][0])
    cfg = arch.parse_config(top)
    model = build_model(arch, cfg, c["dtype"], DEVICE)
    params, w = model.named_parameters(), Weights(c, seed)
    for b in arch.bindings(cfg, model.plan):
        place(params[b.target], b, w(b.name, tuple(b.shape)))
    model.finalize()
    prompts, forced = tokens(c, seed)
    longest = max(len(p) for p in prompts) + c["steps"]
    engine = Engine(model, cache_tokens=c["requests"] * (longest + 32), decode_batch_size=c["requests"],
                    max_num_batched_tokens=c["portion"])
    return {"engine": engine, "prompts": prompts, "forced": forced}


def run(state):
    engine = state["engine"]
    _, logits, ids = engine.prefill(state["prompts"])
    out = [logits]
    for last in state["forced"]:
        out.append(engine.decode_step(last, ids)[1])
    engine.release(ids)
    return out


# ------------------------------------------------------------------------------------------------ what it costs at least
def matrices(c):
    """(elements of the matrices that every token meets, of one expert, experts a token takes, layers with experts)."""
    z, d = SIZES[c["size"]], c["design"]
    D, H, G, dh, ff, r, rot = z["width"], z["heads"], z["kv"], z["dim"], z["ff"], z["rank"], z["rot"]
    if d.startswith("llama4"):
        per = D * dh * (2 * H + 2 * G)
        if d == "llama4-dense":
            return LAYERS * (per + 3 * D * ff), 0, 0, 0
        return LAYERS * (per + 3 * D * (ff // 2)), 3 * D * (ff // 2), 1, LAYERS
    latent = r * H * 2 * dh + H * dh * D
    if d == "rovidra":
        per = D * H * (dh + rot) + latent + 2 * D * D + 2 * D * ff
        return LAYERS * per + (LAYERS // 2) * D * (r + rot), 0, 0, 0
    if d == "sudilorn":
        pair = D * dh * (2 * H + 2 * G) + D * dh * (3 * H + 2 * G)
        maps = D * dh * (H + G + G + H + H)
        return 3 * pair + maps, 2 * D * (ff // 2), 2, LAYERS
    inner = 2 * D
    mem = D * (2 * inner + 2 * 8 * 128 + D // 32) + inner * D
    lat = D * 3 * r + 3 * r * H * (dh + rot) + D * (r + rot) + latent
    return 2 * mem + D * dh * (2 * H + 2 * G) + lat + LAYERS * 3 * D * (ff // 2), 3 * D * (ff // 2), 1.6, LAYERS


def work(c):
    """Every step reads the weights its tokens meet once and the cached rows its queries see, and writes its logits."""
    z, item = SIZES[c["size"]], 4 if c["dtype"] == "float32" else 2
    prompts, _ = tokens(c, 0)
    lengths = [len(p) for p in prompts]
    dense, expert, top, routed = matrices(c)
    head = z["width"] * z["vocab"]
    calls = [(c["portion"], 0)] * (sum(lengths) // c["portion"]) + [(sum(lengths) % c["portion"], c["requests"])]
    calls = [x for x in calls if x[0]] + [(c["requests"], c["requests"])] * c["steps"]
    bytes_, flops = 0.0, 0.0
    kept = {"llama4-moe": 2, "llama4-dense": 2, "rovidra": 2, "sudilorn": 2, "folivik": 1}[c["design"]]
    row = 2 * z["kv"] * z["dim"] if c["design"] != "rovidra" else (z["rank"] + z["rot"]) * 2 // 2
    for n, wanted in calls:
        met = routed * z["experts"] * (1.0 - (1.0 - top / z["experts"]) ** n) if routed else 0.0
        bytes_ += item * (dense + met * expert + (head if wanted else 0)) + 4.0 * wanted * z["vocab"]
        flops += 2.0 * n * (dense + routed * top * expert) + 2.0 * wanted * head
    for length in lengths:
        seen = lambda p: min(p + 1, z["span"])
        pairs = sum(seen(p) for p in range(length + c["steps"]))
        flops += kept / 2 * LAYERS * 4.0 * z["heads"] * z["dim"] * pairs
        bytes_ += item * LAYERS * row * (length + c["steps"] + sum(seen(length + s) for s in range(c["steps"])))
    return {"bytes": bytes_, "flops": flops}


def tolerance(c):
    """Four layers of bfloat16 products and caches, or of float32 sums and angles: against exact() 2.4e-3 (Llama 4)
    to 4.9e-3 (Rovidra) in bfloat16, 1.5e-7 (tiny) to 1.2e-6 (2,048 wide) in float32; four to eight times that."""
    return {"rel": 1e-5, "max": 4e-4} if c["dtype"] == "float32" else {"rel": 2e-2, "max": 0.2}


# ------------------------------------------------------------------------------------------------ the same in 64 bits
def rms(x):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + EPS)


def silu(x):
    return x * torch.sigmoid(x)


def causal_conv(u, taps, bias=0.0):
    K = taps.shape[1]
    rows = torch.cat([u.new_zeros(K - 1, u.shape[1]), u])
    return sum(taps[:, j] * rows[j: j + u.shape[0]] for j in range(K)) + bias


def turn(x, rates, adjacent, grow=1.0):
    """x [T, heads, d]: its leading 2 * len(rates) elements turned, in pairs of neighbours or of halves."""
    n = len(rates)
    angle = torch.arange(x.shape[0], dtype=x.dtype, device=x.device)[:, None] * torch.tensor(rates, dtype=x.dtype, device=x.device)
    cos, sin = torch.cos(angle)[:, None] * grow, torch.sin(angle)[:, None] * grow
    a, b = (x[..., 0: 2 * n: 2], x[..., 1: 2 * n: 2]) if adjacent else (x[..., :n], x[..., n: 2 * n])
    a, b = a * cos - b * sin, b * cos + a * sin
    turned = torch.stack([a, b], -1).flatten(-2) if adjacent else torch.cat([a, b], -1)
    return torch.cat([turned, x[..., 2 * n:]], -1)


def rates_of(rot, scaling=None):
    dims, base = rot["dims"], rot["base"]
    f = [base ** (-2.0 * i / dims) for i in range(dims // 2)]
    if scaling is None:
        return f, 1.0
    where = lambda t: dims * math.log(scaling["original"] / (2.0 * math.pi * t)) / (2.0 * math.log(base))
    lo, hi = max(math.floor(where(scaling["fast"])), 0), min(math.ceil(where(scaling["slow"])), dims - 1)
    ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(dims // 2)]
    return [x / scaling["factor"] * r + x * (1.0 - r) for x, r in zip(f, ramp)], 0.1 * math.log(scaling["factor"]) + 1.0


def attend(q, k, v, seen, score=lambda s, h: s):
    """q [T, H, d], k and v [T, G, .], seen [T, T]: softmax over the seen keys, head by head."""
    H, G = q.shape[1], k.shape[1]
    out = [torch.softmax(score(q[:, h] @ k[:, h * G // H].T, h).masked_fill(~seen, -math.inf), -1) @ v[:, h * G // H]
           for h in range(H)]
    return torch.stack(out, 1)


def back_of(h):
    """[T, T]: how many places back the key lies."""
    p = torch.arange(h.shape[0], device=h.device)
    return p[:, None] - p[None, :]


class Plain:
    """One sequence through the design, written from its equations, in 64 bits."""

    def __init__(self, c, seed):
        self.c, self.cfg, self.z, self.draw, self.drawn = c, config(c), SIZES[c["size"]], Weights(c, seed), {}

    def weights(self, name, shape):
        if name not in self.drawn:
            self.drawn[name] = self.draw(name, shape)
        return self.drawn[name]

    def w(self, name, *shape):
        return self.weights(name, shape).double()

    def linear(self, h, name, n):
        return h @ self.w(name, n, h.shape[1]).T

    def logits(self, sequences, wanted):
        """Per sequence [len(wanted of it), vocab]; layer by layer over all sequences, so that weights are drawn once."""
        z, d, D = self.z, self.c["design"], self.z["width"]
        llama = d.startswith("llama4")
        table = self.weights("model.embed_tokens.weight" if llama else "embed", (z["vocab"], D))
        xs = [table[torch.tensor(s, device=DEVICE)].double() for s in sequences]
        del table
        self.drawn.clear()
        if d == "rovidra":
            xs = [x * self.cfg["embedding"]["scale"] for x in xs]
        kept = [{} for _ in xs]
        for i in range(LAYERS):
            for j, x in enumerate(xs):
                xs[j] = (self.llama if llama else getattr(self, d))(x, i, kept[j])
            self.drawn.clear()
        norm = self.w("model.norm.weight" if llama else "final.norm", *(() if d == "folivik" else (D,)))
        rows = torch.cat([rms(x[torch.tensor(n, device=DEVICE)]) * (norm + (1.0 if d == "sudilorn" else 0.0)) for x, n in zip(xs, wanted)])
        head = self.weights("lm_head.weight" if llama else "head", (z["vocab"], D))
        out = torch.cat([rows @ piece.double().T for piece in head.split(16384)], 1)
        return out.split([len(n) for n in wanted])

    def gated(self, h, p, ff, names=("gate", "up", "down")):
        return self.linear(silu(self.linear(h, p + names[0], ff)) * self.linear(h, p + names[1], ff), p + names[2], h.shape[1])

    def llama(self, x, i, kept):
        z, c, p = self.z, self.cfg, f"model.layers.{i}."
        D, H, G, dh = z["width"], z["heads"], z["kv"], z["dim"]
        T = x.shape[0]
        h = rms(x) * self.w(p + "input_layernorm.weight", D)
        q, k, v = (self.linear(h, p + f"self_attn.{n}_proj.weight", m * dh).reshape(T, m, dh) for n, m in (("q", H), ("k", G), ("v", G)))
        back = back_of(h)
        seen = back >= 0
        if c["no_rope_layers"][i]:
            f, sc = rates_of({"base": c["rope_theta"], "dims": dh})[0], c["rope_scaling"]
            if sc is not None:  # (low and high factor are equal: no band between the two)
                f = [r / sc["factor"] if 2 * math.pi / r > sc["original_max_position_embeddings"] / sc["low_freq_factor"] else r for r in f]
            q, k = rms(turn(q, f, True)), rms(turn(k, f, True))
            chunk = torch.arange(T, device=DEVICE) // c["attention_chunk_size"]
            seen = seen & (chunk[:, None] == chunk[None, :])
        else:
            at = torch.arange(T, device=DEVICE, dtype=x.dtype)
            q = q * (1.0 + c["attn_scale"] * torch.log1p(torch.floor((at + 1.0) / c["floor_scale"])))[:, None, None]
        x = x + self.linear(attend(q * dh ** -0.5, k, v, seen).flatten(1), p + "self_attn.o_proj.weight", D)
        h = rms(x) * self.w(p + "post_attention_layernorm.weight", D)
        p += "feed_forward."
        names = ("gate_proj.weight", "up_proj.weight", "down_proj.weight")
        if self.c["design"] == "llama4-dense":
            return x + self.gated(h, p, z["ff"], names)
        E, ff = z["experts"], z["ff"] // 2
        score = h @ self.w(p + "router.weight", E, D).T
        gate_up, down = self.weights(p + "experts.gate_up_proj", (E, D, 2 * ff)), self.weights(p + "experts.down_proj", (E, ff, D))
        best = score.argmax(-1)
        out = self.gated(h, p + "shared_expert.", ff, names)
        for e in range(E):
            rows = (best == e).nonzero()[:, 0]
            if len(rows):
                a = (h[rows] * torch.sigmoid(score[rows, e: e + 1])) @ gate_up[e].double()
                out[rows] += (silu(a[:, :ff]) * a[:, ff:]) @ down[e].double()
        return x + out

    def rovidra(self, x, i, kept):
        z, p, m = self.z, f"l{i}.", self.cfg["layers"][i]["mixer"]
        D, H, dn, dr, r = z["width"], z["heads"], z["dim"], z["rot"], z["rank"]
        T = x.shape[0]
        rates = rates_of(m["rot"])[0]
        gate = lambda y, h, n: rms(y * torch.sigmoid(self.linear(h, p + f"rg{n}", D) + self.w(p + f"rg{n}.b", D))) * self.w(p + f"norm{n}b", D)
        h = rms(x) * self.w(p + "norm1", D)
        hs = h + (torch.cat([torch.zeros_like(h[:1]), h[:-1]]) - h) * self.w(p + "shift", D)
        if m.get("kv_from") is None:
            down = self.linear(hs, p + "mix.dkv", r + dr)
            kept["latent"] = rms(down[:, :r]) * self.w(p + "mix.dkv.norm", r), turn(down[:, None, r:], rates, False)
        y = self.latent(hs, p, m, kept["latent"], self.linear(hs, p + "mix.q", H * (dn + dr)), rates, False)
        x = x + gate(self.linear(y.flatten(1), p + "mix.o", D), h, 1)
        h = rms(x) * self.w(p + "norm2", D)
        a = self.linear(h, p + "mlp.up", z["ff"]) + self.w(p + "mlp.up.b", z["ff"])
        co = self.w(p + "mlp.act", 4)
        a = co[0] * rms(a) + co[1] * rms(a ** 2) + co[2] * rms(a ** 3) + co[3]
        return x + gate(self.linear(a, p + "mlp.down", D) + self.w(p + "mlp.down.b", D), h, 2)

    def latent(self, h, p, m, kept, q, rates, adjacent):
        """Every head's keys and values formed from the latent."""
        z, T = self.z, h.shape[0]
        H, dn, dr, r = z["heads"], z["dim"], z["rot"], z["rank"]
        c, shared = kept
        q = q.reshape(T, H, dn + dr)
        q = torch.cat([q[..., :dn], turn(q[..., dn:], rates, adjacent)], -1) * m["scale"]
        k = torch.cat([self.linear(c, p + "mix.uk", H * dn).reshape(T, H, dn), shared.expand(T, H, dr)], -1)
        back = back_of(h)
        seen = (back >= 0) & (back < m["mask"]["size"]) if m.get("mask") else back >= 0
        return attend(q, k, self.linear(c, p + "mix.uv", H * dn).reshape(T, H, dn), seen)

    def chosen(self, s, correction, groups, keep, best_of):
        """[T, 2]: the two experts of the largest corrected score within the best groups."""
        cs = (s + correction).reshape(s.shape[0], groups, -1)
        score = cs.topk(best_of, -1).values.sum(-1)
        allowed = torch.zeros_like(score, dtype=torch.bool).scatter_(1, score.topk(keep, -1).indices, True)
        return cs.masked_fill(~allowed[..., None], -math.inf).flatten(1).topk(2, -1).indices

    def sudilorn(self, x, i, kept):
        z, p, mult = self.z, f"l{i}.", self.cfg["residual_mult"]
        D, T, layer = z["width"], x.shape[0], self.cfg["layers"][i]
        h = rms(x) * (1.0 + self.w(p + "norm1", D))
        m = layer["mixer"]
        y = self.two_maps(h, p + "mix.", m) if layer["type"] == "attention" else (
            m["left_scale"] * self.kept_window(h, p + "mix.left.", m["left"]) + m["right_scale"] * self.delta(h, p + "mix.right.", m["right"]))
        x = x + mult * self.w(p + "ls1", D) * y
        h = rms(x) * (1.0 + self.w(p + "norm2", D))
        s = torch.sigmoid(h @ self.w(p + "mlp.router", 8, D).T)
        best = self.chosen(s, self.w(p + "mlp.correction", 8), 4, 2, 2)
        out = torch.zeros_like(h)
        for e in range(8):
            rows = (best == e).any(-1).nonzero()[:, 0]
            if len(rows):
                a = torch.relu(self.linear(h[rows], p + f"mlp.e{e}.up", z["ff"] // 2)) ** 2
                out[rows] += s[rows, e: e + 1] * self.linear(a, p + f"mlp.e{e}.down", D)
        return x + mult * self.w(p + "ls2", D) * out

    def two_maps(self, h, p, m):
        T, H, G, dk, dv = h.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        conv = lambda n, width: causal_conv(self.linear(h, p + n, width), self.w(p + n + ".conv", width, 4))
        rates, grow = rates_of(m["rot"], m["rot"]["scaling"])
        q, k = (turn(rms(conv(n, g * 2 * dk).reshape(T, g * 2, dk)) * self.w(p + n + ".norm", dk), rates, False, grow) for n, g in (("q", H), ("k", G)))
        v = conv("v", G * dv).reshape(T, G, dv)
        lam = [torch.exp((self.w(p + f"lq{n}", dk) * self.w(p + f"lk{n}", dk)).sum()) for n in (1, 2)]
        back = back_of(h)
        seen = (back >= 0) & (back < m["mask"]["size"])
        a, b = (attend(q[:, n::2] * m["scale"], k[:, n::2], v, seen) for n in (0, 1))
        o = rms(a - (lam[0] - lam[1] + m["diff"]) * b) * (1.0 - m["diff"])
        return self.linear(o.flatten(1) * torch.sigmoid(self.linear(h, p + "g", H * dv)), p + "o", h.shape[1])

    def kept_window(self, h, p, m):
        T, H, G, dk = h.shape[0], m["heads"], m["kv_heads"], m["dim"]
        q, k, v = ((self.linear(h, p + n, g * dk) + self.w(p + n + ".b", g * dk)).reshape(T, g, dk) for n, g in (("q", H), ("k", G), ("v", G)))
        rates = rates_of(m["rot"])[0]
        back = back_of(h)
        first = (torch.arange(T, device=DEVICE) < m["mask"]["keep_first"])[None, :]
        seen = (back >= 0) & ((back < m["mask"]["size"]) | first)
        o = attend(turn(q, rates, True) * m["scale"], turn(k, rates, True), v, seen)
        return self.linear(o.flatten(1), p + "o", h.shape[1])

    def delta(self, h, p, m):
        T, H, G, dk, dv = h.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q, k, v = (silu(causal_conv(self.linear(h, p + n, g * e), self.w(p + n + ".conv", g * e, 4))).reshape(T, g, e)
                   for n, g, e in (("q", G, dk), ("k", G, dk), ("v", H, dv)))
        unit = lambda u: (u / torch.sqrt((u * u).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 1)
        q, k = unit(q) * dk ** -0.5, unit(k)
        beta = torch.sigmoid(self.linear(h, p + "b", H))
        decay = torch.exp(-torch.exp(self.w(p + "A_log", H)) * torch.nn.functional.softplus(self.linear(h, p + "a", H) + self.w(p + "dt_bias", H)))
        S, out = h.new_zeros(H, dk, dv), []
        for t in range(T):
            S = S * decay[t][:, None, None]
            u = beta[t][:, None] * (v[t] - (k[t][:, None] @ S)[:, 0])
            S = S + k[t][:, :, None] * u[:, None]
            out.append((q[t][:, None] @ S)[:, 0])
        o = rms(torch.stack(out)) * self.w(p + "norm", dv)
        return self.linear(o.flatten(1) * silu(self.linear(h, p + "g", H * dv)), p + "o", h.shape[1])

    def folivik(self, x, i, kept):
        z, p, layer = self.z, f"l{i}.", self.cfg["layers"][i]
        D, ff, m = z["width"], z["ff"] // 2, self.cfg["layers"][i]["mixer"]
        h = rms(x) * self.w(p + "norm1")
        x = x + {"mamba2": self.memory, "attention": self.penalised, "latent_attention": self.through_latent}[layer["type"]](h, p, m)
        h = rms(x) * self.w(p + "norm2")
        s = torch.softmax(h @ self.w(p + "mlp.router", 10, D).T, -1)
        best = self.chosen(s, self.w(p + "mlp.correction", 10), 5, 3, 1)
        share = torch.zeros_like(s).scatter_(1, best, s.gather(1, best))
        share = share / (share.sum(-1, keepdim=True) + 1e-20) * layer["mlp"]["router"]["scale"]
        out = self.gated(h, p + "mlp.shared.", ff) + share[:, 8:].sum(-1, keepdim=True) * h
        for e in range(8):
            rows = share[:, e].nonzero()[:, 0]
            if len(rows):
                out[rows] += share[rows, e: e + 1] * self.gated(h[rows], p + f"mlp.e{e}.", ff)
        return x + out

    def memory(self, h, p, m):
        T, H, P, N, G = h.shape[0], m["heads"], m["vdim"], m["state"], m["groups"]
        inner, p = H * P, p + "mix."
        rows = self.linear(h, p + "in", 2 * inner + 2 * G * N + H)
        gate, u, dt = rows.split([inner, inner + 2 * G * N, H], 1)
        y = silu(causal_conv(u, self.w(p + "conv", u.shape[1], 4), self.w(p + "conv.b", u.shape[1])))
        v, B, C = y.split([inner, G * N, G * N], 1)
        v = v.reshape(T, H, P)
        B, C = (a.reshape(T, G, N).repeat_interleave(H // G, 1) for a in (B, C))
        dt = torch.nn.functional.softplus(dt + self.w(p + "dt_bias", H))
        decay = torch.exp(-torch.exp(self.w(p + "A_log", H)) * dt)
        S, out = h.new_zeros(H, N, P), []
        for t in range(T):
            S = decay[t][:, None, None] * S + (dt[t][:, None] * B[t])[:, :, None] * v[t][:, None]
            out.append((C[t][:, None] @ S)[:, 0])
        y = (torch.stack(out) + self.w(p + "D", H)[:, None] * v).flatten(1) * silu(gate)
        y = rms(y.reshape(T, m["norm_groups"], -1)).flatten(1) * self.w(p + "norm", inner)
        return self.linear(y, p + "o", h.shape[1])

    def penalised(self, h, p, m):
        T, H, G, dk, p = h.shape[0], m["heads"], m["kv_heads"], m["dim"], p + "mix."
        q, k = (rms(self.linear(h, p + n, g * dk).reshape(T, g, dk)) * self.w(p + n + ".norm", dk) for n, g in (("q", H), ("k", G)))
        v = self.linear(h, p + "v", G * dk).reshape(T, G, dk)
        temp, r1, r2 = (self.w(p + n, H) for n in ("temp", "r1", "r2"))
        back = back_of(h)
        away = back.clamp(min=0).double()
        o = attend(q * m["scale"], k, v, (back >= 0) & (back < m["mask"]["size"]),
                   lambda s, hd: s * temp[hd] - r1[hd] * torch.log(1.0 + r2[hd] * away))
        return self.linear(o.flatten(1), p + "o", h.shape[1])

    def through_latent(self, h, p, m):
        T, H, r, dr, qr = h.shape[0], m["heads"], m["kv_rank"], m["rot_dim"], m["q_rank"]
        rates = rates_of(m["rot"])[0]
        q = self.linear(rms(self.linear(h, p + "mix.dq", qr)) * self.w(p + "mix.dq.norm", qr), p + "mix.uq", H * (m["dim"] + dr))
        down = self.linear(h, p + "mix.dkv", r + dr)
        kept = rms(down[:, :r]) * self.w(p + "mix.dkv.norm", r), turn(down[:, None, r:], rates, True)
        o = self.latent(h, p, m, kept, q, rates, True) * torch.sigmoid(self.linear(h, p + "mix.g", H))[..., None]
        return self.linear(o.flatten(1), p + "mix.o", h.shape[1])


@torch.no_grad()
def exact(c, seed):
    prompts, forced = tokens(c, seed)
    sequences = [p + [row[j] for row in forced] for j, p in enumerate(prompts)]
    got = Plain(c, seed).logits(sequences, [list(range(len(p) - 1, len(s))) for p, s in zip(prompts, sequences)])
    return [torch.stack([g[k] for g in got]) for k in range(c["steps"] + 1)]
