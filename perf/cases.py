"""What is timed when this framework's speed is discussed: the calls that a serving program makes, over the sizes it meets.

The dense graph (Qwen3-0.6B and Qwen3-8B shapes) is driven through ModelRunner / BlockManager / Sequence (one model step and its sampled tokens) and
through LLMEngine.generate (whole requests), a layer-list model through LLMEngine.generate.  Weights are synthetic: the framework's own seeded
generator fills the matrices, and the norm gains are chosen so that the token's embedding stands out of the residual stream behind the last layer: the
greedy choice is then as clear as a trained model's usually is (with gains of 1 the two best of 150 thousand random logits lie closer together than
16-bit rounding in some rows of a hundred, and an answer that takes the other one goes its own way from there on).  float16 cases are the reference's
graph (no head norms), bfloat16 ones the published checkpoints' (norms over the heads of q and k).

A case is a dict:
  path   "decode"   one step that extends `batch` sequences of `shortest` .. `longest` cached tokens (spread geometrically) by a token
         "prefill"  one step over `batch` prompts of `shortest` .. `longest` tokens, of which the first `cached` share (0 .. 1) were computed by an earlier step
         "generate" `batch` requests of `prompt` tokens, the first `shared` of them common to all, until each has `new` tokens
         "layers"   the same on a layer-list model (attention and retention layers in turn)
"""
import math

import numpy as np
import torch

import nvr_import

BLOCK = 256
MODELS = {  # the two shapes of nvr.ModelConfig's presets
    "qwen3-0.6b": dict(V=151936, W=1024, F=3072, L=28, H=16, G=8, D=128, base=1e6, gains=(0.006, 0.06)),
    "qwen3-8b": dict(V=151936, W=4096, F=12288, L=36, H=32, G=8, D=128, base=1e6, gains=(0.002, 0.024)),
}
LAYERS = dict(V=32768, W=1024, F=3072, L=4, H=16, G=8, D=128)  # the smallest size of the framework's own model comparison
EPS, STD = 1e-6, 0.02


def listed():
    small, large = "qwen3-0.6b", "qwen3-8b"
    return [
        # one user typing: the smallest step there is, launches and latency
        dict(name="chat", path="decode", model=small, dtype="float16", batch=1, shortest=128, longest=128, temperature=0.0),
        # the framework's headline: a full decode batch of equal contexts
        dict(name="decode-32", path="decode", model=small, dtype="float16", batch=32, shortest=1024, longest=1024, temperature=0.0),
        # a server's mixed batch: contexts of all lengths, tokens drawn with top-k and top-p
        dict(name="mixed-sampled", path="decode", model=small, dtype="bfloat16", batch=27, shortest=64, longest=8100, temperature=0.8),
        # a throughput server
        dict(name="decode-256", path="decode", model=small, dtype="bfloat16", batch=256, shortest=1024, longest=1024, temperature=0.0),
        # one short prompt: the time to its first token
        dict(name="first-token", path="prefill", model=small, dtype="bfloat16", batch=1, shortest=509, longest=509, cached=0.0),
        # the largest step: a full token budget of prompts
        dict(name="prefill-32k", path="prefill", model=small, dtype="float16", batch=32, shortest=1024, longest=1024, cached=0.0),
        # portions of long prompts behind what earlier portions left in the cache
        dict(name="portions", path="prefill", model=small, dtype="bfloat16", batch=3, shortest=3001, longest=7507, cached=0.75),
        # the larger model: a decode batch, and two prompts
        dict(name="large-decode", path="decode", model=large, dtype="float16", batch=32, shortest=2048, longest=2048, temperature=0.0),
        dict(name="large-prefill", path="prefill", model=large, dtype="bfloat16", batch=2, shortest=1531, longest=1531, cached=0.0),
        # 32-bit storage and arithmetic: one prompt and its answer
        dict(name="single-precision", path="generate", model=small, dtype="float32", batch=1, prompt=128, shared=0, new=48),
        # requests behind one system prompt, through the scheduler and the prefix cache
        dict(name="system-prompt", path="generate", model=small, dtype="float16", batch=64, prompt=577, shared=512, new=16),
        # a layer-list model: prompts and their answers
        dict(name="layer-list", path="layers", dtype="bfloat16", batch=16, prompt=1024, shared=0, new=32),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["decode"] * 4 + ["prefill"] * 4 + ["generate"] * 3 + ["layers"])
    dtype = rng.choice(["float16", "bfloat16"])
    if kind == "decode":
        model = rng.choice(["qwen3-0.6b"] * 6 + ["qwen3-8b"])
        batch = _log(rng, 1, 256 if model == "qwen3-0.6b" else 48)
        longest = _log(rng, 48, min(8100, (262144 if model == "qwen3-0.6b" else 65536) // batch))
        return dict(path=kind, model=model, dtype=dtype, batch=batch, shortest=_log(rng, min(longest, 32), longest), longest=longest, temperature=rng.choice([0.0, 0.0, 0.8]))
    if kind == "prefill":
        model = rng.choice(["qwen3-0.6b"] * 6 + ["qwen3-8b"])
        total = _log(rng, 24, 32768 if model == "qwen3-0.6b" else 3000)  # tokens of the step
        batch = _log(rng, 1, max(1, min(64, total // 24)))
        cached = rng.choice([0.0, 0.0, 0.5, 0.8])
        longest = min(8100, int(total / batch / (1 - cached)))
        return dict(path=kind, model=model, dtype=dtype, batch=batch, shortest=_log(rng, max(1, longest // 4), longest), longest=longest, cached=cached)
    if kind == "generate":
        if rng.random() < 0.33:
            return dict(path=kind, model="qwen3-0.6b", dtype="float32", batch=rng.choice([1, 1, 2]), prompt=_log(rng, 9, 120), shared=0, new=_log(rng, 4, 36))
        batch = _log(rng, 1, 64)
        shared = rng.choice([0, 256, 512])
        return dict(path=kind, model="qwen3-0.6b", dtype=dtype, batch=batch, prompt=shared + _log(rng, 8, 128), shared=shared, new=_log(rng, 4, 24))
    return dict(path=kind, dtype=rng.choice(["bfloat16", "bfloat16", "float32"]), batch=_log(rng, 1, 8), prompt=_log(rng, 16, 512), shared=0, new=_log(rng, 4, 32))


# ---------------------------------------------------------------------------------------------------------------- sizes of a case
def _lengths(case):
    """Tokens of each sequence, spread geometrically over the case's range, long and short ones mixed."""
    b, lo, hi = case["batch"], case["shortest"], case["longest"]
    n = [int(round(lo * (hi / lo) ** (i / max(1, b - 1)))) for i in range(b)] if b > 1 else [hi]
    return [n[(i * 7) % b] for i in range(b)] if b % 7 else n


def _cached(case, n):
    """Tokens of a prompt of n that an earlier step computed."""
    return min(n - 1, int(n * case["cached"]))


def _blocks(case):
    """Block tables of the step's sequences: consecutive blocks, one sequence after the other; a decode step's new token may need one more."""
    tables, at = [], 0
    lengths = _lengths(case)
    for n in lengths:
        k = -(-n // BLOCK)
        tables.append(list(range(at, at + k)))
        at += k
    if case["path"] == "decode":
        for t, n in zip(tables, lengths):
            if n % BLOCK == 0:
                t.append(at)
                at += 1
    return tables, at


def _rng(seed):
    return np.random.default_rng([seed, 20])


def _tokens(case, seed):
    """Token ids of each sequence (a decode case's with the token of the step) or request."""
    rng = _rng(seed)
    if case["path"] in ("generate", "layers"):
        V = LAYERS["V"] if case["path"] == "layers" else MODELS[case["model"]]["V"]
        head = rng.integers(0, V, case["shared"])
        return [np.concatenate([head, rng.integers(0, V, case["prompt"] - case["shared"])]).astype(np.int64) for _ in range(case["batch"])]
    V = MODELS[case["model"]]["V"]
    return [rng.integers(0, V, n + (case["path"] == "decode")).astype(np.int64) for n in _lengths(case)]


def _gains(case, seed):
    """The norm gains of a dense model by tensor name, in 32 bits."""
    m, rng = MODELS[case["model"]], np.random.default_rng([seed, 21])

    def g(n, mean):
        return (mean * (1 + 0.2 * rng.standard_normal(n))).astype(np.float32)
    out = {"norm.weight": g(m["W"], 1.0)}
    for l in range(m["L"]):
        p = "layers.%d." % l
        out[p + "input_layernorm.weight"] = g(m["W"], m["gains"][0])
        out[p + "post_attention_layernorm.weight"] = g(m["W"], m["gains"][1])
        if case["dtype"] == "bfloat16":
            out[p + "self_attn.q_norm.weight"] = g(m["D"], 1.0)
            out[p + "self_attn.k_norm.weight"] = g(m["D"], 1.0)
    return out


def _layers_config():
    s, layers = LAYERS, []
    for i in range(s["L"]):
        mixer = {"heads": s["H"], "dim": s["D"], "vdim": s["D"]}
        if i % 2 == 0:
            mixer.update(kv_heads=s["G"], scale=s["D"] ** -0.5)
        else:
            mixer.update(decay=[1.0 - 2.0 ** (-5 - 3 * j / (s["H"] - 1)) for j in range(s["H"])], rot={"dims": s["D"], "base": 10000.0})
        layers.append({"type": "retention" if i % 2 else "attention", "mixer": mixer, "mlp": {"kind": "dense", "ff": s["F"], "limit": 7.0}})
    return {"architecture": "Rugudra", "vocab": s["V"], "width": s["W"], "residual_mult": 0.5, "embedding": {"scale": 1.0}, "norm": {"eps": 1e-5},
            "canon": {"taps": 4}, "layers": layers}


def _layers_weights(seed):
    """Tensors of the layer-list model by name, with values that bfloat16 holds exactly."""
    s = LAYERS
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 2 + 1)

    def t(*shape, std=1.0, mean=0.0):
        return (mean + std * torch.randn(*shape, generator=g, device="cuda")).to(torch.bfloat16)

    def lin(o, i):
        return t(o, i, std=i ** -0.5)
    W, F, H, G, D = s["W"], s["F"], s["H"], s["G"], s["D"]
    out = {"embed": t(s["V"], W), "final.norm": t(1, mean=1.0, std=0.0)}
    out["head"] = out["embed"] * (W ** -0.5)  # (a power of two: exact)
    for i in range(s["L"]):
        p = "l%d." % i
        out[p + "norm1"], out[p + "norm2"] = t(1, mean=1.0, std=0.1), t(1, mean=1.0, std=0.1)
        out[p + "canon1"], out[p + "canon2"] = t(W, 4, std=0.2), t(W, 4, std=0.2)
        kv = H if i % 2 else G
        out[p + "mix.q"], out[p + "mix.k"], out[p + "mix.v"], out[p + "mix.o"] = lin(H * D, W), lin(kv * D, W), lin(kv * D, W), lin(W, H * D)
        if i % 2:
            out[p + "mix.g"] = lin(H * D, W)
        else:
            out[p + "mix.r1"], out[p + "mix.r2"], out[p + "mix.sink"] = t(H, mean=0.5, std=0.1).abs(), t(H, mean=0.25, std=0.05).abs(), t(H)
        out[p + "mlp.gate"], out[p + "mlp.up"], out[p + "mlp.down"] = lin(F, W), lin(F, W), lin(W, F)
    return out


# ---------------------------------------------------------------------------------------------------------------- state and pass
class _Memory:
    """Device memory of a runner as a tensor sees it; the tensor keeps the runner alive."""

    def __init__(self, owner, pointer, shape, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "data": (pointer, False), "version": 3, "strides": None}


def _view(owner, pointer, shape, dtype):
    kinds = {torch.float32: "<f4", torch.float16: "<f2", torch.bfloat16: "<i2"}
    return torch.as_tensor(_Memory(owner, pointer, shape, kinds[dtype]), device="cuda").view(dtype)


class _State:
    pass


def prepare(case, seed):
    nvr = nvr_import.load()
    nvr.lib().nvr_seq_reset_id_counter()  # (the sampler's random numbers go by the sequence's id)
    s, tokens = _State(), _tokens(case, seed)
    s.case = case
    if case["path"] == "layers":
        n = case["prompt"] + case["new"]
        config = nvr.Config(max_num_seqs=case["batch"], max_num_batched_tokens=case["batch"] * case["prompt"], max_model_len=n, kvcache_block_size=BLOCK,
                            num_kvcache_blocks=case["batch"] * (-(-n // BLOCK)), dtype=case["dtype"])
        s.engine = nvr.LLMEngine(config, nvr.ModelSpec(_layers_config()))
        for name, t in _layers_weights(seed).items():
            if t.numel() == 1:
                s.engine.model_runner.load_tensor(name, np.float32(t.item()))
            else:
                s.engine.model_runner.load_tensor(name, t.view(torch.int16).cpu().numpy().view(np.uint16))
    else:
        m = MODELS[case["model"]]
        model = nvr.ModelConfig(case["model"], tie_word_embeddings=1, seed=seed, qk_norm=int(case["dtype"] == "bfloat16"))
        if case["path"] == "generate":
            n = case["prompt"] + case["new"]
            config = nvr.Config(max_num_seqs=case["batch"], max_num_batched_tokens=max(512, case["batch"] * case["prompt"]), max_model_len=n, kvcache_block_size=BLOCK,
                                num_kvcache_blocks=case["batch"] * (-(-n // BLOCK)), dtype=case["dtype"])
            s.engine = nvr.LLMEngine(config, model)
            runner = s.engine.model_runner
        else:
            lengths, (_, blocks) = _lengths(case), _blocks(case)
            budget = min(32768, sum(lengths))
            config = nvr.Config(max_num_seqs=case["batch"], max_num_batched_tokens=max(512, budget, *lengths), max_model_len=max(lengths) + 1, kvcache_block_size=BLOCK,
                                num_kvcache_blocks=blocks, dtype=case["dtype"], enable_chunked_prefill=int(case.get("cached", 0) > 0))
            s.runner = runner = nvr.ModelRunner(config, model)
        for name, gain in _gains(case, seed).items():
            runner.load_tensor(name, gain)
    if case["path"] in ("generate", "layers"):
        s.prompts = tokens
        s.sampling = nvr.SamplingParams(temperature=0.0, max_tokens=case["new"], ignore_eos=True)
        return s
    hot = case.get("temperature", 0.0) > 0
    sampling = nvr.SamplingParams(temperature=case["temperature"], top_k=50, top_p=0.9, ignore_eos=True) if hot else nvr.SamplingParams(temperature=0.0, ignore_eos=True)
    s.manager = nvr.BlockManager(blocks, BLOCK)
    s.seqs = [nvr.Sequence(t[:n], sampling, BLOCK) for t, n in zip(tokens, lengths)]
    for q in s.seqs:
        s.manager.allocate(q)
    decode = case["path"] == "decode"
    earlier = lengths if decode else [_cached(case, n) for n in lengths]  # what earlier steps computed, in steps of the token budget
    group, held = [], 0
    for i, k in enumerate(earlier):
        if k == 0:
            continue
        if held + k > budget and group:
            runner.execute_model(group, True)
            group, held = [], 0
        if not decode:
            s.seqs[i].set_chunk(0, k)
        group.append(s.seqs[i])
        held += k
    if group:
        runner.execute_model(group, True)
    for q, t, k, n in zip(s.seqs, tokens, earlier, lengths):
        if decode:
            q.append_token(int(t[-1]))
            s.manager.may_append(q)
        elif case["cached"] > 0:
            q.set_chunk(k, n - k)
    kind = {"float16": torch.float16, "bfloat16": torch.bfloat16}[case["dtype"]]
    s.k, s.v = (_view(runner, p, (blocks, BLOCK, m["G"], m["D"]), kind) for p in runner.kv_cache(m["L"] - 1))
    s.logits_at, s.logits = None, None
    return s


def run(s):
    """Logits and tokens; of a single step also what it left in the last layer's caches, which all layers have a part in."""
    if s.case["path"] in ("generate", "layers"):
        out = s.engine.generate(s.prompts, s.sampling)
        return {"tokens": np.array([o.completion_token_ids for o in out]), "logits": s.engine.model_runner.logits(len(out))}
    pointer = s.runner.execute_model(s.seqs, s.case["path"] == "prefill")
    tokens = s.runner.sample_tokens(s.seqs)
    if pointer != s.logits_at:
        s.logits_at, s.logits = pointer, _view(s.runner, pointer, (len(s.seqs), MODELS[s.case["model"]]["V"]), torch.float32)
    return {"tokens": np.array(tokens), "logits": s.logits, "k": s.k, "v": s.v}


# ---------------------------------------------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    size = 4 if case["dtype"] == "float32" else 2
    m = LAYERS if case["path"] == "layers" else MODELS[case["model"]]
    qkvo = (2 * m["H"] + 2 * m["G"]) * m["D"] * m["W"]
    if case["path"] == "layers":
        matrices = m["L"] * 3 * m["F"] * m["W"] + m["L"] // 2 * (qkvo + 5 * m["H"] * m["D"] * m["W"])
        caching = m["L"] // 2
    else:
        matrices = m["L"] * (qkvo + 3 * m["F"] * m["W"])
        caching = m["L"]
    head = m["V"] * m["W"]
    row = 2 * m["G"] * m["D"] * size * caching  # cached bytes of a token
    pair = 4 * m["H"] * m["D"] * caching  # operations of a (query, key) pair

    def step(new, before):  # one model step: `new` tokens of each sequence behind `before` cached ones
        t, b = sum(new), len(new)
        pairs = sum(n * p + n * (n + 1) // 2 for n, p in zip(new, before))
        state = 2 * b * m["H"] * m["D"] * m["D"] * 4 * (m["L"] // 2) if case["path"] == "layers" else 0  # (retention's, read and written)
        fed = t * 4 * m["H"] * m["D"] * m["D"] * (m["L"] // 2) if case["path"] == "layers" else 0
        bytes_ = (matrices + head + t * m["W"]) * size + (t + sum(before)) * row + b * m["V"] * 4 + state
        return bytes_, 2 * matrices * t + 2 * head * b + pairs * pair + fed

    if case["path"] == "decode":
        n = _lengths(case)
        steps = [step([1] * len(n), n)]
    elif case["path"] == "prefill":
        n = _lengths(case)
        c = [_cached(case, k) for k in n]
        steps = [step([k - e for k, e in zip(n, c)], c)]
    else:
        b, p = case["batch"], case["prompt"]
        shared = case["shared"] // BLOCK * BLOCK
        steps = [step([p] + [p - shared] * (b - 1), [0] + [shared] * (b - 1))]
        for i in range(case["new"] - 1):
            ctx = [p + i] * b
            by, fl = step([1] * b, ctx)
            steps.append((by - (b - 1) * shared * row, fl))  # (the shared rows are read once)
    return {"bytes": float(sum(x for x, _ in steps)), "flops": float(sum(x for _, x in steps))}


def tolerance(case):
    """About four times what the framework is off the values in 64 bits (bfloat16: twice): 1.6e-3 in float16 and 1.3e-2 in bfloat16 after the 28 to 36 layers of a dense
    model (the last layer's keys and values included; two correct orders of the sums differ by about as much), 5e-3 after the 4 of the layer list, and 8e-7
    in float32 (1e-5: a sum over 3072 products may be taken in any order)."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 4e-4}
    return {"rel": 6e-3, "max": 0.1} if case["dtype"] == "float16" else {"rel": 0.03, "max": 0.5}


# ---------------------------------------------------------------------------------------------------------------- the same in 64 bits
def _signed(x):
    x &= (1 << 64) - 1
    return x - (1 << 64) if x >> 63 else x


def _mix(x):
    """splitmix64 of an integer, or of a tensor of 64-bit integers."""
    def down(z, n):
        return (z >> n) & ((1 << (64 - n)) - 1)
    if isinstance(x, int):
        x = (x + 0x9E3779B97F4A7C15) & ((1 << 64) - 1)
        x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & ((1 << 64) - 1)
        x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & ((1 << 64) - 1)
        return x ^ (x >> 31)
    x = x + _signed(0x9E3779B97F4A7C15)
    x = (x ^ down(x, 30)) * _signed(0xBF58476D1CE4E5B9)
    x = (x ^ down(x, 27)) * _signed(0x94D049BB133111EB)
    return x ^ down(x, 31)


def _matrix(seed, tid, rows, cols, dtype):
    """A matrix of the synthetic weights: four 16-bit fields of a hash of the element's index, summed and scaled to the deviation, in the model's type."""
    key = _mix((_mix(seed) + tid * 0xD1B54A32D192ED03) & ((1 << 64) - 1))
    scale = float(np.float32(np.float64(np.float32(STD)) / math.sqrt(4.0 * (65536.0 * 65536.0 - 1.0) / 12.0)))
    out, step = [], max(1, (1 << 26) // cols)
    for r in range(0, rows, step):
        n = min(step, rows - r)
        z = _mix(torch.arange(r * cols, (r + n) * cols, device="cuda", dtype=torch.int64) ^ _signed(key))
        z = (z & 0xFFFF) + ((z >> 16) & 0xFFFF) + ((z >> 32) & 0xFFFF) + ((z >> 48) & 0xFFFF) - 131070
        out.append((z.to(torch.float32) * torch.tensor(scale, dtype=torch.float32, device="cuda")).to(dtype).view(n, cols))
    return torch.cat(out)


def _attend(q, k, v, first, scale, bias=None, sink=None):
    """Causal attention: q [T, H, D] at positions first .. , k and v [S, G, D]; bias(distance) [H, ..] is added to the scores, the sink to the sum."""
    T, H, D = q.shape
    S, G = k.shape[0], k.shape[1]
    k, v = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    out = torch.empty(T, H, D, dtype=q.dtype, device=q.device)
    at = torch.arange(S, device=q.device)
    part = max(1, min(T, (1 << 28) // (H * S)))
    for a in range(0, T, part):
        b = min(T, a + part)
        x = q[a:b].permute(1, 0, 2).reshape(G, H // G * (b - a), D) @ k * scale
        x = x.view(H, b - a, S)
        far = torch.arange(first + a, first + b, device=q.device)[:, None] - at[None, :]
        if bias is not None:
            x = x + bias(far.clamp(min=0))
        x = x.masked_fill((far < 0)[None], -math.inf)
        if sink is not None:
            x = torch.cat([x, sink.view(H, 1, 1).expand(H, b - a, 1)], 2)
        x = torch.softmax(x, 2)[..., :S]
        out[a:b] = (x.reshape(G, H // G * (b - a), S) @ v).view(H, b - a, D).permute(1, 0, 2)
    return out.reshape(T, H * D)


def _rotate(x, first, base, half_steps=1.0):
    """Rotation of the two halves of each head against each other; angles are products in 32 bits, by the model's definition."""
    T, D = x.shape[0], x.shape[2]
    f = torch.tensor([1.0 / base ** (2 * j / D) for j in range(D // 2)], dtype=torch.float64, device=x.device).float()
    a = (torch.arange(first, first + T, device=x.device).float()[:, None] * f[None]).double()[:, None]
    u, v = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()], -1)


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


class _Dense:
    """The dense graph in 64 bits."""

    def __init__(self, case, seed):
        m, kind = MODELS[case["model"]], {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}[case["dtype"]]
        self.m, self.layers = m, []
        g = {k: torch.from_numpy(v).to("cuda", kind).double() for k, v in _gains(case, seed).items()}
        for l in range(m["L"]):
            p = "layers.%d." % l
            w = [_matrix(seed, l * 8 + t, r, c, kind).double() for t, r, c in ((0, (m["H"] + 2 * m["G"]) * m["D"], m["W"]), (1, m["W"], m["H"] * m["D"]),
                                                                              (2, 2 * m["F"], m["W"]), (3, m["W"], m["F"]))]
            self.layers.append((w, g[p + "input_layernorm.weight"], g[p + "post_attention_layernorm.weight"],
                                g.get(p + "self_attn.q_norm.weight"), g.get(p + "self_attn.k_norm.weight")))
        self.embed, self.norm = _matrix(seed, 1 << 20, m["V"], m["W"], kind).double(), g["norm.weight"]

    def __call__(self, tokens, rows):
        """Logits of the rows from `rows` on, and the last layer's keys and values."""
        m = self.m
        x = self.embed[torch.from_numpy(np.ascontiguousarray(tokens)).cuda()]
        T, H, G, D = x.shape[0], m["H"], m["G"], m["D"]
        for (qkv, o, gu, down), n1, n2, qn, kn in self.layers:
            y = (_rms(x, EPS) * n1) @ qkv.T
            q, k, v = y[:, :H * D].view(T, H, D), y[:, H * D:(H + G) * D].view(T, G, D), y[:, (H + G) * D:].view(T, G, D)
            if qn is not None:
                q, k = _rms(q, EPS) * qn, _rms(k, EPS) * kn
            q, k = _rotate(q, 0, m["base"]), _rotate(k, 0, m["base"])
            x = x + _attend(q, k, v, 0, D ** -0.5) @ o.T
            y = (_rms(x, EPS) * n2) @ gu.T
            x = x + (torch.nn.functional.silu(y[:, :m["F"]]) * y[:, m["F"]:]) @ down.T
        return (_rms(x[rows:], EPS) * self.norm) @ self.embed.T, k, v


class _Layers:
    """The layer-list model in 64 bits."""

    def __init__(self, seed):
        self.w = {k: v.double() for k, v in _layers_weights(seed).items()}

    def __call__(self, tokens, rows):
        s, w = LAYERS, self.w
        H, G, D = s["H"], s["G"], s["D"]
        x = w["embed"][torch.from_numpy(np.ascontiguousarray(tokens)).cuda()]
        T = x.shape[0]

        def canon(g, taps):
            h = _rms(x, 1e-5) * g
            pad = torch.cat([h.new_zeros(3, s["W"]), h])
            return h + sum(pad[j:j + T] * taps[:, j] for j in range(4))
        far = (torch.arange(T, device="cuda")[:, None] - torch.arange(T, device="cuda")[None]).double()
        for i, layer in enumerate(_layers_config()["layers"]):
            p = "l%d." % i
            h = canon(w[p + "norm1"], w[p + "canon1"])
            kv = H if i % 2 else G
            q, k, v = (h @ w[p + "mix.q"].T).view(T, H, D), (h @ w[p + "mix.k"].T).view(T, kv, D), (h @ w[p + "mix.v"].T).view(T, kv, D)
            if i % 2:
                q, k = _rotate(q, 0, 10000.0), _rotate(k, 0, 10000.0) * D ** -0.5
                decay = torch.tensor(layer["mixer"]["decay"], dtype=torch.float64, device="cuda")
                a = (q.transpose(0, 1) @ k.permute(1, 2, 0)) * torch.where(far >= 0, decay[:, None, None] ** far.clamp(min=0), torch.zeros_like(far))
                y = _rms((a @ v.transpose(0, 1)).transpose(0, 1), 1e-5).reshape(T, H * D) * torch.nn.functional.silu(h @ w[p + "mix.g"].T)
            else:
                r1, r2 = w[p + "mix.r1"][:, None, None], w[p + "mix.r2"][:, None, None]
                y = _attend(q, k, v, 0, D ** -0.5, lambda d: -r1 * torch.log1p(r2 * d), w[p + "mix.sink"])
            y = y @ w[p + "mix.o"].T
            h = canon(w[p + "norm2"], w[p + "canon2"])
            g, u = (h @ w[p + "mlp.gate"].T).clamp(max=7.0), (h @ w[p + "mlp.up"].T).clamp(-7.0, 7.0)
            x = x + 0.5 * (y + (g * torch.sigmoid(1.702 * g) * (u + 1)) @ w[p + "mlp.down"].T)
        return (_rms(x[rows:], 1e-5) * w["final.norm"]) @ w["head"].T, None, None


def exact(case, seed):
    if case["path"] in ("decode", "prefill"):
        lengths = _lengths(case)
        if sum(lengths) * (14 if case["model"] == "qwen3-8b" else 1) > 300000:
            return None
    model, tokens = _Layers(seed) if case["path"] == "layers" else _Dense(case, seed), _tokens(case, seed)
    logits = []
    if case["path"] in ("generate", "layers"):
        answers = []
        for t in tokens:
            answer = np.full(case["new"], t[-1])
            while True:  # the greedy answer: a guess is run whole and kept up to its first wrong token
                y, _, _ = model(np.concatenate([t, answer[:-1]]), t.size - 1)
                best = y.argmax(1).cpu().numpy()
                wrong = np.flatnonzero(best != answer)
                if not wrong.size:
                    break
                answer = np.concatenate([answer[:wrong[0]], best[wrong[0]:]])
            answers.append(answer)
            logits.append(y[-1:].cpu())
        return {"tokens": np.array(answers), "logits": torch.cat(logits)}
    m = MODELS[case["model"]]
    tables, blocks = _blocks(case)
    pools = [torch.zeros(blocks * BLOCK, m["G"], m["D"], dtype=torch.float64, device="cuda") for _ in range(2)]
    for t, table in zip(tokens, tables):
        y, k, v = model(t, t.size - 1)
        logits.append(y)
        rows = (torch.tensor(table, device="cuda")[:, None] * BLOCK + torch.arange(BLOCK, device="cuda")[None]).reshape(-1)[:t.size]
        pools[0][rows], pools[1][rows] = k, v
    logits = torch.cat(logits)
    tokens = None if case.get("temperature", 0.0) > 0 else logits.argmax(1)
    return {"tokens": tokens, "logits": logits, "k": pools[0].view(blocks, BLOCK, m["G"], m["D"]), "v": pools[1].view(blocks, BLOCK, m["G"], m["D"])}
