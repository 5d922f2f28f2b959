"""The work that users of this library have it do, as cases that can be timed and checked.

A case is one request (or one batch of them) through the public entry points: a prompt run and continued by a decode
session, several sessions advanced together, draft tokens scored, a mixed layer stack, or the FP8 operators of a layer of
routed experts. Weights are random; a dense model's head is its embedding with the rows permuted, so that a model's next
token is as clear as a trained one's and the same for every correct implementation.
"""
import ctypes
import math
import random

import numpy as np
import torch

from nerva_amd import DecodeSession, ModelWeights, WeightPlan, abi, runtime, stacks

F16, BF16 = 0, 1
WEIGHT_STD = 0.02
VERIFY_ROUNDS = 6


# ---------------------------------------------------------------- the cases

def _dense(name, kind, hidden, heads, kv_heads, head_dim, ff, vocab, layers, prompt, steps, dtype=BF16, theta=1e6, bias=False,
           qk_norm=False, temperature=0.0, top_p=1.0, top_k=0, sequences=1):
    return dict(name=name, kind=kind, hidden=hidden, heads=heads, kv_heads=kv_heads, head_dim=head_dim, ff=ff, vocab=vocab,
                layers=layers, prompt=prompt, steps=steps, dtype=dtype, theta=theta, bias=bias, qk_norm=qk_norm,
                temperature=temperature, top_p=top_p, top_k=top_k, sequences=sequences)


def listed():
    return [
        # a short request to a small model: nothing but latency and launches
        _dense("small model first words", "generate", 512, 8, 4, 64, 1376, 8003, 4, 12, 16, dtype=F16, theta=1e4),
        # the benchmark's model and prompt: a long document read, an answer begun
        _dense("qwen3 8b long prompt", "generate", 4096, 32, 8, 128, 12288, 151936, 36, 8192, 64, qk_norm=True),
        # a turn of a conversation
        _dense("4096 wide chat turn", "generate", 4096, 32, 8, 128, 14336, 128256, 8, 600, 48, theta=5e5),
        # a page of text for a model whose width is no power of two, with projection biases
        _dense("3584 wide a page", "generate", 3584, 28, 4, 128, 18944, 152064, 4, 900, 16, bias=True),
        # an answer drawn from the distribution
        _dense("2560 wide sampled", "generate", 2560, 32, 8, 128, 9728, 151936, 6, 701, 32, qk_norm=True, temperature=0.7, top_p=0.9),
        # narrow heads, half precision
        _dense("2048 wide heads of 64", "generate", 2048, 32, 8, 64, 8192, 128256, 6, 1024, 32, dtype=F16, theta=5e5),
        # a server's batch: 32 short conversations on one set of weights
        _dense("32 sequences 4096 wide", "batch", 4096, 32, 8, 128, 12288, 151936, 6, 130, 24, qk_norm=True, sequences=32),
        # a few sequences on a small model
        _dense("6 sequences 1024 wide", "batch", 1024, 16, 8, 128, 3072, 151936, 12, 75, 24, qk_norm=True, sequences=6),
        # drafts of another model checked: a few given tokens at a time, the logits of every one wanted
        _dense("5120 wide drafts scored", "verify", 5120, 40, 8, 128, 13824, 152064, 2, 240, 5, bias=True),
        # mixed stacks at widths of their benchmark
        dict(name="retorax 4096 wide", kind="retorax", hidden=4096, heads=32, kv_heads=8, ff=12288, channels=4096, chunk=1536,
             vocab=65536, layers=6, prompt=3000, steps=24),
        dict(name="kavuvik 2048 wide", kind="kavuvik", hidden=2048, heads=16, q_rank=768, kv_rank=512, window=1024, experts=64,
             top=6, expert_ff=768, shared_ff=1536, vocab=65536, layers=5, prompt=1800, steps=24),
        # one token through a layer of FP8 experts and the projections around it
        dict(name="fp8 experts one token", kind="fp8", hidden=7168, expert_ff=2048, experts=48, top=8, q_rank=1536, heads=128,
             head_dim=192, dtype=BF16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _multiple(rng, lo, hi, unit):
    return max(1, round(_log_int(rng, lo, hi) / unit)) * unit


def draw(rng):
    """One more case: widths of dense models from 512 to 5120 in steps of 64 or 128, with one to eight query heads a key head,
    prompts from a few tokens to a few thousand, one to 32 sequences; mixed stacks and expert layers of 512 to 7168."""
    kind = rng.choice(["generate"] * 5 + ["batch"] * 2 + ["verify", "retorax", "kavuvik", "fp8"])
    if kind == "fp8":
        return dict(kind=kind, hidden=_multiple(rng, 2048, 7168, 128), expert_ff=_multiple(rng, 512, 2048, 128),
                    experts=rng.randint(10, 40), top=rng.randint(1, 8), q_rank=_multiple(rng, 512, 1536, 64),
                    heads=_multiple(rng, 16, 96, 16), head_dim=rng.choice([128, 192]), dtype=rng.choice([F16, BF16, BF16]))
    if kind in ("retorax", "kavuvik"):
        heads = rng.randint(4, 32)
        out = dict(kind=kind, hidden=_multiple(rng, 512, 3584, 128), heads=heads, vocab=rng.randint(8000, 65536), layers=rng.randint(2, 5),
                   prompt=_log_int(rng, 30, 2000), steps=rng.randint(4, 24))
        if kind == "retorax":
            kv_heads = rng.choice([k for k in range(1, heads + 1) if heads % k == 0 and heads // k <= 8])
            out.update(kv_heads=kv_heads, ff=_multiple(rng, 2 * out["hidden"], 4 * out["hidden"], 128),
                       channels=_multiple(rng, out["hidden"] // 2, out["hidden"], 128), chunk=_log_int(rng, 100, 4096))
        else:
            out.update(heads=rng.choice([8, 16, 32]), q_rank=_multiple(rng, 256, 1024, 64), kv_rank=512, window=_log_int(rng, 100, 4096),
                       experts=rng.randint(8, 48), top=rng.randint(1, 6), expert_ff=_multiple(rng, 256, 768, 64),
                       shared_ff=_multiple(rng, 256, 1536, 64))
        return out
    head_dim = rng.choice([64, 128, 128])
    group = rng.randint(1, 8)
    hidden = _multiple(rng, 512, 5120, 64 if head_dim == 64 else 128)
    kv_heads = max(1, round(hidden / head_dim / group * rng.uniform(0.7, 1.3)))
    ff = _multiple(rng, 2.5 * hidden, 5 * hidden, 64)
    layer = hidden * (2 * group + 2) * kv_heads * head_dim + 3 * hidden * ff
    sampled = kind == "generate" and rng.random() < 0.3
    case = _dense("", kind, hidden, kv_heads * group, kv_heads, head_dim, ff, rng.randint(8000, 152064),
                  max(1, min(rng.randint(2, 12), int(5e8 // layer))), _log_int(rng, 8, 1000), rng.randint(8, 32), rng.choice([F16, BF16, BF16]),
                  rng.choice([1e4, 5e5, 1e6]), rng.random() < 0.3, rng.random() < 0.5)
    del case["name"]
    if sampled:
        case.update(temperature=rng.uniform(0.5, 1.0), top_p=rng.choice([0.9, 0.95, 1.0]), top_k=rng.choice([0, 0, 40]))
    if kind == "batch":
        case.update(sequences=rng.randint(2, 32), steps=rng.randint(4, 16))
        case.update(prompt=_log_int(rng, 8, 600 // case["sequences"] + 9))
    if kind == "verify":
        case.update(steps=rng.randint(2, 8), prompt=_log_int(rng, 8, 400))
    return case


# ---------------------------------------------------------------- weights and tokens, from the seed alone

class _Pool:
    """Random 16-bit matrices cut out of one run of normal values per standard deviation, at places of their own."""

    def __init__(self, seed, dtype, largest):
        self.generator = torch.Generator("cuda").manual_seed(seed)
        self.rng = random.Random(seed)
        self.dtype = torch.float16 if dtype == F16 else torch.bfloat16
        self.slack = 1 << 22
        self.unit = self.normal([largest + self.slack], 1.0)
        self.runs = {}

    def normal(self, shape, std, mean=0.0):
        return (torch.randn(shape, generator=self.generator, device="cuda") * std + mean).to(self.dtype)

    def matrix(self, shape, std):
        if std not in self.runs:
            self.runs[std] = _host(self.unit * std)
        at = self.rng.randrange(self.slack // 8) * 8
        return self.runs[std][at:at + math.prod(shape)].reshape(shape)

    def vector(self, shape, std, mean=0.0):
        return _host(self.normal(shape, std, mean))


def _host(tensor):
    """The bits of a device tensor in host memory that the library's uploads read fast."""
    out = torch.empty(tensor.shape, dtype=tensor.dtype, pin_memory=True)
    out.copy_(tensor)
    return out


def _bits(tensor):
    return tensor.view(torch.int16).numpy().view(np.uint16)


def _value(tensor):
    return tensor.cuda().double()


def _permutation(pool, vocab):
    return torch.randperm(vocab, generator=pool.generator, device="cuda")


def _embedding_and_head(pool, vocab, hidden, scale, mark=None):
    """Rows of std 2 (`mark` added), and a head whose row follow[t] is row t, `scale` times."""
    embed = pool.normal([vocab, hidden], 2.0)
    if mark is not None:
        embed = (embed.float() + mark).to(pool.dtype)
    follow = _permutation(pool, vocab)
    head = torch.empty_like(embed)
    head[follow] = embed * scale
    return _host(embed), _host(head), follow.cpu().numpy()


def _dense_model(case, seed):
    """({tensor name: host tensor}, per layer the same, follow)."""
    H, I, V, L = case["hidden"], case["ff"], case["vocab"], case["layers"]
    A, KV, hd = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"], case["head_dim"]
    pool = _Pool(seed, case["dtype"], max(I * H, A * H))
    embed, head, follow = _embedding_and_head(pool, V, H, WEIGHT_STD / 2)
    into = WEIGHT_STD / math.sqrt(2 * L)     # matrices that write the residual stream
    layers = []
    for _ in range(L):
        w = dict(rms_attn=pool.vector([H], 0.02, 1.0), rms_mlp=pool.vector([H], 0.02, 1.0),
                 w_q=pool.matrix([A, H], WEIGHT_STD), w_k=pool.matrix([KV, H], WEIGHT_STD), w_v=pool.matrix([KV, H], WEIGHT_STD),
                 w_o=pool.matrix([H, A], into), w_gate=pool.matrix([I, H], WEIGHT_STD), w_up=pool.matrix([I, H], WEIGHT_STD),
                 w_down=pool.matrix([H, I], into))
        if case["qk_norm"]:
            w.update(q_norm=pool.vector([hd], 0.02, 1.0), k_norm=pool.vector([hd], 0.02, 1.0))
        if case["bias"]:
            w.update(q_bias=pool.vector([A], 0.3), k_bias=pool.vector([KV], 0.3), v_bias=pool.vector([KV], 0.3))
        layers.append(w)
    return embed, layers, pool.vector([H], 0.02, 1.0), head, follow


def _prompts(case, seed):
    rng = np.random.default_rng(seed)
    count = case.get("sequences", 1)
    lengths = [case["prompt"]] if count == 1 else [max(1, case["prompt"] * (4 + 7 * i % 9) // 8) for i in range(count)]
    return [rng.integers(0, case["vocab"], n).astype(np.uint32) for n in lengths]


def _stack_config(case):
    if case["kind"] == "retorax":
        layers = []
        for i in range(case["layers"]):
            mixer = stacks.MinGru(case["channels"]) if i % 2 else \
                stacks.Attention(case["heads"], case["kv_heads"], 128, 128, 128, 1e6, 128 ** -0.5, case["chunk"], i - 2 if i % 4 == 2 else None)
            layers.append((mixer, stacks.XieluFeedForward(case["ff"])))
        return stacks.StackConfig(case["hidden"], case["vocab"], 1e-6, layers)
    mixer = stacks.LatentAttention(case["heads"], 128, 64, 128, case["q_rank"], case["kv_rank"], 64, 1e6, 192 ** -0.5, case["window"])
    ff = stacks.ExpertFeedForward(case["experts"], case["top"], case["expert_ff"], 7.0, case["shared_ff"], 7.0)
    return stacks.StackConfig(case["hidden"], case["vocab"], 1e-6, [(mixer, ff)] * case["layers"], stacks.PARALLEL, 1.0, 1.0)


def _stack_model(case, seed):
    """({tensor name: host tensor}, the token that follows each)."""
    config = _stack_config(case)
    manifest = config.manifest()
    pool = _Pool(seed, BF16, max(math.prod(shape) for name, shape in manifest if name not in ("embed", "head")))
    V, H, L = case["vocab"], case["hidden"], case["layers"]
    out = {}
    if case["kind"] == "retorax":
        out["embed"], follow = _host(pool.normal([V, H], 1.0)), np.arange(V)     # the embedding is the head
    else:
        # a token's row points along the router rows of its own experts, as far as a trained router tells them apart
        routes = torch.randn([case["experts"], H], generator=pool.generator, device="cuda")
        chosen = torch.rand([V, case["experts"]], generator=pool.generator, device="cuda").argsort(1)[:, :case["top"]]
        mark = torch.zeros([V, case["experts"]], device="cuda").scatter_(1, chosen, 1.0) @ routes
        out["embed"], out["head"], follow = _embedding_and_head(pool, V, H, WEIGHT_STD / 2, mark * (30.0 / math.sqrt(H)))
    for name, shape in manifest:
        if name in out:
            continue
        if name.endswith("router"):
            order = torch.randperm(case["experts"], generator=pool.generator, device="cuda")
            out[name] = _host((routes[order] * (2.0 / math.sqrt(H))).to(pool.dtype))
        elif name.endswith(".talk"):
            out[name] = _host((torch.eye(shape[0], device="cuda") + pool.normal(shape, 0.1)).to(pool.dtype))
        elif name.endswith(".act"):
            out[name] = pool.vector(shape, 0.5)
        elif name.endswith(".sink"):
            out[name] = pool.vector(shape, 1.0)
        elif name.endswith(("norm1b", "norm2b")):
            out[name] = pool.vector(shape, 0.02, 1.0 / math.sqrt(2 * L))         # what a sublayer adds to the residual
        elif name.endswith((".b",)):
            out[name] = pool.vector(shape, 0.02)
        elif len(shape) == 1:
            out[name] = pool.vector(shape, 0.02, 1.0)
        else:
            out[name] = pool.matrix(shape, WEIGHT_STD / math.sqrt(2 * L) if name.endswith((".o", ".down")) else WEIGHT_STD)
    return config, out, follow


def _fp8(shape, generator):
    """Bytes of e4m3 values that fill the format's range the way quantised normal weights do, and a scale per 128 x 128."""
    w = torch.empty(shape, dtype=torch.uint8, device="cuda")
    for part, whole in zip(w.flatten(0, -3) if len(shape) > 2 else [w], w.flatten(0, -3) if len(shape) > 2 else [w]):
        whole.copy_((torch.randn(part.shape, generator=generator, device="cuda") * 100.0).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8))
    blocks = list(shape[:-2]) + [-(-shape[-2] // 128), -(-shape[-1] // 128)]
    scales = (torch.rand(blocks, generator=generator, device="cuda") + 0.5) * (WEIGHT_STD / 100.0)
    return w, scales


def _fp8_layer(case, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    H, I, E, wide = case["hidden"], case["expert_ff"], case["experts"], case["heads"] * case["head_dim"]
    kind = torch.float16 if case["dtype"] == F16 else torch.bfloat16
    s = dict(gate=_fp8([E + 1, I, H], g), up=_fp8([E + 1, I, H], g), down=_fp8([E + 1, H, I], g),
             q_down=_fp8([case["q_rank"], H], g), q_up=_fp8([wide, case["q_rank"]], g), o=_fp8([H, case["heads"] * 128], g))
    for name, n in (("x", H), ("latent", case["q_rank"]), ("heads16", case["heads"] * 128)):
        s[name] = torch.randn([n], generator=g, device="cuda").to(kind)
    s["logits"] = torch.randn([E], generator=g, device="cuda")
    return s


# ---------------------------------------------------------------- what a program has in hand, and one pass

def _sampler(case, seed):
    cfg = abi.NervaHipHfDecodeSamplerConfig()
    cfg.temperature, cfg.top_p, cfg.top_k, cfg.seed = case["temperature"], case["top_p"], case["top_k"], seed
    return cfg


def prepare(case, seed):
    if case["kind"] == "fp8":
        s = _fp8_layer(case, seed)
        H, I, E, K = case["hidden"], case["expert_ff"], case["experts"], case["top"]
        s.update(ids=torch.zeros([K], dtype=torch.int32, device="cuda"), weights=torch.zeros([K], device="cuda"),
                 activation=torch.zeros([(K + 1) * I], device="cuda"), out=torch.zeros([H], device="cuda"),
                 out_down=torch.zeros([case["q_rank"]], device="cuda"), out_up=torch.zeros([case["heads"] * case["head_dim"]], device="cuda"),
                 out_o=torch.zeros([H], device="cuda"), case=case)
        return s
    prompts = _prompts(case, seed)
    context = max(len(p) for p in prompts) + (VERIFY_ROUNDS if case["kind"] == "verify" else 1) * case["steps"] + 8
    if case["kind"] in ("retorax", "kavuvik"):
        config, tensors, _ = _stack_model(case, seed)
        weights = stacks.StackWeights(config, {k: _bits(t) for k, t in tensors.items()})
        session = DecodeSession.create_stack(config, WeightPlan.from_weights(weights), context)
        return dict(case=case, sessions=[session], prompts=prompts, sampler=None)
    embed, layers, final_norm, head, follow = _dense_model(case, seed)
    weights = ModelWeights(case["dtype"], case["hidden"], case["heads"], case["kv_heads"], case["head_dim"], case["ff"], case["vocab"], 1e-6,
                           case["theta"], _bits(embed), [{k: _bits(t) for k, t in w.items()} for w in layers], _bits(final_norm), _bits(head))
    session = DecodeSession.create(weights, context, plan=WeightPlan.from_weights(weights))
    sessions = [session] + [session.fork_shared_weights() for _ in range(case["sequences"] - 1)]
    state = dict(case=case, sessions=sessions, prompts=prompts, sampler=_sampler(case, seed & 0xFFFF))
    if case["kind"] == "verify":
        state["drafts"] = _drafts(case, seed)
    return state


def _drafts(case, seed):
    rng = np.random.default_rng(seed + 1)
    return [rng.integers(0, case["vocab"], case["steps"]).astype(np.uint32) for _ in range(VERIFY_ROUNDS)]


def _did(rc, result):
    if rc != 0:
        raise RuntimeError("the library refused the call: hip_error=%d" % result.hip_error)


def _start(session, prompt, sampler):
    rc, result = session.start(prompt, sampler=sampler)
    _did(rc, result)


def _advance(session, steps):
    rc, result, tokens = session.advance(steps)
    _did(rc, result)
    return tokens.astype(np.int64)


def run(state):
    case = state["case"]
    if case["kind"] == "fp8":
        return _run_fp8(case, state)
    sessions, prompts = state["sessions"], state["prompts"]
    if case["kind"] == "verify":
        session, logits = sessions[0], []
        session.release_sequence()
        rc, result, _, _ = session.extend(prompts[0])
        _did(rc, result)
        for draft in state["drafts"]:
            rc, result, rows, _ = session.extend(draft, range(len(draft)))
            _did(rc, result)
            logits.append(rows)
        return np.concatenate(logits)
    for session, prompt in zip(sessions, prompts):
        _start(session, prompt, state["sampler"])
    if case["kind"] != "batch":
        tokens = _advance(sessions[0], case["steps"])
        return tokens, sessions[0].logits()
    tokens = [np.concatenate([_advance(session, 1) for session in sessions])]
    for _ in range(case["steps"]):
        rc, result, step = DecodeSession.batch_advance_one(sessions, 32, 2)
        _did(rc, result)
        tokens.append(step.astype(np.int64))
    # the first and the last sequence go on alone
    _advance(sessions[0], 1)
    _advance(sessions[-1], 1)
    return np.stack(tokens), sessions[0].logits(), sessions[-1].logits()


def _run_fp8(case, s):
    lib, error = abi.load(), ctypes.c_int32(0)
    H, I, E, K, wide = case["hidden"], case["expert_ff"], case["experts"], case["top"], case["heads"] * case["head_dim"]

    def gemv(w, x, rows, cols, out):
        runtime.fp8_gemv(s[w][0].data_ptr(), s[w][1].data_ptr(), rows, cols, 128, 128, out.data_ptr(), input16=s[x].data_ptr(),
                         input_dtype=case["dtype"], sync=False)
    gemv("q_down", "x", case["q_rank"], H, s["out_down"])
    gemv("q_up", "latent", wide, case["q_rank"], s["out_up"])
    gemv("o", "heads16", H, case["heads"] * 128, s["out_o"])
    route = abi.NervaHipMoeRouteRequest()
    route.num_experts, route.top_k, route.normalize = E, K, 1
    route.logits, route.expert_ids, route.expert_weights = s["logits"].data_ptr(), s["ids"].data_ptr(), s["weights"].data_ptr()
    if lib.nerva_hip_moe_route_softmax(ctypes.byref(route), None, ctypes.byref(error)) != 0:
        raise RuntimeError("the library refused the call: hip_error=%d" % error.value)
    runtime.moe_fp8_experts(H, I, E + 1, K, 128, s["x"].data_ptr(), s["ids"].data_ptr(), s["weights"].data_ptr(),
                            s["gate"][0].data_ptr(), s["gate"][1].data_ptr(), s["up"][0].data_ptr(), s["up"][1].data_ptr(),
                            s["down"][0].data_ptr(), s["down"][1].data_ptr(), s["activation"].data_ptr(), s["out"].data_ptr(),
                            shared_index=E, input_dtype=case["dtype"], sync=False)
    return s["out"], s["out_down"], s["out_up"], s["out_o"], s["ids"], s["weights"]


# ---------------------------------------------------------------- what a pass cannot do without, and how exact it is

def _layer_sizes(case):
    """(16-bit matrix elements a token uses in one layer, those of a layer, score and value products a visible key costs,
    16-bit elements cached a token), per layer."""
    H = case["hidden"]
    out = []
    for i in range(case["layers"]):
        if case["kind"] == "retorax":
            heads, kv = case["heads"] * 128, case["kv_heads"] * 128
            if i % 2:
                used, keys, cached = 4 * H * case["channels"], 0, 0
            else:
                used, keys, cached = H * (3 * heads + (0 if i % 4 == 2 else 2 * kv)), 2 * heads, 2 * kv
            out.append((used + 2 * H * case["ff"], used + 2 * H * case["ff"], keys, cached))
        elif case["kind"] == "kavuvik":
            heads, q, c = case["heads"], case["q_rank"], case["kv_rank"]
            mixer = H * (q + c + 64 + 2 * heads * 128) + q * heads * 192 + 2 * c * heads * 128 + case["experts"] * H
            expert, shared = 3 * H * case["expert_ff"], 3 * H * case["shared_ff"]
            out.append((mixer + case["top"] * expert + shared, mixer + case["experts"] * expert + shared, heads * 320, c + 64))
        else:
            heads, kv = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
            used = 2 * H * (heads + kv) + 3 * H * case["ff"]
            out.append((used, used, 2 * heads, 2 * kv))
    return out


def _visible(case, position):
    if case["kind"] == "retorax":
        return position % case["chunk"] + 1
    if case["kind"] == "kavuvik":
        return min(position + 1, case["window"])
    return position + 1


def work(case):
    if case["kind"] == "fp8":
        H, I, K, wide = case["hidden"], case["expert_ff"], case["top"], case["heads"] * case["head_dim"]
        weights = 3 * (K + 1) * I * H + case["q_rank"] * (H + wide) + H * case["heads"] * 128
        return dict(bytes=weights * (1 + 4 / 16384) + 10 * H, flops=2 * weights)
    sizes = _layer_sizes(case)
    head = case["vocab"] * case["hidden"]
    total = dict(bytes=0.0, flops=0.0)

    def steps(blocks):
        """blocks: per sequence (first position, tokens) that one stream of the weights serves; a head row for each's last."""
        tokens = sum(n for _, n in blocks)
        for used, all_, per_key, cached in sizes:
            keys = sum(_visible(case, p) for first, n in blocks for p in (range(first, first + n) if n < 64 else [first + n // 2] * n))
            total["bytes"] += 2.0 * min(all_, used * tokens) + 2.0 * cached * sum(_visible(case, first + n - 1) for first, n in blocks)
            total["flops"] += 2.0 * used * tokens + 2.0 * per_key * keys
        total["bytes"] += 2.0 * head + 4.0 * case["vocab"] * len(blocks)
        total["flops"] += 2.0 * head * len(blocks)
    lengths = [len(p) for p in _prompts(case, 0)]
    for n in lengths:
        steps([(0, n)])
    if case["kind"] == "verify":
        for i in range(VERIFY_ROUNDS):
            steps([(lengths[0] + i * case["steps"], case["steps"])])
            total["bytes"] += 4.0 * case["vocab"] * (case["steps"] - 1)
            total["flops"] += 2.0 * head * (case["steps"] - 1)
    elif case["kind"] == "batch":
        for i in range(case["steps"]):
            steps([(n + i, 1) for n in lengths])
        for n in {0: lengths[0], -1: lengths[-1]}.values():
            steps([(n + case["steps"], 1)])
    else:
        for i in range(case["steps"] - 1):
            steps([(lengths[0] + i, 1)])
    return total


def tolerance(case):
    if case["kind"] == "fp8":
        return dict(rel=2e-6, max=2e-5, differ=0.0)
    # the 16-bit inputs of the products: four times what a pass is seen to be off 64 bits, at any of the sizes above
    return dict(rel=1e-3, max=8e-3, differ=0.0) if case.get("dtype", BF16) == F16 else dict(rel=1.6e-2, max=1e-1, differ=0.0)


# ---------------------------------------------------------------- the same in 64 bits

def _rms(x, gamma):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * gamma


def _turn(x, theta, dims, first=0):
    """x [positions, heads, dim]: element i of the first `dims` goes with element i + dims / 2."""
    half = dims // 2
    angle = torch.arange(first, first + x.shape[0], device="cuda", dtype=torch.float64)[:, None] * \
        theta ** (-2.0 * torch.arange(half, device="cuda", dtype=torch.float64) / dims)
    c, s = angle.cos()[:, None], angle.sin()[:, None]
    u, v = x[..., :half], x[..., half:dims]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., dims:]], -1)


def _attend(q, k, v, scale, first_visible, talk=None, sink=None):
    """q [n, H, d], k [n, G, d], v [n, G, dv]: every query sees the keys from first_visible to its own."""
    n, H = q.shape[:2]
    k, v = (t.permute(1, 0, 2).repeat_interleave(H // k.shape[1], 0) for t in (k, v))
    out, places = [], torch.arange(n, device="cuda")
    for at in range(0, n, 256):
        rows = places[at:at + 256]
        end = int(rows[-1]) + 1
        low = int(first_visible[rows].min())
        scores = q[rows].permute(1, 0, 2) @ k[:, low:end].transpose(1, 2).contiguous() * scale
        if talk is not None:
            scores = (talk @ scores.reshape(H, -1)).reshape(scores.shape)
        keys = places[low:end]
        scores.masked_fill_((keys[None] > rows[:, None]) | (keys[None] < first_visible[rows][:, None]), -math.inf)
        if sink is not None:
            scores = torch.cat([scores, sink[:, None, None].expand(-1, scores.shape[1], 1)], 2)
        weights = scores.softmax(-1)[..., :end - low]
        out.append((weights @ v[:, low:end]).permute(1, 0, 2).reshape(len(rows), -1))
    return torch.cat(out)


def _dense_logits(case, model, tokens, wanted):
    embed, layers, final_norm, head, _ = model
    H, A, KV, hd = case["hidden"], case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"], case["head_dim"]
    x = _value(embed[torch.from_numpy(tokens.astype(np.int64))])
    n = len(tokens)
    zero = torch.zeros(n, dtype=torch.int64, device="cuda")
    for w in layers:
        w = {k: _value(t) for k, t in w.items()}
        h = _rms(x, w["rms_attn"])
        q, k, v = (h @ w["w_" + name].T + w.get(name + "_bias", 0.0) for name in "qkv")
        q, k, v = q.reshape(n, -1, hd), k.reshape(n, -1, hd), v.reshape(n, -1, hd)
        if "q_norm" in w:
            q, k = _rms(q, w["q_norm"]), _rms(k, w["k_norm"])
        q, k = _turn(q, case["theta"], hd), _turn(k, case["theta"], hd)
        x = x + _attend(q, k, v, hd ** -0.5, zero) @ w["w_o"].T
        h = _rms(x, w["rms_mlp"])
        x = x + (torch.nn.functional.silu(h @ w["w_gate"].T) * (h @ w["w_up"].T)) @ w["w_down"].T
        del w, h, q, k, v
    return _head(_rms(x[wanted], _value(final_norm)), head)


def _head(x, head):
    return torch.cat([x @ _value(part).T for part in head.split(32768)], -1)


def _layer_norm(x, w, b):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], w, b, 1e-6)


def _retorax_logits(case, config, t, tokens):
    w = lambda name: _value(t[name])                             # noqa: E731
    norm = lambda x, name: _layer_norm(x, w(name), w(name + ".b"))   # noqa: E731
    n = len(tokens)
    x = _value(t["embed"][torch.from_numpy(tokens.astype(np.int64))])
    places = torch.arange(n, device="cuda")
    first = places // case["chunk"] * case["chunk"]
    cache = {}
    for i, (mixer, _) in enumerate(config.layers):
        m = "l%d.mix." % i
        h = norm(x, "l%d.norm1" % i)
        if isinstance(mixer, stacks.Attention):
            if mixer.kv_layer is None:
                cache[i] = (_turn((h @ w(m + "k").T).reshape(n, -1, 128), 1e6, 128), (h @ w(m + "v").T).reshape(n, -1, 128))
            k, v = cache[i if mixer.kv_layer is None else mixer.kv_layer]
            q = _turn((h @ w(m + "q").T).reshape(n, -1, 128), 1e6, 128)
            y = _attend(q, k, v, 128 ** -0.5, first, w(m + "talk"), w(m + "sink")) * (h @ w(m + "g").T).sigmoid()
        else:
            z = (h @ w(m + "z").T + w(m + "z.b")).sigmoid()
            u = h @ w(m + "x").T + w(m + "x.b")
            u = torch.where(u >= 0, u + 0.5, u.sigmoid()) * z
            z, y = 1.0 - z, torch.empty_like(u)
            state = torch.zeros_like(u[0])
            for p in range(n):
                state = torch.addcmul(u[p], z[p], state)
                y[p] = state
            y = y * torch.nn.functional.silu(h @ w(m + "g").T)
        x = x + norm(y @ w(m + "o").T, "l%d.norm1b" % i)
        m = "l%d.mlp." % i
        p, q = torch.nn.functional.softplus(w(m + "act"))
        z = norm(x, "l%d.norm2" % i) @ w(m + "up").T
        low = z.clamp(max=0.0)
        z = torch.where(z > 0, p * z * z, (q + 0.5) * (low.expm1() - low)) + 0.5 * z
        x = x + norm(z @ w(m + "down").T, "l%d.norm2b" % i)
    return _head(norm(x[-1:], "final.norm"), t["embed"])


def _bounded_glu(g, u):
    g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0)
    return g * (1.702 * g).sigmoid() * (u + 1.0)


def _kavuvik_logits(case, config, t, tokens):
    w = lambda name: _value(t[name])                             # noqa: E731
    n, heads, rank = len(tokens), case["heads"], case["kv_rank"]
    x = _value(t["embed"][torch.from_numpy(tokens.astype(np.int64))])
    first = (torch.arange(n, device="cuda") - case["window"] + 1).clamp(min=0)
    for i in range(case["layers"]):
        m, f = "l%d.mix." % i, "l%d.mlp." % i
        h = _rms(x, w("l%d.norm1" % i))
        q = (_rms(h @ w(m + "dq").T, w(m + "dq.norm")) @ w(m + "uq").T).reshape(n, heads, 192)
        q = torch.cat([q[..., :128], _turn(q[..., 128:], 1e6, 64)], -1)
        down = h @ w(m + "dkv").T
        latent = _rms(down[:, :rank], w(m + "dkv.norm"))
        part = _turn(down[:, None, rank:], 1e6, 64).expand(-1, heads, -1)
        k = torch.cat([(latent @ w(m + "uk").T).reshape(n, heads, 128), part], -1)
        v = (latent @ w(m + "uv").T).reshape(n, heads, 128)
        y = (_attend(q, k, v, 192 ** -0.5, first) * (h @ w(m + "g").T).sigmoid()) @ w(m + "o").T
        h = _rms(x, w("l%d.norm2" % i))
        s = (h @ w(f + "router").T).sigmoid()
        best, chosen = s.topk(case["top"], -1)
        weights = torch.zeros_like(s).scatter_(1, chosen, best / best.sum(-1, keepdim=True))

        def expert(name, rows):
            return _bounded_glu(rows @ w(f + name + ".gate").T, rows @ w(f + name + ".up").T) @ w(f + name + ".down").T
        for e in range(case["experts"]):
            rows = weights[:, e].nonzero()[:, 0]
            if len(rows):
                y.index_add_(0, rows, expert("e%d" % e, h[rows]) * weights[rows, e][:, None])
        x = x + y + expert("shared", h)
    return _head(_rms(x[-1:], w("final.norm")), t["head"])


def _chain(prompt, follow, steps):
    """The tokens that follow a prompt, and what the model reads to make the last of them."""
    out, token = [], int(prompt[-1])
    for _ in range(steps):
        token = int(follow[token])
        out.append(token)
    return np.array(out, np.int64), np.concatenate([prompt.astype(np.int64), out[:-1]])


def _block_scaled(pair):
    w, s = pair
    s = s.double().repeat_interleave(128, -2).repeat_interleave(128, -1)
    return w.view(torch.float8_e4m3fn).to(torch.float32).double() * s[..., :w.shape[-2], :w.shape[-1]]


def exact(case, seed):
    if case["kind"] == "fp8":
        s = _fp8_layer(case, seed)
        x = s["x"].double()
        weights = s["logits"].double().softmax(-1)
        best, ids = weights.sort(descending=True, stable=True)
        best, ids = best[:case["top"]] / best[:case["top"]].sum(), ids[:case["top"]]
        out = torch.zeros_like(x)
        for e, a in list(zip(ids.tolist(), best.tolist())) + [(case["experts"], 1.0)]:
            g, u, d = (_block_scaled((s[name][0][e], s[name][1][e])) for name in ("gate", "up", "down"))
            out += a * (d @ (torch.nn.functional.silu(g @ x) * (u @ x)))
        return (out, _block_scaled(s["q_down"]) @ x, _block_scaled(s["q_up"]) @ s["latent"].double(),
                _block_scaled(s["o"]) @ s["heads16"].double(), ids.to(torch.int32), best)
    prompts = _prompts(case, seed)
    if case["kind"] in ("retorax", "kavuvik"):
        config, tensors, follow = _stack_model(case, seed)
        tokens, read = _chain(prompts[0], follow, case["steps"])
        logits = (_retorax_logits if case["kind"] == "retorax" else _kavuvik_logits)(case, config, tensors, read)
        return tokens, logits[0]
    model = _dense_model(case, seed)
    if case["kind"] == "verify":
        read = np.concatenate([prompts[0]] + _drafts(case, seed))
        return _dense_logits(case, model, read, slice(len(prompts[0]), None))
    if case["kind"] == "batch":
        chains = [_chain(p, model[-1], case["steps"] + 2) for p in prompts]
        tokens = np.stack([tokens[:-1] for tokens, _ in chains], 1)
        return (tokens,) + tuple(_dense_logits(case, model, chains[i][1], slice(-1, None))[0] for i in (0, -1))
    tokens, read = _chain(prompts[0], model[-1], case["steps"])
    return tokens, _dense_logits(case, model, read, slice(-1, None))[0]
