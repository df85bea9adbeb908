"""What the framework's speed is measured on: serving a batch of requests with a decoder.

A pass takes a batch of requests through the model as the engine does: the prompts in steps of at most 8192
token rows (a prompt may be cut over two steps, short ones share a step), then ``new`` decode steps of one row
per request, replayed from a captured HIP graph whose batch is rounded up to the engine's next graph size. The
tokens of the decode steps are given, so that two implementations see the same inputs throughout; the output
is the 32-bit logits that the engine would sample from, [new + 1, requests, vocab]. Later logits depend on the
paged caches and the recurrent states that earlier steps wrote.

The models: Llama-3-8B's layers (the headline benchmark's model), and two of the layer-list decoders of
``bench.py --layer-compare`` at its widths: Fikizen (window attention with sinks, a gated delta rule, a
generalized delta rule, dense feed-forwards) and Kesirax (latent attention, minGRU, experts chosen by token).
Few layers of each, as there: the cost per layer is what counts.
"""
import functools
import math
import os
import tempfile

import torch
import torch.nn.functional as F

BLOCK = 16            # tokens of a cache page
STEP_ROWS = 8192      # token rows of a prompt step
VOCAB = 32000
GRAPH_SIZES = (1, 2, 4, 8, 16, 24, 32, 48, 64)
SIZES = {   # by width, as bench.py --layer-compare has them
    1024: dict(width=1024, heads=8, window=512, experts=8, top=2, ff=512, gru=2048, vocab=VOCAB, dense_ff=3072),
    2048: dict(width=2048, heads=16, window=1024, experts=16, top=2, ff=1024, gru=4096, vocab=VOCAB, dense_ff=6144),
    4096: dict(width=4096, heads=32, window=1024, experts=8, top=2, ff=2048, gru=8192, vocab=VOCAB, dense_ff=12288),
}
LLAMA = dict(width=4096, layers=2, heads=32, kv_heads=8, dim=128, ff=14336, theta=500000.0, eps=1e-5)


def listed():
    def case(name, model, width, requests, prompt, new, dtype="bfloat16"):
        return dict(name=name, model=model, width=width, requests=requests, prompt=prompt, new=new, dtype=dtype)

    return [
        # one user's short question: every step is a handful of rows, latency and launches count
        case("llama one short chat", "llama", 4096, 1, 61, 16),
        # the headline benchmark's batch of 64, mostly decoding
        case("llama 64 chats", "llama", 4096, 64, 96, 24),
        # the headline benchmark's prompts: one full step
        case("llama long prompts", "llama", 4096, 8, 1024, 2),
        # the same three situations for the layer-list designs
        case("fikizen one short chat", "fikizen", 1024, 1, 33, 16),
        case("fikizen 16 chats", "fikizen", 2048, 16, 200, 32),
        case("fikizen long prompts", "fikizen", 2048, 4, 2048, 1),
        # 32-bit weights and activations (--dtype float32): numerics work, a few medium prompts
        case("fikizen float32", "fikizen", 1024, 3, 300, 6, "float32"),
        # ragged prompts cut over several steps at the widest size
        case("fikizen wide ragged", "fikizen", 4096, 13, 1500, 4),
        case("kesirax one chat", "kesirax", 2048, 1, 700, 24),
        case("kesirax 41 chats", "kesirax", 2048, 41, 150, 32),
        case("kesirax long prompts", "kesirax", 2048, 4, 2048, 1),
        case("kesirax wide ragged", "kesirax", 4096, 11, 1300, 4),
    ]


def draw(rng):
    model = rng.choice(("llama", "fikizen", "fikizen", "kesirax", "kesirax"))
    width = 4096 if model == "llama" else rng.choice((1024, 2048, 2048, 4096))
    dtype = "float32" if model != "llama" and width == 1024 and rng.random() < 0.4 else "bfloat16"
    rows = 1200 if dtype == "float32" else 6000 if width == 4096 and model != "llama" else 8192 if model == "llama" else 12000
    requests = min(64, int(math.exp(rng.uniform(0.0, math.log(64.99)))))
    prompt = int(math.exp(rng.uniform(math.log(16), math.log(min(2048, rows // requests)))))
    new = int(math.exp(rng.uniform(0.0, math.log(12.99 if width == 4096 and model != "llama" else 24.99))))
    return dict(model=model, width=width, requests=requests, prompt=prompt, new=new, dtype=dtype)


def lengths(case):
    """Prompt lengths: the longest is ``prompt``, the others down to two thirds of it; all full for single steps of long prompts."""
    n, p = case["requests"], case["prompt"]
    if n * p <= STEP_ROWS and p % 1024 == 0:
        return [p] * n
    return [max(1, p - (i * 37) % (p // 3 + 1)) for i in range(n)]


# ---------------------------------------------------------------- weights, tokens
def shapes(case):
    """{tensor name: (shape, kind)}: kinds are "lin" (a projection, standard deviation 1 / sqrt of its inputs, times a
    number), "one" (norm weights around 1), "vec" (others)."""
    if case["model"] == "llama":
        m, t = LLAMA, {}
        H, q, kv, I = m["width"], m["heads"] * m["dim"], m["kv_heads"] * m["dim"], m["ff"]
        t["model.embed_tokens.weight"] = ((VOCAB, H), "rows", 1.0)
        t["model.norm.weight"] = ((H,), "one", 0.1)
        t["lm_head.weight"] = ((VOCAB, H), "lin", 2.0)
        for i in range(m["layers"]):
            p = f"model.layers.{i}."
            t[p + "input_layernorm.weight"] = t[p + "post_attention_layernorm.weight"] = ((H,), "one", 0.1)
            for n, s, g in (("self_attn.q_proj", (q, H), 1.5), ("self_attn.k_proj", (kv, H), 1.5), ("self_attn.v_proj", (kv, H), 1.0),
                            ("self_attn.o_proj", (H, q), 1.0), ("mlp.gate_proj", (I, H), 1.0), ("mlp.up_proj", (I, H), 1.0),
                            ("mlp.down_proj", (H, I), 1.0)):
                t[f"{p}{n}.weight"] = (s, "lin", g)
        return t
    s = SIZES[case["width"]]
    W, H, G = s["width"], s["heads"], max(1, s["heads"] // 4)
    t = {"embed": ((VOCAB, W), "rows", 1.0), "head": ((VOCAB, W), "lin", 2.0), "final.norm": ((W,), "one", 0.1)}
    lin = lambda o, i, g=1.0: ((o, i), "lin", g)  # noqa: E731
    if case["model"] == "kesirax":
        for l in range(4):
            p = f"l{l}.mix."
            t[f"l{l}.norm1"], t[f"l{l}.ls1"], t[f"l{l}.ls2"] = ((W,), "one", 0.1), ((W,), "half", 0.1), ((W,), "half", 0.1)
            if l % 2 == 0:
                t[p + "dq"], t[p + "dkv"], t[p + "g"] = lin(W // 2, W), lin(576, W), lin(H, W)
                t[p + "dq.norm"], t[p + "dkv.norm"] = ((W // 2,), "one", 0.1), ((512,), "one", 0.1)
                t[p + "uq"], t[p + "uk"], t[p + "uv"] = lin(H * 192, W // 2, 1.5), lin(H * 128, 512, 1.5), lin(H * 128, 512)
                t[p + "o"] = lin(W, H * 128)
            else:
                n = s["gru"]
                t[p + "z"], t[p + "x"], t[p + "g"], t[p + "o"] = lin(n, W), lin(n, W), lin(n, W), lin(W, n)
                t[p + "z.b"], t[p + "x.b"] = ((n,), "vec", 1.0), ((n,), "vec", 0.5)
            t[f"l{l}.mlp.table"] = ((VOCAB, s["top"]), "table", s["experts"])
            for e in range(s["experts"]):
                t[f"l{l}.mlp.e{e}.up"], t[f"l{l}.mlp.e{e}.down"] = lin(s["ff"], W), lin(W, s["ff"])
        return t

    def attention(p, biased):
        t[p + "q"], t[p + "k"], t[p + "v"], t[p + "o"] = lin(H * 128, W, 1.5), lin(G * 128, W, 1.5), lin(G * 128, W), lin(W, H * 128)
        if biased:
            t[p + "q.b"], t[p + "k.b"], t[p + "v.b"] = ((H * 128,), "vec", 0.3), ((G * 128,), "vec", 0.3), ((G * 128,), "vec", 0.3)
            t[p + "q.norm"], t[p + "k.norm"] = ((H * 128,), "one", 0.2), ((G * 128,), "one", 0.2)
        else:
            t[p + "g"] = lin(H, W, 1.5)

    for l, ff in ((0, True), (1, False), (2, True)):   # the fourth layer runs the first one's weights
        t[f"l{l}.norm1"] = ((W,), "one", 0.1)
        if ff:
            t[f"l{l}.norm2"] = ((W,), "one", 0.1)
            t[f"l{l}.mlp.up"], t[f"l{l}.mlp.down"] = lin(s["dense_ff"], W), lin(W, s["dense_ff"], 0.5)
            t[f"l{l}.mlp.act"] = ((2,), "vec", 0.5)
    attention("l0.mix.", False)
    p = "l1.mix."
    for n, c in (("q", G * 128), ("k", G * 128), ("v", H * 128)):
        t[p + n], t[p + n + ".conv"] = lin(c, W, 1.5), ((c, 4), "vec", 0.5)
    t[p + "b"], t[p + "a"], t[p + "g"], t[p + "o"] = lin(H, W), lin(H, W), lin(H * 128, W), lin(W, H * 128)
    t[p + "A_log"], t[p + "dt_bias"], t[p + "norm"] = ((H,), "vec", 0.5), ((H,), "vec", 0.5), ((128,), "one", 0.2)
    attention("l2.mix.left.", True)
    p, N = "l2.mix.right.", W
    for n in ("r", "k", "v", "a", "g"):
        t[p + n] = lin(N, W)
    t[p + "w1"], t[p + "w2"], t[p + "o"] = lin(64, W), lin(N, 64), lin(W, N)
    t[p + "a.b"], t[p + "w0"], t[p + "norm"] = ((N,), "vec", 0.5), ((N,), "vec", 1.0), ((N,), "one", 0.2)
    return t


def make_tensors(case, seed):
    """The checkpoint: values that bf16 holds, on the GPU."""
    g = torch.Generator("cuda").manual_seed(1000003 * seed + 17)
    out = {}
    for name, (shape, kind, x) in shapes(case).items():
        if kind == "table":
            out[name] = torch.rand(shape[0], x, device="cuda", generator=g).topk(shape[1], 1).indices.int()
            continue
        v = torch.randn(shape, device="cuda", generator=g, dtype=torch.float32)
        v *= x / math.sqrt(shape[1]) if kind == "lin" else x
        if kind in ("one", "half"):
            v += 1.0 if kind == "one" else 0.5
        out[name] = v.bfloat16()
    return out


def make_tokens(case, seed):
    """[requests, longest prompt + new] ids; a request's row starts with its prompt, followed by its ``new`` tokens."""
    g = torch.Generator("cuda").manual_seed(1000003 * seed + 29)
    return torch.randint(3, VOCAB, (case["requests"], case["prompt"] + case["new"]), device="cuda", generator=g)


# ---------------------------------------------------------------- the framework's side
def build(case, tensors):
    """(model, paged caches, recurrent states, attention scratch) with room for the case's requests and a scratch page and slot."""
    from hipserve.config import PRESETS, EngineConfig
    from hipserve.ops import get_ops
    from hipserve.parallel.comm import TPGroup

    dev, tp = torch.device("cuda", torch.cuda.current_device()), TPGroup(0, 1, None, torch.device("cuda", torch.cuda.current_device()))
    n, longest = case["requests"], case["prompt"] + case["new"]
    pages = n * -(-longest // BLOCK) + 1
    if case["model"] == "llama":
        from hipserve.engine.model_runner import ModelRunner
        from hipserve.ops import load_library
        from hipserve.weights.safetensors_loader import save_hf_checkpoint

        m = LLAMA
        load_library()
        cfg = PRESETS["llama-3-8b"].replace(name="llama-3-few-layers", num_layers=m["layers"], vocab_size=VOCAB)
        with tempfile.TemporaryDirectory(dir="/dev/shm" if os.path.isdir("/dev/shm") else None) as d:
            save_hf_checkpoint(d, cfg, {k: v.cpu() for k, v in tensors.items()})
            runner = ModelRunner(EngineConfig(model=d, load_format="safetensors", device="cuda", max_num_seqs=graph_size(case),
                                              max_num_batched_tokens=STEP_ROWS, max_model_len=4096, num_kv_blocks=pages,
                                              enforce_eager=True), cfg, tp)
        return runner.model, runner.kv, None, (runner.tmp_out, runner.tmp_ml)
    from hipserve.bench.layer_compare import MODELS
    from hipserve.models.registry import build_model

    cfg = MODELS[case["model"]](f"w{case['width']}", SIZES[case["width"]])
    model = build_model(cfg, tp, dev, getattr(torch, case["dtype"]), get_ops(dev), max_pos=4096)
    small = {k: v.cpu() for k, v in tensors.items() if v.dim() == 1}
    model.load_tensors(lambda k: small[k] if k in small else tensors[k])
    return model, model.allocate_kv_cache(pages, BLOCK), model.allocate_state(n + 1), (None, None)


def graph_size(case):
    return next(b for b in GRAPH_SIZES if b >= case["requests"])


def plan_steps(case):
    """Prompt steps as the scheduler cuts them: lists of (request, first token, past the last token)."""
    steps, left = [[]], STEP_ROWS
    for r, n in enumerate(lengths(case)):
        at = 0
        while at < n:
            if left == 0:
                steps.append([])
                left = STEP_ROWS
            take = min(left, n - at)
            steps[-1].append((r, at, at + take))
            at, left = at + take, left - take
    return steps


def prepare(case, seed):
    from hipserve.models.llama import AttnMeta

    model, kv, states, (tmp_out, tmp_ml) = build(case, make_tensors(case, seed))
    tokens = make_tokens(case, seed)
    n, size, lens = case["requests"], graph_size(case), lengths(case)
    dev = tokens.device
    width = -(-(case["prompt"] + case["new"]) // BLOCK)
    order = torch.randperm(n * width, generator=torch.Generator().manual_seed(seed)).int()   # pages in no order, as in use
    tables = order.view(n, width).to(dev)
    scratch_page, listed_model = n * width, case["model"] != "llama"

    def slots_of(pos, rows):
        return tables[rows, pos // BLOCK].long() * BLOCK + pos % BLOCK

    def int32(v):
        return torch.tensor(v, dtype=torch.int32, device=dev)

    prompts = []
    for step in plan_steps(case):
        pos = torch.cat([torch.arange(a, b, device=dev) for _, a, b in step])
        req = torch.cat([torch.full((b - a,), r, device=dev) for r, a, b in step])
        rows = torch.tensor([r for r, _, _ in step], device=dev)
        cu = [0]
        for _, a, b in step:
            cu.append(cu[-1] + b - a)
        tiles = sorted(((i, t) for i, (_, a, b) in enumerate(step) for t in range(0, b - a, 128)), key=lambda x: -(step[x[0]][1] + x[1]))
        ctx = int32([b for _, _, b in step])
        meta = AttnMeta(num_prefill_tokens=cu[-1], num_decode=0, positions=pos, slot_mapping=slots_of(pos, req), bt_prefill=tables[rows],
                        cu_q=int32(cu), ctx_prefill=ctx, tiles=int32(tiles).view(-1, 2), tmp_out=tmp_out, tmp_ml=tmp_ml)
        if listed_model:
            meta.seq_cu, meta.seq_ctx, meta.seq_bt, meta.seq_state, meta.state = meta.cu_q, ctx, meta.bt_prefill, rows.int(), states
            meta.max_q, meta.max_ctx = max(b - a for _, a, b in step), max(b for _, _, b in step)
        ends = [(j, r) for j, (r, _, b) in enumerate(step) if b == lens[r]]   # prompts that are complete after this step
        prompts.append((tokens[req, pos], meta, torch.tensor([cu[j + 1] - 1 for j, _ in ends], device=dev),
                        torch.tensor([r for _, r in ends], device=dev)))

    # decode steps: [ids | positions | slots | context lengths] of every step, and the graph's own copy of one of them
    first = torch.tensor(lens, device=dev)
    inputs = torch.zeros(case["new"], 4, size, dtype=torch.long, device=dev)
    inputs[:, 2], inputs[:, 3] = scratch_page * BLOCK, 1
    for t in range(case["new"]):
        pos = first + t
        inputs[t, 0, :n], inputs[t, 1, :n] = tokens.gather(1, pos[:, None])[:, 0], pos
        inputs[t, 2, :n], inputs[t, 3, :n] = slots_of(pos, torch.arange(n, device=dev)), pos + 1
    now = inputs[0].clone() if case["new"] else None
    ctx32 = torch.ones(size, dtype=torch.int32, device=dev)
    bt = torch.full((size, width), scratch_page, dtype=torch.int32, device=dev)
    bt[:n] = tables
    slot = torch.full((size,), n, dtype=torch.int32, device=dev)
    slot[:n] = torch.arange(n, device=dev)
    meta = AttnMeta(num_prefill_tokens=0, num_decode=size, positions=now[1], slot_mapping=now[2], bt_decode=bt, ctx_decode=ctx32,
                    tmp_out=tmp_out, tmp_ml=tmp_ml)
    if listed_model:
        meta.seq_cu, meta.seq_ctx, meta.seq_bt = torch.arange(size + 1, dtype=torch.int32, device=dev), ctx32, bt
        meta.seq_state, meta.state, meta.max_q, meta.max_ctx = slot, states, 1, case["prompt"] + case["new"]

    def decode():
        ctx32.copy_(now[3])
        return model.compute_logits(model.forward(now[0], meta, kv))

    with torch.inference_mode():
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            decode()
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            logits = decode()
    # the graph reads and writes the tensors it was captured with: they live as long as it does
    return dict(model=model, kv=kv, prompts=prompts, inputs=inputs, now=now, graph=graph, step_meta=meta, step_logits=logits,
                out=torch.empty(case["new"] + 1, n, VOCAB, device=dev))


@torch.inference_mode()
def run(state):
    model, out = state["model"], state["out"]
    for ids, meta, rows, requests in state["prompts"]:
        hidden = model.forward(ids, meta, state["kv"])
        if len(rows):
            out[0].index_copy_(0, requests, model.compute_logits(hidden.index_select(0, rows)).float())
    for t in range(out.shape[0] - 1):
        state["now"].copy_(state["inputs"][t])
        state["graph"].replay()
        out[t + 1].copy_(state["step_logits"][: out.shape[1]])
    return out


# ---------------------------------------------------------------- work, tolerance
def work(case):
    """Every weight once per step that uses it (the steps depend on each other), the visible cache rows once per request and
    decode step and once per prompt step, written cache rows and states, embedding rows and logits."""
    el = 4 if case["dtype"] == "float32" else 2
    lens, new, n = lengths(case), case["new"], case["requests"]
    sh = shapes(case)
    numel = lambda k: sh[k][0][0] * (sh[k][0][1] if len(sh[k][0]) > 1 else 1)  # noqa: E731
    embed = "model.embed_tokens.weight" if case["model"] == "llama" else "embed"
    head = "lm_head.weight" if case["model"] == "llama" else "head"
    experts = [k for k in sh if ".mlp.e" in k]
    shared = sum(numel(k) * (2 if case["model"] == "fikizen" and k.startswith("l0.") else 1) for k in sh
                 if k not in (embed, head) and k not in experts and not k.endswith(".table"))
    steps = [sum(b - a for _, a, b in s) for s in plan_steps(case)] + [n] * new
    rows = sum(steps)
    flops = 2.0 * shared * rows + 2.0 * numel(head) * n * (new + 1)
    bytes_ = 0.0
    for t in steps:
        used = 0.0
        if experts:
            E, top = SIZES[case["width"]]["experts"], SIZES[case["width"]]["top"]
            used = sum(numel(k) for k in experts) * (1 - (1 - top / E) ** t)
        bytes_ += el * (shared + used + numel(head)) + t * (numel(embed) // VOCAB) * el
    if experts:
        flops += 2.0 * rows * SIZES[case["width"]]["top"] * sum(numel(k) for k in experts) / SIZES[case["width"]]["experts"]
    bytes_ += 4.0 * VOCAB * n * (new + 1)
    seen = lambda a, b, w: sum(min(p + 1, w) for p in range(a, b))  # noqa: E731  (keys the rows a .. b - 1 see)
    if case["model"] == "llama":
        layers, window, per_key, row = LLAMA["layers"], 1 << 30, 4 * 4096, 2 * 1024
    elif case["model"] == "fikizen":
        s = SIZES[case["width"]]
        layers, window, per_key, row = 3, s["window"], 4 * s["heads"] * 128, 2 * max(1, s["heads"] // 4) * 128
        state = s["heads"] * 128 * 128 + s["width"] * 64
        flops += 8.0 * state * rows
        bytes_ += 8.0 * state * (n * new + sum(len(p) for p in plan_steps(case)))
    else:
        s = SIZES[case["width"]]
        layers, window, per_key, row = 2, s["window"], 2 * s["heads"] * 320, 576
    for length in lens:
        flops += float(layers) * per_key * seen(0, length + new, window)
        bytes_ += float(layers) * row * el * (length + new + sum(min(length + t + 1, window) for t in range(new)))
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """Measured against ``exact``: 1.3e-6 - 1.5e-6 in float32, 0.0031 - 0.006 in bf16, 0.0065 - 0.0076
    where the residual stream is bf16 too (llama); two implementations stand on either side."""
    return {"rel": 1e-5 if case["dtype"] == "float32" else 0.03 if case["model"] == "llama" else 0.02}


# ---------------------------------------------------------------- the same in 64 bits
D = torch.float64


def _rms(x, w, eps, groups=1):
    y = x.unflatten(-1, (groups, -1))
    return (y * torch.rsqrt(y.square().mean(-1, keepdim=True) + eps)).flatten(-2) * w


def _rotate(x, dims, base):
    """x [B, L, heads, d]: entry i of the first ``dims`` pairs with i + dims / 2, angle position * base^(-2 i / dims)."""
    h = dims // 2
    f = base ** (-2.0 * torch.arange(h, device=x.device, dtype=D) / dims)
    a = torch.arange(x.shape[1], device=x.device, dtype=D)[:, None] * f
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    return torch.cat([x[..., :h] * c - x[..., h:dims] * s, x[..., h:dims] * c + x[..., :h] * s, x[..., dims:]], -1)


def _attend(q, k, v, scale, window=0, sink=False):
    """q [B, L, H, d], k, v [B, L, G, .]: causal, the last ``window`` keys; with ``sink`` one more key of score 0 without a value."""
    B, L, H, _ = q.shape
    i = torch.arange(L, device=q.device)
    back = i[:, None] - i
    hidden = (back < 0) | (back >= window) if window else back < 0
    out = torch.empty(B, L, H, v.shape[-1], device=q.device, dtype=D)
    for b in range(B):
        for g in range(k.shape[2]):
            hs = slice(g * (H // k.shape[2]), (g + 1) * (H // k.shape[2]))
            s = torch.matmul(q[b, :, hs].transpose(0, 1), k[b, :, g].t()).mul_(scale).masked_fill_(hidden, -math.inf)
            if sink:
                m = s.amax(-1, keepdim=True).clamp_(min=0.0)
                e = torch.exp(s.sub_(m))
                s = e / (e.sum(-1, keepdim=True) + torch.exp(-m))
            else:
                s = torch.softmax(s, -1)
            out[b, :, hs] = torch.matmul(s, v[b, :, g].contiguous()).transpose(0, 1)
    return out.flatten(2)


def _llama(W, tokens):
    m = LLAMA
    x = W("model.embed_tokens.weight")[tokens]
    for i in range(m["layers"]):
        w = lambda n: W(f"model.layers.{i}.{n}.weight")  # noqa: E731
        h = _rms(x, w("input_layernorm"), m["eps"])
        q, k, v = (F.linear(h, w(f"self_attn.{n}_proj")).unflatten(-1, (-1, m["dim"])) for n in "qkv")
        q, k = _rotate(q, m["dim"], m["theta"]), _rotate(k, m["dim"], m["theta"])
        x = x + F.linear(_attend(q, k, v, m["dim"] ** -0.5), w("self_attn.o_proj"))
        h = _rms(x, w("post_attention_layernorm"), m["eps"])
        x = x + F.linear(F.silu(F.linear(h, w("mlp.gate_proj"))) * F.linear(h, w("mlp.up_proj")), w("mlp.down_proj"))
    return _rms(x, W("model.norm.weight"), m["eps"]), "lm_head.weight"


def _window_attention(W, p, h, s, biased):
    q, k, v = (F.linear(h, W(p + n), W(f"{p}{n}.b") if biased else None) for n in "qkv")
    if biased:
        q, k = _rms(q, W(p + "q.norm"), 1e-6), _rms(k, W(p + "k.norm"), 1e-6)
    q, k, v = (_rotate(x.unflatten(-1, (-1, 128)), 64, 5e5) if x is not v else x.unflatten(-1, (-1, 128)) for x in (q, k, v))
    if biased:
        v = _rms(v, 1.0, 1e-6)
    o = _attend(q, k, v, 128 ** -0.5, s["window"], True)
    if not biased:
        o = (o.unflatten(-1, (-1, 128)) * torch.sigmoid(F.linear(h, W(p + "g")))[..., None]).flatten(2)
    return F.linear(o, W(p + "o"))


def _unit(x):
    return x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6)


def _gated_delta(W, p, h, s):
    def conv(n):
        y, w = F.linear(h, W(p + n)), W(f"{p}{n}.conv")
        y = F.pad(y, (0, 0, 3, 0))
        return F.silu(sum(y[:, j:j + h.shape[1]] * w[:, j] for j in range(4))).unflatten(-1, (-1, 128))

    H = s["heads"]
    q, k, v = _unit(conv("q")) * 128 ** -0.5, _unit(conv("k")), conv("v")
    q, k = (x.repeat_interleave(H // x.shape[2], 2) for x in (q, k))
    beta = torch.sigmoid(F.linear(h, W(p + "b")))
    g = torch.exp(-torch.exp(W(p + "A_log")) * F.softplus(F.linear(h, W(p + "a")) + W(p + "dt_bias")))
    S = torch.zeros(h.shape[0], H, 128, 128, device=h.device, dtype=D)
    o = torch.empty_like(v)
    for t in range(h.shape[1]):
        S = S * g[:, t, :, None, None]
        u = beta[:, t, :, None] * (v[:, t] - (S * k[:, t, :, :, None]).sum(2))
        S = S + k[:, t, :, :, None] * u[:, :, None]
        o[:, t] = (S * q[:, t, :, :, None]).sum(2)
    o = _rms(o, W(p + "norm"), 1e-6).flatten(2) * F.silu(F.linear(h, W(p + "g")))
    return F.linear(o, W(p + "o"))


def _delta_rule(W, p, h, s):
    r, k, v = (F.linear(h, W(p + n)).unflatten(-1, (-1, 64)) for n in "rkv")
    w = F.linear(torch.tanh(F.linear(h, W(p + "w1"))), W(p + "w2")) + W(p + "w0")
    w = torch.exp(-math.exp(-0.5) * torch.sigmoid(w)).unflatten(-1, (-1, 64))
    u = _unit(k)
    au = u * torch.sigmoid(F.linear(h, W(p + "a")) + W(p + "a.b")).unflatten(-1, (-1, 64))
    S = torch.zeros(h.shape[0], r.shape[2], 64, 64, device=h.device, dtype=D)
    o = torch.empty_like(v)
    for t in range(h.shape[1]):
        us = (S * u[:, t, :, :, None]).sum(2)
        S = S * w[:, t, :, :, None] - au[:, t, :, :, None] * us[:, :, None] + k[:, t, :, :, None] * v[:, t, :, None]
        o[:, t] = (S * r[:, t, :, :, None]).sum(2)
    o = _rms(o, 1.0, 1e-6).flatten(2) * W(p + "norm") * torch.sigmoid(F.linear(h, W(p + "g")))
    return F.linear(o, W(p + "o"))


def _fikizen(W, tokens, s):
    x = W("embed")[tokens]
    for l in (0, 1, 2, 0):
        h, p = _rms(x, W(f"l{l}.norm1"), 1e-6), f"l{l}.mix."
        if l == 0:
            y = _window_attention(W, p, h, s, False)
        elif l == 1:
            y = _gated_delta(W, p, h, s)
        else:
            y = 0.75 * _window_attention(W, p + "left.", h, s, True) + 1.25 * _delta_rule(W, p + "right.", h, s)
        x = x + y
        if l != 1:
            z = F.linear(_rms(x, W(f"l{l}.norm2"), 1e-6), W(f"l{l}.mlp.up"))
            a, b = F.softplus(W(f"l{l}.mlp.act"))
            z = torch.where(z > 0, a * z * z, (0.5 + b) * (torch.expm1(z.clamp(max=0.0)) - z)) + z / 2
            x = x + F.linear(z, W(f"l{l}.mlp.down"))
    return _rms(x, W("final.norm"), 1e-6), "head"


def _kesirax(W, tokens, s):
    B, L = tokens.shape
    x = W("embed")[tokens]
    for l in range(4):
        h, p = _rms(x, W(f"l{l}.norm1"), 1e-6, 4), f"l{l}.mix."
        if l % 2 == 0:
            q = F.linear(_rms(F.linear(h, W(p + "dq")), W(p + "dq.norm"), 1e-6), W(p + "uq")).unflatten(-1, (-1, 192))
            q = torch.cat([q[..., :128], _rotate(q[..., 128:], 64, 10000.0)], -1)
            c, kr = F.linear(h, W(p + "dkv")).split([512, 64], -1)
            c, kr = _rms(c, W(p + "dkv.norm"), 1e-6), _rotate(kr[:, :, None], 64, 10000.0)
            k, v = (F.linear(c, W(p + n)).unflatten(-1, (-1, 128)) for n in ("uk", "uv"))
            k = torch.cat([k, kr.expand(B, L, k.shape[2], 64)], -1)
            o = _attend(q, k, v, 192 ** -0.5, s["window"]).unflatten(-1, (-1, 128))
            y = (o * torch.sigmoid(F.linear(h, W(p + "g")))[..., None]).flatten(2)
        else:
            z, g = torch.sigmoid(F.linear(h, W(p + "z"), W(p + "z.b"))), F.silu(F.linear(h, W(p + "g")))
            u = F.linear(h, W(p + "x"), W(p + "x.b"))
            u = torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
            S = torch.zeros_like(u[:, 0])
            y = torch.empty_like(u)
            for t in range(L):
                S = S + z[:, t] * (u[:, t] - S)
                y[:, t] = S
            y = y * g
        y = F.linear(y, W(p + "o")) * W(f"l{l}.ls1")
        rows, chosen = h.flatten(0, 1), W(f"l{l}.mlp.table")[tokens].flatten(0, 1)
        f = torch.zeros_like(rows)
        for e in range(s["experts"]):
            at = (chosen == e).any(1).nonzero()[:, 0]
            a = F.relu(F.linear(rows[at], W(f"l{l}.mlp.e{e}.up"))).square()
            f[at] += F.linear(a, W(f"l{l}.mlp.e{e}.down")) / s["top"]
        x = x + y + f.view_as(x) * W(f"l{l}.ls2")
    return _rms(x, W("final.norm"), 1e-6, 4), "head"


@torch.inference_mode()
def exact(case, seed):
    tensors, tokens = make_tensors(case, seed), make_tokens(case, seed)

    @functools.lru_cache(maxsize=2)
    def W(name):
        t = tensors[name]
        return t if t.dtype == torch.int32 else t.to(D)

    if case["model"] == "llama":
        hidden, head = _llama(W, tokens)
    else:
        hidden, head = (_fikizen if case["model"] == "fikizen" else _kesirax)(W, tokens, SIZES[case["width"]])
    # a request's logits after its prompt and after each of its new tokens (rows past a request's end are never read)
    at = torch.tensor(lengths(case), device=tokens.device)[:, None] - 1 + torch.arange(case["new"] + 1, device=tokens.device)
    rows = torch.stack([hidden[r, at[r]] for r in range(case["requests"])], 1)
    logits = F.linear(rows, W(head))
    return 25.0 * torch.tanh(logits / 25.0) if case["model"] == "fikizen" else logits
