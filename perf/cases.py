"""The calls whose speed is followed: what a program that decodes with this library makes, by size.

listed() names them, draw() gives more of the same ranges, prepare() builds what such a program holds before
the call, run() is one pass, work() what the pass cannot do without, exact() the same in 64 bits.

Op-level passes go over several layers' weights (or K/V pages) captured once in a graph, as a decode loop does,
so weights come from memory and not from a cache that the previous call left warm; every layer has inputs and
outputs of its own.  Engine passes go through Transformer and Engine.
"""
import math

import numpy as np
import torch  # before qraf_amd: the library then shares torch's HIP runtime

from qraf_amd import F16, F32, Q4_0, Q8_0, lib
from qraf_amd._lib import I8, SamplingParams, call
from qraf_amd.backend import Graph, Stream, backend_init
from qraf_amd.engine import Engine, Transformer, model_config

QUANT = {"q8": Q8_0, "q4": Q4_0}
PAGES = {"f32": F32, "f16": F16, "i8": I8}

# the two architectures the benchmark decodes (random weights)
SMOLLM2 = dict(vocab=49152, hidden=576, layers=30, heads=9, kv_heads=3, inter=1536, theta=1e5, eps=1e-5, tied=False,
               bias=False, weights="q8")
QWEN25_3B = dict(vocab=151936, hidden=2048, layers=36, heads=16, kv_heads=2, inter=11008, theta=1e6, eps=1e-6,
                 tied=True, bias=True, weights="q4")


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # one sequence, one token: Transformer.forward of the small model, the latency a chat user sees
        dict(name="forward smollm2 b1", kind="forward", context=160, **SMOLLM2),
        # single projections at batch 1, the product every decoded token is made of
        dict(name="matvec q8 11008x4096", kind="matvec", weights="q8", n=11008, k=4096, layers=10),
        dict(name="matvec q4 4096x4096", kind="matvec", weights="q4", n=4096, k=4096, layers=40),
        # batched projections: a few dozen concurrent sequences, 128 of them (gate and up in one product), and a
        # ragged count in a step that mixes decoding with a prompt chunk
        dict(name="gemm q4 11008x2048 b32", kind="gemm", weights="q4", n=11008, k=2048, batch=32, layers=16),
        dict(name="gemm q4 22016x2048 b128", kind="gemm", weights="q4", n=22016, k=2048, batch=128, layers=8),
        dict(name="gemm q8 2048x11008 b203", kind="gemm", weights="q8", n=2048, k=11008, batch=203, layers=8),
        # the MLP of a prompt chunk: gate/up with the SiLU-gate in its epilogue, down with the residual
        dict(name="mlp q4 2048-11008 b512", kind="mlp", weights="q4", hidden=2048, inter=11008, batch=512, layers=4),
        # decode attention over long ragged contexts (the reference's f32 cache) and over chat-length fp16 ones
        dict(name="attention f32 128x4096", kind="attention", pages="f32", seqs=128, least=128, most=4096, heads=16,
             kv_heads=2, head_dim=128, page=16, layers=2),
        dict(name="attention f16 128x768", kind="attention", pages="f16", seqs=128, least=16, most=768, heads=16,
             kv_heads=2, head_dim=128, page=16, layers=12),
        # sampled decoding: temperature, top-k, top-p over the vocabulary for every sequence of the batch
        dict(name="sample 128x151936", kind="sample", rows=128, vocab=151936, temperature=0.8, top_k=40, top_p=0.9),
        # a 512-row prompt step through a few layers of the larger model: four prompts, 128 rows of each
        dict(name="prompt 512 rows", kind="stack", rows=512, seqs=4, least=0, most=256, pages="f32",
             **dict(QWEN25_3B, layers=4, vocab=8192)),
        # 128 sequences decoding through the whole larger model, four pipelined steps
        dict(name="decode qwen2.5-3b b128", kind="decode", seqs=128, least=16, most=640, steps=4, **QWEN25_3B),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec", "matvec", "rows", "gemm", "gemm", "gemm", "mlp", "attention", "attention", "sample",
                       "stack", "stack"])
    w = rng.choice(["q8", "q4"])
    if kind == "matvec":
        n, k = _log(rng, 192, 22016), _log(rng, 576, 11008)
        return dict(kind=kind, weights=w, n=n, k=k, layers=max(2, min(30, (200 << 20) // (n * k))))
    if kind == "rows":  # a handful of sequences, below the matrix cores' batch
        n, k = _log(rng, 192, 11008), 64 * _log(rng, 9, 48)
        return dict(kind=kind, weights=w, n=n, k=k, batch=rng.randint(2, 8),
                    layers=max(2, min(24, (200 << 20) // (n * k))))
    if kind == "gemm":
        n, k = _log(rng, 256, 22016), 32 * _log(rng, 18, 344)
        n = min(n, (46 << 20) // k)
        b = _log(rng, 9, 512)
        return dict(kind=kind, weights=w, n=n, k=k, batch=b, layers=max(2, min(12, (200 << 20) // (n * max(k, 4 * b)))))
    if kind == "mlp":
        h, f, b = 32 * _log(rng, 18, 64), 32 * _log(rng, 48, 344), _log(rng, 16, 512)
        return dict(kind=kind, weights=w, hidden=h, inter=f, batch=b, layers=max(2, min(8, (150 << 20) // (h * f))))
    if kind == "attention":
        hd, kv = rng.choice([64, 128]), rng.choice([1, 2, 3, 4, 8])
        group = rng.choice([1, 2, 3, 4, 6, 8])
        seqs, most = _log(rng, 1, 160), _log(rng, 48, 4096)
        seqs = max(1, min(seqs, (128 * 4096 * 256) // (most * kv * hd)))
        pages = rng.choice(["f32", "f16", "i8"])
        return dict(kind=kind, pages=pages, seqs=seqs, least=1 + most // 32, most=most, heads=kv * group, kv_heads=kv,
                    head_dim=hd, page=rng.choice([16, 16, 32]),
                    layers=max(2, min(12, (128 * 4096 * 256) // (seqs * most * kv * hd))))
    if kind == "sample":
        rows, vocab = _log(rng, 1, 160), 4 * _log(rng, 8000, 40000)
        return dict(kind=kind, rows=rows, vocab=vocab, temperature=round(rng.uniform(0.5, 1.2), 2),
                    top_k=rng.choice([20, 40, 50, 100, 400]), top_p=rng.choice([0.8, 0.9, 0.95, 1.0]))
    heads, hd = rng.choice([(9, 64), (8, 64), (12, 64), (8, 128), (16, 128)])
    kv = rng.choice([d for d in (1, 2, 3, 4) if heads % d == 0])
    seqs = _log(rng, 1, 128)
    rows = seqs * rng.choice([1, 1, max(1, _log(rng, 2, 256) // seqs)])
    return dict(kind="stack", rows=rows, seqs=seqs, least=0, most=_log(rng, 32, 512),
                pages=rng.choice(["f32", "f32", "f16"]), hidden=heads * hd, heads=heads, kv_heads=kv,
                inter=32 * _log(rng, 48, 256), layers=rng.randint(2, 4), vocab=4 * _log(rng, 500, 3000), theta=1e6,
                eps=1e-6, tied=rng.random() < 0.5, bias=rng.random() < 0.5, weights=w)


# ------------------------------------------------------------------ inputs

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape, std=1.0):
    return torch.empty(shape, device="cuda").normal_(0.0, std, generator=g)


def _quantized(g, weights, n, k, std=0.02):
    """N(0, std) weights [n][k] in the library's block layout (blocks of 32 along a row): (bytes, integers, scales)."""
    nb = -(-k // 32)
    w = _normal(g, n, nb, 32, std=std)
    if k % 32:
        w.view(n, nb * 32)[:, k:] = 0
    top = w.abs().amax(2)
    if weights == "q8":
        s = top / 127
        q = torch.round(w / s.unsqueeze(2)).clamp_(-127, 127)
        out = torch.empty((n, nb, 36), dtype=torch.uint8, device="cuda")
        out[:, :, :4] = s.unsqueeze(2).view(torch.uint8).view(n, nb, 4)
        out[:, :, 4:] = q.to(torch.int8).view(torch.uint8)
    else:
        s = (top / 7).half()
        q = torch.round(w / s.float().unsqueeze(2)).clamp_(-8, 7)
        u = (q + 8).to(torch.uint8)
        out = torch.empty((n, nb, 18), dtype=torch.uint8, device="cuda")
        out[:, :, :2] = s.unsqueeze(2).view(torch.uint8).view(n, nb, 2)
        out[:, :, 2:] = u[:, :, 0::2] | (u[:, :, 1::2] << 4)
    return out.view(-1), q, s


def _double(q, s, k):
    return (q.double() * s.double().unsqueeze(2)).view(q.shape[0], -1)[:, :k]


class _Plan:
    """The calls of body(stream) captured in a graph."""

    stream = None

    def __init__(self, body):
        backend_init(0)
        torch.cuda.synchronize()
        if _Plan.stream is None:
            _Plan.stream = Stream()
        self.graph = Graph(_Plan.stream)
        with self.graph:
            body(_Plan.stream.h)

    def launch(self):
        self.graph.launch()

    def __del__(self):
        try:
            self.graph.destroy()
        except Exception:
            pass


def _weights(case, g, shapes):
    """Per layer, per shape: (bytes, q, s)."""
    return [[_quantized(g, case["weights"], n, k) for n, k in shapes] for _ in range(case["layers"])]


def _tiled(dt, raw, n, k):
    t = torch.empty(lib.qraf_hip_tiled_weight_bytes(dt, n, k), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    call("qraf_hip_repack_tiles_dev", raw.data_ptr(), dt, n, k, t.data_ptr(), None)
    call("qraf_hip_device_synchronize")
    return t


def _product_inputs(case, seed):
    g, c = _generator(seed), case
    if c["kind"] == "mlp":
        shapes, k = [(2 * c["inter"], c["hidden"]), (c["hidden"], c["inter"])], c["hidden"]
    else:
        shapes, k = [(c["n"], c["k"])], c["k"]
    return shapes, _weights(c, g, shapes), _normal(g, c["layers"], c.get("batch", 1), k)


def _prepare_product(case, seed):
    backend_init(0)
    c, dt = case, QUANT[case["weights"]]
    shapes, weights, x = _product_inputs(c, seed)
    (n, k), batch, layers = shapes[0], c.get("batch", 1), c["layers"]
    if c["kind"] in ("matvec", "rows"):
        raw = [w[0][0] for w in weights]
        y = torch.empty((layers, batch, n), device="cuda")

        def body(s):
            for i in range(layers):
                if c["kind"] == "matvec":
                    call("qraf_hip_matvec_q_dev", raw[i].data_ptr(), dt, 32, n, k, x[i].data_ptr(), y[i].data_ptr(), s)
                else:
                    call("qraf_hip_matvec_q_batch_dev", raw[i].data_ptr(), dt, n, k, x[i].data_ptr(), batch,
                         y[i].data_ptr(), s)
        keep = (raw, x, y)
    else:
        tiles = [[_tiled(dt, w[j][0], *shapes[j]) for j in range(len(shapes))] for w in weights]
        planes = torch.empty((2, batch, k), dtype=torch.int16, device="cuda")
        n_out, k_out = shapes[-1]
        y = torch.empty((layers, batch, n_out), device="cuda")
        act = torch.empty((2, batch, k_out), dtype=torch.int16, device="cuda")
        need = int(lib.qraf_hip_qgemm_tiled_workspace_bytes(dt, n_out, k_out, batch))
        ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
        hi, lo, ahi, alo = planes[0].data_ptr(), planes[1].data_ptr(), act[0].data_ptr(), act[1].data_ptr()

        def body(s):
            for i in range(layers):
                call("qraf_hip_split_bf16_dev", x[i].data_ptr(), hi, lo, batch, k, s)
                if c["kind"] == "gemm":
                    call("qraf_hip_qgemm_tiled_dev", tiles[i][0].data_ptr(), dt, n, k, hi, lo, batch, y[i].data_ptr(),
                         None, ws.data_ptr(), need, s)
                else:
                    call("qraf_hip_qgemm_tiled_silu_dev", tiles[i][0].data_ptr(), dt, n, k, hi, lo, batch, ahi, alo, s)
                    call("qraf_hip_qgemm_tiled_dev", tiles[i][1].data_ptr(), dt, n_out, k_out, ahi, alo, batch,
                         y[i].data_ptr(), x[i].data_ptr(), ws.data_ptr(), need, s)
        keep = (tiles, planes, act, ws, x, y)
    del weights
    return dict(plan=_Plan(body), out=y, keep=keep)


def _exact_product(case, seed):
    shapes, weights, x = _product_inputs(case, seed)
    out = []
    for layer, xi in zip(weights, x.double()):
        if case["kind"] == "mlp":
            gu = xi @ _double(*layer[0][1:], shapes[0][1]).T
            a = torch.nn.functional.silu(gu[:, 0::2]) * gu[:, 1::2]
            out.append(xi + a @ _double(*layer[1][1:], shapes[1][1]).T)
        else:
            out.append(xi @ _double(*layer[0][1:], shapes[0][1]).T)
    return torch.stack(out)


def _attention_inputs(case, seed):
    c, g = case, _generator(seed)
    r = np.random.default_rng(seed)
    ctx = r.integers(c["least"], c["most"] + 1, c["seqs"]).astype(np.int32)
    ps, hkv, hd, layers = c["page"], c["kv_heads"], c["head_dim"], c["layers"]
    per = (ctx + ps - 1) // ps
    pages = int(per.sum())
    table = np.zeros((c["seqs"], -(-c["most"] // ps)), np.int32)
    ids, at = r.permutation(pages).astype(np.int32), 0
    for s, m in enumerate(per):
        table[s, :m] = ids[at:at + m]
        at += m
    q = _normal(g, layers, c["seqs"], c["heads"], hd)
    shape = (pages, hkv, ps, hd)
    kv = []
    for _ in range(layers):
        pair = []
        for v in (False, True):
            if c["pages"] == "i8":  # a cached head's values: bytes of its own scale
                b = (_normal(g, *shape) * 40).round().clamp(-127, 127)
                sc = torch.empty(shape[:3], device="cuda").uniform_(0.01, 0.04, generator=g)
                pair.append((b, sc))
            else:
                t = _normal(g, *shape)
                pair.append((t.half() if c["pages"] == "f16" else t, None))
        kv.append(pair)
    return ctx, table, q, kv


def _page_bytes(c, t, sc, v):
    """Positions x dims [pages][kv heads][position][dim] as the library's pages: V of fp16 and int8 pages lies
    dimension-major, int8 pages end in a scale per position."""
    if c["pages"] == "f32":
        return t
    t = t.transpose(2, 3) if v else t
    if c["pages"] == "f16":
        return t.contiguous()
    p = t.shape[0] * t.shape[1]
    return torch.cat([t.to(torch.int8).reshape(p, -1).view(torch.uint8),
                      sc.reshape(p, -1).contiguous().view(torch.uint8)], 1).contiguous()


def _prepare_attention(case, seed):
    backend_init(0)
    c = case
    ctx, table, q, kv = _attention_inputs(c, seed)
    kv = [[_page_bytes(c, t, sc, v) for v, (t, sc) in enumerate(pair)] for pair in kv]
    ctx, table = torch.from_numpy(ctx).cuda(), torch.from_numpy(table).cuda()
    n, h, hkv, hd = c["seqs"], c["heads"], c["kv_heads"], c["head_dim"]
    need = int(lib.qraf_hip_attention_workspace_bytes(n, h, hkv, hd, c["most"]))
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    out = torch.empty_like(q)

    def body(s):
        for i in range(c["layers"]):
            call("qraf_hip_paged_attention_dev", q[i].data_ptr(), kv[i][0].data_ptr(), kv[i][1].data_ptr(),
                 PAGES[c["pages"]], table.data_ptr(), table.shape[1], ctx.data_ptr(), n, h, hkv, hd, c["page"],
                 1.0 / math.sqrt(hd), c["most"], out[i].data_ptr(), ws.data_ptr(), need, s)
    return dict(plan=_Plan(body), out=out, keep=(q, kv, ctx, table, ws))


def _exact_attention(case, seed):
    c = case
    ctx, table, q, kv = _attention_inputs(c, seed)
    group, out = c["heads"] // c["kv_heads"], torch.empty(q.shape, dtype=torch.float64, device="cuda")
    scale = float(np.float32(1.0 / math.sqrt(c["head_dim"])))
    for s in range(c["seqs"]):
        ids = torch.from_numpy(table[s, :-(-int(ctx[s]) // c["page"])].astype(np.int64)).cuda()
        for i, pair in enumerate(kv):
            k, v = ((t[ids].double() if sc is None else t[ids].double() * sc[ids].double().unsqueeze(3))
                    .transpose(0, 1).reshape(c["kv_heads"], -1, c["head_dim"])[:, :ctx[s]] for t, sc in pair)
            qs = q[i, s].double().view(c["kv_heads"], group, -1)
            for h in range(c["kv_heads"]):
                p = torch.softmax(qs[h] @ k[h].T * scale, 1)
                out[i, s, h * group:(h + 1) * group] = p @ v[h]
    return out


def _prepare_sample(case, seed):
    backend_init(0)
    c, g = case, _generator(seed)
    logits = _normal(g, c["rows"], c["vocab"], std=2.0)
    uniforms = torch.rand(c["rows"], device="cuda", generator=g)
    tokens = torch.empty(c["rows"], dtype=torch.int32, device="cuda")
    # no repetition penalty: it is applied in place, and a pass leaves its inputs as they were
    params = SamplingParams(c["temperature"], c["top_k"], c["top_p"], 1.0)
    torch.cuda.synchronize()
    return dict(logits=logits, uniforms=uniforms, out=tokens, params=params)


# ------------------------------------------------------------------ engines

def _model(case, seed):
    """The model's tensors by the names a .qraf file gives them: name -> (kind, shape, bytes, q, s), one at a time."""
    c, g = case, _generator(seed)
    d, hd = c["hidden"], c["hidden"] // c["heads"]
    kv, f = c["kv_heads"] * hd, c["inter"]

    def mat(name, n, k):
        return name, c["weights"], (n, k), _quantized(g, c["weights"], n, k)

    def vec(name, n, mean, std):
        return name, "f32", (n,), _normal(g, n, std=std) + mean

    yield mat("model.embed_tokens.weight", c["vocab"], d)
    if not c["tied"]:
        yield mat("lm_head.weight", c["vocab"], d)
    yield vec("model.norm.weight", d, 1.0, 0.1)
    for i in range(c["layers"]):
        p = "model.layers.%d." % i
        yield vec(p + "input_layernorm.weight", d, 1.0, 0.1)
        yield vec(p + "post_attention_layernorm.weight", d, 1.0, 0.1)
        for x, n in (("q", d), ("k", kv), ("v", kv)):
            yield mat(p + "self_attn.%s_proj.weight" % x, n, d)
            if c["bias"]:
                yield vec(p + "self_attn.%s_proj.bias" % x, n, 0.0, 0.1)
        yield mat(p + "self_attn.o_proj.weight", d, d)
        yield mat(p + "mlp.gate_proj.weight", f, d)
        yield mat(p + "mlp.up_proj.weight", f, d)
        yield mat(p + "mlp.down_proj.weight", d, f)


def _schedule(case, seed):
    """(tokens already held by each sequence, tokens of the timed rows by sequence)."""
    c, r = case, np.random.default_rng(seed)
    if c["kind"] == "forward":
        return [r.integers(0, c["vocab"], c["context"])], [r.integers(0, c["vocab"], 1)]
    held = [r.integers(0, c["vocab"], int(m)) for m in r.integers(c["least"], c["most"] + 1, c["seqs"])]
    rows = c["steps"] if c["kind"] == "decode" else c["rows"] // c["seqs"]
    return held, [r.integers(0, c["vocab"], rows) for _ in range(c["seqs"])]


def _prepare_engine(case, seed):
    backend_init(0)
    c = case
    held, new = _schedule(c, seed)
    page, most = 16, max(512, c.get("rows", 1))
    need = sum(-(-(len(h) + len(t)) // page) for h, t in zip(held, new))
    cfg = model_config(c["vocab"], c["hidden"], c["layers"], c["heads"], c["kv_heads"], c["inter"], 2048, c["theta"],
                       c["eps"])
    if c["kind"] == "forward":  # the reference's own loop: one engine row, its default sequence
        most, need = 1, 2048 // page
    e = Engine(cfg, kv_dtype=PAGES[c.get("pages", "f32")], page_size=page, max_batch=most, num_pages=need + 8)
    for name, kind, shape, t in _model(c, seed):
        if kind == "f32":
            e.set_tensor(name, F32, shape, t.cpu().numpy())
        else:
            e.set_tensor(name, QUANT[kind], shape, t[0].cpu().numpy())
    e.finalize()
    if c["kind"] == "forward":
        t = Transformer(e)
        for pos, tok in enumerate(held[0]):
            t.forward(int(tok), pos)
        return dict(model=t, token=int(new[0][0]), pos=len(held[0]))
    ids = [e.seq_create() for _ in held]
    sid, tok, pos = (np.concatenate(v) if sum(map(len, held)) else np.zeros(0, np.int64) for v in (
        [np.full(len(h), i) for i, h in zip(ids, held)], held, [np.arange(len(h)) for h in held]))
    for a in range(0, len(sid), most):
        b = slice(a, a + most)
        e.step(sid[b], tok[b], pos[b], want_logits=np.zeros(len(sid[b]), np.uint8), argmax=False)
    if c["kind"] == "decode":
        steps = [([t[j] for t in new], [len(h) + j for h in held]) for j in range(c["steps"])]
        return dict(engine=e, ids=ids, steps=steps)
    sid = np.concatenate([np.full(len(t), i) for i, t in zip(ids, new)])
    pos = np.concatenate([len(h) + np.arange(len(t)) for h, t in zip(held, new)])
    want = np.concatenate([np.arange(len(t)) == len(t) - 1 for t in new]).astype(np.uint8)
    return dict(engine=e, ids=sid, tokens=np.concatenate(new), positions=pos, want=want)


def _exact_engine(case, seed):
    """Logits of each sequence's last new token."""
    c = case
    held, new = _schedule(c, seed)
    rows = [np.concatenate(v) for v in zip(held, new)]
    if sum(map(len, rows)) * c["layers"] * c["hidden"] * c["inter"] > 3e13:
        return None
    heads, kvh, hd = c["heads"], c["kv_heads"], c["hidden"] // c["heads"]
    ends = np.cumsum([len(r) for r in rows])
    pos = torch.from_numpy(np.concatenate([np.arange(len(r)) for r in rows])).cuda()
    freq = 1.0 / torch.pow(torch.tensor(c["theta"]), torch.arange(0, hd, 2).float() / hd)  # the model's f32 angles
    ang = (pos.float().unsqueeze(1) * freq.cuda()).double()
    cos, sin = ang.cos().unsqueeze(1), ang.sin().unsqueeze(1)

    def norm(x, w):
        return x / torch.sqrt((x * x).mean(1, keepdim=True) + c["eps"]) * w.double()

    def rope(x):
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)

    it, x, head, final, t = _model(c, seed), None, None, None, {}
    for name, kind, shape, v in it:
        if name == "model.embed_tokens.weight":
            x = _double(*v[1:], shape[1])[torch.from_numpy(np.concatenate(rows)).cuda()]
            if c["tied"]:
                head = v
            continue
        if name == "lm_head.weight":
            head = v
            continue
        if name == "model.norm.weight":
            final = v
            continue
        t[name.split(".", 3)[3]] = v if kind == "f32" else _double(*v[1:], shape[1])
        if not name.endswith("mlp.down_proj.weight"):
            continue
        h = norm(x, t["input_layernorm.weight"])
        q, k, v = (h @ t["self_attn.%s_proj.weight" % n].T +
                   (t["self_attn.%s_proj.bias" % n].double() if c["bias"] else 0.0) for n in "qkv")
        q, k, v = rope(q.view(-1, heads, hd)), rope(k.view(-1, kvh, hd)), v.view(-1, kvh, hd)
        o, a = torch.empty_like(q), 0
        for b in ends:
            mask = torch.ones((b - a, b - a), dtype=torch.bool, device="cuda").triu(1)
            for j in range(heads):
                s = (q[a:b, j] @ k[a:b, j * kvh // heads].T / math.sqrt(hd)).masked_fill(mask, -math.inf)
                o[a:b, j] = torch.softmax(s, 1) @ v[a:b, j * kvh // heads]
            a = b
        x = x + o.flatten(1) @ t["self_attn.o_proj.weight"].T
        h = norm(x, t["post_attention_layernorm.weight"])
        x = x + (torch.nn.functional.silu(h @ t["mlp.gate_proj.weight"].T) * (h @ t["mlp.up_proj.weight"].T)) @ \
            t["mlp.down_proj.weight"].T
        t = {}
    last = norm(x[torch.from_numpy(ends - 1).cuda()], final)
    out = (last @ _double(*head[1:], c["hidden"]).T).cpu().numpy()
    return out[0] if c["kind"] == "forward" else out


# ------------------------------------------------------------------ the contract

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("matvec", "rows", "gemm", "mlp"):
        return dict(_prepare_product(case, seed), kind=kind)
    if kind == "attention":
        return dict(_prepare_attention(case, seed), kind=kind)
    if kind == "sample":
        return dict(_prepare_sample(case, seed), kind=kind)
    return dict(_prepare_engine(case, seed), kind=kind)


def run(state):
    s, kind = state, state["kind"]
    if "plan" in s:
        s["plan"].launch()
        return s["out"]
    if kind == "sample":
        call("qraf_hip_sample_dev", s["logits"].data_ptr(), s["logits"].shape[0], s["logits"].shape[1], s["params"],
             None, None, 0, s["uniforms"].data_ptr(), s["out"].data_ptr(), None)
        return s["out"]
    if kind == "forward":
        return s["model"].forward(s["token"], s["pos"])
    e = s["engine"]
    if kind == "stack":
        return e.step(s["ids"], s["tokens"], s["positions"], want_logits=s["want"], logits=True, argmax=False)[0]
    tokens = []  # decode: step j + 1 is issued before step j's tokens are read, as the scheduler does
    for j, (tok, pos) in enumerate(s["steps"]):
        e.step_async(s["ids"], tok, pos)
        if j:
            tokens.append(e.collect())
    tokens.append(e.collect())
    return dict(tokens=tokens, logits=e.read_logits(0, 4))  # the rows that a program inspects


def _row_bytes(weights, k):
    return -(-k // 32) * (36 if weights == "q8" else 18)


def work(case):
    c, kind = case, case["kind"]
    if kind in ("matvec", "rows", "gemm"):
        b = c.get("batch", 1)
        return dict(bytes=c["layers"] * (c["n"] * _row_bytes(c["weights"], c["k"]) + 4 * b * (c["n"] + c["k"])),
                    flops=c["layers"] * 2.0 * b * c["n"] * c["k"])
    if kind == "mlp":
        h, f, b = c["hidden"], c["inter"], c["batch"]
        weights = 2 * f * _row_bytes(c["weights"], h) + h * _row_bytes(c["weights"], f)
        return dict(bytes=c["layers"] * (weights + 8 * b * h),
                    flops=c["layers"] * 6.0 * b * h * f)
    if kind == "attention":
        tokens = c["seqs"] * (c["least"] + c["most"]) / 2
        elem = {"f32": 4.0, "f16": 2.0, "i8": 1.0 + 4.0 / c["head_dim"]}[c["pages"]]
        return dict(bytes=c["layers"] * (2 * tokens * c["kv_heads"] * c["head_dim"] * elem +
                                         8 * c["seqs"] * c["heads"] * c["head_dim"]),
                    flops=c["layers"] * 4.0 * tokens * c["heads"] * c["head_dim"])
    if kind == "sample":
        return dict(bytes=4.0 * c["rows"] * c["vocab"], flops=2.0 * c["rows"] * c["vocab"])
    d, f = c["hidden"], c["inter"]
    hd = d // c["heads"]
    kv = c["kv_heads"] * hd
    shapes = [(d + 2 * kv, d), (d, d), (2 * f, d), (d, f)]
    layer_bytes = sum(n * _row_bytes(c["weights"], k) for n, k in shapes)
    layer_macs = sum(n * k for n, k in shapes)
    if kind == "forward":
        steps, rows, outs, held = 1, 1, 1, c["context"]
    elif kind == "decode":
        steps, rows, outs, held = c["steps"], c["seqs"], c["seqs"], c["seqs"] * (c["least"] + c["most"]) / 2
    else:
        steps, rows, outs, held = 1, c["rows"], c["seqs"], c["seqs"] * (c["least"] + c["most"]) / 2
    elem = 2 if c.get("pages") == "f16" else 4
    seen = held * (rows / c.get("seqs", 1))  # positions that the rows attend to
    return dict(bytes=steps * (c["layers"] * (layer_bytes + 2 * (held + rows) * kv * elem) +
                               c["vocab"] * _row_bytes(c["weights"], d) + 4.0 * outs * c["vocab"]),
                flops=steps * (2.0 * rows * c["layers"] * layer_macs + 4.0 * c["layers"] * seen * d +
                               2.0 * outs * c["vocab"] * d))


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":  # tokens, reproduced to the bit
        return "exact"
    if kind == "decode":  # 36 layers deep; greedy tokens may differ where two logits tie to within that
        return {"rel": 4e-5, "max": 4e-4, "differ": 0.004}
    if kind == "stack" and case["pages"] == "f16":  # a last-bit change of k or v can move its rounding to fp16
        return {"rel": 1e-4, "max": 1e-3}
    return {"rel": 1e-5, "max": 1e-4}  # 32-bit sums: 1e-7 to 2e-6 from the sums in 64 bits


def exact(case, seed):
    kind = case["kind"]
    if kind in ("matvec", "rows", "gemm", "mlp"):
        return _exact_product(case, seed)
    if kind == "attention":
        return _exact_attention(case, seed)
    if kind in ("sample", "decode"):  # tokens of a draw, and a whole model over tens of thousands of positions
        return None
    return _exact_engine(case, seed)
