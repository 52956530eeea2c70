"""The work a user of this library has it do, as cases that can be timed and compared: whole decode steps and whole
prefill chunks of the model shapes the library is used with, through its public entry points.

  token    One token through a model, as an engine's decode step makes it: the token's embedding row, the rotary
           angles, every decode layer, the last norm and the output matrix.  Captured once as a HIP graph (the
           position is read on the device) and replayed.
  prefill  One chunk of a prompt through the attention of every layer: rotary embedding of its Q and K rows, the store
           into the fp16 cache, causal attention over the cache so far.  Launched call by call: depth and chunk size
           are arguments by value, so an engine cannot keep a graph of it.

`calls`: the operators one by one, in the order and under the names an engine written against them already has;
otherwise the entry points that fuse them.
"""
import math

import torch

from orin_llm_amd import kernels, layer

# Attention, feed-forward and vocabulary sizes; rotary pairing and base; q/k/v biases; per-head q/k norms; K channels
# that stand out per KV head (as trained K projections have them); per-pair frequency factors; the longest context used.
SHAPES = {
    "qwen1.5b": dict(n_head=12, n_kv=2, head_dim=128, n_embd=1536, n_ff=8960, layers=28, vocab=151936, neox=1, theta=1.0e6,
                     bias=True, qk_norm=False, outliers=4, factors=False, max_ctx=32768),
    "qwen7b": dict(n_head=28, n_kv=4, head_dim=128, n_embd=3584, n_ff=18944, layers=28, vocab=152064, neox=1, theta=1.0e6,
                   bias=True, qk_norm=False, outliers=4, factors=False, max_ctx=32768),
    "llama8b": dict(n_head=32, n_kv=8, head_dim=128, n_embd=4096, n_ff=14336, layers=32, vocab=128256, neox=0, theta=5.0e5,
                    bias=False, qk_norm=False, outliers=0, factors=False, max_ctx=8192),
    "llama1b": dict(n_head=32, n_kv=8, head_dim=64, n_embd=2048, n_ff=8192, layers=16, vocab=128256, neox=0, theta=5.0e5,
                    bias=False, qk_norm=False, outliers=0, factors=True, max_ctx=32768),
    "qwen3": dict(n_head=16, n_kv=8, head_dim=128, n_embd=1024, n_ff=3072, layers=28, vocab=151936, neox=1, theta=1.0e6,
                  bias=False, qk_norm=True, outliers=0, factors=False, max_ctx=32768),
}
EPS = 1.0e-6

# Weight types of a model file: (most matrices, attn_v and ffn_down, embedding and output).  The K mixes keep the
# matrices that matter most in Q6_K, as quantised files do.
FILES = {
    "q4_k_m": (layer.Q4_K, layer.Q6_K, layer.Q6_K),
    "q5_k_m": (layer.Q5_K, layer.Q6_K, layer.Q6_K),
    "q6_k": (layer.Q6_K, layer.Q6_K, layer.Q6_K),
    "q8_0": (layer.Q8_0, layer.Q8_0, layer.Q8_0),
    "f16": (layer.F16, layer.F16, layer.F16),
}
BLOCK = {layer.F16: (1, 2), layer.Q8_0: (32, 34), layer.Q4_K: (256, 144), layer.Q5_K: (256, 176), layer.Q6_K: (256, 210)}
TABLE_ROWS = 64  # rows kept of the embedding table: a step reads one
CHUNK = 512      # the longest chunk a prompt is cut into


def listed():
    return [
        # a short question to the smallest model in common use: latency and launches
        dict(name="prefill-qwen1.5b-45", kind="prefill", shape="qwen1.5b", n_ctx=4096, n_past=0, batch=45, calls=False),
        # the last whole chunk of a 4k prompt
        dict(name="prefill-qwen1.5b-512-at-3584", kind="prefill", shape="qwen1.5b", n_ctx=4096, n_past=3584, batch=512, calls=False),
        # a whole chunk in the middle of the context of the model most often served
        dict(name="prefill-llama8b-512-at-4096", kind="prefill", shape="llama8b", n_ctx=8192, n_past=4096, batch=512, calls=False),
        # the last chunk of a full 32k context, seven query heads per KV head: the most arithmetic
        dict(name="prefill-qwen7b-512-at-32256", kind="prefill", shape="qwen7b", n_ctx=32768, n_past=32256, batch=512, calls=False),
        # a ragged follow-up question in a chat, head size 64, from an engine that makes the calls one by one
        dict(name="prefill-llama1b-301-at-1501-calls", kind="prefill", shape="llama1b", n_ctx=8192, n_past=1501, batch=301, calls=True),
        # chat with a small quantised model, a few hundred tokens in: the shortest steps
        dict(name="token-qwen1.5b-q4km-at-200", kind="token", shape="qwen1.5b", file="q4_k_m", n_ctx=4096, pos=200, calls=False),
        # the same model at the end of a full context
        dict(name="token-qwen1.5b-q4km-at-32767", kind="token", shape="qwen1.5b", file="q4_k_m", n_ctx=32768, pos=32767, calls=False),
        # the model most often served, at the end of its context
        dict(name="token-llama8b-q4km-at-8191", kind="token", shape="llama8b", file="q4_k_m", n_ctx=8192, pos=8191, calls=False),
        # a larger file and seven query heads per KV head, half way
        dict(name="token-qwen7b-q5km-at-16001", kind="token", shape="qwen7b", file="q5_k_m", n_ctx=32768, pos=16001, calls=False),
        # head size 64, frequency factors, the format small models are shipped in
        dict(name="token-llama1b-q8_0-at-1777", kind="token", shape="llama1b", file="q8_0", n_ctx=8192, pos=1777, calls=False),
        # unquantised weights, which 288 GB leave room for: the most bytes
        dict(name="token-llama8b-f16-at-8191", kind="token", shape="llama8b", file="f16", n_ctx=8192, pos=8191, calls=False),
        # an engine that makes the operator calls one by one, as it did before it linked this library
        dict(name="token-qwen1.5b-q4km-at-1000-calls", kind="token", shape="qwen1.5b", file="q4_k_m", n_ctx=4096, pos=1000, calls=True),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 5.0e12, w["flops"] / 6.0e14)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        shape = rng.choice(sorted(SHAPES))
        n_ctx = rng.choice([n for n in (2048, 4096, 8192, 16384, 32768) if n <= SHAPES[shape]["max_ctx"]])
        calls = rng.random() < 0.2
        if rng.random() < 0.55:
            case = dict(kind="token", shape=shape, file=rng.choice(sorted(FILES)), n_ctx=n_ctx, pos=_log_int(rng, 16, n_ctx - 1), calls=calls)
        else:
            batch = _log_int(rng, 4, CHUNK) if rng.random() < 0.6 else CHUNK
            n_past = 0 if rng.random() < 0.25 else _log_int(rng, 16, n_ctx - batch)
            case = dict(kind="prefill", shape=shape, n_ctx=n_ctx, n_past=n_past, batch=batch, calls=calls)
        if _cost(case) <= most:
            return case


def _matrices(s, file):
    """{name: (type, n_in, n_out)} of a layer."""
    most, some, _ = FILES[file]
    ne, nff, nq, nkv = s["n_embd"], s["n_ff"], s["n_head"] * s["head_dim"], s["n_kv"] * s["head_dim"]
    return dict(wq=(most, ne, nq), wk=(most, ne, nkv), wv=(some, ne, nkv), wo=(most, nq, ne), ffn_gate=(most, ne, nff),
                ffn_up=(most, ne, nff), ffn_down=(some, nff, ne))


def _row_bytes(wtype, n):
    per, size = BLOCK[wtype]
    return n // per * size


def work(case):
    s = SHAPES[case["shape"]]
    d, h, g, layers = s["head_dim"], s["n_head"], s["n_kv"], s["layers"]
    if case["kind"] == "token":
        rows = case["pos"] + 1
        mats = list(_matrices(s, case["file"]).values()) * layers + [(FILES[case["file"]][2], s["n_embd"], s["vocab"])]
        weights = sum(_row_bytes(t, n_in) * n_out for t, n_in, n_out in mats)
        flops = sum(2.0 * n_in * n_out for _, n_in, n_out in mats) + 4.0 * d * h * rows * layers
        return {"bytes": float(weights + 4 * g * rows * d * layers + 4 * s["vocab"]), "flops": flops}
    b, p = case["batch"], case["n_past"]
    q_rows, kv_rows = b * h * d, b * g * d
    # q and k are read and written back rotated, v is read; K and V go to the cache; the cache is read once; out is written
    per_layer = 4 * (3 * q_rows + 3 * kv_rows) + 2 * 2 * kv_rows + 2 * 2 * g * (p + b) * d
    return {"bytes": float(per_layer * layers), "flops": 4.0 * d * h * (b * p + b * (b + 1) / 2.0) * layers}


def tolerance(case):
    # token: 32-bit sums throughout, but every layer's new K and V row is rounded to fp16, where last bits flip whole fp16
    # steps, and later layers carry that on.  prefill: the softmax weights enter the second product as fp16.
    return {"rel": 2e-4, "max": 1e-2} if case["kind"] == "token" else {"rel": 1e-3, "max": 4e-2}


def _weight(gen, wtype, n_in, n_out, std=0.03):
    """Random rows of a weight type: block scales such that the decoded values spread by about `std`, every other byte random."""
    if wtype == layer.F16:
        return (torch.randn((n_out, n_in), generator=gen, device="cuda") * std).half().view(torch.uint8).reshape(-1)
    per, size = BLOCK[wtype]
    raw = torch.randint(0, 256, (n_in // per * n_out, size), generator=gen, device="cuda", dtype=torch.uint8)
    halves = raw.view(torch.float16)
    u = torch.rand(raw.shape[0], generator=gen, device="cuda") + 0.5
    if wtype == layer.Q8_0:
        halves[:, 0] = (std / 74.0 * u).half()
    elif wtype == layer.Q4_K:
        halves[:, 0], halves[:, 1] = (std / 166.0 * u).half(), (std / 166.0 * 7.5 * u).half()
    elif wtype == layer.Q5_K:
        halves[:, 0], halves[:, 1] = (std / 340.0 * u).half(), (std / 340.0 * 15.5 * u).half()
    else:
        halves[:, 104] = (std / 1369.0 * u).half()
    return raw.reshape(-1)


def _caches(gen, s, n_ctx):
    """The K and V caches of every layer, [layer][2][n_kv][n_ctx][head_dim]: whatever they will be asked for is there."""
    kv = torch.empty((s["layers"], 2, s["n_kv"], n_ctx, s["head_dim"]), device="cuda", dtype=torch.float16)
    for one in kv.unbind(0):
        one.copy_(torch.randn(one.shape, generator=gen, device="cuda"))
        for head in one[0].unbind(0):
            head[:, torch.randperm(s["head_dim"], generator=gen, device="cuda")[: s["outliers"]]] *= 8.0
    return kv


def _use_current_stream():
    kernels.set_stream(torch.cuda.current_stream().cuda_stream)


def prepare(case, seed):
    kernels.init(torch.cuda.current_device())
    _use_current_stream()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    s = SHAPES[case["shape"]]
    return (_prepare_token if case["kind"] == "token" else _prepare_prefill)(case, s, gen)


def _factors(s):
    # (the long-context scaling of a model trained with it: low frequencies slowed down)
    return torch.linspace(1.0, 8.0, s["head_dim"] // 2, device="cuda") if s["factors"] else None


def _prepare_token(case, s, gen):
    d, h, g, ne, nff, n_ctx = s["head_dim"], s["n_head"], s["n_kv"], s["n_embd"], s["n_ff"], case["n_ctx"]
    randn = lambda *shape: torch.randn(shape, generator=gen, device="cuda")  # noqa: E731
    table_type = FILES[case["file"]][2]
    hp = dict(n_embd=ne, n_head=h, n_kv=g, head_dim=d, n_ff=nff, n_rot=d, neox=s["neox"], rms_eps=EPS, rope_theta=s["theta"],
              freq_factors_dev=_factors(s))
    cache = _caches(gen, s, n_ctx)
    model = []
    for _ in range(s["layers"]):
        one = {k: (t, _weight(gen, t, n_in, n_out)) for k, (t, n_in, n_out) in _matrices(s, case["file"]).items()}
        one["attn_norm"], one["ffn_norm"] = 1.0 + 0.1 * randn(ne), 1.0 + 0.1 * randn(ne)
        if s["bias"]:
            one["bq"], one["bk"], one["bv"] = 0.1 * randn(h * d), 0.1 * randn(g * d), 0.1 * randn(g * d)
        if s["qk_norm"]:
            one["q_norm"], one["k_norm"] = 1.0 + 0.1 * randn(d), 1.0 + 0.1 * randn(d)
        model.append(one)
    table = _weight(gen, table_type, ne, TABLE_ROWS, std=1.0)
    output, output_norm = _weight(gen, table_type, ne, s["vocab"]), 1.0 + 0.1 * randn(ne)
    zeros = lambda n: torch.zeros(n, device="cuda")  # noqa: E731
    bufs = dict(x=zeros(ne), xn=zeros(ne), xn2=zeros(ne), q=zeros(h * d), k=zeros(g * d), v=zeros(g * d), attn=zeros(h * d),
                act=zeros(nff), up_tmp=zeros(nff))
    logits, angles = zeros(s["vocab"]), torch.zeros((d // 2, 2), device="cuda")
    pos = torch.tensor([case["pos"]], dtype=torch.int32, device="cuda")
    kv = [(c[0].view(torch.int16), c[1].view(torch.int16)) for c in cache]
    descs = [layer.make_desc(hp, one, bufs, kc, vc, pos, n_ctx, rope_angles=angles) for one, (kc, vc) in zip(model, kv)]
    row = table[7 * _row_bytes(table_type, ne):]

    def step():
        layer.dequant_row(table_type, row, bufs["x"], ne)
        if case["calls"]:
            for one, (kc, vc) in zip(model, kv):
                layer.decode_layer_calls(hp, one, bufs, kc, vc, pos, n_ctx)
        else:
            kernels.rope_angles_ind(angles, d, s["theta"], pos, hp["freq_factors_dev"])
            for desc in descs:
                layer.decode_layer(desc)
        layer.rms_norm(bufs["x"], output_norm, ne, EPS, bufs["xn"])
        layer.gemv(table_type, output, bufs["xn"], logits, ne, s["vocab"])

    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    try:
        with torch.cuda.graph(graph):
            _use_current_stream()
            step()
    finally:
        _use_current_stream()
    return dict(graph=graph, out=dict(logits=logits, x=bufs["x"], cache=cache),
                keep=(model, table, output, output_norm, bufs, angles, pos, descs, hp))


def _prepare_prefill(case, s, gen):
    d, h, g, b, layers = s["head_dim"], s["n_head"], s["n_kv"], case["batch"], s["layers"]
    randn = lambda *shape: torch.randn(shape, generator=gen, device="cuda")  # noqa: E731
    cache = _caches(gen, s, case["n_ctx"])
    q, k, v = randn(layers, b, h, d), randn(layers, b, g, d), randn(layers, b, g, d)
    out = torch.empty((layers, b, h, d), device="cuda")
    per_layer = [(q[i], k[i], v[i], cache[i, 0].view(torch.int16), cache[i, 1].view(torch.int16), out[i]) for i in range(layers)]
    return dict(case=case, s=s, layers=per_layer, factors=_factors(s), scale=1.0 / math.sqrt(d), out=dict(out=out, q=q, k=k, cache=cache))


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    case, s, factors, scale = state["case"], state["s"], state["factors"], state["scale"]
    h, g, d, theta, n_ctx, n_past, b = s["n_head"], s["n_kv"], s["head_dim"], s["theta"], case["n_ctx"], case["n_past"], case["batch"]
    rope = kernels.rope_neox_batch if s["neox"] else kernels.rope_normal_batch
    for q, k, v, kc, vc, out in state["layers"]:
        if case["calls"]:
            rope(q, b * h, d, d, theta, n_past, h, factors)
            rope(k, b * g, d, d, theta, n_past, g, factors)
            kernels.kv_store_batch(kc, vc, k, v, g, d, n_ctx, n_past, b)
        else:
            kernels.rope_store_batch(q, k, v, kc, vc, b, h, g, d, n_ctx, n_past, d, theta, factors, bool(s["neox"]))
        kernels.flash_attention(q, kc, vc, out, h, g, d, n_ctx, n_past, b, scale)
    return state["out"]
