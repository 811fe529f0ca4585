"""The work that programs give this framework, as measurable cases.

A decode step of a Qwen3-shaped model at batch 1, through the torch front end (llminfer_amd.ops): attention of one layer
("attend"), a step's attention over all layers with a launch per layer ("step"), the same with QK-Norm + RoPE as a call of
its own ("unfused"), in one call for all layers ("stack"), the whole attention block with its projections ("block"), a
projection alone ("project"), and the conversion of a prompt's position-major cache to the decode layout ("restride").

`listed()` holds the measured cases, `draw()` gives more of the same ranges, `prepare()` makes what a program has in hand
before the call (caches, weights, tables, workspace, captured graph), `run()` is one pass, `work()` the bytes and operations
a pass cannot do without, `tolerance()` what another correct implementation of the same precision may differ by.
"""
import torch

from llminfer_amd import _binding as B
from llminfer_amd import ops

HEAD_DIM = 128
BF16, F32 = torch.bfloat16, torch.float32
LAYOUTS = {"pos": B.KV_LAYOUT_POS_MAJOR, "head": B.KV_LAYOUT_HEAD_MAJOR}
# Query heads, KV heads, hidden size: the Qwen3-0.6B, Qwen3-4B and Qwen3-32B layer shapes ...
MODELS = [(16, 8, 1024), (32, 8, 2560), (64, 8, 5120)]
# ... and the head layouts that else occur: shards by KV head of the last two, one query head per KV head, odd groups.
OTHER_HEADS = [(16, 4), (16, 2), (8, 2), (8, 1), (8, 8), (24, 8), (40, 8), (32, 2)]


def listed():
    return [
        # the first tokens of a short chat on the smallest model: one layer, nothing but latency
        dict(name="attend-16q8kv-57", kind="attend", n_q=16, n_kv=8, ctx=57, max_seq_len=4096, layout="head"),
        # one layer in the reference engine's own cache layout, a few thousand tokens in
        dict(name="attend-32q8kv-6007-pos", kind="attend", n_q=32, n_kv=8, ctx=6007, max_seq_len=8192, layout="pos"),
        # one GPU's share (2 of 8 KV heads) of the largest model's layer at a long context
        dict(name="attend-16q2kv-40001", kind="attend", n_q=16, n_kv=2, ctx=40001, max_seq_len=40960, layout="head"),
        # the longest context: one layer of the largest model
        dict(name="attend-64q8kv-131072", kind="attend", n_q=64, n_kv=8, ctx=131072, max_seq_len=131072, layout="head"),
        # the reference's call sequence (norm + rope, then attention), smallest model, all layers, issued one by one
        dict(name="unfused-16q8kv-28x300-pos", kind="unfused", n_q=16, n_kv=8, layers=28, ctx=300, max_seq_len=4096, layout="pos",
             graph=False),
        # a serving loop: the step captured once with the position in device memory and replayed for every token
        dict(name="step-32q8kv-36x1100-graph", kind="step", n_q=32, n_kv=8, layers=36, ctx=1100, max_seq_len=4096, layout="head",
             graph=True),
        dict(name="step-64q8kv-64x5000-graph", kind="step", n_q=64, n_kv=8, layers=64, ctx=5000, max_seq_len=8192, layout="head",
             graph=True),
        # the attention of all 36 layers at 4096 cached positions in one call
        dict(name="stack-32q8kv-36x4096", kind="stack", n_q=32, n_kv=8, layers=36, ctx=4097, max_seq_len=4104, layout="head"),
        # the attention blocks of a step with their projections, issued call by call ...
        dict(name="block-32q8kv-36x700", kind="block", n_q=32, n_kv=8, layers=36, hidden=2560, ctx=700, max_seq_len=4096,
             layout="head", graph=False),
        # ... and replayed, for a part of the layers of the largest model (one stage of a pipeline)
        dict(name="block-64q8kv-8x3001-graph", kind="block", n_q=64, n_kv=8, layers=8, hidden=5120, ctx=3001, max_seq_len=4096,
             layout="head", graph=True),
        # the projection onto the vocabulary, fp32 logits
        dict(name="project-152000x2560-f32", kind="project", n=152000, k=2560, mode="f32"),
        # a prompt's caches (K and V, all layers) brought into the decode layout
        dict(name="restride-36x3777", kind="restride", n_kv=8, layers=36, ctx=3777, max_seq_len=4096),
    ]


MOST_BYTES = 2.0e9  # a drawn case reads and writes no more than this


def _log_int(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm; odd ones as likely as even ones."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _window(rng, ctx):
    """Positions a cache is sized for: the context window, a round number, or just what is needed."""
    return rng.choice([max(4096, -(-ctx // 4096) * 4096), -(-ctx // 1024) * 1024, ctx + rng.randrange(1, 40)])


def draw(rng):
    kind = rng.choice(["attend"] * 4 + ["unfused", "step", "step", "stack", "block", "block", "project", "restride"])
    n_q, n_kv, hidden = rng.choice(MODELS)
    layout = rng.choice(["head", "head", "pos"])
    if kind == "attend":
        if rng.random() < 0.4:
            n_q, n_kv = rng.choice(OTHER_HEADS)
        ctx = _log_int(rng, 16, 131072)
        return dict(kind=kind, n_q=n_q, n_kv=n_kv, ctx=ctx, max_seq_len=_window(rng, ctx), layout=layout)
    if kind in ("unfused", "step", "stack"):
        layers = _log_int(rng, 4, 64)
        ctx = _log_int(rng, 32, max(64, min(32768, int(MOST_BYTES / (layers * n_kv * 2 * HEAD_DIM * 2)))))
        case = dict(kind=kind, n_q=n_q, n_kv=n_kv, layers=layers, ctx=ctx, max_seq_len=_window(rng, ctx), layout=layout)
        return case if kind == "stack" else dict(case, graph=rng.random() < 0.5)
    if kind == "block":
        weights = ((n_q + 2 * n_kv) + n_q) * HEAD_DIM * hidden * 2
        layers = _log_int(rng, 2, min(36, int(0.75 * MOST_BYTES / weights)))
        ctx = _log_int(rng, 32, 4096)
        return dict(kind=kind, n_q=n_q, n_kv=n_kv, layers=layers, hidden=hidden, ctx=ctx, max_seq_len=_window(rng, ctx),
                    layout=layout, graph=rng.random() < 0.5)
    if kind == "project":
        k = 8 * _log_int(rng, 64, 1216)
        n = _log_int(rng, 500, min(152000, int(0.9 * MOST_BYTES / (2 * k))))
        return dict(kind=kind, n=n, k=k, mode=rng.choice(["bf16", "f32", "add"]))
    layers = _log_int(rng, 4, 64)
    ctx = _log_int(rng, 16, min(32768, int(MOST_BYTES / (layers * n_kv * 8 * HEAD_DIM))))
    return dict(kind=kind, n_kv=n_kv, layers=layers, ctx=ctx, max_seq_len=_window(rng, ctx))


class _Inputs:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.dev = torch.device("cuda")
        self.gen = torch.Generator(device=self.dev)
        self.gen.manual_seed(seed)

    def normal(self, *shape, scale=1.0, mean=0.0):
        x = torch.randn(shape, generator=self.gen, device=self.dev, dtype=BF16)
        if scale != 1.0:
            x.mul_(scale)
        return x.add_(mean) if mean else x

    def keys(self, *shape):
        """Key rows as QK-Norm leaves them: unit root mean square over a head's 128 values."""
        x = self.normal(*shape)
        for part in x:  # (a layer at a time: the float copies stay small)
            f = part.float()
            part.copy_(f * torch.rsqrt(f.square().mean(-1, keepdim=True)))
        return x

    def zeros(self, *shape, dtype=BF16):
        return torch.zeros(shape, device=self.dev, dtype=dtype)


def _caches(case, rnd, s, layers):
    n_kv, msl = case["n_kv"], case["max_seq_len"]
    shape = (layers, msl, n_kv, HEAD_DIM) if case["layout"] == "pos" else (layers, n_kv, msl, HEAD_DIM)
    s["kc"], s["vc"] = rnd.keys(*shape), rnd.normal(*shape)
    pos = case["ctx"] - 1  # the position the step is at: it attends to 0..pos
    s["rows"] = [c[:, pos] if case["layout"] == "pos" else c[:, :, pos] for c in (s["kc"], s["vc"])]
    s["ws"] = torch.empty(ops.workspace_bytes(case["n_q"], HEAD_DIM, msl) // 4, dtype=F32, device=rnd.dev)
    s["cache"] = dict(kv_dim=n_kv * HEAD_DIM, head_num=case["n_q"], head_dim=HEAD_DIM, max_seq_len=msl,
                      kv_layout=LAYOUTS[case["layout"]])
    s["attention"] = dict(s["cache"], kv_mul=case["n_q"] // n_kv, workspace_side=ops.workspace_side(s["ws"]))


def prepare(case, seed):
    rnd, kind = _Inputs(seed), case["kind"]
    s = {"kind": kind}
    if kind == "project":
        n, k = case["n"], case["k"]
        s["x"], s["w"] = rnd.normal(k), rnd.normal(n, k, scale=k ** -0.5)
        s["mode"] = {"bf16": B.GEMV_OUT_BF16, "f32": B.GEMV_OUT_F32, "add": B.GEMV_ADD_BF16}[case["mode"]]
        s["out"] = rnd.zeros(n, dtype=F32 if case["mode"] == "f32" else BF16)
        if case["mode"] == "add":
            s["residual"] = rnd.normal(n)
        return s
    if kind == "restride":
        shape = (case["layers"], case["max_seq_len"], case["n_kv"], HEAD_DIM)
        s["src"] = [rnd.normal(*shape), rnd.normal(*shape)]
        s["dst"] = [torch.zeros_like(c) for c in s["src"]]
        s["args"] = dict(layer_num=case["layers"], max_seq_len=case["max_seq_len"], kv_dim=case["n_kv"] * HEAD_DIM, head_dim=HEAD_DIM,
                         num_pos=case["ctx"])
        return s

    n_q, n_kv, pos = case["n_q"], case["n_kv"], case["ctx"] - 1
    dim, kv_dim = n_q * HEAD_DIM, n_kv * HEAD_DIM
    if kind == "attend":
        _caches(case, rnd, s, 1)
        s["q"], s["out"] = rnd.normal(dim), rnd.zeros(dim)
        s["attention"].update(layer_id=0, pos=pos)
        return s

    layers = case["layers"]
    _caches(case, rnd, s, layers)
    s["norm"] = rnd.normal(layers, 2 * HEAD_DIM, scale=0.02, mean=1.0)
    s["sin"], s["cos"] = ops.sincos_table(HEAD_DIM, case["max_seq_len"])
    s["out"] = rnd.zeros(layers, dim)
    s["q"], s["k"], s["v"] = rnd.normal(layers, dim), rnd.normal(layers, kv_dim), rnd.normal(layers, kv_dim)
    s["layers"] = range(layers)
    if kind == "block":
        hidden = case["hidden"]
        s["hidden"] = rnd.normal(layers, hidden)
        s["wqkv"] = rnd.normal(layers, dim + 2 * kv_dim, hidden, scale=hidden ** -0.5)
        s["wo"] = rnd.normal(layers, hidden, dim, scale=dim ** -0.5)
        s["token"], s["residual"] = rnd.normal(hidden), rnd.zeros(hidden)
    if kind == "unfused":
        s["q_rot"] = rnd.zeros(dim)
    if kind == "stack":
        s["attention"].update(layer_id=0, pos=pos, layer_count=layers, query_stride=dim, key_new_stride=kv_dim,
                              value_new_stride=kv_dim, norm_weight_stride=2 * HEAD_DIM, output_stride=dim)
        return s
    s["pos"] = pos
    if case["graph"]:
        if kind != "unfused":  # one captured step serves every token of the window
            s["attention"]["pos_device"] = torch.full((1,), pos, dtype=torch.int32, device=rnd.dev)
            s["pos"] = case["max_seq_len"] - 1
        _issue(s)
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            _issue(s)
    return s


def _issue(s):
    """The calls of one decode step, layer by layer."""
    pos, at, sin, cos, kc, vc, ws = s["pos"], s["attention"], s["sin"], s["cos"], s["kc"], s["vc"], s["ws"]
    q, k, v, norm, out = s["q"], s["k"], s["v"], s["norm"], s["out"]
    if s["kind"] == "step":
        for l in s["layers"]:
            ops.mha_decode_append(q[l], k[l], v[l], norm[l], sin, cos, kc, vc, out[l], ws, layer_id=l, pos=pos, **at)
    elif s["kind"] == "unfused":
        for l in s["layers"]:
            ops.qk_norm_rope_append(s["q_rot"], k[l], v[l], kc, vc, norm[l], sin, cos, layer_id=l, pos=pos, query_src=q[l],
                                    **s["cache"])
            ops.mha_decode(s["q_rot"], kc, vc, out[l], ws, layer_id=l, pos=pos, **at)
    else:
        s["residual"].copy_(s["token"])
        for l in s["layers"]:
            ops.qkv_gemv(s["hidden"][l], s["wqkv"][l], q[l], k[l], v[l])
            ops.mha_decode_append(q[l], k[l], v[l], norm[l], sin, cos, kc, vc, out[l], ws, layer_id=l, pos=pos,
                                  o_weight=s["wo"][l], residual=s["residual"], **at)


def run(s):
    kind = s["kind"]
    if kind == "attend":
        return ops.mha_decode(s["q"], s["kc"], s["vc"], s["out"], s["ws"], **s["attention"])
    if kind == "project":
        if "residual" in s:
            s["out"].copy_(s["residual"])
        return ops.gemv(s["x"], s["w"], s["out"], mode=s["mode"])
    if kind == "restride":
        return [ops.kv_restride(src, dst, **s["args"]) for src, dst in zip(s["src"], s["dst"])]
    if kind == "stack":
        ops.mha_decode_append_stack(s["q"], s["k"], s["v"], s["norm"], s["sin"], s["cos"], s["kc"], s["vc"], s["out"], s["ws"],
                                    **s["attention"])
    elif "graph" in s:
        s["graph"].replay()
    else:
        _issue(s)
    result = {"out": s["out"], "caches": [s["kc"], s["vc"]], "rows": s["rows"]}
    if kind == "block":
        result.update(residual=s["residual"], qkv=[s["q"], s["k"], s["v"]])
    return result


def work(case):
    kind = case["kind"]
    if kind == "project":
        n, k = case["n"], case["k"]
        out = {"bf16": 2, "f32": 4, "add": 4}[case["mode"]]
        return {"bytes": 2 * n * k + 2 * k + out * n, "flops": 2 * n * k}
    if kind == "restride":
        return {"bytes": 2 * 2 * case["layers"] * case["ctx"] * case["n_kv"] * HEAD_DIM * 2, "flops": 0}
    n_q, n_kv, layers = case["n_q"], case["n_kv"], case.get("layers", 1)
    row = n_kv * HEAD_DIM * 2
    head_bytes = 2 * n_q * HEAD_DIM * 2  # query in, output out
    flops = 4 * n_q * HEAD_DIM * case["ctx"]
    if kind == "attend":
        return {"bytes": 2 * case["ctx"] * row + head_bytes, "flops": flops}
    # the cached rows; the new rows in and out, the norm weights and the position's sines and cosines
    nbytes = 2 * (case["ctx"] - 1) * row + head_bytes + 4 * row + 4 * HEAD_DIM + 4 * HEAD_DIM
    if kind == "block":
        n = (n_q + 2 * n_kv) * HEAD_DIM
        nbytes += 2 * case["hidden"] * (n + n_q * HEAD_DIM) + 6 * case["hidden"]
        flops += 2 * case["hidden"] * (n + n_q * HEAD_DIM)
    return {"bytes": layers * nbytes, "flops": layers * flops}


def tolerance(case):
    """Four times what the paths differ by from the same steps in float64 with bf16 rounding where the results are bf16
    (measured over the listed and a dozen drawn cases: attention outputs rel 2.4e-4, max 7.7e-3 -- single values that round
    the other way --, the residual stream of 36 blocks rel 8.8e-4, max 8.2e-3, fp32 projections rel 7.7e-8, max 3.8e-7)."""
    kind = case["kind"]
    if kind == "restride":
        return "exact"
    if kind == "project" and case["mode"] == "f32":
        return {"rel": 3e-7, "max": 1.5e-6}
    return {"rel": 3.5e-3 if kind == "block" else 1e-3, "max": 3e-2}
