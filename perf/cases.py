"""What this package is timed and checked on: the work a training run, a
prompt and a decoding loop have it do, through its public entry points.

Paths (``case["path"]``):
  op_train       chunk_nested_gdn2 forward and backward, every gradient
  op_prefill     chunk_nested_gdn2 forward alone, output and final state
  decode         step_nested_gdn2, one token for a batch of sequences
  layer_train    NestedGDN2Attention forward and backward under bf16 autocast
  mlp_train      add_rms_norm and GatedMLP forward and backward, bf16 autocast
  loss_train     FusedLinearCrossEntropyLoss forward and backward, bf16 autocast
  model_prefill  NestedGDN2ForCausalLM on a prompt, logits, bf16 autocast

Sizes are those of the benchmark configurations, the model's defaults and the
tests; lists (firing intervals, queries per level) are texts, "1,4,16".
``exact`` restates each path in float64 with torch alone.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F
from torch.utils.checkpoint import checkpoint

import nested_recurrent_memory_amd as ngdn
from nested_recurrent_memory_amd import model as ngdn_model
from nested_recurrent_memory_amd import model_ops

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
EPS = 1e-5


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # the benchmark's training shape: long sequences, 16 heads of 128
        _op("op_train", "train_three_levels", B=4, T=8192, H=16, K=128, intervals="1,4,16",
            queries="64,64"),
        # the model's default heads: 16 of 64, two levels
        _op("op_train", "train_heads64", B=8, T=2048, H=16, K=64, intervals="1,4", queries="64"),
        # the four-level merge arm of the experiments on a ragged length, a state carried in
        # and out (truncated backpropagation)
        _op("op_train", "train_merge_ragged", B=2, T=3000, H=8, K=64, intervals="1,2,4,8",
            queries="16,32,64", promotion="merge", inputs="reftest", state=True),
        # fp32 training at the two-level configuration
        _op("op_train", "train_fp32", B=2, T=2048, H=8, K=128, intervals="1,4", queries="32",
            dtype="fp32"),
        # a very long document read once: 65536 tokens in one sequence
        _op("op_prefill", "prefill_long", B=1, T=65536, H=16, K=128, intervals="1,8,64",
            queries="64,64", g_scale=1.0, state=True),
        # a short prompt before decoding, odd length
        _op("op_prefill", "prefill_prompt", B=1, T=333, H=16, K=64, intervals="1,4", queries="64",
            state=True),
        # a serving batch, every sequence at its own position, the state updated in place
        dict(path="decode", name="decode_batch", B=256, H=16, K=128, intervals="1,4,16",
             queries="64,64", promotion="learned", dtype="bf16", inplace=True, rows=True),
        # one sequence being generated, as the layer's own decoding calls the step
        dict(path="decode", name="decode_one", B=1, H=16, K=64, intervals="1,4", queries="64",
             promotion="learned", dtype="bf16", inplace=False, rows=False),
        # one token-mixing layer of the 12-layer model in training
        dict(path="layer_train", name="layer_train", B=2, T=4096, hidden=1024, H=8, K=128,
             intervals="1,4,16", queries="64,64", promotion="learned", read_mix="softmax"),
        # the same model's channel mixing: residual add, norm, SwiGLU MLP
        dict(path="mlp_train", name="mlp_train", tokens=8192, hidden=1024, inner=4096),
        # its head: logits, cross entropy and their gradients
        dict(path="loss_train", name="loss_train", tokens=8192, hidden=1024, vocab=32000),
        # a whole call: a batch of prompts through a small stack to the logits
        dict(path="model_prefill", name="model_prefill", B=4, T=600, layers=2, hidden=1024, H=16,
             K=64, intervals="1,4", queries="64", inner=2816, vocab=32000),
    ]


def _op(path, name, *, B, T, H, K, intervals, queries, dtype="bf16", promotion="learned",
        inputs="baseline", g_scale=0.1, state=False):
    c = dict(path=path, B=B, T=T, H=H, K=K, intervals=intervals, queries=queries, dtype=dtype,
             promotion=promotion, inputs=inputs, g_scale=g_scale, state=state)
    return dict(c, name=name) if name else c


_LEVELS = [("1", ""), ("1,4", "64"), ("1,4", "32"), ("1,2,4", "16,32"), ("1,4,16", "64,64"),
           ("1,8,64", "64,64"), ("1,2,4,8", "16,32,64")]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    path = rng.choice(["op_train"] * 4 + ["op_prefill"] * 2 + ["decode"] * 2
                      + ["layer_train", "mlp_train", "loss_train", "model_prefill"])
    if path == "op_train":
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
        most = 4 * 8192 * 16 * 128 if dtype == "bf16" else 2 * 2048 * 8 * 128
        return _draw_op(rng, path, dtype, most, 8192)
    if path == "op_prefill":
        return _draw_op(rng, path, rng.choice(["bf16", "bf16", "bf16", "fp32"]),
                        65536 * 16 * 128 // 2, 65536)
    if path == "decode":
        levels, queries = rng.choice(_LEVELS)
        return dict(path=path, B=_log_int(rng, 1, 256), H=rng.choice([4, 8, 16]),
                    K=rng.choice([64, 128]), intervals=levels, queries=queries,
                    promotion=rng.choice(["learned", "learned", "merge"]),
                    dtype=rng.choice(["bf16", "bf16", "fp32"]), inplace=rng.random() < 0.5,
                    rows=rng.random() < 0.5)
    if path == "layer_train":
        levels, queries = rng.choice(_LEVELS)
        H, K = rng.choice([(16, 64), (8, 128), (8, 64), (4, 128)])
        T = _log_int(rng, 64, 4096)
        return dict(path=path, B=_log_int(rng, 1, max(1, min(16, 8192 // T))), T=T, hidden=H * K,
                    H=H, K=K, intervals=levels, queries=queries,
                    promotion=rng.choice(["learned", "learned", "merge"]),
                    read_mix=rng.choice(["softmax", "sigmoid"]))
    if path == "mlp_train":
        hidden = rng.choice([512, 1024, 2048])
        return dict(path=path, tokens=_log_int(rng, 100, 8192 * 1024 // hidden), hidden=hidden,
                    inner=rng.choice([2, 3, 4]) * hidden)
    if path == "loss_train":
        return dict(path=path, tokens=_log_int(rng, 64, 8192), hidden=rng.choice([512, 1024]),
                    vocab=rng.choice([8000, 16000, 32000]))
    levels, queries = rng.choice(_LEVELS[1:5])
    T = _log_int(rng, 64, 1200)
    return dict(path=path, B=_log_int(rng, 1, max(1, 2400 // T)), T=T, layers=rng.choice([1, 2]),
                hidden=1024, H=16, K=64, intervals=levels, queries=queries, inner=2816,
                vocab=32000)


def _draw_op(rng, path, dtype, most, longest):
    H, K = rng.choice([4, 8, 16]), rng.choice([64, 128])
    T = _log_int(rng, 64, min(longest, most // (H * K)))
    levels, queries = rng.choice(_LEVELS)
    return _op(path, None, B=_log_int(rng, 1, max(1, min(16, most // (T * H * K)))), T=T, H=H, K=K,
               intervals=levels, queries=queries, dtype=dtype,
               promotion=rng.choice(["learned", "learned", "merge"]),
               inputs=rng.choice(["baseline", "baseline", "reftest"]),
               g_scale=rng.choice([0.1, 0.5, 1.0]), state=rng.random() < 0.5)


# ------------------------------------------------------------------ inputs

def _ints(text):
    return tuple(int(x) for x in text.split(",") if x)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _promotion_params(r, L, H, K, n):
    s = K ** -0.5
    return dict(query_banks=r(L - 1, H, n, K) * s, key_projections=r(L - 1, H, K, K) * s,
                b_projections=r(L - 1, H, K, K) * s, w_projections=r(L - 1, H, K, K) * s,
                g_projections=r(L - 1, H, K, K) * s)


def _op_inputs(case, seed):
    """The op's tensor arguments (K = V), drawn on the GPU; ``baseline`` and
    ``reftest`` are the distributions of the benchmark and of the reference's
    op tests."""
    gen = _gen(seed)
    B, T, H, K = (case[x] for x in ("B", "T", "H", "K"))
    L = len(_ints(case["intervals"]))
    dt = DTYPES[case["dtype"]]
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV)  # noqa: E731
    u = lambda *s: torch.rand(*s, generator=gen, device=DEV)  # noqa: E731
    if case["inputs"] == "baseline":
        x = dict(q=F.normalize(r(B, T, H, L, K), dim=-1), k=F.normalize(r(B, T, H, K), dim=-1),
                 v=r(B, T, H, K), g=-F.softplus(r(B, T, H, K)) * case["g_scale"],
                 b=torch.sigmoid(r(B, T, H, K)), w=torch.sigmoid(r(B, T, H, K)))
    else:
        x = dict(q=r(B, T, H, L, K), k=F.normalize(r(B, T, H, K), dim=-1), v=r(B, T, H, K) * 0.5,
                 g=F.logsigmoid(r(B, T, H, K)), b=u(B, T, H, K), w=u(B, T, H, K))
    x["mix_weights"] = torch.softmax(r(B, T, H, L), dim=-1)
    x.update(_promotion_params(r, L, H, K, max(_ints(case["queries"]), default=1)))
    g = x.pop("g")
    x = {n: t.to(dt) for n, t in x.items()}
    x["g"] = g if case["inputs"] == "baseline" else g.to(dt)
    if case["state"]:
        x["initial_state"] = r(B, H, L, K, K) * 0.3
    return x, r(B, T, H, K).to(dt), r(B, H, L, K, K) * 0.1 if case["state"] else None


def _op_kw(case):
    f, nq = _ints(case["intervals"]), _ints(case["queries"])
    return dict(n_queries_per_level=nq, firing_intervals=f, L=len(f), promotion=case["promotion"])


def _decode_inputs(case, seed):
    B, H, K = (case[x] for x in ("B", "H", "K"))
    gen = _gen(seed)
    L = len(_ints(case["intervals"]))
    x, _, _ = _op_inputs(dict(case, T=1, inputs="baseline", g_scale=0.1, state=False), seed + 1000)
    x = {n: (t[:, 0].contiguous() if n in ("q", "k", "v", "g", "b", "w", "mix_weights") else t)
         for n, t in x.items()}
    x["state"] = torch.randn(B, H, L, K, K, generator=gen, device=DEV) * 0.3
    # sequences of a serving batch are at unrelated positions: one in 64 ends a chunk
    x["position"] = (torch.randint(0, 8192, (B,), generator=gen, device=DEV) if case["rows"]
                     else seed % 8192)
    return x


def _layer_params(case, seed):
    """A NestedGDN2Attention state dict: linear and convolution weights as the
    model initialises them, the rest as the layer does."""
    gen = _gen(seed + 2000)
    d, H, K = (case[x] for x in ("hidden", "H", "K"))
    L = len(_ints(case["intervals"]))
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV)  # noqa: E731
    u = lambda *s: torch.rand(*s, generator=gen, device=DEV)  # noqa: E731
    p = {n: r(*s) * 0.02 for n, s in {
        "q_proj.weight": (L * H * K, d), "k_proj.weight": (H * K, d), "v_proj.weight": (H * K, d),
        "f_proj.0.weight": (K, d), "f_proj.1.weight": (H * K, K), "b_proj.weight": (H * K, d),
        "w_proj.weight": (H * K, d), "mix_proj.weight": (H * L, d), "g_proj.0.weight": (K, d),
        "g_proj.1.weight": (H * K, K), "g_proj.1.bias": (H * K,), "o_proj.weight": (d, H * K)}.items()}
    for n, width in (("q", L * H * K), ("k", H * K), ("v", H * K)):
        p[f"{n}_conv1d.weight"] = (u(width, 1, 4) - 0.5)
    p["A_log"] = torch.log(1 + 15 * u(H))
    dt = torch.exp(u(H * K) * (math.log(0.1) - math.log(0.001)) + math.log(0.001))
    p["dt_bias"] = dt + torch.log(-torch.expm1(-dt))
    p["o_norm.weight"] = 1 + 0.1 * r(K)
    if L > 1:
        p.update(_promotion_params(r, L, H, K, max(_ints(case["queries"]))))
    return p


def _layer_cfg(case):
    f = _ints(case["intervals"])
    return dict(hidden_size=case["hidden"], num_heads=case["H"], head_dim=case["K"],
                num_levels=len(f), firing_intervals=f,
                n_queries_per_level=_ints(case["queries"]), promotion=case["promotion"],
                read_mix=case["read_mix"])


def _layer_io(case, seed):
    gen = _gen(seed)
    shape = (case["B"], case["T"], case["hidden"])
    # after the block's norm, in the dtype autocast has the norm write
    x = torch.randn(shape, generator=gen, device=DEV).bfloat16()
    return x, (torch.randn(shape, generator=gen, device=DEV) * 1e-3).bfloat16()


def _mlp_inputs(case, seed):
    gen = _gen(seed)
    n, d, m = (case[x] for x in ("tokens", "hidden", "inner"))
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV)  # noqa: E731
    x = dict(x=r(n, d), r=(r(n, d) * 0.5).bfloat16())
    p = {"norm": 1 + 0.1 * r(d), "gate_proj.weight": r(m, d) * 0.02,
         "up_proj.weight": r(m, d) * 0.02, "down_proj.weight": r(d, m) * 0.02}
    return x, p, r(n, d) * 1e-3, (r(n, d) * 1e-3).bfloat16()


def _loss_inputs(case, seed):
    gen = _gen(seed)
    n, d, v = (case[x] for x in ("tokens", "hidden", "vocab"))
    x = torch.randn(n, d, generator=gen, device=DEV)
    w = torch.randn(v, d, generator=gen, device=DEV) * 0.02
    y = torch.randint(0, v, (n,), generator=gen, device=DEV)
    y[:: 97] = -100            # sequence ends carry no target
    return x, w, y


def _model_params(case, seed):
    """The model's state dict by name."""
    gen = _gen(seed + 3000)
    d, m, v = (case[x] for x in ("hidden", "inner", "vocab"))
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV)  # noqa: E731
    p = {"model.embeddings.weight": r(v, d) * 0.02, "model.norm.weight": 1 + 0.1 * r(d),
         "lm_head.weight": r(v, d) * 0.02}
    for i in range(case["layers"]):
        at = f"model.layers.{i}."
        p[at + "attn_norm.weight"] = 1 + 0.1 * r(d)
        p[at + "mlp_norm.weight"] = 1 + 0.1 * r(d)
        for n, s in (("gate_proj", (m, d)), ("up_proj", (m, d)), ("down_proj", (d, m))):
            p[at + f"mlp.{n}.weight"] = r(*s) * 0.02
        lp = _layer_params(dict(case, promotion="learned"), seed + 10 * i)
        p.update({at + "attn." + n: t for n, t in lp.items()})
    return p


def _model_ids(case, seed):
    return torch.randint(0, case["vocab"], (case["B"], case["T"]), generator=_gen(seed), device=DEV)


def _build_model(case, params):
    cfg = ngdn_model.NestedGDN2Config(
        vocab_size=case["vocab"], num_hidden_layers=case["layers"],
        intermediate_size=case["inner"],
        **_layer_cfg(dict(case, promotion="learned", read_mix="softmax")))
    with torch.device(DEV):
        m = ngdn_model.NestedGDN2ForCausalLM(cfg)
    m.load_state_dict(params)
    return m.eval()


# ------------------------------------------------------------------ one pass

def prepare(case, seed):
    path = case["path"]
    if path in ("op_train", "op_prefill"):
        x, do, dfinal = _op_inputs(case, seed)
        if path == "op_train":
            x = {n: t.requires_grad_(True) for n, t in x.items()}
        return dict(path=path, x=x, do=do, dfinal=dfinal, kw=_op_kw(case), state=case["state"])
    if path == "decode":
        x, kw = _decode_inputs(case, seed), _op_kw(case)
        if case["inplace"] and kw["L"] > 1:    # a serving loop lays the parameters out once
            kw["params"] = ngdn.prepare_step_params(
                x["query_banks"], x["key_projections"], x["b_projections"], x["w_projections"],
                x["g_projections"], x["q"].dtype)
        return dict(path=path, x=x, kw=dict(kw, inplace=case["inplace"]))
    if path == "layer_train":
        with torch.device(DEV):
            layer = ngdn.NestedGDN2Attention(ngdn.NestedGDN2LayerConfig(**_layer_cfg(case)),
                                             layer_idx=0)
        p = _layer_params(case, seed)
        if case["promotion"] == "merge":       # the bank and key projections are buffers there
            p = {n: t for n, t in p.items() if n not in ("query_banks", "key_projections")}
        layer.load_state_dict(p)
        x, dy = _layer_io(case, seed)
        return dict(path=path, module=layer.train(), x=x.requires_grad_(True), dy=dy)
    if path == "mlp_train":
        x, p, dh, dy = _mlp_inputs(case, seed)
        with torch.device(DEV):
            mlp = model_ops.GatedMLP(case["hidden"], intermediate_size=case["inner"])
            norm = model_ops.RMSNorm(case["hidden"], eps=EPS)
        mlp.load_state_dict({n: t for n, t in p.items() if n != "norm"})
        norm.load_state_dict({"weight": p["norm"]})
        return dict(path=path, x={n: t.requires_grad_(True) for n, t in x.items()}, mlp=mlp,
                    norm=norm, dh=dh, dy=dy)
    if path == "loss_train":
        x, w, y = _loss_inputs(case, seed)
        return dict(path=path, x=x.requires_grad_(True), w=w.requires_grad_(True), y=y,
                    loss=model_ops.FusedLinearCrossEntropyLoss())
    return dict(path=path, model=_build_model(case, _model_params(case, seed)),
                ids=_model_ids(case, seed))


def run(s):
    path = s["path"]
    if path == "op_train":
        x = s["x"]
        for t in x.values():
            t.grad = None
        o, final = ngdn.chunk_nested_gdn2(**x, **s["kw"], output_final_state=s["state"])
        if s["state"]:
            torch.autograd.backward([o, final], [s["do"], s["dfinal"]])
        else:
            o.backward(s["do"])
        return {"o": o, "final": final, **{"d" + n: t.grad for n, t in x.items() if t.numel()}}
    if path == "op_prefill":
        with torch.no_grad():
            o, final = ngdn.chunk_nested_gdn2(**s["x"], **s["kw"], output_final_state=s["state"])
        return {"o": o, "final": final}
    if path == "decode":
        with torch.no_grad():
            o, state = ngdn.step_nested_gdn2(**s["x"], **s["kw"])
        return {"o": o, "state": state}
    if path == "layer_train":
        layer, x = s["module"], s["x"]
        layer.zero_grad(set_to_none=True)
        x.grad = None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y, _, _ = layer(x)
        y.backward(s["dy"])
        return {"y": y, "dx": x.grad, **{"d" + n: p.grad for n, p in layer.named_parameters()}}
    if path == "mlp_train":
        x, mlp, norm = s["x"], s["mlp"], s["norm"]
        mlp.zero_grad(set_to_none=True)
        norm.zero_grad(set_to_none=True)
        for t in x.values():
            t.grad = None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            h, y = model_ops.add_rms_norm(x["x"], x["r"], norm.weight, norm.eps, torch.bfloat16)
            y = mlp(y)
        torch.autograd.backward([h, y], [s["dh"], s["dy"]])
        return {"h": h, "y": y, **{"d" + n: t.grad for n, t in x.items()},
                "dnorm": norm.weight.grad, **{"d" + n: p.grad for n, p in mlp.named_parameters()}}
    if path == "loss_train":
        x, w = s["x"], s["w"]
        x.grad = w.grad = None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            loss = s["loss"](x, s["y"], w)
        loss.backward()
        return {"loss": loss, "dx": x.grad, "dw": w.grad}
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        out = s["model"](input_ids=s["ids"], use_cache=True)
    states = [out.past_key_values[i]["recurrent_state"][0] for i in sorted(out.past_key_values)]
    return {"logits": out.logits, "states": states}


# ------------------------------------------------------------------ what a pass cannot do without

def _op_work(case, train):
    """Inputs, parameters and outputs once (and for training the output
    gradient, the inputs again and every gradient); the flops of the chunk
    form's dense products at 64 tokens a chunk."""
    B, T, H, K = (case[x] for x in ("B", "T", "H", "K"))
    f, nq = _ints(case["intervals"]), _ints(case["queries"])
    L, es, C = len(f), 2 if case.get("dtype", "bf16") == "bf16" else 4, 64
    NT, tok, kv = -(-T // C), B * T * H, K * K * 4
    gs = 4 if case.get("inputs", "baseline") == "baseline" else es
    n_par = sum((0 if case["promotion"] == "merge" else nq[l - 1] * K + K * K) + 3 * K * K
                for l in range(1, L))
    ins = tok * ((L + 4) * K * es + K * gs + L * es) + H * n_par * es
    st = B * H * L * kv if case.get("state") else 0
    fwd = ins + tok * K * es + 2 * st
    units = B * H * NT
    pairs = sum(B * H * (NT // f[l]) * (K if case["promotion"] == "merge" else nq[l - 1])
                for l in range(1, L))
    fl_f = units * (2 * C * C * 5 * K + 6 * C * K * K) + tok * (L - 1) * 2 * K * K + pairs * 14 * K * K
    fl_b = units * (2 * C * C * 10 * K + 12 * C * K * K) + tok * (L - 1) * 4 * K * K + pairs * 28 * K * K
    if not train:
        return fwd, fl_f
    return fwd + 2 * ins + tok * K * es + 2 * st, fl_f + fl_b


def work(case):
    path = case["path"]
    if path in ("op_train", "op_prefill"):
        b, f = _op_work(case, path == "op_train")
        return {"bytes": b, "flops": f}
    if path == "decode":
        B, H, K = (case[x] for x in ("B", "H", "K"))
        L, es = len(_ints(case["intervals"])), 2 if case["dtype"] == "bf16" else 4
        kv = K * K * 4
        # every level read; level 0 written in place, every level out of place
        return {"bytes": B * H * ((L + (1 if case["inplace"] else L)) * kv
                                  + ((L + 5) * K + L) * es + K * 4),
                "flops": B * H * (L + 2) * 2 * K * K}
    if path == "layer_train":
        B, T, d, H, K = (case[x] for x in ("B", "T", "hidden", "H", "K"))
        L, n = len(_ints(case["intervals"])), B * T
        lin = d * H * K * (L + 5) + 2 * K * (d + H * K) + d * H * L
        _, f = _op_work(case, True)
        # x and dy in, y and dx out, weights in and their gradients out (fp32)
        return {"bytes": 4 * n * d * 2 + 2 * lin * 4, "flops": f + 6 * n * lin}
    if path == "mlp_train":
        n, d, m = (case[x] for x in ("tokens", "hidden", "inner"))
        return {"bytes": n * d * (4 * 4 + 4 * 2) + 2 * 3 * d * m * 4, "flops": 6 * n * 3 * d * m}
    if path == "loss_train":
        n, d, v = (case[x] for x in ("tokens", "hidden", "vocab"))
        return {"bytes": 2 * n * d * 4 + 2 * v * d * 4 + n * 8, "flops": 6 * n * d * v}
    B, T, d, H, K, m, v = (case[x] for x in ("B", "T", "hidden", "H", "K", "inner", "vocab"))
    L, n = len(_ints(case["intervals"])), B * T
    lin = d * H * K * (L + 5) + 2 * K * (d + H * K) + d * H * L + 3 * d * m
    _, f = _op_work(dict(case, promotion="learned"), False)
    return {"bytes": n * v * 2 + v * d * 4 + case["layers"] * lin * 4 + n * (8 + d * 4),
            "flops": case["layers"] * (f + 2 * n * lin) + 2 * n * d * v}


def tolerance(case):
    """About four times the error against ``exact``: results rounded to bf16
    are 1.7e-3 off by that rounding alone, fp32 ones up to 1.1e-6; through
    the bf16 GEMMs of a layer gradients are 1.1e-2 off, of the MLP 5e-3, of
    the loss 3.5e-3, and the logits of two layers 1.6e-2."""
    path = case["path"]
    if path in ("op_train", "op_prefill", "decode"):
        return {"rel": 7e-3} if case["dtype"] == "bf16" else {"rel": 5e-6}
    return {"rel": {"layer_train": 4e-2, "mlp_train": 2e-2, "loss_train": 1.5e-2,
                    "model_prefill": 6e-2}[path]}


# ------------------------------------------------------------------ the same in float64

def _firing(S_below, S, i, P, n, merge):
    """One firing of level i + 1: probe the level below, write the pairs."""
    K = S.shape[-2]
    if merge:
        vals, keys = S_below, torch.eye(K, device=S.device, dtype=S.dtype)
    else:
        vals = P["query_banks"][i][:, :n] @ S_below
        u = vals @ P["key_projections"][i].transpose(-1, -2)
        keys = u / u.norm(dim=-1, keepdim=True).clamp_min(1e-12)
    b = torch.sigmoid(vals @ P["b_projections"][i] - 4.0)
    w = torch.sigmoid(vals @ P["w_projections"][i])
    g = -F.softplus(vals @ P["g_projections"][i] - 4.0).mean(-2)
    Sd = g.exp().unsqueeze(-1) * S
    return Sd + keys.transpose(-1, -2) @ (vals * w - (keys * b) @ Sd)


def _op64(x, kw, initial_state=None, fire_partial=True):
    """The chunk form in float64: x by argument name, [B,T,H,...]."""
    L, f, nq, merge = (kw["L"], kw["firing_intervals"], kw["n_queries_per_level"],
                       kw["promotion"] == "merge")
    B, T, H, K = x["k"].shape
    C, scale = 64, K ** -0.5
    NT = -(-T // C)
    NF = NT if fire_partial else T // C

    def chunks(t):
        t = t.transpose(1, 2)
        t = F.pad(t, (0, 0) * (t.dim() - 3) + (0, NT * C - T))
        return t.reshape(B, H, NT, C, *t.shape[3:]).unbind(2)

    rows = [chunks(x[n]) for n in ("q", "k", "v", "g", "b", "w", "mix_weights")]
    i = torch.arange(C, device=x["k"].device)
    strict = (i[:, None] > i).to(torch.float64)
    causal = (i[:, None] >= i).to(torch.float64)
    eye = torch.eye(C, device=x["k"].device, dtype=torch.float64)

    def chunk(q, k, v, g, b, w, mix, *S):
        S = list(S)
        gc = g.cumsum(-2)
        dec = (gc.unsqueeze(-2) - gc.unsqueeze(-3)).clamp(max=0.0).exp() * k.unsqueeze(-3)
        A = (dec @ (b * k).unsqueeze(-1)).squeeze(-1) * strict
        Aqk = (dec @ (q[..., 0, :] * scale).unsqueeze(-1)).squeeze(-1) * causal
        inv, P = eye - A, A @ A                   # (I + A)^-1: A is nilpotent
        for _ in range(5):
            inv, P = inv + inv @ P, P @ P
        vn = inv @ (w * v) - (inv @ (b * k * gc.exp())) @ S[0]
        reads = [Aqk @ vn + (scale * q[..., 0, :] * gc.exp()) @ S[0]]
        reads += [(scale * q[..., l, :]) @ S[l] for l in range(1, L)]
        o = sum(mix[..., l:l + 1] * reads[l] for l in range(L))
        last = gc[..., -1:, :]
        S[0] = last.transpose(-1, -2).exp() * S[0] + (k * (last - gc).exp()).transpose(-1, -2) @ vn
        return (o, S[0])

    def fire(l, below, S):
        return _firing(below, S, l - 1, x, nq[l - 1], merge)

    S = [initial_state[:, :, l] if initial_state is not None
         else torch.zeros(B, H, K, K, device=x["k"].device, dtype=torch.float64) for l in range(L)]
    grad = torch.is_grad_enabled()
    once = (lambda fn, *a: checkpoint(fn, *a, use_reentrant=False)) if grad else (lambda fn, *a: fn(*a))
    outs = []
    for n in range(NT):
        o, S[0] = once(chunk, *(r[n] for r in rows), *S)
        outs.append(o)
        for l in range(1, L):
            if (n + 1) % f[l] == 0 and n < NF:
                S[l] = once(fire, l, S[l - 1], S[l])
    o = torch.stack(outs, 2).reshape(B, H, NT * C, K)[:, :, :T].transpose(1, 2)
    return o, torch.stack(S, 2)


def _step64(x, kw):
    L, K = kw["L"], x["k"].shape[-1]
    S = list(x["state"].unbind(2))
    k, Sd = x["k"].unsqueeze(-1), x["g"].exp().unsqueeze(-1) * S[0]
    pred = ((x["k"] * x["b"]).unsqueeze(-2) @ Sd)
    S[0] = Sd + k @ ((x["v"] * x["w"]).unsqueeze(-2) - pred)
    o = sum(x["mix_weights"][..., l:l + 1] * K ** -0.5 * (x["q"][:, :, l].unsqueeze(-2) @ S[l]).squeeze(-2)
            for l in range(L))
    pos = x["position"]
    end = (pos if torch.is_tensor(pos) else torch.full((k.shape[0],), pos, device=k.device)) + 1
    for l in range(1, L):
        rows = torch.nonzero(end % (64 * kw["firing_intervals"][l]) == 0).flatten()
        if rows.numel():
            new = _firing(S[l - 1][rows], S[l][rows], l - 1, x, kw["n_queries_per_level"][l - 1],
                          kw["promotion"] == "merge")
            S[l] = S[l].index_copy(0, rows, new)
    return o, torch.stack(S, 2)


def _conv64(x, w):
    W = w.shape[-1]
    return F.silu(sum(w[:, 0, i] * F.pad(x, (0, 0, W - 1 - i, 0))[:, :x.shape[1]] for i in range(W)))


def _layer64(p, x, case):
    B, T, _ = x.shape
    H, K = case["H"], case["K"]
    f = _ints(case["intervals"])
    L = len(f)
    lin = lambda n, t: t @ p[n + ".weight"].t()  # noqa: E731
    q, k, v = (_conv64(lin(n + "_proj", x), p[n + "_conv1d.weight"]) for n in "qkv")
    heads = lambda t: t.reshape(B, T, H, -1)  # noqa: E731
    q = F.normalize(q.reshape(B, T, L, H, K).transpose(2, 3), dim=-1)
    dec = F.softplus(lin("f_proj.1", lin("f_proj.0", x)) + p["dt_bias"])
    ml = heads(lin("mix_proj", x))
    a = dict(q=q, k=F.normalize(heads(k), dim=-1), v=heads(v),
             g=-p["A_log"].exp().unsqueeze(-1) * heads(dec), b=torch.sigmoid(heads(lin("b_proj", x))),
             w=torch.sigmoid(heads(lin("w_proj", x))),
             mix_weights=ml.softmax(-1) if case["read_mix"] == "softmax" else torch.sigmoid(ml))
    if L > 1:
        a.update({n: p[n] for n in ("query_banks", "key_projections", "b_projections",
                                    "w_projections", "g_projections")})
    o, final = _op64(a, _op_kw(case), fire_partial=False)
    gate = heads(lin("g_proj.1", lin("g_proj.0", x)) + p["g_proj.1.bias"])
    o = _norm64(o, p["o_norm.weight"]) * torch.sigmoid(gate)
    return lin("o_proj", o.reshape(B, T, H * K)), final


def _norm64(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w


def _mlp64(p, y):
    return (F.silu(y @ p["gate_proj.weight"].t()) * (y @ p["up_proj.weight"].t())) @ p["down_proj.weight"].t()


def _wide(d, grad):
    return {n: t.detach().double().requires_grad_(grad) if torch.is_tensor(t) and t.is_floating_point()
            else t for n, t in d.items()}


def exact(case, seed):
    path = case["path"]
    if path in ("op_train", "op_prefill"):
        x, do, dfinal = _op_inputs(case, seed)
        train = path == "op_train"
        x = _wide(x, train)
        with torch.set_grad_enabled(train):
            o, final = _op64(x, _op_kw(case), x.get("initial_state"))
        out = {"o": o, "final": final if case["state"] else None}
        if train:
            torch.autograd.backward([o] + ([final] if case["state"] else []),
                                    [do.double()] + ([dfinal.double()] if case["state"] else []))
            # a parameter that the promotion does not read has a zero gradient, one level has none
            out.update({"d" + n: t.grad if t.grad is not None else torch.zeros_like(t)
                        for n, t in x.items() if t.numel()})
        return out
    if path == "decode":
        with torch.no_grad():
            o, state = _step64(_wide(_decode_inputs(case, seed), False), _op_kw(case))
        return {"o": o, "state": state}
    if path == "layer_train":
        p = _wide(_layer_params(case, seed), True)
        x, dy = _layer_io(case, seed)
        x = x.double().requires_grad_(True)
        y, _ = _layer64(p, x, case)
        y.backward(dy.double())
        if case["promotion"] == "merge":
            p = {n: t for n, t in p.items() if n not in ("query_banks", "key_projections")}
        return {"y": y, "dx": x.grad, **{"d" + n: t.grad if t.grad is not None else torch.zeros_like(t)
                                         for n, t in p.items()}}
    if path == "mlp_train":
        x, p, dh, dy = _mlp_inputs(case, seed)
        x, p = _wide(x, True), _wide(p, True)
        h = x["x"] + x["r"]
        y = _mlp64(p, _norm64(h, p["norm"]))
        torch.autograd.backward([h, y], [dh.double(), dy.double()])
        return {"h": h, "y": y, **{"d" + n: t.grad for n, t in {**x, **p}.items()}}
    if path == "loss_train":
        x, w, y = _loss_inputs(case, seed)
        x, w = x.double().requires_grad_(True), w.double().requires_grad_(True)
        loss = F.cross_entropy(x @ w.t(), y, ignore_index=-100)
        loss.backward()
        return {"loss": loss, "dx": x.grad, "dw": w.grad}
    p = _wide(_model_params(case, seed), False)
    c = dict(case, promotion="learned", read_mix="softmax")
    states = []
    with torch.no_grad():
        h = p["model.embeddings.weight"][_model_ids(case, seed)]
        for i in range(case["layers"]):
            at = f"model.layers.{i}."
            part = lambda s: {n[len(at + s):]: t for n, t in p.items() if n.startswith(at + s)}  # noqa: E731
            y, final = _layer64(part("attn."), _norm64(h, p[at + "attn_norm.weight"]), c)
            states.append(final)
            h = h + y
            h = h + _mlp64(part("mlp."), _norm64(h, p[at + "mlp_norm.weight"]))
        return {"logits": _norm64(h, p["model.norm.weight"]) @ p["lm_head.weight"].t(), "states": states}
