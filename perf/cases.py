"""The work a user of this framework has it do, as cases that can be timed and
checked: Q4_0 linears from one decode row to a prefill chunk, the LM head with
greedy sampling, split-KV decode attention for one and for several sequences,
the per-layer decode seam, whole decode steps of the 4B model on the step
runner, and the element-wise ops around a prefill chunk.

  listed()              the cases, dicts of plain values
  draw(rng)             one more case of the same ranges
  prepare(case, seed)   inputs, weights and handles on the GPU, from the seed
  run(state)            one pass through the public entry points
  work(case)            bytes and flops that the pass cannot do without
  tolerance(case)       how far another correct implementation may be
  exact(case, seed)     the outputs in 64 bits, in plain torch

Shapes are the 4B decoder's (hidden 2560, 32 q / 8 kv heads of 128,
intermediate 9728, vocab 151936, BF16 paged KV of 128-token blocks), the
contexts those of the benchmark (2048..6144 for one sequence, 512..32768 for
several), and generic odd sizes.
"""
from __future__ import annotations

import importlib
import itertools
import math
import os

import torch

os.environ.setdefault("SMX_ALLOW_UNVALIDATED", "1")  # the library as built is what is measured

import __graft_entry__  # noqa: E402

PKG = __graft_entry__.load_package().__name__


def _mod(name: str):
    return importlib.import_module(f"{PKG}.{name}")


BF16 = torch.bfloat16
HIDDEN, N_Q, N_KV, HD, INTER, VOCAB = 2560, 32, 8, 128, 9728, 151936
QKV_ROWS = (N_Q + 2 * N_KV) * HD
BLOCK = 128
EPS, THETA = 1e-6, 1e6
SCALE = 1.0 / math.sqrt(HD)
CAP_1SEQ = 6272  # 49 pages: the benchmark's block table for one sequence
MODEL_STEPS = 8


# --------------------------------------------------------------------- cases
def listed() -> list[dict]:
    return [
        # one decode row through a linear's quant method: the smallest call, latency
        dict(name="linear_1row", kind="linear", m=1, n=9728, k=2560, packed=False, bias=False),
        # eight sequences' rows through a linear packed for batched decode (down projection)
        dict(name="linear_8rows_packed", kind="linear", m=8, n=2560, k=9728, packed=True,
             bias=False),
        # a few rows of a linear whose sizes are multiples of nothing but Q4_0's 32, with bias
        dict(name="linear_odd", kind="linear", m=5, n=4001, k=2592, packed=False, bias=True),
        # a short prompt, or the verification of drafted tokens
        dict(name="linear_48rows", kind="linear", m=48, n=6144, k=2560, packed=False, bias=False),
        # a prompt of odd length
        dict(name="linear_193rows", kind="linear", m=193, n=9728, k=2560, packed=False,
             bias=False),
        # a prefill chunk through the widest linear of the model (gate|up)
        dict(name="linear_2048rows", kind="linear", m=2048, n=19456, k=2560, packed=False,
             bias=False),
        # one token's logits and its greedy id
        dict(name="head_1row", kind="head", rows=1, vocab=VOCAB, hidden=HIDDEN),
        # the attention backend for one sequence at the benchmark's longest context
        dict(name="attn_1seq", kind="attn", seqs=1, lo=6144, hi=6144, planned=False),
        # eight ragged sequences, one split plan per step
        dict(name="attn_8seq", kind="attn", seqs=8, lo=512, hi=32768, planned=True),
        # the per-layer decode seam for a batch of chat-length sequences
        dict(name="layer_16seq", kind="layer", seqs=16, lo=200, hi=4000),
        # decode of the 4B model at its mean context, teacher-forced, on the step runner
        dict(name="model_1seq", kind="model", layers=36, context=4096, vocab=VOCAB),
        # the element-wise ops around a prefill chunk
        dict(name="prefill_ops", kind="prefill_ops", tokens=2047, act="swiglu"),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["linear", "linear", "linear", "linear", "head", "attn", "attn", "layer",
                       "model", "prefill_ops"])
    if kind == "linear":
        m = _log_int(rng, 1, 2048)
        if rng.random() < 0.5:
            n, k = rng.choice([(QKV_ROWS, HIDDEN), (HIDDEN, N_Q * HD), (2 * INTER, HIDDEN),
                               (HIDDEN, INTER), (INTER, HIDDEN)])
        else:
            n, k = _log_int(rng, 256, 19456), 32 * _log_int(rng, 16, 304)
            while m * n * k > 2048 * 2 * INTER * HIDDEN:
                m = max(1, m // 2)
        return dict(kind=kind, m=m, n=n, k=k, packed=rng.random() < 0.5,
                    bias=rng.random() < 0.3)
    if kind == "head":
        return dict(kind=kind, rows=_log_int(rng, 1, 16), vocab=_log_int(rng, 8000, VOCAB),
                    hidden=256 * _log_int(rng, 2, 10))
    if kind == "attn":
        if rng.random() < 0.5:
            ctx = _log_int(rng, 16, 8192)
            return dict(kind=kind, seqs=1, lo=ctx, hi=ctx, planned=False)
        seqs = _log_int(rng, 2, 32)
        hi = _log_int(rng, 256, min(32768, 262144 // seqs))
        return dict(kind=kind, seqs=seqs, lo=max(1, hi // 64), hi=hi,
                    planned=rng.random() < 0.75)
    if kind == "layer":
        seqs = _log_int(rng, 1, 16)
        hi = _log_int(rng, 64, 8192)
        return dict(kind=kind, seqs=seqs, lo=max(1, hi // 16), hi=hi)
    if kind == "model":
        return dict(kind=kind, layers=_log_int(rng, 1, 12), context=_log_int(rng, 32, 6000),
                    vocab=_log_int(rng, 8000, VOCAB))
    return dict(kind=kind, tokens=_log_int(rng, 17, 4096), act=rng.choice(["swiglu", "gelu"]))


# -------------------------------------------------------------------- inputs
def _gen(seed: int, *salt: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    s = int(seed) & 0x7FFFFFFF
    for x in salt:
        s = (s * 1000003 + 12345 + int(x)) & 0x7FFFFFFFFFFF
    g.manual_seed(s)
    return g


def _randn(g: torch.Generator, *shape: int) -> torch.Tensor:
    return torch.randn(shape, generator=g, device="cuda").to(BF16)


def _blocks(g: torch.Generator, n: int, k: int) -> torch.Tensor:
    """Random GGUF Q4_0 rows uint8 [n, k/32*18]: d = fp16(0.02 |N(0, 1)|),
    uniform codes (the single-GEMV workload's weights)."""
    out = torch.randint(0, 256, (n, k // 32, 18), generator=g, device="cuda", dtype=torch.uint8)
    d = (torch.randn((n, k // 32), generator=g, device="cuda").abs_() * 0.02).half()
    out[:, :, :2] = d.view(torch.uint8).view(n, k // 32, 2)
    return out.view(n, k // 32 * 18)


def _norm(g: torch.Generator, n: int) -> torch.Tensor:
    return (1.0 + 0.1 * torch.randn(n, generator=g, device="cuda")).to(BF16)


def _dequant64(blocks: torch.Tensor, k: int) -> torch.Tensor:
    n = blocks.shape[0]
    b = blocks.view(n, k // 32, 18)
    d = b[:, :, :2].contiguous().view(torch.float16).to(torch.float64)  # [n, k/32, 1]
    q = torch.cat((b[:, :, 2:] & 15, b[:, :, 2:] >> 4), dim=-1).to(torch.float64) - 8.0
    return (d * q).view(n, k)


def _lengths(case: dict) -> list[int]:
    """Ragged context lengths of a case: lo..hi, the same for every seed (a
    seed's inputs must not change how much work a pass is)."""
    s, lo, hi = case["seqs"], case["lo"], case["hi"]
    if s == 1:
        return [hi]
    return [lo + (hi - lo) * ((7 * i + 3) % s) // (s - 1) for i in range(s)]


def _pages(g: torch.Generator, seqs: int, per_seq: int) -> torch.Tensor:
    """Shuffled physical pages, int32 [seqs, per_seq]."""
    return torch.randperm(seqs * per_seq, generator=g, device="cuda").to(torch.int32).view(
        seqs, per_seq)


def _slots(table: torch.Tensor, pos: torch.Tensor) -> torch.Tensor:
    rows = torch.arange(pos.numel(), device="cuda")
    return table[rows, pos // BLOCK].to(torch.int64) * BLOCK + pos % BLOCK


def _layer_weights(seed: int, i: int) -> dict:
    w = {}
    for j, (name, n, k) in enumerate((("qkv", QKV_ROWS, HIDDEN), ("o_proj", HIDDEN, N_Q * HD),
                                      ("gate_up", 2 * INTER, HIDDEN), ("down", HIDDEN, INTER))):
        w[f"layers.{i}.{name}"] = _blocks(_gen(seed, 1, i, j), n, k)
    for j, n in enumerate((HIDDEN, HIDDEN, HD, HD)):
        w[f"layers.{i}.norm{j}"] = _norm(_gen(seed, 2, i, j), n)
    return w


_unique = itertools.count()


def prepare(case: dict, seed: int) -> dict:
    return _PREPARE[case["kind"]](case, seed)


def run(state: dict):
    return state["run"](state)


def _prep_linear(case, seed):
    lin = _mod("integration.linear")
    m, n, k = case["m"], case["n"], case["k"]
    layer = lin.Q4_0Linear(k, [n], device="cuda")
    layer.quant_method = lin.Q4_0Config(
        pack_for_batch=case["packed"]).get_quant_method(layer)
    layer.qweight.data.copy_(_blocks(_gen(seed, 1), n, k))
    layer.quant_method.process_weights_after_loading(layer)
    bias = _randn(_gen(seed, 3), n) if case["bias"] else None
    return dict(run=_run_linear, layer=layer, x=_randn(_gen(seed, 2), m, k), bias=bias)


def _run_linear(s):
    return s["layer"].quant_method.apply(s["layer"], s["x"], bias=s["bias"])


def _prep_head(case, seed):
    head = _mod("integration.head").TiedQ4_0Head(
        _blocks(_gen(seed, 1), case["vocab"], case["hidden"]), case["vocab"], case["hidden"])
    return dict(run=_run_head, head=head, x=_randn(_gen(seed, 2), case["rows"], case["hidden"]),
                sample=_mod("integration.head").greedy_sample)


def _run_head(s):
    logits = s["head"].logits(s["x"])
    return logits, s["sample"](logits)


def _attn_inputs(case, seed):
    S = case["seqs"]
    L = torch.tensor(_lengths(case), dtype=torch.int64, device="cuda")
    hi = case["hi"]
    per_seq = -(-max(hi, CAP_1SEQ if S == 1 else 1) // BLOCK)
    table = _pages(_gen(seed, 1), S, per_seq)
    kv = torch.empty((2, S * per_seq, BLOCK, N_KV, HD), dtype=BF16, device="cuda")
    kv.normal_(0.0, 1.0, generator=_gen(seed, 2))
    g = _gen(seed, 3)
    q, k, v = _randn(g, S, N_Q * HD), _randn(g, S, N_KV * HD), _randn(g, S, N_KV * HD)
    return L, per_seq, table, kv, q, k, v


def _prep_attn(case, seed):
    att = _mod("integration.attention")
    S = case["seqs"]
    L, per_seq, table, kv, q, k, v = _attn_inputs(case, seed)
    md = att.SplitKVDecodeMetadata(block_tables=table, seq_lens=L.to(torch.int32),
                                   slot_mapping=_slots(table, L - 1), num_splits=1)
    if case["planned"]:
        md.num_items, md.num_splits = att.choose_plan(S, N_KV)
    else:
        md.num_splits = att.choose_num_splits(per_seq * BLOCK, num_seqs=S)
    impl = att.SplitKVDecodeImpl(N_Q, HD, SCALE, N_KV)
    return dict(run=_run_attn, impl=impl, md=md, kv=kv, q=q, k=k, v=v, planned=case["planned"],
                backend=att.SplitKVDecodeBackend)


def _run_attn(s):
    if s["planned"]:  # once per decode step
        s["backend"].plan(s["md"], BLOCK, N_Q, HD)
    out = s["impl"].forward(None, s["q"], s["k"], s["v"], s["kv"], s["md"])
    return out, s["kv"]


def _prep_layer(case, seed):
    att, model, lr = (_mod("integration.attention"), _mod("integration.model"),
                      _mod("integration.layer_run"))
    S = case["seqs"]
    L = torch.tensor(_lengths(case), dtype=torch.int64, device="cuda")
    max_len = -(-(case["hi"] + 1) // BLOCK) * BLOCK
    cfg = model.DecoderConfig(n_layers=1, vocab=1024)
    w = _layer_weights(seed, 0)
    w["final_norm"] = _norm(_gen(seed, 4), HIDDEN)
    m = model.DecodeModel(cfg, "cuda", max_len=max_len, weights=w, batch=S)
    m.layers[0].name = f"perf.{next(_unique)}.attn"
    m.layers[0].kv_cache.normal_(0.0, 1.0, generator=_gen(seed, 5))
    lr.install(m)
    _mod("integration.custom_ops").register()
    table = m.state.block_table
    md = att.SplitKVDecodeMetadata(block_tables=table, seq_lens=L.to(torch.int32),
                                   slot_mapping=_slots(table, L - 1),
                                   num_splits=m.num_splits, num_items=m.num_items)
    g = _gen(seed, 6)
    return dict(run=_run_layer, model=m, md=md, positions=L - 1, x=_randn(g, S, HIDDEN),
                residual=_randn(g, S, HIDDEN), lr=lr, backend=att.SplitKVDecodeBackend)


def _run_layer(s):
    md = s["md"]
    if md.num_items:  # once per decode step
        s["backend"].plan(md, BLOCK, N_Q, HD, positions=s["positions"])
    s["lr"].set_attention_metadata(md)
    L = s["model"].layers[0]
    y, r = torch.ops.smx.layer_run(s["x"], s["residual"], s["positions"], L.name)
    return y, r, L.kv_cache


def _model_tokens(case, seed):
    g = _gen(seed, 7)
    return torch.randint(0, case["vocab"], (MODEL_STEPS,), generator=g, device="cuda")


def _model_weights(case, seed):
    w = {}
    for i in range(case["layers"]):
        w.update(_layer_weights(seed, i))
    w["final_norm"] = _norm(_gen(seed, 4), HIDDEN)
    w["head"] = _blocks(_gen(seed, 8), case["vocab"], HIDDEN)
    return w


def _prep_model(case, seed):
    model = _mod("integration.model")
    cfg = model.DecoderConfig(n_layers=case["layers"], vocab=case["vocab"])
    m = model.DecodeModel(cfg, "cuda", max_len=CAP_1SEQ, weights=_model_weights(case, seed))
    m.fill_kv(int(seed) + 1)
    m.record_runner()
    toks = _model_tokens(case, seed)
    c = case["context"]
    # the given tokens at their positions, as a prompt's are fed
    forced = torch.zeros_like(m.state.forced)
    forced[0, c:c + MODEL_STEPS] = toks
    m.state.forced.copy_(forced)
    flen = torch.tensor([c + MODEL_STEPS], dtype=torch.int32, device="cuda")
    return dict(run=_run_model, model=m, context=c, first=toks[:1].cpu(), flen=flen)


def _run_model(s):
    m = s["model"]
    m.set_context([s["context"]], ids=s["first"])
    m.state.forced_len.copy_(s["flen"])
    m.run_steps(MODEL_STEPS, fences="acquire")
    return [m.logits] + [L.kv_cache for L in m.layers]


def _prefill_inputs(case, seed):
    T = case["tokens"]
    g = _gen(seed, 1)
    per_seq = -(-T // BLOCK)
    return dict(
        table=_randn(g, 32000, HIDDEN),
        ids=torch.randint(0, 32000, (T,), generator=g, device="cuda"),
        residual=_randn(g, T, HIDDEN), gamma=_norm(g, HIDDEN), qkv=_randn(g, T, QKV_ROWS),
        q_gamma=_norm(g, HD), k_gamma=_norm(g, HD), gate_up=_randn(g, T, 2 * INTER),
        block_table=_pages(g, 1, per_seq), pos=torch.arange(T, device="cuda"),
        qsl=torch.tensor([0, T], dtype=torch.int32, device="cuda"),
        kv=torch.zeros((2, per_seq, BLOCK, N_KV, HD), dtype=BF16, device="cuda"))


def _cos_sin(max_pos: int) -> torch.Tensor:
    inv = 1.0 / (THETA ** (torch.arange(0, HD, 2, dtype=torch.float32) / HD))
    f = torch.outer(torch.arange(max_pos, dtype=torch.float32), inv)
    return torch.cat((f.cos(), f.sin()), dim=-1).to(BF16).cuda()


def _prep_prefill(case, seed):
    s = _prefill_inputs(case, seed)
    ops = _mod("native.torch_ops")
    s.update(run=_run_prefill, ops=ops, cos_sin=_cos_sin(case["tokens"]),
             lut=ops.gelu_table("cuda") if case["act"] == "gelu" else None)
    return s


def _run_prefill(s):
    ops = s["ops"]
    h = ops.embedding(s["table"], s["ids"])
    y, res = ops.add_rmsnorm(h, s["residual"], s["gamma"], EPS)
    slots = ops.compute_slot_mapping(s["qsl"], s["pos"], s["block_table"], BLOCK)
    q = ops.qknorm_rope_kv_write(s["qkv"], s["q_gamma"], s["k_gamma"], s["cos_sin"], s["pos"],
                                 slots, s["kv"][0], s["kv"][1], N_Q, N_KV, EPS)
    act = (ops.silu_mul(s["gate_up"]) if s["lut"] is None
           else ops.gelu_mul(s["gate_up"], s["lut"]))
    return h, y, res, slots, q, s["kv"], act


_PREPARE = {"linear": _prep_linear, "head": _prep_head, "attn": _prep_attn,
            "layer": _prep_layer, "model": _prep_model, "prefill_ops": _prep_prefill}


# ---------------------------------------------------------------------- work
def _linear_work(m: int, n: int, k: int) -> tuple[int, int]:
    return n * k // 32 * 18 + 2 * m * k + 2 * m * n, 2 * m * n * k


def _attn_work(lengths) -> tuple[int, int]:
    t, s = sum(lengths), len(lengths)
    return (t * 2 * N_KV * HD * 2 + s * (2 * N_Q + 4 * N_KV) * HD * 2, 4 * t * N_Q * HD)


def _layer_work(lengths) -> tuple[int, int]:
    s = len(lengths)
    parts = [_linear_work(s, n, k) for n, k in ((QKV_ROWS, HIDDEN), (HIDDEN, N_Q * HD),
                                                (2 * INTER, HIDDEN), (HIDDEN, INTER))]
    a = _attn_work(lengths)
    weights = sum((QKV_ROWS, 2 * INTER)) * HIDDEN // 32 * 18 \
        + HIDDEN * (N_Q * HD + INTER) // 32 * 18
    return (weights + a[0] + 4 * s * HIDDEN * 2 + 2 * HIDDEN * 2,
            sum(p[1] for p in parts) + a[1])


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "linear":
        b, f = _linear_work(case["m"], case["n"], case["k"])
    elif kind == "head":
        b, f = _linear_work(case["rows"], case["vocab"], case["hidden"])
    elif kind == "attn":
        b, f = _attn_work(_lengths(case))
    elif kind == "layer":
        b, f = _layer_work(_lengths(case))
    elif kind == "model":
        b = f = 0
        for t in range(MODEL_STEPS):
            lb, lf = _layer_work([case["context"] + t + 1])
            hb, hf = _linear_work(1, case["vocab"], HIDDEN)
            b += case["layers"] * lb + hb
            f += case["layers"] * lf + hf
    else:
        t = case["tokens"]
        # embedding row in/out, residual in, norm and residual out; qkv in, q and K/V out;
        # gate|up in, activation out
        b = 2 * t * (5 * HIDDEN + 2 * QKV_ROWS + 3 * INTER)
        f = t * (10 * HIDDEN + 10 * QKV_ROWS + 8 * INTER)
    return {"bytes": b, "flops": f}


def tolerance(case: dict):
    # About four times what was measured on an MI355X for another correct way to the same
    # result; the outputs are bf16, so one differently rounded value is up to 2^-7 of itself.
    kind = case["kind"]
    if kind == "linear":
        # up to 16 rows multiply the exact Q4_0 weights (other sum orders: rel 4e-5, max
        # 7e-3); more rows may take their bf16 roundings (rel 2.6e-3, max 1.3e-2)
        return ({"rel": 1e-3, "max": 0.03} if case["m"] <= 16 else {"rel": 1e-2, "max": 0.05})
    if kind == "head":  # as the linears; ids differ where two logits tie
        return ({"rel": 1e-3, "max": 0.03, "differ": 0.01} if case["rows"] == 1
                else {"rel": 1e-2, "max": 0.05, "differ": 0.01})
    if kind == "attn":  # splits of other lengths: bf16 probabilities at other maxima
        return {"rel": 1e-2, "max": 0.05}  # seen 2.4e-3, 1.2e-2
    if kind == "layer":  # the GGUF GEMMs and another split plan
        return {"rel": 1.5e-2, "max": 0.08}  # seen 3.9e-3, 1.9e-2
    if kind == "model":  # one launch per op instead of the fused step, other splits
        return {"rel": 5e-3, "max": 0.06}  # seen 1.1e-3, 1.4e-2
    # the q/k norm rounded to bf16 before the rotation or not: seen 2.7e-3, 1.5e-2
    return {"rel": 1e-2, "max": 0.06}


# --------------------------------------------------------------------- exact
def exact(case: dict, seed: int):
    with torch.no_grad():
        return _EXACT[case["kind"]](case, seed)


def _exact_linear(case, seed):
    m, n, k = case["m"], case["n"], case["k"]
    y = _randn(_gen(seed, 2), m, k).double() @ _dequant64(_blocks(_gen(seed, 1), n, k), k).T
    if case["bias"]:
        y = y + _randn(_gen(seed, 3), n).double()
    return y


def _exact_head(case, seed):
    w = _dequant64(_blocks(_gen(seed, 1), case["vocab"], case["hidden"]), case["hidden"])
    return _randn(_gen(seed, 2), case["rows"], case["hidden"]).double() @ w.T, None


def _attn64(q, K, V):
    """q [T, n_q, hd] at the last T of K, V [L, n_kv, hd]: causal attention."""
    T, L = q.shape[0], K.shape[0]
    out = torch.empty_like(q)
    mask = (torch.arange(L, device="cuda")[None, :]
            > torch.arange(L - T, L, device="cuda")[:, None])
    g = q.shape[1] // K.shape[1]
    for h in range(q.shape[1]):
        s = (q[:, h] @ K[:, h // g].T) * SCALE
        p = torch.softmax(s.masked_fill(mask, -math.inf), dim=-1)
        out[:, h] = p @ V[:, h // g]
    return out


def _gather_kv(kv, table_row, length):
    t = torch.arange(length, device="cuda")
    p = table_row[t // BLOCK].to(torch.int64)
    return (kv[0][p, t % BLOCK].double(), kv[1][p, t % BLOCK].double())


def _exact_attn(case, seed):
    L, _, table, kv, q, k, v = _attn_inputs(case, seed)
    slots = _slots(table, L - 1)
    kv[0].view(-1, N_KV, HD)[slots] = k.view(-1, N_KV, HD)
    kv[1].view(-1, N_KV, HD)[slots] = v.view(-1, N_KV, HD)
    outs = []
    for i, n in enumerate(L.tolist()):
        K, V = _gather_kv(kv, table[i], n)
        outs.append(_attn64(q[i].double().view(1, N_Q, HD), K, V).view(-1))
    return torch.stack(outs), kv


def _rms64(x, gamma):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * gamma.double()


def _rope64(x, pos, cs):
    c = cs[pos, None, :HD // 2].double()
    s = cs[pos, None, HD // 2:].double()
    a, b = x[..., :HD // 2], x[..., HD // 2:]
    return torch.cat((a * c - b * s, b * c + a * s), dim=-1)


def _layer64(w, i, h, res, pos, cs, kv, tables, groups):
    """One decoder layer on h [T, hidden] (normalised input) with residual
    res: (mlp out, residual).  groups: [(row of tables, first, last + 1)] of
    consecutive tokens; kv (bf16) gets the new K/V rows."""
    d = {n: _dequant64(w[f"layers.{i}.{n}"], k) for n, k in
         (("qkv", HIDDEN), ("o_proj", N_Q * HD), ("gate_up", HIDDEN), ("down", INTER))}
    T = h.shape[0]
    qkv = (h @ d["qkv"].T).view(T, N_Q + 2 * N_KV, HD)
    q = _rope64(_rms64(qkv[:, :N_Q], w[f"layers.{i}.norm2"]), pos, cs)
    k = _rope64(_rms64(qkv[:, N_Q:N_Q + N_KV], w[f"layers.{i}.norm3"]), pos, cs)
    v = qkv[:, N_Q + N_KV:]
    o = torch.empty_like(q)
    for r, a, b in groups:
        L = int(pos[b - 1]) + 1
        K, V = _gather_kv(kv, tables[r], L)
        K[L - (b - a):], V[L - (b - a):] = k[a:b], v[a:b]
        o[a:b] = _attn64(q[a:b], K, V)
        p = tables[r][pos[a:b] // BLOCK].to(torch.int64) * BLOCK + pos[a:b] % BLOCK
        kv[0].view(-1, N_KV, HD)[p] = k[a:b].to(BF16)
        kv[1].view(-1, N_KV, HD)[p] = v[a:b].to(BF16)
    res = o.reshape(T, -1) @ d["o_proj"].T + res
    gu = _rms64(res, w[f"layers.{i}.norm1"]) @ d["gate_up"].T
    act = torch.nn.functional.silu(gu[:, :INTER]) * gu[:, INTER:]
    return act @ d["down"].T, res


def _model_pages(num_blocks: int, batch: int) -> torch.Tensor:
    """The block table a DecodeModel hands out (its pages are shuffled by its
    own seed, 0)."""
    perm = torch.randperm(num_blocks, generator=torch.Generator().manual_seed(0))
    return perm[:num_blocks - 1].view(batch, -1).cuda()


def _exact_layer(case, seed):
    S = case["seqs"]
    L = torch.tensor(_lengths(case), dtype=torch.int64, device="cuda")
    per_seq = -(-(case["hi"] + 1) // BLOCK)
    tables = _model_pages(S * per_seq + 1, S)
    kv = torch.empty((2, S * per_seq + 1, BLOCK, N_KV, HD), dtype=BF16, device="cuda")
    kv.normal_(0.0, 1.0, generator=_gen(seed, 5))
    g = _gen(seed, 6)
    x, res = _randn(g, S, HIDDEN).double(), _randn(g, S, HIDDEN).double()
    w = _layer_weights(seed, 0)
    d, res = _layer64(w, 0, x, res, L - 1, _cos_sin(per_seq * BLOCK), kv, tables,
                      [(i, i, i + 1) for i in range(S)])
    res = d + res
    return _rms64(res, _norm(_gen(seed, 4), HIDDEN)), res, kv


def _exact_model(case, seed):
    c, n = case["context"], case["layers"]
    per_seq = -(-CAP_1SEQ // BLOCK)
    tables = _model_pages(per_seq + 1, 1)
    fill = torch.Generator(device="cuda").manual_seed(int(seed) + 1)
    w = _model_weights(case, seed)
    toks = _model_tokens(case, seed)
    head = _dequant64(w["head"], HIDDEN)
    pos = torch.arange(c, c + MODEL_STEPS, device="cuda")
    cs = _cos_sin(CAP_1SEQ)
    d, res, caches = None, head[toks].to(BF16).double(), []
    for i in range(n):
        kv = torch.empty((2, per_seq + 1, BLOCK, N_KV, HD), dtype=BF16, device="cuda")
        kv.normal_(0.0, 1.0, generator=fill)
        if d is not None:
            res = d + res
        d, res = _layer64(w, i, _rms64(res, w[f"layers.{i}.norm0"]), res, pos, cs, kv, tables,
                          [(0, 0, MODEL_STEPS)])
        caches.append(kv)
    h = _rms64((d + res)[-1:], w["final_norm"])
    return [h @ head.T] + caches


def _exact_prefill(case, seed):
    s = _prefill_inputs(case, seed)
    T = case["tokens"]
    h = s["table"][s["ids"]]
    res = h.double() + s["residual"].double()
    pos = s["pos"]
    slots = s["block_table"][0][pos // BLOCK].to(torch.int64) * BLOCK + pos % BLOCK
    qkv = s["qkv"].double().view(T, N_Q + 2 * N_KV, HD)
    cs = _cos_sin(T)
    q = _rope64(_rms64(qkv[:, :N_Q], s["q_gamma"]), pos, cs)
    k = _rope64(_rms64(qkv[:, N_Q:N_Q + N_KV], s["k_gamma"]), pos, cs)
    kv = s["kv"]
    kv[0].view(-1, N_KV, HD)[slots] = k.to(BF16)
    kv[1].view(-1, N_KV, HD)[slots] = s["qkv"].view(T, N_Q + 2 * N_KV, HD)[:, N_Q + N_KV:]
    g, u = s["gate_up"][:, :INTER].double(), s["gate_up"][:, INTER:].double()
    act = (torch.nn.functional.silu(g) if case["act"] == "swiglu"
           else 0.5 * g * (1.0 + torch.erf(g / math.sqrt(2.0)))) * u
    return h, _rms64(res, s["gamma"]), res, slots, q, kv, act


_EXACT = {"linear": _exact_linear, "head": _exact_head, "attn": _exact_attn,
          "layer": _exact_layer, "model": _exact_model, "prefill_ops": _exact_prefill}
