"""The calls that this framework's time is judged by: what a thinker and a Talker have it do, through its public entry
points, from one decode token to a 2048-token prompt.

  moe_decode   one decode MoE block of 1..8 tokens (fused_moe.moe_block_decode), replayed from the graph that a decode
               loop keeps
  moe_prefill  one prompt MoE block of 9..2048 tokens (fused_moe.moe_block_prefill) on stacks whose prefill copies were
               made at load
  kda          the KDA core of one layer over a prompt (thinker_attn.chunk_kda past thinker_step.KDA_CHUNK_ABOVE tokens,
               fused_recurrent_kda up to it, the thinker's own switch), the layer's state updated in place
  mla          the MLA attention of one layer over a prompt behind a context of `pos` tokens (thinker_attn.mla_prefill_attn)
  step         one greedy decode token of a hybrid thinker (3 KDA layers, 1 MLA layer, MoE blocks, LM head), replayed
  prompt       a padded prompt through the same thinker (FastThinkerStep.prefill with n_valid), replayed from the graph
               of its bucket
  talker       one decode token of the Talker's Qwen2 (fast_talker.FastQwen2Step), replayed
  tail         one latent of the Talker's flow-matching tail (fast_talker.FastTail), replayed

Two shapes of MoE block: "lite" (hidden 2048, 64 routed experts of 1408, softmax top-6) and "tiny" (hidden 1536, 128
routed experts of 512, sigmoid top-8 in 8 groups of which 4 are kept, scale 2.5), each with one shared expert. Weights
are bf16, or int8 with fp32 or bf16 row scales. Attention: 16 heads, KDA 128 x 128 with gate rank 128 and window 4, MLA
192 / 128. exact() is the same mathematics in 64 bits without any intermediate rounding, except where the interface
itself rounds (cache rows held in bf16).
"""
import math
import os
import sys
from types import SimpleNamespace as NS

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ming-voice_amd"))

import fast_talker  # noqa: E402
import fused_moe  # noqa: E402
import thinker_attn  # noqa: E402
import thinker_step  # noqa: E402

DEV = "cuda"
BF, F32, F64 = torch.bfloat16, torch.float32, torch.float64
EPS = 1e-6
MOE = {
    "lite": dict(H=2048, I=1408, E=64, top_k=6, scoring="softmax", n_group=1, topk_group=1, scale=1.0),
    "tiny": dict(H=1536, I=512, E=128, top_k=8, scoring="sigmoid", n_group=8, topk_group=4, scale=2.5),
}
HEADS, KDIM, VDIM, RANK, WINDOW = 16, 128, 128, 128, 4  # a KDA layer
MLA_QK, MLA_V = 192, 128                                # an MLA layer, also 16 heads
HIDDEN, VOCAB, LAYERS, MLA_EVERY = 2048, 126464, 4, 4   # the hybrid thinker
MLA_LEN = 4096                                          # rows of an MLA cache
KDA_SWITCH = 192
TALKER = dict(hidden=896, heads=14, kv_heads=2, inter=4864, layers=24, max_len=1024)
TAIL = dict(dim=1024, heads=16, mlp=4096, depth=4, agg=2, latent=64)


# ------------------------------------------------------------------------------------------------------- the cases

def listed():
    return [
        # every generated token, once a layer: the smallest call and the most frequent one
        dict(name="moe_decode_1", kind="moe_decode", shape="lite", tokens=1, weights="bf16", scales="none"),
        # several streams decoded together, on the quantised experts that small cards are served with
        dict(name="moe_decode_5_int8", kind="moe_decode", shape="lite", tokens=5, weights="int8", scales="f32"),
        # a short spoken turn
        dict(name="moe_prefill_37_int8", kind="moe_prefill", shape="lite", tokens=37, weights="int8", scales="bf16",
             routing="ragged"),
        # a turn with tool results or audio features: the benchmarked prompt
        dict(name="moe_prefill_512", kind="moe_prefill", shape="lite", tokens=512, weights="bf16", scales="none",
             routing="ragged"),
        # a long prompt whose routing prefers a few experts
        dict(name="moe_prefill_2048_zipf", kind="moe_prefill", shape="lite", tokens=2048, weights="bf16",
             scales="none", routing="zipf"),
        # the thinker's own block shape: many small experts, grouped sigmoid selection
        dict(name="moe_prefill_tiny_300", kind="moe_prefill", shape="tiny", tokens=300, weights="bf16", scales="none",
             routing="ragged"),
        # a KDA layer's core over a prompt (three of four layers)
        dict(name="kda_700", kind="kda", tokens=700, bound=0.0),
        # an MLA layer's attention over a prompt behind a conversation
        dict(name="mla_500_at_611", kind="mla", tokens=500, pos=611),
        # a whole decode token
        dict(name="step_at_700", kind="step", pos=700, weights="bf16"),
        # a whole prompt in its padded bucket
        dict(name="prompt_150", kind="prompt", tokens=150, bucket=160, pos=512, weights="bf16"),
        # the Talker's decode token and the latent that follows it: once for every 80 ms of speech
        dict(name="talker_at_300", kind="talker", pos=300),
        dict(name="tail_10", kind="tail", steps=10),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["moe_decode", "moe_prefill", "moe_prefill", "moe_prefill", "kda", "mla", "step", "prompt",
                       "talker", "tail"])
    if kind in ("moe_decode", "moe_prefill"):
        w = rng.choice(["bf16", "int8"])
        c = dict(kind=kind, shape=rng.choice(["lite", "tiny"]), weights=w,
                 scales=rng.choice(["f32", "bf16"]) if w == "int8" else "none",
                 tokens=rng.randint(1, 8) if kind == "moe_decode" else _log_int(rng, 9, 2048))
        if kind == "moe_prefill":
            c["routing"] = rng.choice(["ragged", "zipf"])
        return c
    if kind == "kda":
        return dict(kind=kind, tokens=_log_int(rng, 3, 2048), bound=rng.choice([0.0, -5.0]))
    if kind == "mla":
        n = _log_int(rng, 3, 2048)
        return dict(kind=kind, tokens=n, pos=rng.choice([0, _log_int(rng, 1, MLA_LEN - n)]))
    if kind == "step":
        return dict(kind=kind, pos=_log_int(rng, 10, MLA_LEN - 1), weights=rng.choice(["bf16", "int8"]))
    if kind == "prompt":
        n = _log_int(rng, 3, 150)
        return dict(kind=kind, tokens=n, bucket=n if n <= 16 else -(-n // 32) * 32, pos=rng.choice([0, rng.randint(1, 2000)]),
                    weights=rng.choice(["bf16", "int8"]))
    if kind == "talker":
        return dict(kind=kind, pos=rng.randint(0, TALKER["max_len"] - 1))
    return dict(kind=kind, steps=rng.randint(2, 16))


# ------------------------------------------------------------------------------------------------ inputs from a seed

class _Draw:
    """Tensors drawn one after the other from one seeded generator on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0, dtype=BF):
        return torch.randn(shape, generator=self.g, device=DEV).mul_(std).add_(mean).to(dtype)

    def uniform(self, *shape, lo=0.0, hi=1.0, dtype=F32):
        return torch.rand(shape, generator=self.g, device=DEV).mul_(hi - lo).add_(lo).to(dtype)

    def ints(self, hi, *shape):
        return torch.randint(hi, shape, generator=self.g, device=DEV)

    def order(self, n):
        return torch.randperm(n, generator=self.g, device=DEV)

    def gamma(self, n):
        return self.normal(n, std=0.02, mean=1.0)


def _quantised(w, scale_dtype):
    """Symmetric int8 rows of w and their scales."""
    s = (w.abs().amax(-1).float().clamp_min(1e-8) / 127.0).to(scale_dtype)
    q = torch.empty(w.shape, dtype=torch.int8, device=w.device)
    for e in range(w.shape[0]):
        q[e] = torch.round(w[e].float() / s[e].float()[:, None]).clamp_(-127, 127).to(torch.int8)
    return q, s


def _block(d, shape, weights, scales, routing="ragged"):
    """One MoE block's weights. routing: router biases that give ragged or Zipf-like (rank^-1.2) expert counts."""
    m = MOE[shape]
    H, I, E = m["H"], m["I"], m["E"]
    b = dict(m, norm_w=d.gamma(H), w32=d.normal(E, H, std=0.02, dtype=F32), s_gu=None, s_d=None)
    b["w_gu"] = d.normal(E + 1, 2 * I, H, std=0.02)
    b["w_d"] = d.normal(E + 1, H, I, std=0.02)
    if weights == "int8":
        t = F32 if scales == "f32" else BF
        b["w_gu"], b["s_gu"] = _quantised(b["w_gu"], t)
        b["w_d"], b["s_d"] = _quantised(b["w_d"], t)
    if routing == "zipf":
        p = torch.arange(1, E + 1, device=DEV, dtype=F32).pow(-1.2)[d.order(E)]
        b["bias"] = (p / p.sum()).log().contiguous() * (1.0 if m["scoring"] == "softmax" else 0.1)
    else:
        b["bias"] = d.normal(E, std=0.5 if m["scoring"] == "softmax" else 0.05, dtype=F32)
    return b


def _route_args(b):
    return dict(top_k=b["top_k"], bias=b["bias"], scoring=b["scoring"], n_group=b["n_group"],
                topk_group=b["topk_group"], scale=b["scale"], s_gu=b["s_gu"], s_d=b["s_d"])


def _kda_gate_params(d):
    """A_log and dt_bias as trained gates have them: from channels that hardly decay to ones that forget at once."""
    return d.uniform(HEADS, lo=0.0, hi=math.log(16.0)), d.uniform(HEADS * KDIM, lo=-6.0, hi=0.5)


def _kda_inputs(d, n):
    A_log, dt_bias = _kda_gate_params(d)
    return dict(q=d.normal(1, n, HEADS, KDIM), k=d.normal(1, n, HEADS, KDIM), v=d.normal(1, n, HEADS, VDIM),
                g=d.normal(1, n, HEADS, KDIM), beta=d.normal(1, n, HEADS), A_log=A_log, dt_bias=dt_bias,
                state=d.normal(1, HEADS, KDIM, VDIM, std=0.1, dtype=F32))


def _mla_inputs(d, n, pos):
    s = dict(q=d.normal(n, HEADS * MLA_QK), k=d.normal(n, HEADS * MLA_QK), v=d.normal(n, HEADS * MLA_V),
             kc=torch.zeros(1, HEADS, MLA_LEN, MLA_QK, device=DEV, dtype=BF),
             vc=torch.zeros(1, HEADS, MLA_LEN, MLA_V, device=DEV, dtype=BF))
    s["kc"][:, :, :pos] = d.normal(1, HEADS, pos, MLA_QK)
    s["vc"][:, :, :pos] = d.normal(1, HEADS, pos, MLA_V)
    return s


def _lin(w, b=None):
    return NS(weight=w, bias=b)


def _thinker(d, pos, weights):
    """A hybrid thinker as a loaded model holds it: every MLA_EVERY-th layer MLA, the others KDA, then a MoE block."""
    H, nq, nv = HIDDEN, HEADS * KDIM, HEADS * VDIM
    layers, caches, raw = [], [], []
    for li in range(LAYERS):
        b = _block(d, "lite", weights, "f32")
        p = dict(blk=b, ln1=d.gamma(H))
        if (li + 1) % MLA_EVERY == 0:
            m = _mla_inputs(d, 1, pos)
            p.update(kind="mla", wq=d.normal(HEADS * MLA_QK, H, std=0.02), wk=d.normal(HEADS * MLA_QK, H, std=0.02),
                     wv=d.normal(HEADS * MLA_V, H, std=0.02), wo=d.normal(H, HEADS * MLA_V, std=0.02), kc=m["kc"], vc=m["vc"])
            attn = NS(q_proj=_lin(p["wq"]), k_proj=_lin(p["wk"]), v_proj=_lin(p["wv"]), o_proj=_lin(p["wo"]),
                      num_heads=HEADS, qk_head_dim=MLA_QK, v_head_dim=MLA_V)
            caches.append(NS(k=p["kc"], v=p["vc"]))
        else:
            A_log, dt_bias = _kda_gate_params(d)
            p.update(kind="kda", wq=d.normal(nq, H, std=0.02), wk=d.normal(nq, H, std=0.02), wv=d.normal(nv, H, std=0.02),
                     fa=d.normal(RANK, H, std=0.02), ga=d.normal(RANK, H, std=0.02), wb=d.normal(HEADS, H, std=0.02),
                     fb=d.normal(nq, RANK, std=0.05), gb=d.normal(nv, RANK, std=0.05),
                     cw=[d.normal(n, 1, WINDOW, std=0.5) for n in (nq, nq, nv)],
                     conv=[d.normal(1, n, WINDOW) for n in (nq, nq, nv)], A_log=A_log, dt_bias=dt_bias,
                     o_norm=d.gamma(VDIM), wo=d.normal(H, nv, std=0.02),
                     state=d.normal(1, HEADS, KDIM, VDIM, std=0.1, dtype=F32))
            c = [NS(weight=w, bias=None) for w in p["cw"]]
            attn = NS(q_proj=_lin(p["wq"]), k_proj=_lin(p["wk"]), v_proj=_lin(p["wv"]), f_a_proj=_lin(p["fa"]),
                      g_a_proj=_lin(p["ga"]), b_proj=_lin(p["wb"]), f_b_proj=_lin(p["fb"]), g_b_proj=_lin(p["gb"]),
                      q_conv1d=c[0], k_conv1d=c[1], v_conv1d=c[2], o_norm=NS(weight=p["o_norm"], eps=1e-5),
                      o_proj=_lin(p["wo"]), A_log=A_log, dt_bias=dt_bias, lower_bound=None, num_heads=HEADS,
                      head_k_dim=KDIM, head_dim=VDIM, no_kda_lora=False)
            caches.append(NS(keys=p["state"], values=tuple(p["conv"])))
        gate = NS(w32=b["w32"], expert_bias=b["bias"], top_k=b["top_k"], n_group=1, topk_group=1, routed_scaling_factor=1.0)
        mlp = NS(gate=gate, w_gu=None, w_d=None)
        if weights == "int8":
            mlp.q_gu, mlp.q_d, mlp.s_gu, mlp.s_d = b["w_gu"], b["w_d"], b["s_gu"], b["s_d"]
        else:
            mlp.w_gu, mlp.w_d = b["w_gu"], b["w_d"]
        layers.append(NS(attention=attn, attention_layer_type="attention" if p["kind"] == "mla" else "kda", mlp=mlp,
                         input_layernorm=NS(weight=p["ln1"], variance_epsilon=EPS),
                         post_attention_layernorm=NS(weight=b["norm_w"], variance_epsilon=EPS)))
        raw.append(p)
    embed, norm, head = d.normal(VOCAB, H), d.gamma(H), d.normal(VOCAB, H, std=0.02)
    model = NS(model=NS(word_embeddings=NS(weight=embed), layers=layers, norm=NS(weight=norm, variance_epsilon=EPS)),
               lm_head=_lin(head))
    return dict(model=model, caches=caches, layers=raw, embed=embed, norm=norm, head=head,
                tok=d.ints(VOCAB, 1, 1), pos=torch.tensor([pos], device=DEV))


def _thinker_state(t):
    """The tensors that a call of the thinker updates, but the token and the position."""
    out = []
    for p in t["layers"]:
        out += [p["kc"], p["vc"]] if p["kind"] == "mla" else [p["state"], *p["conv"]]
    return out


def _talker(d, pos):
    t = TALKER
    H, hd = t["hidden"], t["hidden"] // t["heads"]
    layers = []
    for _ in range(t["layers"]):
        def w(*shape):
            return d.normal(*shape, std=0.02)
        at = NS(q_proj=_lin(w(t["heads"] * hd, H), w(t["heads"] * hd)), k_proj=_lin(w(t["kv_heads"] * hd, H), w(t["kv_heads"] * hd)),
                v_proj=_lin(w(t["kv_heads"] * hd, H), w(t["kv_heads"] * hd)), o_proj=_lin(w(H, t["heads"] * hd)))
        mlp = NS(gate_proj=_lin(w(t["inter"], H)), up_proj=_lin(w(t["inter"], H)), down_proj=_lin(w(H, t["inter"])))
        layers.append(NS(self_attn=at, mlp=mlp, input_layernorm=NS(weight=d.gamma(H), variance_epsilon=EPS),
                         post_attention_layernorm=NS(weight=d.gamma(H), variance_epsilon=EPS)))
    k = torch.zeros(t["layers"], 1, t["kv_heads"], t["max_len"], hd, device=DEV, dtype=BF)
    v = torch.zeros_like(k)
    k[:, :, :, :pos] = d.normal(t["layers"], 1, t["kv_heads"], pos, hd)
    v[:, :, :, :pos] = d.normal(t["layers"], 1, t["kv_heads"], pos, hd)
    inv = 1.0 / (1e6 ** (torch.arange(0, hd, 2, device=DEV, dtype=F32) / hd))
    return NS(m=NS(layers=layers, norm=NS(weight=d.gamma(H), variance_epsilon=EPS)), nh=t["heads"], nkv=t["kv_heads"],
              hd=hd, max_len=t["max_len"], k=k, v=v, inv_freq=inv), d.normal(1, 1, H), torch.tensor([pos], device=DEV)


class _Rotary:
    """Interleaved rotary angles, each pair's angle twice."""

    def __init__(self, hd):
        self.inv = 1.0 / (1e4 ** (torch.arange(0, hd, 2, device=DEV, dtype=F32) / hd))

    def forward_from_seq_len(self, n):
        f = torch.arange(n, device=DEV, dtype=F32)[:, None] * self.inv[None]
        return torch.stack([f, f], -1).reshape(1, n, -1), 1.0


def _dit_block(d, D, heads, mlp):
    def w(*shape):
        return d.normal(*shape, std=0.02)
    attn = NS(heads=heads, to_q=_lin(w(D, D), w(D)), to_k=_lin(w(D, D), w(D)), to_v=_lin(w(D, D), w(D)),
              to_out=[_lin(w(D, D), w(D))], q_norm=None, pe_attn_head=None)
    ff = [[_lin(w(mlp, D), w(mlp)), NS(approximate="tanh")], None, _lin(w(D, mlp), w(D))]
    return NS(attn=attn, mlp=NS(ff=ff), norm1=NS(weight=d.gamma(D), eps=EPS), norm2=NS(weight=d.gamma(D), eps=EPS))


def _tail(d, steps):
    c, llm = TAIL, TALKER["hidden"]
    D, hd, z = c["dim"], c["dim"] // c["heads"], c["latent"]

    def w(*shape):
        return d.normal(*shape, std=0.02)

    def final(out):
        return NS(norm_final=NS(weight=d.gamma(D), eps=EPS), linear=_lin(w(out, D), w(out)))
    temb = d.normal(steps, D, std=0.5)
    ts = torch.linspace(0, 1, steps + 1, device=DEV).to(BF)
    at = {float(ts[i]): temb[i:i + 1] for i in range(steps)}
    dit = NS(spk_embedder=None, t_embedder=lambda t: at[float(t)], c_embedder=NS(cond_embedder=_lin(w(D, llm), w(D))),
             x_embedder=_lin(w(D, z), w(D)), blocks=[_dit_block(d, D, c["heads"], c["mlp"]) for _ in range(c["depth"])],
             rotary_embed=_Rotary(hd), final_layer=final(z))
    cls = d.normal(1, 1, D)
    agg = NS(word_embedder=lambda ids: cls, x_embedder=_lin(w(D, z), w(D)),
             blocks=[_dit_block(d, D, c["heads"], c["mlp"]) for _ in range(c["agg"])], rotary_embed=_Rotary(hd),
             final_layer=final(llm))
    t = NS(cfm=NS(model=dit), aggregator=agg, stop_head=_lin(d.normal(2, llm, std=0.05), w(2)))
    dts = [ts[i + 1] - ts[i] for i in range(steps)]
    return dict(talker=NS(t=t), ts=ts, dts=dts, temb=temb, cls=cls, hidden=d.normal(1, 1, llm), hist=d.normal(1, 1, z),
                noise=d.normal(1, 1, z))


# --------------------------------------------------------------------------------------------- prepare and run a pass

def _captured(fn, keep=()):
    """fn in a graph of its own, as a serving loop keeps it: warmed up, captured, and the state in `keep` put back."""
    saved = [t.clone() for t in keep]
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(2):
            fn()
        s.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            out = fn()
    torch.cuda.current_stream().wait_stream(s)
    for t, old in zip(keep, saved):
        t.copy_(old)
    return g, out


def prepare(case, seed):
    kind, d = case["kind"], _Draw(seed)
    if kind in ("moe_decode", "moe_prefill"):
        b = _block(d, case["shape"], case["weights"], case["scales"], case.get("routing", "ragged"))
        x = d.normal(case["tokens"], b["H"])
        s = dict(kind=kind, x=x, b=b)
        if kind == "moe_prefill":
            s["copies"] = fused_moe.prefill_copies(b["w_gu"], b["w_d"])
        else:
            s["graph"], s["out"] = _captured(lambda: fused_moe.moe_block_decode(
                x, b["norm_w"], EPS, b["w32"], b["w_gu"], b["w_d"], **_route_args(b)))
        return s
    if kind == "kda":
        return dict(_kda_inputs(d, case["tokens"]), kind=kind, bound=case["bound"] or None, n=case["tokens"])
    if kind == "mla":
        return dict(_mla_inputs(d, case["tokens"], case["pos"]), kind=kind, pos=torch.tensor([case["pos"]], device=DEV))
    if kind in ("step", "prompt"):
        t = _thinker(d, case["pos"], case["weights"])
        s = dict(kind=kind, t=t, start=t["pos"].clone(), tok0=t["tok"].clone(), state=_thinker_state(t))
        fast = thinker_step.FastThinkerStep(t["model"], t["caches"], t["tok"], t["pos"], scoring="softmax")
        if kind == "step":
            call = fast
        else:
            s["ids"] = d.ints(VOCAB, case["bucket"])
            s["n"] = torch.tensor([case["tokens"]], device=DEV)
            s["copies"] = [fused_moe.prefill_copies(p["blk"]["w_gu"], p["blk"]["w_d"]) for p in t["layers"]]

            def call():
                return fast.prefill(ids=s["ids"], n_valid=s["n"])

        def turn():  # the conversation's position and token, then the call
            t["pos"].copy_(s["start"])
            t["tok"].copy_(s["tok0"])
            return call()
        s["fast"] = fast
        s["graph"], s["out"] = _captured(turn, [t["pos"], t["tok"], *s["state"]])
        return s
    if kind == "talker":
        llm, x, pos = _talker(d, case["pos"])
        step = fast_talker.FastQwen2Step(llm)
        s = dict(kind=kind, llm=llm, step=step, x=x, pos=pos)
        s["graph"], s["out"] = _captured(lambda: step(x, pos))
        return s
    m = _tail(d, case["steps"])
    tail = fast_talker.FastTail(m["talker"], m["ts"], m["dts"], 2.0)
    s = dict(kind=kind, tail=tail, m=m)
    s["graph"], s["out"] = _captured(lambda: tail(m["hidden"], m["hist"], m["noise"]))
    return s


def run(s):
    kind = s["kind"]
    if kind == "moe_prefill":
        b = s["b"]
        return fused_moe.moe_block_prefill(s["x"], b["norm_w"], EPS, b["w32"], b["w_gu"], b["w_d"], **_route_args(b))
    if kind == "kda":
        f = thinker_attn.chunk_kda if s["n"] > KDA_SWITCH else thinker_attn.fused_recurrent_kda
        return f(s["q"], s["k"], s["v"], s["g"], s["beta"], A_log=s["A_log"], dt_bias=s["dt_bias"],
                 initial_state=s["state"], inplace=True, use_qk_l2norm_in_kernel=True, use_gate_in_kernel=True,
                 beta_is_logits=True, lower_bound=s["bound"])
    if kind == "mla":
        y = thinker_attn.mla_prefill_attn(s["q"], s["k"], s["v"], s["kc"], s["vc"], s["pos"])
        return y, s["kc"], s["vc"]
    s["graph"].replay()
    if kind in ("step", "prompt"):
        return [s["out"], *s["state"]]
    if kind == "talker":
        return s["out"], s["llm"].k, s["llm"].v
    return s["out"]


# ------------------------------------------------------------------------------------------------- what a pass needs

def _experts_used(E, k, n, zipf):
    """Expected number of distinct routed experts that n tokens with k picks each reach."""
    p = [1.0] * E
    if zipf:
        p = [(i + 1) ** -1.2 for i in range(E)]
    t = sum(p)
    return sum(1 - (1 - min(1.0, k * x / t)) ** n for x in p)


def _moe_work(shape, n, weights, scales, routing="ragged"):
    m = MOE[shape]
    H, I, E, k = m["H"], m["I"], m["E"], m["top_k"]
    used = _experts_used(E, k, n, routing == "zipf") + 1
    each = 3 * H * I * (1 if weights == "int8" else 2) + (0 if weights == "bf16" else (2 * I + H) * (4 if scales == "f32" else 2))
    return used * each + E * H * 4 + 2 * n * H * 2 + n * (E * 4 + (k + 1) * 12), n * (k + 1) * 6 * H * I + 2 * n * E * H


def _kda_work(n):
    state = HEADS * KDIM * VDIM
    return n * HEADS * (3 * KDIM + 2 * VDIM + 1) * 2 + 2 * state * 4, n * 6 * state


def _mla_work(n, pos):
    rows = HEADS * (MLA_QK + MLA_V) * 2
    return n * HEADS * (MLA_QK + MLA_V) * 2 + (pos + 2 * n) * rows, 2 * HEADS * (MLA_QK + MLA_V) * (n * pos + n * (n + 1) / 2)


def _thinker_work(n, pos, weights):
    H = HIDDEN
    kda_w = H * (2 * HEADS * KDIM + HEADS * VDIM + 2 * RANK + HEADS) + RANK * HEADS * (KDIM + VDIM) + H * HEADS * VDIM
    mla_w = H * HEADS * (2 * MLA_QK + MLA_V) + H * HEADS * MLA_V
    by = fl = 0
    for li in range(LAYERS):
        mla = (li + 1) % MLA_EVERY == 0
        w = mla_w if mla else kda_w
        b1, f1 = _mla_work(n, pos) if mla else _kda_work(n)
        b2, f2 = _moe_work("lite", n, weights, "f32")
        by += w * 2 + b1 + b2
        fl += 2 * n * w + f1 + f2
    return by + VOCAB * H * 2 + VOCAB * 2 + n * H * 2, fl + 2 * VOCAB * H


def work(case):
    kind = case["kind"]
    if kind in ("moe_decode", "moe_prefill"):
        by, fl = _moe_work(case["shape"], case["tokens"], case["weights"], case["scales"], case.get("routing", "ragged"))
    elif kind == "kda":
        by, fl = _kda_work(case["tokens"])
    elif kind == "mla":
        by, fl = _mla_work(case["tokens"], case["pos"])
    elif kind in ("step", "prompt"):
        by, fl = _thinker_work(case.get("tokens", 1), case["pos"], case["weights"])
    elif kind == "talker":
        t = TALKER
        hd = t["hidden"] // t["heads"]
        w = t["hidden"] * hd * (2 * t["heads"] + 2 * t["kv_heads"]) + 3 * t["hidden"] * t["inter"]
        kv = 2 * t["kv_heads"] * (case["pos"] + 2) * hd
        by, fl = t["layers"] * (w + kv) * 2, t["layers"] * (2 * w + 4 * t["heads"] * hd * (case["pos"] + 1))
    else:
        c = TAIL
        blk = c["dim"] * (4 * c["dim"] + 2 * c["mlp"])
        one = c["depth"] * blk + 2 * c["dim"] * c["latent"]
        by = (one + c["agg"] * blk + 2 * c["dim"] * TALKER["hidden"]) * 2
        fl = 2 * (case["steps"] * 6 * one + 2 * c["agg"] * blk)
    return {"bytes": int(by), "flops": int(fl)}


def tolerance(case):
    # About four times the error against exact() (bf16 results of one layer 0.002-0.003 off it, their fp32 state 3e-7).
    # Blocks and models are further off it where a 16-bit rounding moves a router score past the next one: up to
    # 0.013 (a prompt's block), 0.016 (a prompt's states) and 0.017 (the Talker's 24 layers).
    return {"moe_decode": {"rel": 0.01, "max": 0.2}, "moe_prefill": {"rel": 0.02, "max": 0.5},
            "kda": {"rel": 0.007, "max": 0.2}, "mla": {"rel": 0.008, "max": 0.2}, "step": {"rel": 0.03, "max": 0.5},
            "prompt": {"rel": 0.03, "max": 0.5}, "talker": {"rel": 0.03, "max": 0.5},
            "tail": {"rel": 0.024, "max": 0.5}}[case["kind"]]


# --------------------------------------------------------------------------------------------- the same in 64 bits

def _rms64(x, w, eps=EPS):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _route64(b, xn):
    logits = xn @ b["w32"].double().t()
    n, E = logits.shape
    if b["scoring"] == "softmax":
        score = torch.softmax(logits + b["bias"].double(), -1)
        key = logits + b["bias"].double()
    else:
        score = torch.sigmoid(logits)
        key = score + b["bias"].double()
        if b["n_group"] > 1:
            g = key.view(n, b["n_group"], -1).topk(2, -1).values.sum(-1).topk(b["topk_group"], -1).indices
            kept = torch.zeros(n, b["n_group"], dtype=torch.bool, device=DEV).scatter_(1, g, True)
            key = key.masked_fill(~kept.repeat_interleave(E // b["n_group"], 1), -math.inf)
    ids = key.topk(b["top_k"], -1).indices
    w = score.gather(1, ids)
    w = w / (w.sum(-1, keepdim=True) + 1e-20) * b["scale"]
    shared = torch.full((n, 1), E, device=DEV)
    return logits, torch.cat([ids, shared], 1), torch.cat([w, torch.ones(n, 1, device=DEV, dtype=F64)], 1)


def _moe64(b, x):
    """One MoE block with its norm and residual on x (64 bits): (y, weights, logits)."""
    xn = _rms64(x, b["norm_w"])
    logits, ids, w = _route64(b, xn)
    y = x.clone()
    for e in range(b["E"] + 1):
        t, k = (ids == e).nonzero(as_tuple=True)
        if not t.numel():
            continue
        gu, dn = b["w_gu"][e].double(), b["w_d"][e].double()
        if b["s_gu"] is not None:
            gu, dn = gu * b["s_gu"][e].double()[:, None], dn * b["s_d"][e].double()[:, None]
        h = xn[t] @ gu.t()
        a = F.silu(h[:, :b["I"]]) * h[:, b["I"]:]
        y.index_add_(0, t, w[t, k][:, None] * (a @ dn.t()))
    return y, w, logits


def _kda64(q, k, v, f, beta, A_log, dt_bias, state, bound=None):
    """q, k, f [T, heads, K], v [T, heads, V], beta logits [T, heads], state [heads, K, V]: (outputs, last state)."""
    q, k = (x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6) for x in (q, k))
    q = q * KDIM ** -0.5
    x, a = f + dt_bias.double().view(HEADS, KDIM), A_log.double().exp()[:, None]
    decay = torch.exp(-a * F.softplus(x) if bound is None else bound * torch.sigmoid(a * x))
    beta, S, o = torch.sigmoid(beta), state.double().clone(), []
    for t in range(q.shape[0]):
        S = S * decay[t][:, :, None]
        u = beta[t][:, None] * (v[t] - (k[t][:, None] @ S)[:, 0])
        S = S + k[t][:, :, None] * u[:, None]
        o.append((q[t][:, None] @ S)[:, 0])
    return torch.stack(o), S


def _mla64(q, k, v, kc, vc, pos):
    """T tokens of [heads * d] rows over caches whose rows pos .. pos + T - 1 they fill: (outputs, caches)."""
    T = q.shape[0]
    kc, vc = kc.clone(), vc.clone()
    kc[0, :, pos:pos + T] = k.view(T, HEADS, MLA_QK).transpose(0, 1).to(BF)
    vc[0, :, pos:pos + T] = v.view(T, HEADS, MLA_V).transpose(0, 1).to(BF)
    out = torch.empty(T, HEADS, MLA_V, device=DEV, dtype=F64)
    hidden = torch.arange(pos + T, device=DEV)[None] > pos + torch.arange(T, device=DEV)[:, None]
    for h in range(HEADS):
        s = q.view(T, HEADS, MLA_QK)[:, h] @ kc[0, h, :pos + T].double().t() * MLA_QK ** -0.5
        out[:, h] = torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ vc[0, h, :pos + T].double()
    return out.view(T, -1), kc, vc


def _conv64(x, cache, w):
    """Causal depthwise convolution over [T, C] behind the cache's last inputs, SiLU: (y, the cache after it)."""
    win = torch.cat([cache[0].double().t()[1:], x], 0)
    y = sum(win[j:j + x.shape[0]] * w[:, 0, j].double() for j in range(WINDOW))
    return F.silu(y), torch.cat([cache[0].double().t(), x], 0)[-WINDOW:].t()[None]


def _thinker64(t, h, pos):
    """T rows h through the thinker's layers: (the last row's logits, the updated state in _thinker_state's order)."""
    state, T = [], h.shape[0]
    for p in t["layers"]:
        x = _rms64(h, p["ln1"])
        q, k, v = (x @ p[n].double().t() for n in ("wq", "wk", "wv"))
        if p["kind"] == "mla":
            o, kc, vc = _mla64(q, k, v, p["kc"], p["vc"], pos)
            state += [kc, vc]
        else:
            y, conv = zip(*(_conv64(r, c, w) for r, c, w in zip((q, k, v), p["conv"], p["cw"])))
            f, g = (x @ p[a].double().t() @ p[b].double().t() for a, b in (("fa", "fb"), ("ga", "gb")))
            o, S = _kda64(*(r.view(T, HEADS, -1) for r in y), f.view(T, HEADS, KDIM), x @ p["wb"].double().t(),
                          p["A_log"], p["dt_bias"], p["state"][0])
            o = (_rms64(o, p["o_norm"], 1e-5) * torch.sigmoid(g.view(T, HEADS, VDIM))).view(T, -1)
            state += [S[None], *conv]
        h = _moe64(p["blk"], h + o @ p["wo"].double().t())[0]
    return _rms64(h[-1:], t["norm"]) @ t["head"].double().t(), state


def _talker64(s, x, pos):
    nh, nkv, hd = s.nh, s.nkv, s.hd
    ang = pos * torch.cat([s.inv_freq, s.inv_freq]).double()
    h, kc, vc = x.double().view(1, -1), s.k.clone(), s.v.clone()

    def rot(r):
        return r * ang.cos() + torch.cat([-r[:, hd // 2:], r[:, :hd // 2]], 1) * ang.sin()
    for i, layer in enumerate(s.m.layers):
        at, mlp = layer.self_attn, layer.mlp
        xn = _rms64(h, layer.input_layernorm.weight)
        q, k, v = ((xn @ p.weight.double().t() + p.bias.double()).view(-1, hd) for p in (at.q_proj, at.k_proj, at.v_proj))
        kc[i, 0, :, pos], vc[i, 0, :, pos] = rot(k).to(BF), v.to(BF)
        K, V = (c[i, 0, :, :pos + 1].double().repeat_interleave(nh // nkv, 0) for c in (kc, vc))
        a = torch.softmax((K @ rot(q)[:, :, None])[..., 0] * hd ** -0.5, -1)
        h = h + (a[:, None] @ V).reshape(1, -1) @ at.o_proj.weight.double().t()
        xn = _rms64(h, layer.post_attention_layernorm.weight)
        act = F.silu(xn @ mlp.gate_proj.weight.double().t()) * (xn @ mlp.up_proj.weight.double().t())
        h = h + act @ mlp.down_proj.weight.double().t()
    return _rms64(h, s.m.norm.weight).view(1, 1, -1), kc, vc


def _tail64(m, steps):
    def lin(x, p):
        return x @ p.weight.double().t() + p.bias.double()

    def blocks(h, blks):
        B, S, D = h.shape
        for b in blks:
            at, hd = b.attn, D // b.attn.heads
            x = _rms64(h, b.norm1.weight)
            q, k, v = (lin(x, p).view(B, S, at.heads, hd).transpose(1, 2) for p in (at.to_q, at.to_k, at.to_v))
            ang = torch.arange(S, device=DEV, dtype=F64)[:, None] * _Rotary(hd).inv.double()[None]
            rot = torch.polar(torch.ones_like(ang), ang)
            q, k = (torch.view_as_real(torch.view_as_complex(r.reshape(B, at.heads, S, hd // 2, 2)) * rot).flatten(-2)
                    for r in (q, k))
            p = torch.softmax(q @ k.transpose(-1, -2) * hd ** -0.5, -1)
            h = h + lin((p @ v).transpose(1, 2).reshape(B, S, D), at.to_out[0])
            ff = b.mlp.ff
            h = h + lin(F.gelu(lin(_rms64(h, b.norm2.weight), ff[0][0]), approximate="tanh"), ff[2])
        return h
    t = m["talker"].t
    dit, agg = t.cfm.model, t.aggregator
    hid = m["hidden"].double().view(1, -1)
    cond = torch.cat([lin(hid, dit.c_embedder.cond_embedder), dit.c_embedder.cond_embedder.bias.double()[None]])
    hist = lin(m["hist"].double().view(1, -1), dit.x_embedder).expand(2, -1)
    y = m["noise"].double().view(1, -1)
    for i in range(steps):
        h = torch.stack([cond + m["temb"][i].double(), hist, lin(y, dit.x_embedder).expand(2, -1)], 1)
        o = lin(_rms64(blocks(h, dit.blocks)[:, -1], dit.final_layer.norm_final.weight), dit.final_layer.linear)
        y = y + (o[:1] + (o[:1] - o[1:]) * 2.0) * m["dts"][i].double()
    a = blocks(torch.stack([m["cls"].double().view(1, -1), lin(y, agg.x_embedder)], 1), agg.blocks)
    nxt = lin(_rms64(a[:, 0], agg.final_layer.norm_final.weight), agg.final_layer.linear)
    return y.view(1, 1, -1), nxt.view(1, 1, -1), torch.softmax(lin(hid, t.stop_head), -1)[0, 1]


def exact(case, seed):
    kind, d = case["kind"], _Draw(seed)
    if kind in ("moe_decode", "moe_prefill"):
        b = _block(d, case["shape"], case["weights"], case["scales"], case.get("routing", "ragged"))
        y, w, logits = _moe64(b, d.normal(case["tokens"], b["H"]).double())
        return y, None, w, logits
    if kind == "kda":
        s = _kda_inputs(d, case["tokens"])
        o, S = _kda64(*(s[n][0].double() for n in ("q", "k", "v", "g", "beta")), s["A_log"], s["dt_bias"], s["state"][0],
                      case["bound"] or None)
        return o[None], S[None]
    if kind == "mla":
        s = _mla_inputs(d, case["tokens"], case["pos"])
        return _mla64(s["q"].double(), s["k"].double(), s["v"].double(), s["kc"], s["vc"], case["pos"])
    if kind in ("step", "prompt"):
        t = _thinker(d, case["pos"], case["weights"])
        if kind == "step":
            ids = t["tok"].view(1)
        else:
            ids = d.ints(VOCAB, case["bucket"])[:case["tokens"]]
        logits, state = _thinker64(t, t["embed"][ids].double(), case["pos"])
        if kind == "prompt":  # the cache rows of the padding hold what the padding gives: no exact value
            state = [None if s.dtype == BF and s.dim() == 4 else s for s in state]
        return [logits, *state]
    if kind == "talker":
        return _talker64(*_talker(d, case["pos"])[:2], case["pos"])
    return _tail64(_tail(d, case["steps"]), case["steps"])
