"""Timed cases of the packed-training hot path, through the package's public entry points.

Every case is one call (or one forward and backward) that a training or scoring
program makes: document-masked attention, the block mask, the norms, SwiGLU, the
LM-head cross-entropy, and a whole captured training step.  Sizes come from the
benchmark configurations (packs of 256, 2048 and 8192 tokens; the 100M decoder's
768 / 12 heads / 4 KV heads / head dim 64; 32 / 8 heads of 128; [32768, 14336]
activations; the 32000- and 128256-entry vocabularies), from the tests, or are
the same with lengths that are not multiples of a tile: a batch is cut at its
longest pack, and a prompt to be scored has whatever length it has.

``exact`` restates each case in float64 with plain torch.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from packbalance_amd.data import workloads as W

DEV = "cuda"
_DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


# ---------------------------------------------------------------- cases
def listed() -> list[dict]:
    return [
        # The tiny fp32 model's attention (2 layers, head dim 32), one pack of 256:
        # the smallest call, forward and backward.
        dict(name="attn_tiny_f32", kind="attn", B=1, S=256, hq=4, hkv=2, d=32, dtype="f32",
             mu=48.0, sigma=0.8, lo=4, dense=False, train=True),
        # One training step's four packs of the 100M model, forward and backward.
        dict(name="attn_train_2k", kind="attn", B=4, S=2048, hq=12, hkv=4, d=64, dtype="bf16",
             mu=200.0, sigma=1.1, lo=8, dense=False, train=True),
        # Long packs at 32 / 8 heads of 128, the first pack one whole document.
        dict(name="attn_train_8k", kind="attn", B=8, S=8192, hq=32, hkv=8, d=128, dtype="bf16",
             mu=512.0, sigma=1.0, lo=16, dense=True, train=True),
        # The 100M model fine-tuned on a batch cut at its longest pack.
        dict(name="attn_train_ragged", kind="attn", B=4, S=1999, hq=12, hkv=4, d=64,
             dtype="bf16", mu=200.0, sigma=1.1, lo=8, dense=False, train=True),
        # Scoring one long prompt: forward only, whatever length it has.
        dict(name="attn_score_prompt", kind="attn", B=1, S=6001, hq=32, hkv=8, d=128,
             dtype="bf16", mu=512.0, sigma=1.0, lo=16, dense=True, train=False),
        # The FlexAttention block mask of one 8192-token pack for 32 heads.
        dict(name="block_mask_8k", kind="mask", S=8192, heads=32, block=128, mu=512.0,
             sigma=1.0, lo=16),
        # The residual add + norm of a decoder layer at width 4096, one 8192-token pack:
        # fp32 residual stream, bf16 sublayer output and norm output.
        dict(name="add_norm_4k", kind="addnorm", rows=8192, n=4096, out="bf16"),
        # The final / layer norm of a wide decoder, bf16 activations.
        dict(name="rmsnorm_wide", kind="norm", rows=8192, n=8192, dtype="bf16"),
        # SwiGLU at [32768, 14336] bf16.
        dict(name="swiglu_mlp", kind="swiglu", rows=32768, n=14336, dtype="bf16"),
        # LM-head CE of a 135M-class model (d 576, vocabulary 49152) on a batch cut
        # at its longest sequence.
        dict(name="lm_ce_small", kind="ce", n=2999, d=576, v=49152, dtype="bf16"),
        # LM-head CE at 16384 tokens, d 4096, vocabulary 128256.
        dict(name="lm_ce_large", kind="ce", n=16384, d=4096, v=128256, dtype="bf16"),
        # One training step of the 100M model: four packs of 2048 built on the device,
        # forward, backward, clip and AdamW, replayed from its captured graph.
        dict(name="train_step_100m", kind="step", layers=12, dm=768, hq=12, hkv=4, ff=2048,
             v=32000, S=2048, packs=4, mu=200.0, sigma=1.1, lo=8),
    ]


def _log(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["attn", "attn", "attn", "attn_f32", "mask", "addnorm", "norm", "swiglu",
                       "ce", "ce", "step"])
    docs = dict(mu=float(_log(rng, 64, 1024)), sigma=round(rng.uniform(0.6, 1.3), 2), lo=8)
    if kind == "attn":
        hq, hkv, d = rng.choice([(12, 4, 64), (9, 3, 64), (16, 16, 64), (16, 4, 64), (32, 8, 128),
                                 (16, 4, 128), (8, 8, 128), (12, 6, 96)])
        S = _log(rng, 500, 8192)
        if rng.random() < 0.35:
            S = max(512, S // 64 * 64)
        B = rng.randint(1, max(1, min(8, 65536 // S)))
        return dict(kind="attn", B=B, S=S, hq=hq, hkv=hkv, d=d, dtype="bf16",
                    dense=rng.random() < 0.3, train=rng.random() < 0.75, **docs)
    if kind == "attn_f32":
        hq, hkv, d = rng.choice([(4, 2, 32), (12, 4, 64), (8, 2, 128)])
        return dict(kind="attn", B=rng.randint(1, 3), S=_log(rng, 200, 2048), hq=hq, hkv=hkv, d=d,
                    dtype="f32", dense=False, train=True, **docs)
    if kind == "mask":
        S = _log(rng, 1500, 16384)
        return dict(kind="mask", S=S, heads=rng.choice([4, 12, 32]), block=128,
                    mu=min(docs["mu"], S / 8.0), sigma=docs["sigma"], lo=docs["lo"])
    if kind == "addnorm":
        return dict(kind="addnorm", rows=_log(rng, 256, 32768),
                    n=rng.choice([576, 768, 1024, 2048, 3072, 4096, 5120]),
                    out=rng.choice(["bf16", "bf16", "f32"]))
    if kind == "norm":
        dtype = rng.choice(["bf16", "bf16", "f32"])
        return dict(kind="norm", rows=_log(rng, 256, 32768),
                    n=rng.choice([576, 768, 1024, 2048, 4096, 5120, 6144, 8192]), dtype=dtype)
    if kind == "swiglu":
        return dict(kind="swiglu", rows=_log(rng, 256, 32768),
                    n=rng.choice([344, 1536, 2048, 3333, 8192, 14336]),
                    dtype=rng.choice(["bf16", "bf16", "f32"]))
    if kind == "ce":
        d, v = rng.choice([(576, 49152), (768, 32000), (768, 50257), (1000, 32000),
                           (2048, 128256), (4096, 32000), (4096, 128256)])
        return dict(kind="ce", n=_log(rng, 500, 16384), d=d, v=v, dtype="bf16")
    S = rng.choice([512, 1024, 2048])
    return dict(kind="step", layers=rng.choice([2, 4, 8, 12]), dm=768, hq=12, hkv=4, ff=2048,
                v=32000, S=S, packs=4, mu=min(docs["mu"], S / 4.0), sigma=docs["sigma"],
                lo=docs["lo"])


# ---------------------------------------------------------------- inputs
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, dtype=torch.float32, scale=1.0, mean=0.0):
    t = torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)
    return t.mul_(scale).add_(mean).to(dtype)


def _packs(case: dict, n_packs: int, seed: int) -> list[list[int]]:
    """Document lengths of each pack: lognormal, filling the sequence; with ``dense``
    the first pack is one document.  The shape of a case's work is the same for
    every seed (the lengths come from the case), only the values differ."""
    S = case["S"]
    rng = np.random.default_rng(1000 + S)
    packs = []
    for i in range(n_packs):
        if i == 0 and case.get("dense"):
            packs.append([S])
        else:
            packs.append(W.fill_sequential(rng, S, math.log(case["mu"]), case["sigma"],
                                           min(case["lo"], S), S))
    # which pack of the batch is which depends on the seed
    order = np.random.default_rng(seed).permutation(n_packs)
    return [packs[i] for i in order]


def _attn_inputs(case, seed):
    g = _gen(seed)
    dt = _DTYPES[case["dtype"]]
    B, S, hq, hkv, d = (case[k] for k in ("B", "S", "hq", "hkv", "d"))

    def heads(h):  # the model's [B, S, H, D] memory seen as [B, H, S, D]
        return _randn(g, B, S, h, d, dtype=dt).transpose(1, 2)

    q, k, v, do = heads(hq), heads(hkv), heads(hkv), heads(hq)
    packs = _packs(case, B, seed)
    return q, k, v, do, W.doc_ids_from_lengths(packs, S).to(DEV), packs


def _mask_inputs(case, seed):
    """One pack's document ids [1, S], its documents drawn from the seed."""
    S = case["S"]
    lens = W.fill_sequential(np.random.default_rng(seed), S, math.log(case["mu"]), case["sigma"],
                             min(case["lo"], S), S)
    return W.doc_ids_from_lengths([lens], S).to(DEV)


def _ce_inputs(case, seed):
    g = _gen(seed)
    dt = _DTYPES[case["dtype"]]
    x = _randn(g, case["n"], case["d"], dtype=dt)
    w = _randn(g, case["v"], case["d"], dtype=dt, scale=0.02)
    t = torch.randint(0, case["v"], (case["n"],), generator=g, device=DEV)
    t[torch.rand(case["n"], generator=g, device=DEV) < 0.01] = -100
    return x, w, t


def _addnorm_inputs(case, seed):
    g = _gen(seed)
    r, n = case["rows"], case["n"]
    out = _DTYPES[case["out"]]
    return (_randn(g, r, n), _randn(g, r, n, dtype=out), _randn(g, n, scale=0.1, mean=1.0),
            _randn(g, r, n, scale=0.5), _randn(g, r, n, dtype=out))


def _norm_inputs(case, seed):
    g = _gen(seed)
    r, n, dt = case["rows"], case["n"], _DTYPES[case["dtype"]]
    return (_randn(g, r, n, dtype=dt), _randn(g, n, dtype=dt, scale=0.1, mean=1.0),
            _randn(g, r, n, dtype=dt))


def _swiglu_inputs(case, seed):
    g = _gen(seed)
    r, n, dt = case["rows"], case["n"], _DTYPES[case["dtype"]]
    return tuple(_randn(g, r, n, dtype=dt) for _ in range(3))


EPS = 1e-5
THETA = 10000.0


def _step_shapes(case) -> dict[str, tuple[int, ...]]:
    dm, ff, hd = case["dm"], case["ff"], case["dm"] // case["hq"]
    s = {"embed_tokens.weight": (case["v"], dm)}
    for i in range(case["layers"]):
        p = f"layers.{i}."
        s[p + "input_layernorm.weight"] = (dm,)
        s[p + "self_attn.q_proj.weight"] = (case["hq"] * hd, dm)
        s[p + "self_attn.k_proj.weight"] = (case["hkv"] * hd, dm)
        s[p + "self_attn.v_proj.weight"] = (case["hkv"] * hd, dm)
        s[p + "self_attn.o_proj.weight"] = (dm, case["hq"] * hd)
        s[p + "post_attention_layernorm.weight"] = (dm,)
        s[p + "mlp.gate_proj.weight"] = (ff, dm)
        s[p + "mlp.up_proj.weight"] = (ff, dm)
        s[p + "mlp.down_proj.weight"] = (dm, ff)
    s["norm.weight"] = (dm,)
    return s


def _step_inputs(case, seed):
    """Weights by parameter name, the corpus, and the step's packs as (start, length) lists."""
    g = _gen(seed)
    deep = 1.0 / math.sqrt(2 * case["layers"])
    w = {}
    for name, shape in _step_shapes(case).items():
        if len(shape) == 1:
            w[name] = _randn(g, *shape, scale=0.02, mean=1.0)
        else:
            out = name.endswith(("o_proj.weight", "down_proj.weight"))
            w[name] = _randn(g, *shape, scale=0.02 * (deep if out else 1.0))
    lens = _packs(case, case["packs"], seed)
    rng = np.random.default_rng(seed)
    corpus = rng.integers(0, case["v"], size=sum(map(sum, lens))).astype(np.uint32)
    packs, pos = [], 0
    for p in lens:
        packs.append([(pos + sum(p[:i]), n) for i, n in enumerate(p)])
        pos += sum(p)
    return w, corpus, packs


# ---------------------------------------------------------------- prepare / run
def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "attn":
        from packbalance_amd.model.attention import DocPlans, attention_forward

        q, k, v, do, doc, _ = _attn_inputs(case, seed)
        if case["train"]:
            q, k, v = (t.requires_grad_(True) for t in (q, k, v))
        return dict(kind=kind, train=case["train"], fn=attention_forward, q=q, k=k, v=v, do=do,
                    doc=doc, mask=DocPlans(doc))
    if kind == "mask":
        from packbalance_amd.model.attention import build_doc_block_mask

        return dict(kind=kind, fn=build_doc_block_mask, doc=_mask_inputs(case, seed),
                    heads=case["heads"], block=case["block"])
    if kind == "addnorm":
        from packbalance_amd.kernels.rmsnorm import add_rmsnorm

        x, delta, w, dh, dy = _addnorm_inputs(case, seed)
        x, delta, w = (t.requires_grad_(True) for t in (x, delta, w))
        return dict(kind=kind, fn=add_rmsnorm, x=x, delta=delta, w=w, dh=dh, dy=dy,
                    out=_DTYPES[case["out"]])
    if kind == "norm":
        from packbalance_amd.kernels.rmsnorm import rmsnorm

        x, w, dy = _norm_inputs(case, seed)
        return dict(kind=kind, fn=rmsnorm, x=x.requires_grad_(True), w=w.requires_grad_(True),
                    dy=dy)
    if kind == "swiglu":
        from packbalance_amd.kernels.swiglu import swiglu

        g, u, dy = _swiglu_inputs(case, seed)
        return dict(kind=kind, fn=swiglu, g=g.requires_grad_(True), u=u.requires_grad_(True),
                    dy=dy)
    if kind == "ce":
        from packbalance_amd.kernels.fused_ce import linear_cross_entropy

        x, w, t = _ce_inputs(case, seed)
        return dict(kind=kind, fn=linear_cross_entropy, x=x.requires_grad_(True),
                    w=w.requires_grad_(True), t=t)
    from packbalance_amd.data.device_packs import DeviceTokenStore
    from packbalance_amd.model.llama import ModelConfig
    from packbalance_amd.model.step import TrainStep

    w, corpus, packs = _step_inputs(case, seed)
    cfg = ModelConfig(vocab_size=case["v"], d_model=case["dm"], n_layers=case["layers"],
                      n_heads=case["hq"], n_kv_heads=case["hkv"], d_ff=case["ff"],
                      max_seq_len=case["S"], rope_theta=THETA, norm_eps=EPS)
    # Learning rate 0 is the first step of a linear warm-up: the whole update runs,
    # and every replay of the step sees the same weights.
    ts = TrainStep(cfg, torch.device(DEV), packs_per_step=case["packs"], seq_len=case["S"],
                   lr=0.0, store=DeviceTokenStore(corpus, DEV), streams=2,
                   packs_per_micro_batch=2)
    with torch.no_grad():
        for name, p in ts.model.named_parameters():
            p.copy_(w[name])
    ts.flat.invalidate()
    ts.capture_packs(packs)
    return dict(kind=kind, ts=ts, packs=packs)


def run(state: dict):
    kind = state["kind"]
    if kind == "attn":
        q, k, v = state["q"], state["k"], state["v"]
        if not state["train"]:
            with torch.no_grad():
                return state["fn"](q, k, v, state["doc"], block_mask=state["mask"])
        out = state["fn"](q, k, v, state["doc"], block_mask=state["mask"])
        return (out.detach(),) + torch.autograd.grad(out, (q, k, v), state["do"])
    if kind == "mask":
        m = state["fn"](state["doc"], state["heads"], state["block"])
        return {t: getattr(m, t) for t in _TABLES}
    if kind == "addnorm":
        x, d, w = state["x"], state["delta"], state["w"]
        h, y = state["fn"](x, d, w, EPS, state["out"])
        return (h.detach(), y.detach()) + torch.autograd.grad((h, y), (x, d, w),
                                                              (state["dh"], state["dy"]))
    if kind == "norm":
        y = state["fn"](state["x"], state["w"], EPS)
        return (y.detach(),) + torch.autograd.grad(y, (state["x"], state["w"]), state["dy"])
    if kind == "swiglu":
        y = state["fn"](state["g"], state["u"])
        return (y.detach(),) + torch.autograd.grad(y, (state["g"], state["u"]), state["dy"])
    if kind == "ce":
        loss = state["fn"](state["x"], state["w"], state["t"])
        return (loss.detach(),) + torch.autograd.grad(loss, (state["x"], state["w"]))
    ts = state["ts"]
    ts.replay_packs(state["packs"])
    # the step's whole gradient: every parameter's, in registration order
    return {"loss": ts.loss_sum, "grad_norm": ts.grad_norm, "grad": ts.flat.grad}


_TABLES = ("kv_num_blocks", "kv_indices", "full_kv_num_blocks", "full_kv_indices",
           "q_num_blocks", "q_indices", "full_q_num_blocks", "full_q_indices")


# ---------------------------------------------------------------- what a pass cannot do without
def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "attn":
        e = 2 if case["dtype"] == "bf16" else 4
        B, S, hq, hkv, d = (case[k] for k in ("B", "S", "hq", "hkv", "d"))
        pairs = W.attention_pairs(_packs(case, B, 0))
        qb, kb = B * S * hq * d * e, B * S * hkv * d * e
        if not case["train"]:
            return dict(bytes=2 * qb + 2 * kb + 8 * B * S, flops=4.0 * d * hq * pairs)
        # forward: q, k, v -> out; backward: q, k, v, out, do -> dq, dk, dv
        return dict(bytes=6 * qb + 6 * kb + 8 * B * S, flops=12.0 * d * hq * pairs)
    if kind == "mask":
        nb = -(-case["S"] // case["block"])
        return dict(bytes=8 * case["S"] + 4 * case["heads"] * (4 * nb * nb + 4 * nb), flops=0.0)
    if kind == "addnorm":
        e, o = case["rows"] * case["n"], 2 if case["out"] == "bf16" else 4
        # forward x, delta -> h, y; backward h, dh, dy -> dx, ddelta
        return dict(bytes=e * (4 + o + 4 + o + 4 + 4 + o + 4 + o), flops=12.0 * e)
    if kind in ("norm", "swiglu"):
        e = case["rows"] * case["n"] * (2 if case["dtype"] == "bf16" else 4)
        return dict(bytes=(5 if kind == "norm" else 8) * e,
                    flops=15.0 * case["rows"] * case["n"])
    if kind == "ce":
        n, d, v = case["n"], case["d"], case["v"]
        return dict(bytes=2.0 * (3 * n * d + 3 * v * d) + 8 * n, flops=6.0 * n * d * v)
    hd = case["dm"] // case["hq"]
    per_layer = case["dm"] * hd * (2 * case["hq"] + 2 * case["hkv"]) + 3 * case["dm"] * case["ff"]
    mats = case["layers"] * per_layer + case["v"] * case["dm"]
    lens = _packs(case, case["packs"], 0)
    tokens = sum(map(sum, lens))
    return dict(bytes=34.0 * mats,  # the optimizer's own traffic
                flops=6.0 * mats * tokens
                + 12.0 * hd * case["hq"] * case["layers"] * W.attention_pairs(lens))


def tolerance(case: dict):
    """About four times the 2-norm error against ``exact`` that these paths show (bf16
    attention 3.0e-3, bf16 norms, SwiGLU and CE 1.7e-3, the whole step's bf16
    gradient 1.1e-2); 1e-5 for 32-bit sums."""
    kind = case["kind"]
    if kind == "mask":
        return "exact"
    if kind == "step":
        return {"rel": 4e-2}
    if case.get("dtype", case.get("out")) == "f32":
        return {"rel": 1e-5}
    return {"rel": 1.2e-2 if kind == "attn" else 7e-3}


# ---------------------------------------------------------------- float64
def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "attn":
        return _exact_attn(case, seed)
    if kind == "mask":
        return _exact_mask(case, seed)
    if kind == "addnorm":
        x, d, w, dh, dy = (t.double() for t in _addnorm_inputs(case, seed))
        h = x + d
        y, dn, dw = _norm64(h, w, dy)
        return h, y, dn + dh, dn + dh, dw
    if kind == "norm":
        x, w, dy = (t.double() for t in _norm_inputs(case, seed))
        return _norm64(x, w, dy)
    if kind == "swiglu":
        g, u, dy = (t.double() for t in _swiglu_inputs(case, seed))
        s = torch.sigmoid(g)
        return g * s * u, dy * u * s * (1 + g * (1 - s)), dy * g * s
    if kind == "ce":
        return _exact_ce(case, seed)
    return _exact_step(case, seed)


def _norm64(x, w, dy):
    r = torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS)
    xh = x * r
    g = dy * w
    return xh * w, r * (g - xh * (g * xh).mean(-1, keepdim=True)), (dy * xh).sum(0)


def _attn64(q, k, v, do=None):
    """One document: q [G, L, D], k / v [L, D] -> out, and with ``do`` dq, dk, dv."""
    L = q.shape[-2]
    sc = 1.0 / math.sqrt(q.shape[-1])
    s = torch.matmul(q, k.t()).mul_(sc)
    s.masked_fill_(torch.ones(L, L, dtype=torch.bool, device=q.device).triu_(1), -math.inf)
    p = torch.softmax(s, -1)
    out = torch.matmul(p, v)
    if do is None:
        return (out,)
    dp = torch.matmul(do, v.t())
    ds = p * (dp - (do * out).sum(-1, keepdim=True))
    g = q.shape[0] * L
    dk = torch.mm(ds.reshape(g, L).t().contiguous(), q.reshape(g, -1)).mul_(sc)
    dv = torch.mm(p.reshape(g, L).t().contiguous(), do.reshape(g, -1))
    return out, torch.matmul(ds, k).mul_(sc), dk, dv


def _exact_attn(case, seed):
    q, k, v, do, _, packs = _attn_inputs(case, seed)
    G = case["hq"] // case["hkv"]
    outs = [torch.zeros(q.shape, dtype=torch.float64, device=DEV)]
    if case["train"]:
        outs += [torch.zeros(t.shape, dtype=torch.float64, device=DEV) for t in (q, k, v)]
    for b, lens in enumerate(packs):
        o = 0
        for n in lens:
            for h in range(case["hkv"]):
                hs = slice(h * G, (h + 1) * G)
                r = _attn64(q[b, hs, o:o + n].double().contiguous(),
                            k[b, h, o:o + n].double().contiguous(),
                            v[b, h, o:o + n].double().contiguous(),
                            do[b, hs, o:o + n].double().contiguous() if case["train"] else None)
                outs[0][b, hs, o:o + n] = r[0]
                if case["train"]:
                    outs[1][b, hs, o:o + n] = r[1]
                    outs[2][b, h, o:o + n] = r[2]
                    outs[3][b, h, o:o + n] = r[3]
            o += n
    return tuple(outs) if case["train"] else outs[0]


def _exact_mask(case, seed):
    doc = _mask_inputs(case, seed)[0]
    S, H = case["S"], case["heads"]
    bs = min(case["block"], max(32, 1 << max(0, S - 1).bit_length()))
    nb = -(-S // bs)
    allowed = torch.zeros(nb * bs, nb * bs, dtype=torch.bool, device=DEV)
    pos = torch.arange(S, device=DEV)
    allowed[:S, :S] = (doc[:, None] == doc[None]) & (pos[:, None] >= pos[None])
    cnt = allowed.view(nb, bs, nb, bs).sum((1, 3))
    full = cnt == bs * bs
    part = (cnt > 0) & ~full
    out = {}
    for kv, fkv, p, f in (("kv", "full_kv", part, full), ("q", "full_q", part.t(), full.t())):
        for name, m in ((kv, p), (fkv, f)):
            m = m.contiguous()
            idx = torch.argsort(m.to(torch.int32), dim=-1, descending=True, stable=True)
            out[name + "_num_blocks"] = m.sum(-1).to(torch.int32).expand(1, H, nb).contiguous()
            out[name + "_indices"] = idx.to(torch.int32).expand(1, H, nb, nb).contiguous()
    return out


def _ce64(x, w, t, dw=None):
    """Summed CE and its gradients, token rows in chunks (x, w float64)."""
    dx = torch.empty_like(x)
    dw = torch.zeros_like(w) if dw is None else dw
    total = torch.zeros((), dtype=torch.float64, device=x.device)
    for r0 in range(0, x.shape[0], 2048):
        xs, ts = x[r0:r0 + 2048], t[r0:r0 + 2048]
        p = torch.mm(xs, w.t())
        lse = torch.logsumexp(p, -1)
        ok = ts != -100
        tt = torch.where(ok, ts, torch.zeros_like(ts))[:, None]
        total += ((lse - p.gather(1, tt)[:, 0]) * ok).sum()
        p.sub_(lse[:, None]).exp_().scatter_add_(1, tt, -torch.ones_like(lse)[:, None])
        p.mul_(ok[:, None])
        dx[r0:r0 + 2048] = torch.mm(p, w)
        dw.addmm_(p.t(), xs)
    return total, dx, dw


def _exact_ce(case, seed):
    x, w, t = _ce_inputs(case, seed)
    return _ce64(x.double(), w.double(), t)


def _rope64(x, c, s):
    h = x.shape[-1] // 2
    x1, x2 = x[..., :h], x[..., h:]
    return torch.cat((x1 * c - x2 * s, x2 * c + x1 * s), -1)


def _exact_step(case, seed):
    w, corpus, packs = _step_inputs(case, seed)
    w = {k: t.double().requires_grad_(True) for k, t in w.items()}
    hd, hq, hkv = case["dm"] // case["hq"], case["hq"], case["hkv"]
    G = hq // hkv
    tokens = sum(n for p in packs for _, n in p)
    inv = 1.0 / THETA ** (torch.arange(0, hd, 2, dtype=torch.float64, device=DEV) / hd)

    def norm(x, g):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * g

    ids = torch.from_numpy(corpus.astype(np.int64)).to(DEV)
    loss_sum = 0.0
    for pack in packs:
        toks = torch.cat([ids[a:a + n] for a, n in pack])
        labels = torch.cat([torch.cat((ids[a + 1:a + n], ids.new_full((1,), -100)))
                            for a, n in pack])
        pos = torch.cat([torch.arange(n, device=DEV) for _, n in pack])
        doc = torch.cat([torch.full((n,), i, device=DEV) for i, (_, n) in enumerate(pack)])
        S = toks.numel()
        at = torch.arange(S, device=DEV)
        bad = ~((doc[:, None] == doc[None]) & (at[:, None] >= at[None]))
        ang = pos[:, None].double() * inv
        c, s = ang.cos(), ang.sin()
        h = w["embed_tokens.weight"][toks]
        for i in range(case["layers"]):
            p = f"layers.{i}."
            x = norm(h, w[p + "input_layernorm.weight"])
            q, k, v = ((x @ w[p + f"self_attn.{n}_proj.weight"].t()).view(S, -1, hd).transpose(0, 1)
                       for n in "qkv")
            q, k = _rope64(q, c, s), _rope64(k, c, s)
            k, v = (t.repeat_interleave(G, 0).contiguous() for t in (k, v))
            a = torch.matmul(q.contiguous(), k.transpose(1, 2).contiguous()) / math.sqrt(hd)
            o = torch.matmul(torch.softmax(a.masked_fill(bad, -math.inf), -1), v)
            h = h + o.transpose(0, 1).reshape(S, -1) @ w[p + "self_attn.o_proj.weight"].t()
            x = norm(h, w[p + "post_attention_layernorm.weight"])
            g = x @ w[p + "mlp.gate_proj.weight"].t()
            u = x @ w[p + "mlp.up_proj.weight"].t()
            h = h + (torch.nn.functional.silu(g) * u) @ w[p + "mlp.down_proj.weight"].t()
        y = norm(h, w["norm.weight"])
        lg = y @ w["embed_tokens.weight"].t()
        loss = torch.nn.functional.cross_entropy(lg, labels, ignore_index=-100, reduction="sum")
        (loss / tokens).backward()
        loss_sum += loss.detach()
    # Parameters sit back to back in the store: every size is a multiple of its alignment.
    grad = torch.cat([t.grad.reshape(-1) for t in w.values()])
    return {"loss": loss_sum, "grad_norm": grad.pow(2).sum().sqrt(), "grad": grad}
