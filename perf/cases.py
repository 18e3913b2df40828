"""The work a program does with this framework, as cases that can be timed and checked.

A case is a dict of plain values: ``kind`` and the sizes and options of one call. ``prepare`` builds what such a program
holds before the call (seeded random weights of the model family's shapes, the cache so far, the engine or the
recorded graph), ``run`` makes one pass through the public entry points, ``exact`` is the same pass in 64-bit torch and
numpy without the package's code. Weights are N(0, 0.02) as checkpoints hold them (bf16), norms 1 + 0.1 N(0, 1), caches N(0, 1),
the shapes those of the package's 0.6B and 1.7B talkers and its code predictor.

Kinds:
  sample  a frame's 16 samplings (15 sub-codes, then code 0 with the talker processor) on ``FusedSampler``
  perop   embed -> decoder layers -> norm -> head on the per-op C entry points, one recorded graph (f32 weights, caches
          longer than the frame kernel takes, teacher forcing, callers of the C interface)
  blayer  half a batched decoder layer on the C entry points: qkv -> ragged attention -> o, or gate/up -> down
  bstep   steps of ``BatchedTalker`` (up to 16 streams at their own positions)
  frames  greedy or sampled frames of a talker fed by its own codes, one ``run_frames`` launch
  cp      a frame's sub-codes on ``CodePredictor``
  tts     ``generate_codes`` of a talker with its code predictor: the frame loop of a sentence
  prompt  ``generate_codes`` up to the first code: the prefill of a prompt
"""

from __future__ import annotations

import math
from types import SimpleNamespace as NS

import numpy as np
import torch

HD, EPS, THETA, EOS, EMB_V = 128, 1e-6, 1e6, 2150, 3072
SHAPES = {"0.6b": (1024, 3072), "1.7b": (2048, 6144)}  # hidden, intermediate; 16 q and 8 kv heads of 128 in both
NQ, NKV = 16, 8
CP = (1024, 3072)      # the code predictor's hidden and intermediate, vocabulary 2048, 5 layers
CP_V, CP_LAYERS = 2048, 5
F64 = torch.float64


# ---- cases -------------------------------------------------------------------------------------------------------
def listed() -> list[dict]:
    return [
        # the smallest calls: the reference's default settings, 16 one-block kernels in a row
        dict(name="sample_frame", kind="sample", groups=16, do_sample=True, top_k=50),
        # a single int8 decoder layer of the 0.6B talker at 257 positions: launches and latency
        dict(name="perop_06b_layer", kind="perop", shape="0.6b", wd="i8row", layers=1, pos=256, max_len=320),
        # a cache longer than the frame kernel takes at this shape, odd position, the serving weight format
        dict(name="perop_06b_long", kind="perop", shape="0.6b", wd="i8g32", layers=4, pos=1601, max_len=2048),
        # f32 weights and cache (the accuracy check's engine) run on these kernels only
        dict(name="perop_17b_f32", kind="perop", shape="1.7b", wd="f32", layers=2, pos=1023, max_len=1280),
        # sixteen ragged streams: the attention half and the MLP half of a layer
        dict(name="blayer_17b_attn", kind="blayer", part="attn", shape="1.7b", batch=16, lo=64, hi=2048),
        dict(name="blayer_17b_mlp", kind="blayer", part="mlp", shape="1.7b", batch=16, lo=0, hi=0),
        # serving sixteen streams on the 1.7B talker; a few short streams on the 0.6B talker
        dict(name="bstep_17b_16", kind="bstep", shape="1.7b", layers=8, batch=16, lo=64, hi=2048, steps=4),
        dict(name="bstep_06b_5", kind="bstep", shape="0.6b", layers=12, batch=5, lo=8, hi=200, steps=6),
        # the headline decode: 0.6B int8, KV 512, 64 greedy frames in a launch
        dict(name="frames_06b", kind="frames", shape="0.6b", wd="i8row", layers=28, pos=512, frames=64, do_sample=False),
        # the reference's default format and settings at the larger shape
        dict(name="frames_17b_bf16", kind="frames", shape="1.7b", wd="bf16", layers=8, pos=1024, frames=16, do_sample=True),
        # a sentence's frame loop with the code predictor, sampled, the serving weight format (few frames: a pick between two
        # scores within rounding of each other changes every later one)
        dict(name="tts_06b", kind="tts", shape="0.6b", wd="i8g32", layers=14, pos=41, frames=3, do_sample=True),
        # the prompt of a sentence (bf16 modules)
        dict(name="prompt_06b", kind="prompt", shape="0.6b", layers=4, rows=45),
    ]


def _log(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["sample", "perop", "perop", "blayer", "blayer", "bstep", "bstep", "frames", "frames", "cp", "tts", "prompt"])
    shape = rng.choice(["0.6b", "1.7b"])
    wd = rng.choice(["i8row", "i8g32", "bf16"])
    if kind == "sample":
        return dict(kind=kind, groups=rng.randint(2, 33), do_sample=rng.random() < 0.75, top_k=rng.choice([0, 1, 20, 50, 50, 63, 100, 400]))
    if kind == "perop":
        pos = _log(rng, 1, 4000)
        return dict(kind=kind, shape=shape, wd=rng.choice([wd, wd, "f32"]), layers=rng.randint(1, 3 if shape == "0.6b" else 2), pos=pos,
                    max_len=pos + _log(rng, 1, 1000))
    if kind == "blayer":
        part = rng.choice(["attn", "attn", "mlp"])
        hi = _log(rng, 64, 2048)
        return dict(kind=kind, part=part, shape=shape, batch=rng.randint(1, 16), lo=rng.randint(1, hi) if part == "attn" else 0,
                    hi=hi if part == "attn" else 0)
    if kind == "bstep":
        hi = _log(rng, 32, 2048)
        return dict(kind=kind, shape=shape, layers=rng.randint(2, 10) if shape == "0.6b" else rng.randint(2, 5),
                    batch=rng.choice([16, 16, rng.randint(1, 16)]), lo=rng.randint(8, hi), hi=hi, steps=rng.randint(1, 5))
    if kind == "frames":
        frames = _log(rng, 1, 40)
        top = (1024 if shape == "0.6b" else 2048) - frames - 1
        return dict(kind=kind, shape=shape, wd=wd, layers=rng.randint(2, 12) if shape == "0.6b" else rng.randint(2, 5),
                    pos=_log(rng, 1, top), frames=frames, do_sample=rng.random() < 0.5)
    if kind == "cp":
        return dict(kind=kind, wd=wd, proj=rng.random() < 0.4, positions=rng.choice([16, 16, rng.randint(3, 32)]),
                    do_sample=rng.random() < 0.5)
    if kind == "tts":
        return dict(kind=kind, shape=shape, wd=wd, layers=rng.randint(2, 8) if shape == "0.6b" else rng.randint(2, 4),
                    pos=_log(rng, 4, 900), frames=rng.randint(1, 3), do_sample=rng.random() < 0.6)
    return dict(kind=kind, shape=shape, layers=rng.randint(2, 4) if shape == "0.6b" else 2, rows=_log(rng, 6, 250))


# ---- seeded weights ------------------------------------------------------------------------------------------------
def _gen(seed: int, *tag: int) -> torch.Generator:
    s = int(seed) & 0x7FFFFFFF
    for t in tag:
        s = (s * 1000003 + t + 7919) % (1 << 62)
    return torch.Generator(device="cuda").manual_seed(s)


def _normal(g, *shape, std=1.0, mean=0.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device="cuda") * std + mean).to(dtype)


def _layer_weights(seed: int, i: int, H: int, I: int) -> dict:
    g = _gen(seed, 1, i)
    w = {k: _normal(g, n, m, std=0.02, dtype=torch.bfloat16) for k, n, m in
         (("q", NQ * HD, H), ("k", NKV * HD, H), ("v", NKV * HD, H), ("o", H, NQ * HD), ("gate", I, H), ("up", I, H), ("down", H, I))}
    for k, n in (("in_norm", H), ("post_norm", H), ("qn", HD), ("kn", HD)):
        w[k] = _normal(g, n, std=0.1, mean=1.0)
    return w


def _model_weights(seed: int, layers: int, H: int, I: int, V: int, emb: int | None = None) -> dict:
    g = _gen(seed, 2)
    return {"layers": [_layer_weights(seed, i, H, I) for i in range(layers)], "norm": _normal(g, H, std=0.1, mean=1.0),
            "head": _normal(g, V, H, std=0.02, dtype=torch.bfloat16),
            "emb": _normal(g, EMB_V, emb or H, std=0.02, dtype=torch.bfloat16), "H": H, "I": I}


def _cp_weights(seed: int, positions: int, win: int) -> dict:
    w = _model_weights(seed + 77, CP_LAYERS, CP[0], CP[1], CP_V, emb=win)
    g = _gen(seed, 3)
    w["heads"] = [_normal(g, CP_V, CP[0], std=0.02, dtype=torch.bfloat16) for _ in range(positions - 1)]
    w["cemb"] = [_normal(g, CP_V, win, std=0.02, dtype=torch.bfloat16) for _ in range(positions - 1)]
    if win != CP[0]:
        w["proj"] = _normal(g, CP[0], win, std=0.02, dtype=torch.bfloat16)
        w["proj_b"] = _normal(g, CP[0], std=0.02)
    return w


def _inv_freq() -> torch.Tensor:
    return 1.0 / THETA ** (torch.arange(0, HD, 2, dtype=torch.int64).float() / HD)


def _prior(seed: int, layers: int, T: int):
    g = _gen(seed, 4)
    return [_normal(g, layers, NKV, T, HD, dtype=torch.bfloat16) for _ in range(2)]


def _lengths(case: dict, seed: int) -> list[int]:
    r = np.random.RandomState(seed & 0x7FFFFFFF)
    return [int(t) for t in r.randint(case["lo"], case["hi"] + 1, case["batch"])]


# ---- Hugging Face-shaped objects, as the engines read them ------------------------------------------------------------
def _lin(w):
    return NS(weight=w, bias=None)


def _stack(w: dict, V: int):
    layers = [NS(self_attn=NS(q_proj=_lin(x["q"]), k_proj=_lin(x["k"]), v_proj=_lin(x["v"]), o_proj=_lin(x["o"]), q_norm=_lin(x["qn"]),
                              k_norm=_lin(x["kn"])),
                 mlp=NS(gate_proj=_lin(x["gate"]), up_proj=_lin(x["up"]), down_proj=_lin(x["down"])),
                 input_layernorm=_lin(x["in_norm"]), post_attention_layernorm=_lin(x["post_norm"])) for x in w["layers"]]
    cfg = NS(hidden_size=w["H"], intermediate_size=w["I"], num_attention_heads=NQ, num_key_value_heads=NKV, head_dim=HD,
             rms_norm_eps=EPS, rope_theta=THETA, num_hidden_layers=len(layers), vocab_size=V)
    return NS(config=cfg, layers=layers, norm=_lin(w["norm"]), rotary_emb=NS(inv_freq=_inv_freq().cuda(), attention_scaling=1.0))


def _code_predictor(w: dict):
    proj = torch.nn.Identity()
    if "proj" in w:
        proj = torch.nn.Linear(w["proj"].shape[1], CP[0]).cuda()
        with torch.no_grad():
            proj.weight.copy_(w["proj"])
            proj.bias.copy_(w["proj_b"])
    return NS(model=_stack(w, CP_V), lm_head=[_lin(h) for h in w["heads"]], small_to_mtp_projection=proj,
              config=NS(vocab_size=CP_V), get_input_embeddings=lambda: [_lin(t) for t in w["cemb"]])


def _talker(w: dict, cp=None):
    return NS(model=_stack(w, EMB_V), config=None, codec_head=_lin(w["head"]), code_predictor=cp, device=torch.device("cuda", torch.cuda.current_device()),
              dtype=torch.bfloat16, get_input_embeddings=lambda: _lin(w["emb"]))


def _tts(talker, H: int, groups: int):
    tc = NS(num_code_groups=groups, vocab_size=EMB_V, hidden_size=H, codec_eos_token_id=EOS)
    return NS(model=NS(talker=talker, config=NS(talker_config=tc)))


def _sampling(do_sample: bool):
    from sokutou_amd.fast import Sampling

    return Sampling(max_new_tokens=4096) if do_sample else Sampling.greedy(processor=False, max_new_tokens=4096)


def _kw(s) -> dict:
    return dict(do_sample=s.do_sample, temperature=s.temperature, top_k=s.top_k, repetition_penalty=s.repetition_penalty,
                min_new_tokens=s.min_new_tokens, max_new_tokens=s.max_new_tokens, subtalker_dosample=s.sub_do_sample,
                subtalker_temperature=s.sub_temperature, subtalker_top_k=s.sub_top_k)


def _record(fn):
    """One pass of ``fn`` as a HIP graph."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        fn()
    return g


# ---- prepare ------------------------------------------------------------------------------------------------------
@torch.no_grad()
def prepare(case: dict, seed: int):
    return {"sample": _prepare_sample, "perop": _prepare_perop, "blayer": _prepare_blayer, "bstep": _prepare_bstep,
            "frames": _prepare_frames, "cp": _prepare_cp, "tts": _prepare_tts, "prompt": _prepare_prompt}[case["kind"]](case, seed)


def _sample_inputs(case, seed):
    g, n = _gen(seed, 5), case["groups"]
    sub = _normal(g, n - 1, CP_V, std=3.0)
    code0 = _normal(g, EMB_V, std=3.0)
    seen = torch.rand(EMB_V, generator=g, device="cuda") < 0.1
    sup = torch.zeros(EMB_V, dtype=torch.bool, device="cuda")
    sup[EMB_V - 1024:] = True
    sup[EOS] = False
    return sub, code0, seen, sup


def _prepare_sample(case, seed):
    from sokutou_amd.sampler import FusedSampler

    sub, code0, seen, sup = _sample_inputs(case, seed)
    fs = FusedSampler(torch.device("cuda"))
    i64 = dict(dtype=torch.int64, device="cuda")
    st = NS(codes=torch.zeros(case["groups"], **i64), id0=torch.zeros(1, **i64), ngen=torch.ones(1, **i64),
            pos=torch.zeros(1, **i64), seen=seen.clone(), fs=fs, keep=(sub, code0, sup))
    temp, ds, k = (0.9 if case["do_sample"] else 1.0), case["do_sample"], case["top_k"]

    def frame():
        for i in range(case["groups"] - 1):
            fs(sub[i], st.codes.data_ptr() + 8 * (i + 1), ds, temp, k)
        fs(code0, st.codes.data_ptr(), ds, temp, k,
           talker=dict(seen=st.seen, rep_pen=1.05, suppress=sup, ngen=st.ngen, min_new=2, eos=EOS, id0=st.id0, pos=st.pos))

    st.graph = _record(frame)
    fs.set_seed(seed)
    st.seen.copy_(seen)
    st.ngen.fill_(1)
    st.pos.zero_()
    return st


def _pack(w: dict, wd: str):
    from sokutou_amd.kernels import _Lin

    out = []
    for x in w["layers"]:
        gu = torch.stack([x["gate"], x["up"]], dim=1).reshape(-1, x["gate"].shape[1])
        out.append(dict(qkv=_Lin(torch.cat([x["q"], x["k"], x["v"]]), wd), o=_Lin(x["o"], wd), gu=_Lin(gu, wd), down=_Lin(x["down"], wd),
                        in_norm=x["in_norm"], post_norm=x["post_norm"], qn=x["qn"], kn=x["kn"]))
    return out


def _rope(max_len: int) -> torch.Tensor:
    f = torch.arange(max_len, device="cuda", dtype=torch.float32)[:, None] * _inv_freq().cuda()[None, :]
    return torch.cat([f.cos(), f.sin()], dim=1).contiguous()


def _prepare_perop(case, seed):
    from sokutou_amd import _lib
    from sokutou_amd.kernels import _Lin

    H, I = SHAPES[case["shape"]]
    wd, ct = case["wd"], ("f32" if case["wd"] == "f32" else "bf16")
    cdt = torch.float32 if ct == "f32" else torch.bfloat16
    w = _model_weights(seed, case["layers"], H, I, EMB_V)
    layers, head = _pack(w, wd), _Lin(w["head"], wd)
    for m in [head] + [x[k] for x in layers for k in ("qkv", "o", "gu", "down")]:
        m.pol = 1  # read once per frame, as the engine sets it
    f32 = dict(dtype=torch.float32, device="cuda")
    kp, vp = _prior(seed, case["layers"], case["pos"])
    st = NS(kc=torch.zeros((case["layers"], NKV, case["max_len"], HD), dtype=cdt, device="cuda"), h=torch.zeros(H, **f32),
            x=torch.zeros(H, **f32), logits=torch.zeros(EMB_V, **f32))
    st.vc = torch.zeros_like(st.kc)
    st.kc[:, :, :case["pos"]].copy_(kp)
    st.vc[:, :, :case["pos"]].copy_(vp)
    qkv, att, act = torch.zeros((NQ + 2 * NKV) * HD, **f32), torch.zeros(NQ * HD, **f32), torch.zeros(I, **f32)
    ws = torch.zeros(int(_lib.load().sk_attn_workspace_size(NQ, NKV, case["max_len"])), dtype=torch.uint8, device="cuda")
    emb, rope, pos = w["emb"].to(cdt), _rope(case["max_len"]), torch.tensor([case["pos"]], device="cuda")
    tok = torch.tensor([seed % EMB_V], device="cuda")
    st.keep = (w["norm"], layers, head, emb, rope, pos, tok, ws, qkv, att, act)
    p, c = _lib.ptr, _lib.call

    def frame():
        s = _lib.stream()
        c("sk_embed", p(emb), p(tok), p(st.h), H, _lib.CT[ct], s)
        for i, x in enumerate(layers):
            c("sk_rms_gemv", p(st.h), p(x["in_norm"]), EPS, p(x["qkv"].w), p(x["qkv"].s), p(qkv), x["qkv"].N, H, 0, _lib.WD[wd], x["qkv"].pol, s)
            c("sk_attn", p(qkv), p(x["qn"]), p(x["kn"]), EPS, p(rope), p(st.kc[i]), p(st.vc[i]), p(pos), 0, case["max_len"], NQ, NKV, p(att),
              p(ws), ws.numel(), _lib.CT[ct], s)
            c("sk_gemv", p(att), p(x["o"].w), p(x["o"].s), None, p(st.h), H, NQ * HD, 1, _lib.WD[wd], x["o"].pol, s)
            c("sk_rms_gemv", p(st.h), p(x["post_norm"]), EPS, p(x["gu"].w), p(x["gu"].s), p(act), 2 * I, H, 1, _lib.WD[wd], x["gu"].pol, s)
            c("sk_gemv", p(act), p(x["down"].w), p(x["down"].s), None, p(st.h), H, I, 1, _lib.WD[wd], x["down"].pol, s)
        c("sk_rmsnorm", p(st.h), p(w["norm"]), EPS, p(st.x), H, s)
        c("sk_gemv", p(st.x), p(head.w), p(head.s), None, p(st.logits), EMB_V, H, 0, _lib.WD[wd], head.pol, s)

    st.graph = _record(frame)
    return st


def _terms(x: torch.Tensor, n: int) -> torch.Tensor:
    """fp32 [16, K] as n bf16 planes whose sum is the value."""
    out, v = [], x.clone()
    for _ in range(n):
        b = v.to(torch.bfloat16)
        out.append(b)
        v = v - b.float()
    return torch.stack(out).contiguous()


def _blayer_inputs(case, seed):
    H, I = SHAPES[case["shape"]]
    g = _gen(seed, 6)
    h = _normal(g, 16, H)
    h[case["batch"]:] = 0
    x = _layer_weights(seed, 0, H, I)
    nw_next = _normal(g, H, std=0.1, mean=1.0)
    T = _lengths(case, seed)
    ml = case["hi"] + 1
    kv = [_normal(g, case["batch"], NKV, ml, HD, dtype=torch.bfloat16) for _ in range(2)] if case["part"] == "attn" else None
    return h, x, nw_next, T, ml, kv


def _prepare_blayer(case, seed):
    from sokutou_amd import _lib
    from sokutou_amd.batch import tile

    L = _lib.load()
    H, I = SHAPES[case["shape"]]
    h0, x, nw_next, T, ml, kv = _blayer_inputs(case, seed)
    lay = _pack({"layers": [x]}, "i8row")[0]
    attn = case["part"] == "attn"
    w = {k: tile(lay[k]) for k in (("qkv", "o") if attn else ("gu", "down"))}
    nt = int(L.sk_batch_terms())
    nw = x["in_norm"] if attn else x["post_norm"]
    planes = _terms(h0 * nw, nt)
    ssp = h0.square().view(16, H // 16, 16).sum(2).t().contiguous()
    f32, b16 = dict(dtype=torch.float32, device="cuda"), dict(dtype=torch.bfloat16, device="cuda")
    st = NS(h=h0.clone(), h0=h0, qkv=torch.zeros(16, (NQ + 2 * NKV) * HD, **f32), ss=torch.zeros(H // 16, 16, **f32))
    xn = torch.zeros(nt, 16, H, **b16)
    ws = {k: torch.zeros(int(L.sk_bgemm_workspace_size(lay[k].N, lay[k].K)), dtype=torch.uint8, device="cuda") for k in w}
    st.keep = (lay, w, planes, ssp, xn, ws, nw_next, x)
    p, c = _lib.ptr, _lib.call
    if attn:
        st.kc, st.vc = (t.clone() for t in kv)
        att = torch.zeros(nt, 16, NQ * HD, **b16)
        aws = torch.zeros(int(L.sk_batch_attn_workspace_size(NKV)), dtype=torch.uint8, device="cuda")
        pos, rope = torch.tensor(T, device="cuda"), _rope(ml)
        st.keep += (att, aws, pos, rope)

    def half():
        s = _lib.stream()
        torch.mul(h0, 1.0, out=st.h)  # the residual as the part before leaves it
        if attn:
            c("sk_bgemm", p(planes), p(ssp), H // 16, EPS, p(w["qkv"]), p(lay["qkv"].s), lay["qkv"].N, H, 0, p(st.qkv), None, None, None, None,
              p(ws["qkv"]), ws["qkv"].numel(), s)
            c("sk_batch_attn", p(st.qkv), p(x["qn"]), p(x["kn"]), EPS, p(rope), p(st.kc), p(st.vc), p(pos), case["batch"], ml, NQ, NKV, p(att),
              p(aws), aws.numel(), s)
            c("sk_bgemm", p(att), None, 0, EPS, p(w["o"]), p(lay["o"].s), H, NQ * HD, 2, p(st.h), None, p(xn), p(x["post_norm"]), p(st.ss),
              p(ws["o"]), ws["o"].numel(), s)
        else:
            c("sk_bgemm", p(planes), p(ssp), H // 16, EPS, p(w["gu"]), p(lay["gu"].s), 2 * I, H, 1, None, p(act), None, None, None,
              p(ws["gu"]), ws["gu"].numel(), s)
            c("sk_bgemm", p(act), None, 0, EPS, p(w["down"]), p(lay["down"].s), H, I, 2, p(st.h), None, p(xn), p(nw_next), p(st.ss),
              p(ws["down"]), ws["down"].numel(), s)

    act = None if attn else torch.zeros(nt, 16, I, **b16)
    st.keep += (act,)
    st.graph = _record(half)
    return st


def _prepare_bstep(case, seed):
    from sokutou_amd.batch import BatchedTalker

    H, I = SHAPES[case["shape"]]
    w = _model_weights(seed, case["layers"], H, I, EMB_V)
    T = _lengths(case, seed)
    eng = BatchedTalker(_talker(w), case["batch"], case["hi"] + case["steps"] + 1, max_frames=case["steps"] + 1)
    for b, t in enumerate(T):
        eng.load_kv(b, *_prior(seed * 16 + b, case["layers"], t))
    eng.logits = torch.zeros(16, EMB_V, device="cuda")
    tok = [(seed * 31 + 97 * b) % EMB_V for b in range(case["batch"])]
    eng.reset(T, tok)
    eng.capture()
    return NS(eng=eng, T=T, tok=tok, steps=case["steps"])


def _engine(case, w, seed, cp=None, groups=1, max_cache=None):
    from sokutou_amd.kernels import Qwen3Kernels

    eng = Qwen3Kernels(_tts(_talker(w, cp), w["H"], groups), _sampling(case["do_sample"]), max_cache=max_cache, wd=case["wd"], sampler="fused",
                       suppress_tail=1024 if case["do_sample"] else 0)
    eng.load_kv(*_prior(seed, case["layers"], case["pos"]))
    return eng


def _prepare_frames(case, seed):
    H, I = SHAPES[case["shape"]]
    w = _model_weights(seed, case["layers"], H, I, EMB_V)
    eng = _engine(case, w, seed, max_cache=case["pos"] + case["frames"] + 1)
    return NS(eng=eng, pos=case["pos"], tok=seed % EMB_V, frames=case["frames"], seed=seed)


def _prepare_cp(case, seed):
    from sokutou_amd.kernels import CodePredictor

    w = _cp_weights(seed, case["positions"], 2048 if case["proj"] else CP[0])
    i64 = dict(dtype=torch.int64, device="cuda")
    eng = CodePredictor(_code_predictor(w), w["emb"], n_positions=case["positions"], wd=case["wd"])
    eng.x0.copy_(_normal(_gen(seed, 7), eng.in_width))
    eng.id0.fill_(seed % EMB_V)
    st = NS(eng=eng, counter=torch.zeros(1, **i64))
    if case["do_sample"]:
        eng.set_sampling(0.9, 50, torch.full((1,), seed, **i64), st.counter)
    return st


def _prepare_tts(case, seed):
    H, I = SHAPES[case["shape"]]
    w, cw = _model_weights(seed, case["layers"], H, I, EMB_V), _cp_weights(seed, 16, H)
    eng = _engine(case, w, seed, cp=_code_predictor(cw), groups=16, max_cache=case["pos"] + max(case["frames"], 4) + 1)
    x0, pad = _tts_inputs(seed, H)
    kw = dict(_kw(eng.s), prefill_len=case["pos"], first_token=seed % 1000, last_hidden=x0, tts_pad_embed=pad)
    eng.pad16.copy_(pad)
    eng.ph32.copy_(x0)
    eng.reset(case["pos"], seed % 1000)
    eng.capture()
    for t in (eng.kc, eng.vc):
        t[:, :, case["pos"]:].zero_()  # what capture's warm-up frames left
    return NS(eng=eng, kw=kw, frames=case["frames"], seed=seed)


def _tts_inputs(seed, H):
    g = _gen(seed, 8)
    return _normal(g, H), _normal(g, H, std=0.02, dtype=torch.bfloat16)


def _prompt_shape(case):
    from sokutou_amd import synthetic as syn

    return syn.shape(case["shape"], n_layers=case["layers"])


def _prompt_weights(case, seed):
    H, I = SHAPES[case["shape"]]
    return _model_weights(seed, case["layers"], H, I, EMB_V), _normal(_gen(seed, 9), 1, case["rows"], H, std=0.02, dtype=torch.bfloat16)


_HF: dict = {}


def _hf_model(case, w):
    """The package's runnable talker modules of this shape in bf16, holding the weights ``w``."""
    import copy

    from sokutou_amd import synthetic as syn

    key = (case["shape"], case["layers"])
    if key not in _HF:  # one host copy per shape: only its module tree is used, every weight is replaced below
        _HF[key] = syn.hf_talker_model(0, _prompt_shape(case)).to(torch.bfloat16)
    m = copy.deepcopy(_HF[key]).cuda()
    for layer, x in zip(m.layers, w["layers"]):
        a, f = layer.self_attn, layer.mlp
        for mod, k in ((a.q_proj, "q"), (a.k_proj, "k"), (a.v_proj, "v"), (a.o_proj, "o"), (f.gate_proj, "gate"), (f.up_proj, "up"),
                       (f.down_proj, "down"), (a.q_norm, "qn"), (a.k_norm, "kn"), (layer.input_layernorm, "in_norm"),
                       (layer.post_attention_layernorm, "post_norm")):
            mod.weight.copy_(x[k])
    m.norm.weight.copy_(w["norm"])
    m.rotary_emb.inv_freq = _inv_freq().cuda()  # kept in fp32, as checkpoints are loaded
    return m


def _prepare_prompt(case, seed):
    from sokutou_amd.kernels import Qwen3Kernels

    H, _ = SHAPES[case["shape"]]
    w, emb = _prompt_weights(case, seed)
    tts = _tts(_talker(w), H, 1)
    tts.model.talker.model = _hf_model(case, w)
    eng = Qwen3Kernels(tts, _sampling(False), max_cache=case["rows"] + 64, wd="bf16", sampler="fused", suppress_tail=0)
    eng.warm_prefill([case["rows"]])
    return NS(eng=eng, kw=dict(_kw(eng.s), inputs_embeds=emb))


# ---- run ----------------------------------------------------------------------------------------------------------
@torch.no_grad()
def run(st):
    kw = getattr(st, "kw", None)
    if kw is not None and "inputs_embeds" in kw:  # prompt
        st.eng.generate_codes(kw, max_frames=0)
        return {"id0": st.eng.id0, "hidden": st.eng.ph32, "k": st.eng.kc, "v": st.eng.vc}
    if kw is not None:  # tts
        torch.manual_seed(st.seed)
        codes = st.eng.generate_codes(kw, max_frames=st.frames)
        return {"codes": codes, "logits": st.eng.logit_t, "hidden": st.eng.ph32, "k": st.eng.kc, "v": st.eng.vc}
    if hasattr(st, "steps"):  # bstep
        st.eng.reset(st.T, st.tok)
        st.eng.replay(st.steps)
        return {"codes": st.eng.codes, "logits": st.eng.logits, "pos": st.eng.pos, "k": st.eng.kc, "v": st.eng.vc}
    if hasattr(st, "frames"):  # frames
        st.eng.reset(st.pos, st.tok)
        if st.eng.s.do_sample:
            st.eng.fs.set_seed(st.seed)
        st.eng.run_frames(st.frames)
        return {"codes": st.eng.frame_ids, "logits": st.eng.logit_t, "seen": st.eng.seen, "pos": st.eng.pos, "k": st.eng.kc, "v": st.eng.vc}
    if hasattr(st, "eng"):  # cp
        st.eng.run()
        return {"codes": st.eng.codes, "logits": st.eng.logits, "counter": st.counter, "k": st.eng.kc, "v": st.eng.vc}
    st.graph.replay()
    if hasattr(st, "fs"):  # sample
        return {"codes": st.codes, "seen": st.seen, "ngen": st.ngen, "pos": st.pos, "counter": st.fs.counter}
    if hasattr(st, "logits"):  # perop
        return {"logits": st.logits, "hidden": st.x, "h": st.h, "k": st.kc, "v": st.vc}
    out = {"h": st.h, "ss": st.ss}  # blayer
    if hasattr(st, "kc"):
        out.update(qkv=st.qkv, k=st.kc, v=st.vc)
    return out


# ---- work ---------------------------------------------------------------------------------------------------------
def _wbytes(n: int, wd: str, rows: int) -> float:
    return {"i8row": n + 2 * rows, "i8g32": n + n / 16, "bf16": 2 * n, "f32": 4 * n}[wd]


def _layer_work(H, I, wd):
    n = (NQ + 2 * NKV) * HD * H + H * NQ * HD + 3 * I * H
    return _wbytes(n, wd, (NQ + 2 * NKV) * HD + 2 * H + 2 * I), 2 * n


def work(case: dict) -> dict:
    k = case["kind"]
    if k == "sample":
        n = (case["groups"] - 1) * CP_V + EMB_V
        return {"bytes": 4 * n + 2 * EMB_V, "flops": 4 * n}
    if k == "cp":
        lb, lf = _layer_work(*CP, case["wd"])
        win = 2048 if case["proj"] else 0
        heads = (case["positions"] - 1) * CP_V * CP[0]
        return {"bytes": CP_LAYERS * lb + _wbytes(heads, case["wd"], (case["positions"] - 1) * CP_V) + _wbytes(win * CP[0], case["wd"], CP[0]),
                "flops": case["positions"] * (CP_LAYERS * lf + 2 * win * CP[0]) + 2 * heads}
    H, I = SHAPES[case["shape"]]
    wd = case.get("wd", "i8row")
    lb, lf = _layer_work(H, I, wd)
    head = _wbytes(EMB_V * H, wd, EMB_V)
    row = 2 * NKV * HD * (4 if wd == "f32" else 2)  # one position's K and V
    qk = 4 * NQ * HD                                # flops per attended position
    if k == "perop":
        T = case["pos"] + 1
        return {"bytes": case["layers"] * (lb + row * (T + 1)) + head, "flops": case["layers"] * (lf + qk * T) + 2 * EMB_V * H}
    if k == "blayer":
        if case["part"] == "mlp":
            return {"bytes": 3 * H * I + 2 * (2 * I + H) + 16 * (6 * H + 14 * H), "flops": 2 * 16 * 3 * H * I}
        T = (case["lo"] + case["hi"]) / 2 * case["batch"]
        n = (NQ + 2 * NKV) * HD * H + H * NQ * HD
        return {"bytes": n + 2 * ((NQ + 2 * NKV) * HD + H) + row * T + 16 * 20 * H, "flops": 2 * 16 * n + qk * T}
    if k == "bstep":
        T = ((case["lo"] + case["hi"]) / 2 + 1) * case["batch"]
        return {"bytes": case["steps"] * (case["layers"] * (lb + row * T) + head),
                "flops": case["steps"] * (case["layers"] * (case["batch"] * lf + qk * T) + 2 * case["batch"] * EMB_V * H)}
    if k == "prompt":
        L = case["rows"]
        lb, lf = _layer_work(H, I, "bf16")
        return {"bytes": case["layers"] * (lb + row * L) + 2 * EMB_V * H + 2 * L * H,
                "flops": case["layers"] * (L * lf + qk * L * (L + 1) / 2) + 2 * EMB_V * H}
    n, T = case["frames"], case["pos"] + (case["frames"] + 1) / 2
    b, f = case["layers"] * (lb + row * (T + 1)) + head, case["layers"] * (lf + qk * T) + 2 * EMB_V * H
    if k == "tts":
        c = work(dict(kind="cp", wd=wd, proj=case["shape"] == "1.7b", positions=16))
        b, f = b + c["bytes"], f + c["flops"]
    return {"bytes": n * b, "flops": n * f}


def tolerance(case: dict):
    # Whole values (codes, counters, positions) agree unless two scores lie within rounding of each other. Floats: fp32 sums
    # in another order, and keys and values that land on the other side of a bf16 rounding after them.
    k = case["kind"]
    if k == "sample":
        return "exact"
    if k == "prompt":
        return {"rel": 2e-2, "max": 0.5, "differ": 0.005}  # bf16 modules
    if k == "blayer":
        return {"rel": 1e-4, "max": 4e-3, "differ": 0.0}
    if k == "perop":
        return {"rel": 2e-4, "max": 1e-2, "differ": 0.0}
    if k in ("cp", "tts"):  # caches of up to 16 positions: one key or value weighs most
        return {"rel": 2e-3, "max": 8e-2, "differ": 0.0}
    return {"rel": 5e-4, "max": 2e-2, "differ": 0.0}


# ---- the same in 64 bits --------------------------------------------------------------------------------------------
def _deq(w: torch.Tensor, wd: str) -> torch.Tensor:
    """float64 weights of the format: the values the kernels multiply with."""
    wf = w.float()
    if wd in ("bf16", "f32"):
        return (w.to(torch.bfloat16) if wd == "bf16" else wf).to(F64)
    g = wf if wd == "i8row" else wf.view(w.shape[0], -1, 32)
    sc = (g.abs().amax(-1) / 127).clamp_min(1e-12).to(torch.bfloat16 if wd == "i8row" else torch.float16)
    q = torch.round(g / sc.float()[..., None]).clamp(-127, 127)
    return (q.to(F64) * sc.to(F64)[..., None]).view(w.shape)


def _rms64(h, w):
    return h * torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS) * w.to(F64)


class _Ref:
    """Decoder stack in float64 over B rows, each with its own cache [layer][kv head][max_len][128] and position."""

    def __init__(self, w: dict, wd: str, kc, vc, bf16_cache: bool):
        self.L = [{k: (_deq(v, wd) if v.dim() == 2 else v) for k, v in x.items()} for x in w["layers"]]
        self.norm, self.kc, self.vc, self.round = w["norm"], kc, vc, bf16_cache
        self.inv = _inv_freq().cuda()
        self.new = []  # (stream, layer, position, k, v) as computed, before the cache's rounding

    def _rot(self, x, pos):
        f = (torch.tensor(pos, device="cuda", dtype=torch.float32)[:, None] * self.inv[None, :]).to(F64)
        c, s = f.cos()[:, None], f.sin()[:, None]
        a, b = x[..., :HD // 2], x[..., HD // 2:]
        return torch.cat([a * c - b * s, b * c + a * s], dim=-1)

    def qkv(self, i, x, pos):
        """Rotated q, k and plain v ([B, heads, 128]) of normalised rows x."""
        W, B = self.L[i], x.shape[0]
        q, k, v = ((x @ W[n].T).view(B, -1, HD) for n in ("q", "k", "v"))
        return self._rot(_rms64(q, W["qn"]), pos), self._rot(_rms64(k, W["kn"]), pos), v

    def put(self, b, i, p, k, v):
        """Row p of stream b's cache, as the cache holds it."""
        self.new.append((b, i, p, k, v))
        self.kc[b][i][:, p], self.vc[b][i][:, p] = ((t.float().to(torch.bfloat16).to(F64) if self.round else t) for t in (k, v))

    def caches(self):
        """The caches with this pass's rows as computed: a row lies one rounding of the cache's type from them."""
        for b, i, p, k, v in self.new:
            self.kc[b][i][:, p], self.vc[b][i][:, p] = k, v
        return self.kc, self.vc

    def attend(self, q, K, V):
        """q [nq, 128] over K, V [nkv, T, 128]."""
        s = (q.view(NKV, 2, HD) @ K.to(F64).transpose(1, 2)) / math.sqrt(HD)
        return (torch.softmax(s, -1) @ V.to(F64)).reshape(-1)

    def layer(self, i, h, pos):
        W = self.L[i]
        q, k, v = self.qkv(i, _rms64(h, W["in_norm"]), pos)
        att = []
        for b, p in enumerate(pos):
            self.put(b, i, p, k[b], v[b])
            att.append(self.attend(q[b], self.kc[b][i][:, :p + 1], self.vc[b][i][:, :p + 1]))
        h = h + torch.stack(att) @ W["o"].T
        return h + self.mlp(i, h)

    def mlp(self, i, h):
        W = self.L[i]
        x = _rms64(h, W["post_norm"])
        return (torch.nn.functional.silu(x @ W["gate"].T) * (x @ W["up"].T)) @ W["down"].T

    def __call__(self, h, pos):
        for i in range(len(self.L)):
            h = self.layer(i, h, pos)
        return h


def _philox_uniform(n: int, draw_no: int, key: int) -> np.ndarray:
    """Philox4x32-10 with counter (index, draw lo, draw hi, 0x51): the uniforms of entries 0..n-1."""
    m = np.uint64(0xFFFFFFFF)
    c = [np.arange(n, dtype=np.uint64), np.full(n, draw_no & 0xFFFFFFFF, np.uint64), np.full(n, draw_no >> 32, np.uint64), np.full(n, 0x51, np.uint64)]
    k0, k1 = key & 0xFFFFFFFF, key >> 32
    for _ in range(10):
        a, b = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
        c = [(b >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), b & m, (a >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), a & m]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return ((c[0] >> np.uint64(8)).astype(np.float64) + 0.5) / 2 ** 24


def _pick64(logits: torch.Tensor, do_sample: bool, key: int, draw_no: int, seen: set | None = None, ngen: int = 0, temp=0.9, top_k=50) -> int:
    """The greedy or sampled pick; with ``seen`` the default processor (penalty 1.05, the last 1024 ids but EOS suppressed, EOS
    blocked for the first 2 codes)."""
    v = logits.detach().double().cpu().numpy().copy()
    if seen is not None and do_sample:
        s = sorted(seen)
        v[s] = np.where(v[s] < 0, v[s] * 1.05, v[s] / 1.05)
        eos = v[EOS]
        v[len(v) - 1024:] = -np.inf
        v[EOS] = eos if ngen >= 2 else -np.inf
    if not do_sample:
        return int(np.argmax(v))
    v = v / temp
    keep = (v >= np.sort(v)[-top_k]) & np.isfinite(v)
    score = np.where(keep, v - np.log(-np.log(_philox_uniform(len(v), draw_no, key))), -np.inf)
    return int(np.argmax(score))


@torch.no_grad()
def exact(case: dict, seed: int):
    return {"perop": _exact_perop, "blayer": _exact_blayer, "bstep": _exact_bstep, "frames": _exact_frames, "cp": _exact_cp,
            "tts": _exact_tts, "prompt": _exact_prompt, "sample": lambda c, s: None}[case["kind"]](case, seed)


def _caches(seed, layers, T, ml, dtype=torch.bfloat16):
    kp, vp = _prior(seed, layers, T)
    out = []
    for t in (kp, vp):
        c = torch.zeros((layers, NKV, ml, HD), dtype=F64, device="cuda")
        c[:, :, :T] = t.to(F64)
        out.append(c)
    return out


def _exact_perop(case, seed):
    H, I = SHAPES[case["shape"]]
    w = _model_weights(seed, case["layers"], H, I, EMB_V)
    kc, vc = _caches(seed, case["layers"], case["pos"], case["max_len"])
    ref = _Ref(w, case["wd"], [kc], [vc], case["wd"] != "f32")
    h = ref(w["emb"][seed % EMB_V].to(F64)[None], [case["pos"]])
    x = _rms64(h, w["norm"])
    ref.caches()
    return {"logits": (x @ _deq(w["head"], case["wd"]).T)[0], "hidden": x[0], "h": h[0], "k": kc, "v": vc}


def _exact_blayer(case, seed):
    h0, x, nw_next, T, ml, kv = _blayer_inputs(case, seed)
    h, out = h0.to(F64), {}
    attn = case["part"] == "attn"
    kc, vc = (t.to(F64) for t in kv) if attn else (None, None)  # [stream][kv head][max_len][128]
    ref = _Ref({"layers": [x], "norm": None}, "i8row", kc[:, None] if attn else None, vc[:, None] if attn else None, True)
    W = ref.L[0]
    if attn:
        z = _rms64(h, W["in_norm"])
        q, k, v = ref.qkv(0, z[:case["batch"]], T)
        att = torch.zeros(16, NQ * HD, dtype=F64, device="cuda")
        for b, p in enumerate(T):
            ref.put(b, 0, p, k[b], v[b])
            att[b] = ref.attend(q[b], kc[b, :, :p + 1], vc[b, :, :p + 1])
        h = h + att @ W["o"].T
        ref.caches()
        out = dict(qkv=torch.cat([z @ W[n].T for n in ("q", "k", "v")], dim=1), k=kc, v=vc)
    else:
        h = h + ref.mlp(0, h)
    return dict(out, h=h, ss=h.square().view(16, -1, 16).sum(2).t())


def _exact_bstep(case, seed):
    H, I = SHAPES[case["shape"]]
    B, ml = case["batch"], case["hi"] + case["steps"] + 1
    w = _model_weights(seed, case["layers"], H, I, EMB_V)
    T = _lengths(case, seed)
    caches = [_caches(seed * 16 + b, case["layers"], t, ml) for b, t in enumerate(T)]
    ref = _Ref(w, "i8row", [c[0] for c in caches], [c[1] for c in caches], True)
    head = _deq(w["head"], "i8row")
    tok = [(seed * 31 + 97 * b) % EMB_V for b in range(B)]
    logits = torch.zeros(16, EMB_V, dtype=F64, device="cuda")
    for n in range(case["steps"]):
        logits[:B] = _rms64(ref(w["emb"][tok].to(F64), [t + n for t in T]), w["norm"]) @ head.T
        tok = logits[:B].argmax(1).tolist()
    k, v = (torch.stack(c, dim=1) for c in ref.caches())
    return {"codes": None, "logits": logits, "pos": None, "k": k, "v": v}


def _exact_frames(case, seed):
    H, I = SHAPES[case["shape"]]
    w = _model_weights(seed, case["layers"], H, I, EMB_V)
    kc, vc = _caches(seed, case["layers"], case["pos"], case["pos"] + case["frames"] + 1)
    ref = _Ref(w, case["wd"], [kc], [vc], True)
    head, tok, seen = _deq(w["head"], case["wd"]), seed % EMB_V, {seed % EMB_V}
    for n in range(case["frames"]):
        logits = (_rms64(ref(w["emb"][tok].to(F64)[None], [case["pos"] + n]), w["norm"]) @ head.T)[0]
        tok = _pick64(logits, case["do_sample"], seed, n, seen, n + 1)
        seen.add(tok)
    ref.caches()
    return {"codes": None, "logits": logits.view(1, -1), "seen": None, "pos": None, "k": kc, "v": vc}


class _CpRef:
    def __init__(self, w: dict, wd: str, positions: int):
        self.w, self.n = w, positions
        self.kc, self.vc = (torch.zeros((CP_LAYERS, NKV, positions, HD), dtype=F64, device="cuda") for _ in range(2))
        self.ref = _Ref(w, wd, [self.kc], [self.vc], True)
        self.heads = [_deq(h, wd) for h in w["heads"]]
        self.proj = _deq(w["proj"], wd) if "proj" in w else None

    def frame(self, x0, id0, do_sample, key, draw_no):
        codes, logits = [id0], None
        for g in range(self.n):
            x = x0 if g == 0 else (self.w["emb"][id0] if g == 1 else self.w["cemb"][g - 2][codes[g - 1]]).to(F64)
            if self.proj is not None:
                x = self.proj @ x + self.w["proj_b"].to(F64)
            h = self.ref(x[None], [g])
            if g:
                logits = (_rms64(h, self.w["norm"]) @ self.heads[g - 1].T)[0]
                codes.append(_pick64(logits, do_sample, key, draw_no + g - 1))
        return codes, logits


def _exact_cp(case, seed):
    w = _cp_weights(seed, case["positions"], 2048 if case["proj"] else CP[0])
    c = _CpRef(w, case["wd"], case["positions"])
    x0 = _normal(_gen(seed, 7), w["emb"].shape[1]).to(F64)
    _, logits = c.frame(x0, seed % EMB_V, case["do_sample"], seed, 0)
    c.ref.caches()
    return {"codes": None, "logits": logits, "counter": None, "k": c.kc, "v": c.vc}


def _exact_tts(case, seed):
    H, I = SHAPES[case["shape"]]
    w, cw = _model_weights(seed, case["layers"], H, I, EMB_V), _cp_weights(seed, 16, H)
    cw["emb"] = w["emb"]
    kc, vc = _caches(seed, case["layers"], case["pos"], case["pos"] + max(case["frames"], 4) + 1)
    ref, cp = _Ref(w, case["wd"], [kc], [vc], True), _CpRef(cw, case["wd"], 16)
    head = _deq(w["head"], case["wd"])
    x0, pad = _tts_inputs(seed, H)
    torch.manual_seed(seed)
    key = int(torch.randint(0, 2 ** 62, (1,)).item())
    ph, tok, draws, ds = x0.to(F64), seed % 1000, 0, case["do_sample"]
    seen = {tok}
    for n in range(case["frames"]):
        if tok == EOS:
            break
        codes, _ = cp.frame(ph, tok, ds, key, draws)
        x = w["emb"][tok].to(F64) + pad.to(F64)
        for g in range(1, 16):
            x = x + cw["cemb"][g - 1][codes[g]].to(F64)
        ph = _rms64(ref(x[None], [case["pos"] + n]), w["norm"])[0]
        logits = head @ ph
        tok = _pick64(logits, ds, key, draws + 15, seen, n + 1)
        seen.add(tok)
        draws += 16
    ref.caches()
    return {"codes": None, "logits": logits.view(1, -1), "hidden": ph, "k": kc, "v": vc}


def _exact_prompt(case, seed):
    w, emb = _prompt_weights(case, seed)
    n, ml = case["rows"], case["rows"] + 64
    w["layers"] = [{k: v.to(torch.bfloat16) for k, v in x.items()} for x in w["layers"]]
    ref = _Ref(w, "bf16", None, None, False)
    kc, vc = (torch.zeros((case["layers"], NKV, ml, HD), dtype=F64, device="cuda") for _ in range(2))
    h, mask = emb[0].to(F64), torch.ones(n, n, dtype=torch.bool, device="cuda").tril()
    for i, W in enumerate(ref.L):
        q, k, v = ref.qkv(i, _rms64(h, W["in_norm"]), list(range(n)))
        kc[i, :, :n], vc[i, :, :n] = k.transpose(0, 1), v.transpose(0, 1)
        s = torch.einsum("tgrd,sgd->grts", q.view(n, NKV, 2, HD), k) / math.sqrt(HD)
        a = torch.softmax(s.masked_fill(~mask, -math.inf), -1)
        h = h + torch.einsum("grts,sgd->tgrd", a, v).reshape(n, NQ * HD) @ W["o"].T
        h = h + ref.mlp(i, h)
    return {"id0": None, "hidden": _rms64(h, w["norm"].to(torch.bfloat16))[-1], "k": kc, "v": vc}
