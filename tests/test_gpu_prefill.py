"""The prompt prefill on the package's kernels (sk_prefill): hidden states, keys and values of whole prompts against a float64
evaluation of the same bf16 weights, and the rule that puts it in place of the talker's modules when a prefill graph is
recorded."""

import math

import numpy as np
import pytest
import torch

from sokutou_amd import prefill
from sokutou_amd import synthetic as syn

pytestmark = pytest.mark.gpu
HD = 128


def _model(shape, seed=3, **kw):
    return syn.hf_talker_model(seed, shape, **kw).to(torch.bfloat16)


def _reference(model, emb, eps=1e-6):
    """float64 forward of the module tree's weights: (final hidden [L, H], keys, values [layer][nkv][L][128])."""
    f = lambda w: w.detach().double().cpu()
    h, L = emb[0].double().cpu(), emb.shape[1]
    pos = torch.arange(L, dtype=torch.float32)[:, None] * model.rotary_emb.inv_freq.float().cpu()[None, :]
    c, s = (torch.cat([t, t], 1).double()[:, None] for t in (pos.cos(), pos.sin()))
    rms = lambda x, w: x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * f(w)
    rot = lambda x: x * c + torch.cat([-x[..., 64:], x[..., :64]], -1) * s
    keys, vals = [], []
    for y in model.layers:
        a, m = y.self_attn, y.mlp
        x = rms(h, y.input_layernorm.weight)
        q, k, v = ((x @ f(p.weight).T).view(L, -1, HD) for p in (a.q_proj, a.k_proj, a.v_proj))
        q, k = rot(rms(q, a.q_norm.weight)), rot(rms(k, a.k_norm.weight))
        keys.append(k.transpose(0, 1))
        vals.append(v.transpose(0, 1))
        sc = torch.einsum("tgrd,sgd->grts", q.view(L, -1, 2, HD), k) / math.sqrt(HD)
        w = torch.softmax(sc.masked_fill(~torch.ones(L, L, dtype=torch.bool).tril(), -math.inf), -1)
        h = h + torch.einsum("grts,sgd->tgrd", w, v).reshape(L, -1) @ f(a.o_proj.weight).T
        x = rms(h, y.post_attention_layernorm.weight)
        h = h + (torch.nn.functional.silu(x @ f(m.gate_proj.weight).T) * (x @ f(m.up_proj.weight).T)) @ f(m.down_proj.weight).T
    return rms(h, model.norm.weight), torch.stack(keys), torch.stack(vals)


def _rel(a, b) -> float:
    return float((a.double().cpu() - b).norm() / b.norm())


@pytest.mark.parametrize("hidden,inter,nq,L", [(1024, 3072, 16, n) for n in (1, 2, 15, 16, 17, 32, 33, 45, 63, 64, 65, 130)] +
                         [(2048, 1024, 8, 31), (2048, 6144, 16, 70), (1024, 1024, 8, 200), (1024, 1024, 8, 500),
                                                     (2048, 1024, 16, 260)])
def test_prefill_against_float64(gpu, hidden, inter, nq, L):
    """Rows on both sides of every tile (16), key tile (32) and row block (64). Inputs of each product are rounded to bf16
    (2^-9 each), so an output is off by about 2^-9 sqrt(number of roundings on its way): 6 per layer and 2 layers, 7e-3,
    and keys and values by one more rounding. Cache rows past the prompt stay as they were."""
    from sokutou_amd.kernels import _Stack

    print(f"prefill hidden {hidden} inter {inter} heads {nq} rows {L}", flush=True)
    s = syn.TalkerShape(hidden=hidden, n_layers=2, nq=nq, nkv=nq // 2, inter=inter, vocab=64)
    model = _model(s).to(gpu)
    with torch.no_grad():
        P = _Stack(model, "bf16", L + 7)
    kc = torch.full((2, nq // 2, L + 7, HD), 5.0, dtype=torch.bfloat16, device=gpu)
    vc = kc.clone()
    emb = torch.from_numpy(syn.prompt_embeds(1, s, L)).to(gpu).to(torch.bfloat16)
    pre = prefill.plan(model, P, kc, vc, L)
    assert pre is not None
    pre.ws.fill_(255)  # NaN in every buffer: nothing is read before it is written
    for _ in range(2):
        out = pre(emb)
    torch.cuda.synchronize()
    h, k, v = _reference(model, emb)
    assert _rel(out[0], h) < 1e-2
    assert _rel(kc[:, :, :L], k) < 1e-2 and _rel(vc[:, :, :L], v) < 1e-2
    assert bool((kc[:, :, L:] == 5).all()) and bool((vc[:, :, L:] == 5).all())


def test_prefill_takes_only_plain_bf16_modules(gpu):
    """What the rule leaves to the modules, and a model whose attention differs, which the probe finds."""
    from sokutou_amd.kernels import _Stack

    print("prefill: the modules it takes", flush=True)
    s = syn.TalkerShape(hidden=1024, n_layers=1, nq=16, nkv=8, inter=1024, vocab=64)
    kc = torch.zeros((1, 8, 40, HD), dtype=torch.bfloat16, device=gpu)
    m = _model(s).to(gpu).eval()
    P = _Stack(m, "bf16", 40)
    go = lambda **kw: prefill.plan(kw.get("model", m), P, kw.get("kc", kc), kw.get("kc", kc).clone(), kw.get("rows", 9))
    assert go() is not None
    wide = torch.zeros((1, 8, 4100, HD), dtype=torch.bfloat16, device=gpu)
    P.rope = torch.zeros((4100, HD), device=gpu)
    assert go(kc=wide, rows=4096) is not None and go(kc=wide, rows=4097) is None  # the library's from there on
    assert go(rows=41) is None and go(kc=kc.float()) is None
    assert go(model=syn.hf_talker_model(3, s).to(gpu)) is None  # fp32 weights
    m.train()
    assert go() is None
    m.eval()
    hook = m.layers[0].mlp.register_forward_hook(lambda *a: None)
    assert go() is None
    hook.remove()
    m.layers[0].mlp.up_proj = torch.nn.Sequential(m.layers[0].mlp.up_proj)
    m.layers[0].mlp.up_proj.weight = m.layers[0].mlp.up_proj[0].weight
    assert go() is None


def _engine(gpu, L):
    from sokutou_amd.fast import Sampling
    from sokutou_amd.kernels import Qwen3Kernels

    s = syn.shape("0.6b", n_layers=2)
    tts = syn.make_tts(3, s, device=gpu)
    tts.model.talker.model = _model(s).to(gpu)
    eng = Qwen3Kernels(tts, Sampling.greedy(processor=False), max_cache=L + 9, wd="bf16", sampler="fused", suppress_tail=0)
    return eng, torch.from_numpy(syn.prompt_embeds(5, s, L)).to(gpu).to(torch.bfloat16)


@pytest.mark.parametrize("other", ["", "scale", "probe"])
def test_recorded_prefill_is_the_modules(gpu, monkeypatch, other):
    """An engine over bf16 modules records the prompt on the package's kernels, or through the modules where they name another
    attention scale or the probe disagrees. Either way the graph's results are the modules' within two bf16 evaluations, replays repeat them,
    and the transformers cache stands at the prompt's end."""
    L = 21
    print(f"recorded prefill, left to the modules by: {other or 'nothing'}", flush=True)
    eng, emb = _engine(gpu, L)
    if other == "probe":
        monkeypatch.setattr(prefill, "agrees", lambda *a: False)
    if other == "scale":
        for y in eng.talker.model.layers:
            y.self_attn.scaling *= 1.5
    with torch.no_grad():
        ref = eng._prefill_run(emb).float().clone()
    rk, rv = eng.kc.float().clone(), eng.vc.float().clone()
    for _ in range(2):
        eng._prefill(emb)
        torch.cuda.synchronize()
        assert (eng._pf[L][3] is None) == bool(other)
        assert _rel(eng.ph32, ref[0, -1].double().cpu()) < 2e-2
        assert _rel(eng.kc[:, :, :L], rk[:, :, :L].double().cpu()) < 2e-2 and _rel(eng.vc[:, :, :L], rv[:, :, :L].double().cpu()) < 2e-2
        assert int(eng.pos) == L and all(int(y.cumulative_length) == L for y in eng.tcache.layers)


@pytest.mark.parametrize("what", ["scale", "positions", "activation", "residual"])
def test_probe_finds_another_structure(gpu, what):
    """Differences that no attribute check sees at the time (changed after the plan was made) are found by the random prompt."""
    L = 12
    print(f"prefill probe: {what}", flush=True)
    eng, _ = _engine(gpu, L)
    pre = prefill.plan(eng.talker.model, eng.T, eng.kc, eng.vc, L)
    run = lambda e: eng._prefill_run(e)
    with torch.no_grad():
        assert prefill.agrees(pre, run, eng.kc, eng.vc)
        for y in eng.talker.model.layers:
            if what == "scale":
                y.self_attn.scaling *= 1.5
            elif what == "activation":
                y.mlp.act_fn = torch.nn.GELU()
            elif what == "residual":
                y.mlp.register_forward_hook(lambda m, a, o: o * 0.9)
        if what == "positions":
            eng.talker.model.rotary_emb.inv_freq *= 0.97
        assert not prefill.agrees(pre, run, eng.kc, eng.vc)
