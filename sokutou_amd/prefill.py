"""The prompt prefill on the package's own kernels (``sk_prefill``), in place of the talker's modules where a prefill graph is
recorded: about forty small launches per layer become six.

The modules stay what defines the result. ``plan`` takes a model only if every weight it would read is a plain bf16
``nn.Linear`` or norm weight of the structure the decode kernels read (qwen3/kernels.py:454-476), nothing hooks into the
forward pass and the prompt is not so long that the library's large products win; and a recording only uses it after ``agrees`` has run one random prompt of that length through both.
Anything else (fp32 modules, other shapes, biases, wrapped or hooked modules, eager runs) goes through the modules."""

from __future__ import annotations

import ctypes

import torch

from . import _lib
from .kernels import HD


class Prefill:
    """A prompt of ``rows`` rows through ``layers`` (bf16 weight tensors by name, kept alive here and read in place, so a
    weight updated in place is seen) into the caches ``kc`` / ``vc``. Owns its workspace and output."""

    def __init__(self, P, layers: list, norm: torch.Tensor, kc: torch.Tensor, vc: torch.Tensor, rows: int):
        n, max_len = len(layers), int(kc.shape[2])
        size = int(_lib.load().sk_prefill_workspace_size(P.H, P.I, P.nq, P.nkv, rows))
        if size == 0 or rows > max_len or rows > P.rope.shape[0]:
            raise ValueError("sk_prefill does not take this shape")
        self.keep = (P.rope, layers, norm, kc, vc)
        self.ws = torch.empty(size, dtype=torch.uint8, device=kc.device)
        self.out = torch.empty((1, rows, P.H), dtype=torch.bfloat16, device=kc.device)
        self.rows, self.hidden = rows, P.H
        self._layers = (_lib.SkPrefillLayer * n)()
        for i, w in enumerate(layers):
            self._layers[i] = _lib.SkPrefillLayer(kc=kc[i].data_ptr(), vc=vc[i].data_ptr(), **{k: t.data_ptr() for k, t in w.items()})
        self._desc = _lib.SkPrefillDesc(n_layers=n, hidden=P.H, inter=P.I, nq=P.nq, nkv=P.nkv, rows=rows, max_len=max_len, eps=P.eps,
                                        layers=ctypes.cast(self._layers, ctypes.c_void_p), embeds=None, norm=norm.data_ptr(),
                                        rope=P.rope.data_ptr(), out=self.out.data_ptr(), workspace=self.ws.data_ptr(), workspace_bytes=size)

    def __call__(self, embeds: torch.Tensor) -> torch.Tensor:
        """``embeds`` (1, rows, hidden) bf16 -> last hidden states (1, rows, hidden) bf16 (this object's buffer)."""
        if tuple(embeds.shape) != (1, self.rows, self.hidden) or embeds.dtype != torch.bfloat16 or not embeds.is_contiguous():
            raise ValueError("embeds must be contiguous bf16 (1, rows, hidden)")
        self._desc.embeds = embeds.data_ptr()
        _lib.check(_lib.load().sk_prefill(ctypes.byref(self._desc), _lib.stream()), "sk_prefill")
        return self.out


# Rows times hidden size up to which the package's kernels are the faster ones: their products read each weight again for
# every 64 rows, from the caches, where the library's large tiles catch up. Against the modules (us, two layers): 0.6B 17 rows
# 195 : 674, 1900 rows 912 : 1609, 4000 rows 2169 : 3369; 1.7B 33 rows 255 : 777, 900 rows 931 : 1340, 2000 rows
# 1849 : 1999.
MAX_WORK = 1 << 22


def _hooked(model) -> bool:
    names = ("_forward_hooks", "_forward_pre_hooks")
    return any(getattr(m, k, None) for m in model.modules() for k in names) or any(
        getattr(torch.nn.modules.module, "_global" + k, None) for k in names)


@torch.no_grad()
def plan(model, P, kc: torch.Tensor, vc: torch.Tensor, rows: int) -> Prefill | None:
    """The prefill of a prompt of ``rows`` rows on the package's kernels, or None where the modules have to run it."""
    if not isinstance(model, torch.nn.Module) or model.training or kc.dtype != torch.bfloat16 or _hooked(model):
        return None
    if rows * P.H > MAX_WORK or len(model.layers) != len(P.layers) or rows > min(int(kc.shape[2]), int(P.rope.shape[0])):
        return None
    if int(_lib.load().sk_prefill_workspace_size(P.H, P.I, P.nq, P.nkv, rows)) == 0:
        return None

    def ok(w, *shape) -> bool:
        return (type(w) in (torch.nn.Parameter, torch.Tensor) and tuple(w.shape) == shape and w.dtype == torch.bfloat16 and w.device == kc.device
                and w.is_contiguous() and w.data_ptr() % 16 == 0)

    nq, nkv = P.nq * HD, P.nkv * HD
    layers = []
    for x in model.layers:
        a, m = x.self_attn, x.mlp
        lin = dict(q=(a.q_proj, nq, P.H), k=(a.k_proj, nkv, P.H), v=(a.v_proj, nkv, P.H), o=(a.o_proj, P.H, nq), gate=(m.gate_proj, P.I, P.H),
                   up=(m.up_proj, P.I, P.H), down=(m.down_proj, P.H, P.I))
        if any(type(y) is not torch.nn.Linear or y.bias is not None or not ok(y.weight, r, c) for y, r, c in lin.values()):
            return None
        # the parts of an attention module's structure that its attributes name, where it has them
        if (getattr(a, "sliding_window", None) is not None or abs(getattr(a, "scaling", HD ** -0.5) - HD ** -0.5) > 1e-6
                or any(abs(getattr(y, "variance_epsilon", P.eps) - P.eps) > 1e-9 for y in (x.input_layernorm, a.q_norm, a.k_norm))):
            return None
        w = {k: y.weight.detach() for k, (y, _, _) in lin.items()}
        for k, y, size in (("in_norm", x.input_layernorm, P.H), ("post_norm", x.post_attention_layernorm, P.H), ("qn", a.q_norm, HD),
                           ("kn", a.k_norm, HD)):
            if not ok(y.weight, size):
                return None
            w[k] = y.weight.detach()
        layers.append(w)
    if not ok(model.norm.weight, P.H):
        return None
    return Prefill(P, layers, model.norm.weight.detach(), kc, vc, rows)


# Two bf16 evaluations of one decoder differ by their roundings, more with every layer (2-norm, measured on random weights, 3 to
# 200 rows): keys and values of layer 0 by 0.004, of layer 1 by 0.007 to 0.011, of layer 27 by 0.014 (0.6B) to 0.031
# (1.7B), the last hidden states like the last layer's. An attention scale 1.5 times as large, as an example of another
# structure, moves those of layer 1 by 0.11 to 0.45.
def _bound(layer: int) -> float:
    return 0.01 if layer == 0 else 0.02 + 0.001 * layer


@torch.no_grad()
def agrees(pre: Prefill, modules, kc: torch.Tensor, vc: torch.Tensor) -> bool:
    """Whether ``pre`` and ``modules`` (embeds -> last hidden states) give the same keys and values in every layer and the same
    hidden states for a random prompt. Leaves the caches' rows [0, rows) as ``pre`` wrote them."""
    g = torch.Generator(device=kc.device).manual_seed(pre.rows)
    emb = (torch.randn((1, pre.rows, pre.hidden), generator=g, device=kc.device) * 0.02).to(torch.bfloat16)
    ref = [modules(emb).float().clone(), kc[:, :, :pre.rows].float(), vc[:, :, :pre.rows].float()]
    got = [pre(emb).float(), kc[:, :, :pre.rows].float(), vc[:, :, :pre.rows].float()]
    if got[0].shape != ref[0].shape:
        return False
    n = int(kc.shape[0])
    off = [(got[0] - ref[0]).norm() / ref[0].norm()]
    off += [(a[i] - b[i]).norm() / b[i].norm() for a, b in zip(got[1:], ref[1:]) for i in range(n)]
    top = torch.tensor([_bound(n)] + [_bound(i) for _ in range(2) for i in range(n)], device=kc.device)
    return bool((torch.stack(off) <= top).all())  # (a NaN compares false)
