"""Small Pikurax configurations for the tests, their random weights, and the comparison with the plain decoder.

The configurations differ from one another in every size and option: one, several or all query heads to a key head, values
narrower and wider than keys, chunks shorter and longer than a page and of sizes that are multiples of nothing, heads turned
whole, in part and not at all, one to six taps, blocks of one channel and one block, layers without a feed-forward, dense and
routed ones with and without a shared expert, stretches that run again from the first layer, the middle and to the last, a
table of pairs with few rows, widths that are odd.
"""
from __future__ import annotations

import os
from typing import Dict, List

import torch

from llm_rs_amd import PikuraxConfig, random_model_tensors, write_model_folder
from kept_results import kept
from plain_pikurax import bf16_rounding, plain_pikurax_logits


def dense(ff):
    return {"kind": "dense", "ff": ff}


def moe(experts, top, ff, shared=None):
    return {"kind": "moe", "expert": {"ff": ff}, "router": {"experts": experts, "top": top}, "shared": None if shared is None else {"ff": shared}}


def rotation(dims, base=1000.0):
    return {"dims": dims, "base": base}


def chunked(heads, kv_heads, dim, chunk, width, blocks, conv, rot=None, scale=None, mlp=None):
    """A layer of type "parallel": attention over chunks beside a gated linear recurrent unit."""
    left = {"heads": heads, "kv_heads": kv_heads, "dim": dim, "vdim": dim, "scale": 1.5 * dim ** -0.5 if scale is None else scale, "mask": {"size": chunk}}
    if rot is not None:
        left["rot"] = rotation(*rot) if isinstance(rot, tuple) else rotation(rot)
    return {"type": "parallel", "mixer": {"left": left, "right": {"width": width, "blocks": blocks, "conv": conv}}, "mlp": mlp}


def decays(heads):
    return [1.0 - 2.0 ** -(2.0 + 7.0 * h / max(heads - 1, 1)) for h in range(heads)]


def biased(heads, kv_heads, dim, vdim, r_heads, r_dim, r_vdim, rot=None, scale=None, softcap=7.0, temp=(0.4, 9), decay=None, mlp=None):
    """A layer of type "parallel_2": capped and biased attention with a sink beside a retention."""
    left = {"heads": heads, "kv_heads": kv_heads, "dim": dim, "vdim": vdim, "scale": 1.5 * dim ** -0.5 if scale is None else scale, "softcap": softcap,
            "q_temp": {"coef": temp[0], "every": temp[1]}}
    right = {"heads": r_heads, "dim": r_dim, "vdim": r_vdim, "decay": decays(r_heads) if decay is None else decay}
    if rot is not None:
        right["rot"] = rotation(*rot) if isinstance(rot, tuple) else rotation(rot)
    return {"type": "parallel_2", "mixer": {"left": left, "right": right}, "mlp": mlp}


def config(width, vocab, layers, loop=None, eps=1e-5, scale=1.7, bigram=(11, 3, 5), logit_scale=0.5, logit_softcap=9.0):
    return {"architecture": "Pikurax", "vocab": vocab, "width": width,
            "embedding": {"scale": scale, "bigram": dict(zip(("buckets", "mul_prev", "mul_cur"), bigram))}, "norm": {"eps": eps},
            "loop": None if loop is None else dict(zip(("start", "stop", "times"), loop)), "layers": layers, "logit_scale": logit_scale,
            "logit_softcap": logit_softcap}


ODD = config(45, 97, [
    chunked(6, 2, 10, 13, 21, 3, 4, rot=6, mlp=moe(6, 2, 7, 9)),
    biased(3, 1, 9, 20, 3, 5, 7, rot=4, mlp=dense(19)),
    chunked(3, 3, 7, 50, 10, 10, 1, mlp=dense(8)),
    biased(4, 4, 6, 3, 1, 11, 4, temp=(-0.2, 1)),
    chunked(4, 1, 12, 5, 9, 1, 6, rot=12, mlp=moe(5, 5, 6)),
], loop=(1, 4, 3), eps=1e-4)
PLAIN = config(64, 128, [
    biased(4, 2, 16, 16, 2, 16, 32, rot=16, mlp=moe(8, 2, 24, 40)),
    chunked(8, 2, 16, 32, 64, 4, 4, rot=16, mlp=dense(96)),
    chunked(2, 2, 16, 40, 32, 2, 3, rot=8, mlp=moe(4, 1, 16, 16)),
], loop=(0, 3, 2), eps=1e-6, bigram=(203, 31, 7))
# widths at which the bfloat16 products go to the matrix cores, heads the matrix-core attention takes, experts the grouped products take
WIDE = config(384, 352, [
    chunked(8, 2, 32, 80, 192, 4, 4, rot=32, mlp=dense(256)),
    biased(6, 2, 64, 64, 3, 64, 128, rot=32, softcap=11.0, temp=(0.1, 64), mlp=moe(8, 2, 64, 128)),
    chunked(16, 2, 64, 130, 256, 2, 2, rot=(64, 500000.0), mlp=moe(12, 3, 128, 192)),
    biased(4, 4, 96, 96, 2, 128, 128, rot=128, mlp=moe(5, 2, 64)),
    biased(2, 1, 128, 128, 4, 32, 16),
], loop=(2, 5, 2), eps=1e-3, bigram=(1009, 127, 17))
CONFIGS = {"odd": ODD, "plain": PLAIN, "wide": WIDE}
PAGE_SIZE = {"odd": 4, "plain": 16, "wide": 16}


def one_layer(layer, width=40, vocab=61, eps=1e-5, loop=None):
    return config(width, vocab, [layer], loop, eps)


def loud(tensors) -> None:
    """Random weights under which every mechanism shows: scores that differ from key to key, gates that move with the token, a
    table of pairs as large as the token table, biases, and routers enlarged so that the choice of experts is no near tie.  A
    retention's keys lie near its queries, so that a read-out always holds its own token: one that all but cancels is no more than
    rounding, and its norm would make it as large as any other."""
    width = tensors["embed"].shape[1]
    unit = 1.0 / (0.02 * width ** 0.5)              # what makes a matrix keep the size of a normed row
    for name in list(tensors):
        factor = (25.0 if name == "embed" else 40.0 if name == "bigram" else 0.7 * unit if name == "loop.in" else 30.0 if name.endswith(".b")
                  else 40.0 if name.endswith(".mlp.router") else 10.0 if name.endswith(".shared.sg") else 4.0 if name.endswith((".ra", ".ri"))
                  else unit if name.endswith((".q", ".k", ".v", ".x", ".y", ".g", ".gate", ".up")) else None)
        if factor is not None:
            tensors[name] = (tensors[name].double() * factor).to(tensors[name].dtype)
    for name in list(tensors):
        if name.endswith(".right.k"):
            tensors[name] = (0.3 * tensors[name].double() + tensors[name[:-1] + "q"].double()).to(tensors[name].dtype)


def calm_routers(tensors) -> None:
    """Routers under which 16-bit rounding of their input cannot change which experts a token gets (two logits that differ by
    less than the rounding would otherwise fall either way, and an expert swapped for another is no rounding error): one feature
    of the stream is made the same for every token (the same in every row of the table, not touched by the pairs, the
    sublayers or the joins), and the routers read their experts' order from it and hardly anything from the rest.  Which experts a
    token gets by its own logits is what the 32-bit runs check."""
    at = tensors["embed"].shape[1] - 1
    tensors["embed"][:, at] = 12.0
    tensors["bigram"][:, at] = 0.0
    tensors["final.norm"][at] = 0.0                 # (the table is the output matrix, too)
    if "loop.in" in tensors:
        tensors["loop.in"][at] = 0.0
        tensors["loop.in"][at, at] = 1.0
    for name in list(tensors):
        if name.endswith((".norm1b", ".norm2b")):
            tensors[name][at] = 0.0
        elif name.endswith(".mlp.router"):
            n = tensors[name].shape[0]
            tensors[name] = (tensors[name].double() * 0.0005).to(tensors[name].dtype)
            order = torch.tensor([(5 * e + 2) % n if n % 5 else (3 * e + 1) % n for e in range(n)], dtype=torch.float64)
            if len(set(order.tolist())) < n:
                order = torch.arange(n, dtype=torch.float64)
            tensors[name][:, at] = (0.3 * order).to(tensors[name].dtype)


def make_model(cfg: dict, seed: int = 0, change=None, calm_router: bool = False):
    """(typed config, {name: bfloat16 tensor}); `change(tensors)` may put values of its own in."""
    typed = PikuraxConfig.from_dict(cfg)
    tensors = random_model_tensors(typed, seed)
    loud(tensors)
    if calm_router:
        calm_routers(tensors)
    if change is not None:
        change(tensors)
    return typed, tensors


def make_folder(tmp_path, cfg: dict, seed: int = 0, change=None, name: str = "model", calm_router: bool = False) -> str:
    typed, tensors = make_model(cfg, seed, change, calm_router)
    folder = os.path.join(str(tmp_path), name)
    write_model_folder(folder, typed, tensors)
    return folder


@kept
def reference(cfg: dict, tensors, requests: Dict[str, List[int]], rnd=None):
    kw = {} if rnd is None else {"rnd": rnd}
    return {rid: plain_pikurax_logits(cfg, tensors, toks, **kw) for rid, toks in requests.items()}


def allowed_error(dtype: str, cfg: dict, tensors, requests, exact) -> float:
    """How far the engine may be from the exact logits, as a part of a sequence's largest logit.  float32: 3e-5, or four times as
    far as the plain decoder itself gets in 32-bit where that is more.  bfloat16: twice as far as the plain decoder gets when
    every activation that passes through memory between two stages is rounded to bfloat16 (the engine keeps some of those in
    32-bit and sums in other orders; it does not round more often)."""
    kw = {"compute": torch.float32} if dtype == "float32" else {"rnd": bf16_rounding}
    other = {rid: plain_pikurax_logits(cfg, tensors, toks, **kw).double() for rid, toks in requests.items()}
    far = max(float((other[r] - exact[r]).abs().max()) / float(exact[r].abs().max()) for r in requests)
    return max(3e-5, 4.0 * far) if dtype == "float32" else 2.0 * far


def check_rows(rows, exact, requests, allowed: float, what: str = "") -> float:
    """Every position of every request within `allowed` of the exact logits; with 16-bit hand-overs (a bound of 1e-3 or more) one
    position in fifty of a request may be up to 1.5 times as far: a read-out of a retention or a unit whose parts nearly cancel is
    made as large as any other by the norm behind it, and what was rounded before with it, at places that differ with the rounding."""
    worst = 0.0
    for rid, toks in requests.items():
        ref = exact[rid]
        scale = float(ref.abs().max())
        assert sorted(rows[rid]) == list(range(len(toks))), f"{what} request {rid}: not every position came back"
        got = torch.stack([rows[rid][p] for p in range(len(toks))]).double()
        assert torch.isfinite(got).all(), f"{what} request {rid}: logits that are not numbers"
        err = (got - ref).abs().max(dim=1).values / scale
        bad = (err > allowed).nonzero()
        rare = allowed >= 1e-3 and len(bad) <= len(toks) // 50 and float(err.max()) <= 1.5 * allowed
        assert len(bad) == 0 or rare, (f"{what} request {rid}: first wrong position {int(bad[0])} of {len(toks)} (error "
                               f"{float(err[int(bad[0])]):.3e} of the largest logit, allowed {allowed:.1e}); {len(bad)} positions wrong")
        worst = max(worst, float(err.max()))
    return worst


MARK = 7


def only(tensors, branch: str) -> None:
    """Layer 0's mixer reduced to one of its two sides: the other's output matrix is zero, and so is its share of the result."""
    other = {"left": "right", "right": "left"}[branch]
    tensors[f"l0.mix.{other}.o"] = torch.zeros_like(tensors[f"l0.mix.{other}.o"])


def marked_model(layer: dict, width=48, vocab=50):
    """One layer whose attention is alone and in which the key of token MARK stands out for every query, wherever it stands.  Two
    features of the stream are kept: the last is the same for all tokens, and every query's last feature reads it alone; the one before
    it is large in the marked token's row only, and a key's last feature reads it alone.  (The layer's rotation, if any, leaves the
    last feature of a head as it is.)"""
    cfg = config(width, vocab, [layer], logit_softcap=0.0)
    kind, m = layer["type"], layer["mixer"]["left"]
    H, G, d = m["heads"], m["kv_heads"], m["dim"]

    def change(t):
        only(t, "left")
        t["bigram"] = torch.zeros_like(t["bigram"])
        t["embed"][:, width - 2], t["embed"][:, width - 1] = 0.0, 3.0
        t["embed"][MARK, width - 2] = 6.0
        wq = torch.zeros(H, d, width, dtype=torch.float64)
        wq[:, d - 1, width - 1] = 1.0
        wk = t["l0.mix.left.k"].double().view(G, d, width) * 0.3
        wk[:, :, width - 2] = 0.0
        wk[:, d - 1, :] = 0.0
        wk[:, d - 1, width - 2] = 1.0
        if kind == "parallel":                      # (a key is its own value: let the value's other features tell tokens apart, too)
            wk[:, 0, width - 2] = 1.5
        t["l0.mix.left.q"], t["l0.mix.left.k"] = wq.reshape(-1, width).to(torch.bfloat16), wk.reshape(-1, width).to(torch.bfloat16)
        for name in ("q.b", "k.b"):
            if f"l0.mix.left.{name}" in t:
                t[f"l0.mix.left.{name}"] = torch.zeros_like(t[f"l0.mix.left.{name}"])
        for name in ("q.norm", "k.norm"):
            if f"l0.mix.left.{name}" in t:
                t[f"l0.mix.left.{name}"] = torch.ones_like(t[f"l0.mix.left.{name}"])
    typed, tensors = make_model(cfg, seed=11, change=change)
    return cfg, typed, tensors


def state_model(which: str, width=40, vocab=61):
    """One layer whose right side is alone and whose state hardly decays.  What token MARK leaves in it outweighs by far what the
    others leave, through the same two features of the stream as in `marked_model`."""
    layer = chunked(1, 1, 4, 3, 32, 2, 3) if which == "unit" else biased(1, 1, 4, 4, 2, 16, 16, decay=[0.9999, 1.0])
    cfg = config(width, vocab, [layer], logit_softcap=0.0)

    def change(t):
        only(t, "right")
        t["bigram"] = torch.zeros_like(t["bigram"])
        t["embed"][:, width - 2], t["embed"][:, width - 1] = 0.0, 3.0
        t["embed"][MARK, width - 2] = 6.0
        name = "l0.mix.right.x" if which == "unit" else "l0.mix.right.k"
        w = t[name].double() * 0.05
        signs = torch.where(torch.arange(w.shape[0]) % 3 == 0, -1.0, 1.0).double()
        w[:, width - 2], w[:, width - 1] = signs, 0.0
        t[name] = w.to(torch.bfloat16)
        if which == "unit":
            t["l0.mix.right.lam"] = torch.full_like(t["l0.mix.right.lam"], -12.0)
            t["l0.mix.right.x.b"] = torch.zeros_like(t["l0.mix.right.x.b"])
            t["l0.mix.right.conv.b"] = torch.zeros_like(t["l0.mix.right.conv.b"])
        else:
            q = t["l0.mix.right.q"].double() * 0.3
            q[:, width - 1] = signs
            t["l0.mix.right.q"] = q.to(torch.bfloat16)
    typed, tensors = make_model(cfg, seed=7, change=change)
    return cfg, typed, tensors


def sequence_with_mark(vocab, n, at, seed):
    from replay_cases import random_tokens
    toks = [t if t != MARK else (t + 1) % vocab for t in random_tokens(vocab, n, seed)]
    toks[at] = MARK
    return toks


def moves(cfg, tensors, toks, at, exact=None):
    """How far the logits of every position move when the token at `at` is another one, as a part of the largest logit."""
    exact = plain_pikurax_logits(cfg, tensors, toks) if exact is None else exact
    other = [t if i != at else (t + 2) % cfg["vocab"] for i, t in enumerate(toks)]
    return (plain_pikurax_logits(cfg, tensors, other) - exact).abs().max(dim=1).values / float(exact.abs().max())
