"""The workloads this framework's speed is measured on: decode steps of the
HBM partition of a KV cache (GQA, separate key / value widths, absorbed MLA)
with their merges, and the prefill append into it.

A case is a dict of plain values:
  kind      "gqa"     fused append + split-KV attention over paged K/V
            "dense"   the same over contiguous per-row buffers
                      (reference_api.resident_layer)
            "mla"     absorbed MLA over the paged 576-wide latent
            "append"  prefill append of n tokens per sequence
  finish    how the step ends: "full" (bf16 output, no host share), "host"
            (merge with a host partial of the same rows), "uv" (merge and
            W_UV projection), "partial" ((out, lse) for a later merge)
  dist, lo, hi, lens_seed   tokens per sequence already in HBM: "fixed" (hi),
            "uniform" in [lo, hi], "lognormal" around sqrt(lo * hi)
Every decode step appends one token per sequence and attends over it too.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from scope_amd import ops, reference_api

DEV = "cuda:0"
BF16_TOL = 1e-2


def listed():
    return [
        # One user, short context: the latency of a step and its launches.
        dict(name="gqa_b1_4k", kind="gqa", finish="full", B=1, Hkv=4, G=8, D=128, page=64,
             dist="fixed", lo=4096, hi=4096, lens_seed=0),
        # A partitioned step at the Mixtral-8x7B layer shape: half of contexts
        # of 1k to 32k tokens in HBM, merged with the host's normalised triple.
        dict(name="gqa_b16_half", kind="gqa", finish="host", B=16, Hkv=8, G=4, D=128, page=64,
             dist="uniform", lo=512, hi=16384, lens_seed=2000),
        # A few very long contexts at the Qwen3-30B-A3B layer shape.
        dict(name="gqa_b4_128k", kind="gqa", finish="full", B=4, Hkv=4, G=8, D=128, page=64,
             dist="fixed", lo=131072, hi=131072, lens_seed=0),
        # A serving batch of many short, ragged contexts.
        dict(name="gqa_b256_short", kind="gqa", finish="full", B=256, Hkv=8, G=4, D=128, page=64,
             dist="uniform", lo=64, hi=2048, lens_seed=7),
        # The widest heads.
        dict(name="gqa_d256_b8", kind="gqa", finish="full", B=8, Hkv=4, G=2, D=256, page=64,
             dist="uniform", lo=1000, hi=16384, lens_seed=11),
        # A width between the powers of two, 24 query heads over 8 KV heads.
        dict(name="gqa_d96_g3", kind="gqa", finish="host", B=12, Hkv=8, G=3, D=96, page=64,
             dist="uniform", lo=777, hi=9001, lens_seed=13),
        # Decompressed DeepSeek-V2 attention (16 heads, 192-wide keys, 128-wide
        # values) over contiguous buffers of an odd capacity.
        dict(name="dense_192_128", kind="dense", finish="partial", B=8, Hkv=16, G=1, D=192, page=0,
             dist="fixed", lo=4096, hi=4096, lens_seed=0),
        # DeepSeek-V2-Lite, half of 16k contexts in HBM, merged with the host.
        dict(name="mla_b8_half", kind="mla", finish="host", B=8, Hkv=1, G=16, D=576, page=64,
             dist="fixed", lo=8192, hi=8192, lens_seed=0),
        # DeepSeek-V2-Lite, a ragged batch all in HBM, through W_UV.
        dict(name="mla_b32_uv", kind="mla", finish="uv", B=32, Hkv=1, G=16, D=576, page=64,
             dist="lognormal", lo=256, hi=65536, lens_seed=2005),
        # DeepSeek-V2's 128 heads, a few long contexts.
        dict(name="mla_h128_b4_32k", kind="mla", finish="partial", B=4, Hkv=1, G=128, D=576,
             page=64, dist="fixed", lo=32768, hi=32768, lens_seed=0),
        # DeepSeek-V2's 128 heads, a serving batch.
        dict(name="mla_h128_b96", kind="mla", finish="host", B=96, Hkv=1, G=128, D=576, page=64,
             dist="uniform", lo=256, hi=4096, lens_seed=17),
        # Prefill: the trailing 2k tokens of four prompts into the partition.
        dict(name="append_b4_2k", kind="append", finish="kv", B=4, Hkv=8, G=1, D=128, page=64,
             dist="fixed", lo=2048, hi=2048, lens_seed=0),
    ]


# A drawn case reads at most this many bytes and does at most this many
# operations (the largest listed cases').
MAX_BYTES = 1.0e9
MAX_FLOPS = 5.0e10


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(("gqa", "gqa", "gqa", "mla", "mla", "mla", "dense", "append"))
        c = dict(kind=kind, page=rng.choice((32, 64, 128)), lens_seed=rng.randrange(1 << 30))
        if kind == "gqa":
            c.update(finish=rng.choice(("full", "host", "partial")), B=_log_int(rng, 1, 256),
                     Hkv=rng.choice((1, 2, 4, 8)), G=rng.choice((1, 2, 3, 4, 5, 7, 8, 16)),
                     D=rng.choice((64, 80, 96, 112, 128, 128, 128, 160, 192, 256)))
        elif kind == "dense":
            c.update(finish="partial", B=_log_int(rng, 1, 32), Hkv=16, G=1, D=192, page=0)
        elif kind == "mla":
            c.update(finish=rng.choice(("host", "uv", "partial")), B=_log_int(rng, 1, 160), Hkv=1,
                     G=rng.choice((16, 16, 32, 64, 128, 128)), D=576)
        else:
            c.update(finish=rng.choice(("kv", "latent")), B=_log_int(rng, 1, 16),
                     Hkv=rng.choice((1, 2, 4, 8)), G=1, D=rng.choice((64, 128, 256)))
        top = _log_int(rng, 64, 131072) if kind != "append" else _log_int(rng, 1, 16384)
        c.update(dist="fixed", lo=top, hi=top)
        if kind in ("gqa", "mla") and rng.random() < 0.6:
            c.update(dist=rng.choice(("uniform", "lognormal")),
                     lo=max(1, top // rng.choice((2, 8, 32))))
        w = work(c)
        if w["bytes"] <= MAX_BYTES and w["flops"] <= MAX_FLOPS:
            return c


# ---------------------------------------------------------------------------
# sizes


def lengths(case):
    """Tokens per sequence in HBM before the step (of the case alone)."""
    B, lo, hi = case["B"], case["lo"], case["hi"]
    r = np.random.RandomState(case["lens_seed"])
    if case["dist"] == "fixed":
        return np.full(B, hi, np.int64)
    if case["dist"] == "uniform":
        return r.randint(lo, hi + 1, B).astype(np.int64)
    return np.clip(np.exp(r.normal(0.5 * (math.log(lo) + math.log(hi)), 1.0, B)), lo,
                   hi).astype(np.int64)


def _dv(case):
    return {"gqa": case["D"], "dense": 128, "mla": 512}[case["kind"]]


def _scale(case):
    return 1.0 / math.sqrt(192 if case["kind"] == "mla" else case["D"])


DOUT = 128  # W_UV's output width per head


def work(case):
    B, Hkv, G, D = case["B"], case["Hkv"], case["G"], case["D"]
    if case["kind"] == "append":
        row = Hkv * D * 4 if case["finish"] == "kv" else 1152
        return {"bytes": 2.0 * B * case["hi"] * row, "flops": 0.0}
    tokens = float(lengths(case).sum()) + B
    dv = _dv(case)
    rows = B * Hkv * G
    if case["kind"] == "mla":
        kv, new = 1152.0 * tokens, 2 * 1152.0 * B
    else:
        kv, new = 2.0 * (D + dv) * Hkv * tokens, 4.0 * (D + dv) * Hkv * B
    b = kv + new + rows * D * 2.0
    if case["kind"] != "dense":
        b += 4.0 * float(np.ceil((lengths(case) + 1) / case["page"]).sum()) + 8.0 * B
    if case["finish"] == "full":
        b += rows * (dv * 6.0 + 4)
    elif case["finish"] == "partial":
        b += rows * (dv * 4.0 + 4)
    elif case["finish"] == "host":
        b += rows * (dv * 4.0 + 8)  # the host partial in, the bf16 output and lse out
    elif case["finish"] == "uv":
        b += rows * DOUT * 2.0 + G * DOUT * 512 * 2.0
    flops = 2.0 * (D + dv) * G * Hkv * tokens
    if case["finish"] == "uv":
        flops += 2.0 * rows * DOUT * 512
    return {"bytes": b, "flops": flops}


# ---------------------------------------------------------------------------
# inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, sigma=1.0):
    t = torch.randn(shape, generator=g, device=DEV, dtype=torch.bfloat16)
    return t.mul_(sigma) if sigma != 1.0 else t


def _paging(case, g, extra):
    """(page_table, number of pages, max_pages, lengths on the device): the
    sequences' pages scattered over the pool."""
    lens = lengths(case)
    page = case["page"]
    need = (lens + extra + page - 1) // page
    total, max_pages = int(need.sum()), int(need.max())
    order = torch.randperm(total, generator=g, device=DEV).to(torch.int32)
    # every sequence's pages one after another, spread to its row of the table
    first = np.concatenate([[0], np.cumsum(need)[:-1]])
    at = first[:, None] + np.minimum(np.arange(max_pages)[None, :], need[:, None] - 1)
    table = order[torch.from_numpy(at).to(DEV)].contiguous()
    return table, total, max_pages, torch.from_numpy(lens.astype(np.int32)).to(DEV)


def prepare(case, seed):
    g = _gen(seed)
    B, Hkv, G, D = case["B"], case["Hkv"], case["G"], case["D"]
    s = dict(case=case, scale=_scale(case) if case["kind"] != "append" else 0.0)
    if case["kind"] == "dense":
        N, cap = B * Hkv, case["hi"] + 1
        s.update(q=_randn(g, N, G, D), k=_randn(g, N, cap, D), v=_randn(g, N, cap, 128),
                 k_new=_randn(g, N, 1, D), v_new=_randn(g, N, 1, 128))
        return s
    if case["kind"] == "append":
        # an empty partition that takes n tokens per sequence
        n, page = case["hi"], case["page"]
        per = (n + page - 1) // page
        table = torch.randperm(B * per, generator=g, device=DEV).to(torch.int32).view(B, per)
        s.update(table=table, len_in=torch.zeros(B, dtype=torch.int32, device=DEV))
        if case["finish"] == "kv":
            s.update(k_new=_randn(g, B, Hkv, n, D), v_new=_randn(g, B, Hkv, n, D),
                     k=torch.zeros(B * per, Hkv, page, D, dtype=torch.bfloat16, device=DEV),
                     v=torch.zeros(B * per, Hkv, page, D, dtype=torch.bfloat16, device=DEV))
        else:
            s.update(c_new=_randn(g, B, n, 512, sigma=0.5), pe_new=_randn(g, B, n, 64, sigma=0.5),
                     k=torch.zeros(B * per, page, 576, dtype=torch.bfloat16, device=DEV))
        return s
    table, pages, max_pages, len_in = _paging(case, g, 1)
    max_len = int(lengths(case).max()) + 1
    dv, rows = _dv(case), B * Hkv * G
    s.update(table=table, len_in=len_in, len_out=torch.zeros_like(len_in), max_len=max_len)
    if case["kind"] == "mla":
        s.update(q=_randn(g, rows, 512, sigma=0.5), q_pe=_randn(g, rows, 64, sigma=0.5),
                 k=_randn(g, pages, case["page"], 576, sigma=0.5),
                 c_new=_randn(g, B, 1, 512, sigma=0.5), pe_new=_randn(g, B, 1, 64, sigma=0.5))
        nbytes = ops.decode_plan(1, B, G, max_len)[1]
    else:
        s.update(q=_randn(g, B, Hkv * G, D), k=_randn(g, pages, Hkv, case["page"], D),
                 v=_randn(g, pages, Hkv, case["page"], D), k_new=_randn(g, B, Hkv, 1, D),
                 v_new=_randn(g, B, Hkv, 1, D))
        nbytes = ops.gqa_plan(B * Hkv, G, D, D, max_len)[1]
    if case["finish"] in ("host", "uv"):
        s["ws"] = torch.zeros(max(nbytes, 256), dtype=torch.uint8, device=DEV)
    if case["finish"] == "host":
        # the host's share of the rows, about as many tokens as the GPU's: an
        # average over n tokens has components of 1 / sqrt(n)
        n = float(lengths(case).mean()) + 1
        out = _randn(g, rows, dv, sigma=(0.5 if case["kind"] == "mla" else 1.0) / math.sqrt(n))
        lse = torch.randn(rows, generator=g, device=DEV) * 0.1 + math.log(n) + 0.5
        if case["kind"] == "mla":  # the native host partial
            s.update(b=(out, lse), fmt=ops.PARTIAL_LSE_BF16)
        else:  # the reference kernel's bf16 triple
            s.update(b=(out, (lse - 4.0).to(torch.bfloat16),
                        torch.full((rows,), math.exp(4.0), device=DEV).to(torch.bfloat16)),
                     fmt=ops.TRIPLE_NORM_BF16)
    if case["finish"] == "uv":
        s["w_uv"] = _randn(g, G, DOUT, 512, sigma=512 ** -0.5)
    return s


# ---------------------------------------------------------------------------
# one pass


def run(s):
    case, finish = s["case"], s["case"]["finish"]
    kind = case["kind"]
    if kind == "dense":
        o, m, z = reference_api.resident_layer(s["q"], s["k"], s["v"], s["k_new"], s["v_new"],
                                               s["scale"])
        return {"out": o, "max": m, "sum": z, "k": s["k"], "v": s["v"]}
    if kind == "append":
        if finish == "kv":
            ops.kv_append(s["k_new"], s["v_new"], s["k"], s["v"], s["table"], s["len_in"],
                          update_len=False)
            return {"k": s["k"], "v": s["v"]}
        ops.latent_append(s["c_new"], s["pe_new"], s["k"], s["table"], s["len_in"],
                          update_len=False)
        return {"k": s["k"]}
    if kind == "gqa":
        args = (s["q"], s["k_new"], s["v_new"], s["k"], s["v"], s["table"], s["len_in"],
                s["len_out"], s["scale"], s["max_len"])
        got = {"k": s["k"], "v": s["v"], "len": s["len_out"]}
        if finish == "full":
            got["out"], got["lse"] = ops.gqa_append_decode_full(*args)
        elif finish == "partial":
            got["out"], got["lse"] = ops.gqa_append_decode_partial(*args)
        else:
            step = ops.gqa_append_decode_split(*args, workspace=s["ws"])
            got["out"], got["lse"] = ops.merge_split(step, s["b"], s["fmt"])
        return got
    args = (s["q"], s["q_pe"], s["c_new"], s["pe_new"], s["k"], s["table"], s["len_in"],
            s["len_out"], s["scale"], s["max_len"])
    got = {"k": s["k"], "len": s["len_out"]}
    if finish == "partial":
        got["out"], got["lse"] = ops.mla_append_decode_partial(*args)
        return got
    step = ops.mla_append_decode_split(*args, workspace=s["ws"])
    if finish == "host":
        got["out"], got["lse"] = ops.merge_split(step, s["b"], s["fmt"])
    else:
        got["out"], _, got["lse"] = ops.merge_split_uv(step, s["w_uv"], want_lse=True)
    return got


def tolerance(case):
    """The decode steps round probabilities, split pieces and outputs to bf16;
    an append copies bits."""
    if case["kind"] == "append":
        return "exact"
    return {"rel": BF16_TOL, "max": 0.06}


# ---------------------------------------------------------------------------
# 64-bit results


def _attend64(q, k, v, scale):
    """q [.., G, Dk], k [.., L, Dk], v [.., L, Dv] -> (out, lse) in 64 bits."""
    x = torch.matmul(q.double(), k.double().transpose(-1, -2)) * scale
    lse = torch.logsumexp(x, -1)
    return torch.matmul(torch.exp(x - lse.unsqueeze(-1)), v.double()), lse


def exact(case, seed):
    s = prepare(case, seed)
    B, Hkv, G, kind = case["B"], case["Hkv"], case["G"], case["kind"]
    if kind == "append":
        return None
    if kind == "dense":
        s["k"][:, -1:] = s["k_new"]
        s["v"][:, -1:] = s["v_new"]
        got = [_attend64(s["q"][i], s["k"][i], s["v"][i], s["scale"]) for i in range(B * Hkv)]
        lse = torch.stack([x[1] for x in got]).unsqueeze(-1)
        return {"out": torch.stack([x[0] for x in got]), "max": lse, "sum": torch.ones_like(lse),
                "k": None, "v": None}
    outs, lses = [], []
    for b, n in enumerate(lengths(case).tolist()):
        pages = s["table"][b, :(n + 1 + case["page"] - 1) // case["page"]].long()
        if kind == "mla":
            lat = s["k"][pages].reshape(-1, 576)[:n + 1].clone()
            lat[n, :512], lat[n, 512:] = s["c_new"][b, 0], s["pe_new"][b, 0]
            rows = slice(b * G, (b + 1) * G)
            q = torch.cat([s["q"][rows], s["q_pe"][rows]], -1)
            o, l = _attend64(q, lat, lat[:, :512], s["scale"])
        else:
            k, v = (x[pages].transpose(0, 1).reshape(Hkv, -1, case["D"])[:, :n + 1].clone()
                    for x in (s["k"], s["v"]))
            k[:, n], v[:, n] = s["k_new"][b, :, 0], s["v_new"][b, :, 0]
            o, l = _attend64(s["q"][b].view(Hkv, G, -1), k, v, s["scale"])
        outs.append(o.reshape(Hkv * G, -1))
        lses.append(l.reshape(Hkv * G))
    out, lse = torch.cat(outs), torch.cat(lses)
    if case["finish"] == "host":
        b_out, b_lse = s["b"][0].double(), s["b"][1].double()
        if len(s["b"]) == 3:
            b_lse = b_lse + torch.log(s["b"][2].double())
        both = torch.logaddexp(lse, b_lse)
        out = out * torch.exp(lse - both).unsqueeze(-1) + b_out * torch.exp(b_lse - both).unsqueeze(-1)
        lse = both
    elif case["finish"] == "uv":
        out = torch.matmul(out.view(B, G, 1, 512), s["w_uv"].double().transpose(1, 2)).reshape(B, -1)
    got = {"k": None, "len": None, "out": out, "lse": lse}
    if kind == "gqa":
        got["v"] = None
        if case["finish"] != "host":
            got["out"], got["lse"] = out.view(B, Hkv * G, -1), lse.view(B, Hkv * G)
    return got
