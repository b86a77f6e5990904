"""The calls a serving engine makes of this operator set, as measurable cases.

Each case is one public op (``torch.ops.npu.*``) at a size from this repository's
benchmark, tests or gate sweep. ``listed()`` names the fixed ones, ``draw()`` gives
others of the same ranges, ``prepare()`` builds what a serving process holds before
the call (paged K/V pool, block tables, lengths, weights), ``run()`` is one call.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "vllm-hust-cascade-kernel_amd"))
import cascade_amd  # noqa: E402,F401  (registers torch.ops.npu)

DEV = "cuda:0"
D = 128      # head dim of every attention op
PAGE = 128   # tokens per K/V page
SCALE = 1.0 / math.sqrt(D)
MAX_SUFFIX = 4096
EPS = 1e-6
BF16, F32, I32, I64 = 2, 4, 4, 8  # bytes


def listed():
    return [
        # A small decode batch on a short system prompt: the smallest fused call, all
        # launch and start-up latency.
        _cascade("cascade-b8", 8, 32, 8, 2048, 256),
        # The benchmark workload: 64 decode queries on a shared 8192-token prefix,
        # geometric suffixes of mean 512.
        _cascade("cascade-b64", 64, 32, 8, 8192, 512),
        # A 64-head model (8 query heads per kv head) at a batch and a prefix length
        # that are no multiples of anything.
        _cascade("cascade-b47-h64", 47, 64, 8, 6037, 400),
        # The same model with 256 sequences on a 32K shared prefix: the largest call.
        _cascade("cascade-b256-h64", 256, 64, 8, 32768, 512),
        # Stage 1 of the composed cascade: 64 queries flattened into one request.
        _stage1("stage1-flat-t64", 1, 64, 32, 8, 8192, True),
        # Stage 1 per request (q_len 1), each request on its own pages of ragged length.
        _stage1("stage1-b7-ragged", 7, 1, 40, 8, 4096, False),
        # Stage 2 of the composed cascade on the head-major pool its first users have.
        _suffix("suffix-b61-bnsd", 61, 32, 8, 512, 1),
        # The merge of the composed cascade: fp32 stage-1 rows with the padded LSE,
        # bf16 suffix rows, some suffixes empty.
        _merge("merge-r8192", 256, 32, 1, 1),
        # gate_up + SwiGLU: one decode token, a decode batch, a prefill chunk.
        _gateup("gateup-m1", 1, 4096, 14336),
        _gateup("gateup-m64", 64, 4096, 14336),
        _gateup("gateup-m4096", 4096, 4096, 14336),
        # A decoder layer's residual add and norm over a prefill chunk: mode 0 gives the
        # new residual and its statistics, mode 1 the normalised rows.
        _norm("norm-r2048", 2048, 5120, "bf16", False),
    ]


def _cascade(name, batch, heads, kv_heads, prefix, mean, layout=0):
    return {"name": name, "op": "cascade", "batch": batch, "heads": heads, "kv_heads": kv_heads,
            "prefix": prefix, "suffix_mean": mean, "layout": layout}


def _stage1(name, batch, q_len, heads, kv_heads, kv, uniform):
    return {"name": name, "op": "stage1", "batch": batch, "q_len": q_len, "heads": heads, "kv_heads": kv_heads,
            "kv": kv, "uniform": uniform}


def _suffix(name, batch, heads, kv_heads, mean, layout):
    return {"name": name, "op": "suffix", "batch": batch, "heads": heads, "kv_heads": kv_heads,
            "suffix_mean": mean, "layout": layout}


def _merge(name, tokens, heads, out_code, empty):
    return {"name": name, "op": "merge", "tokens": tokens, "heads": heads, "out_code": out_code, "some_empty": empty}


def _gateup(name, m, k, inter):
    return {"name": name, "op": "gateup", "m": m, "k": k, "inter": inter}


def _norm(name, rows, k, dtype, beta):
    return {"name": name, "op": "norm", "rows": rows, "k": k, "dtype": dtype, "beta": beta}


def draw(rng):
    """One more case of the ranges the listed ones stand for."""
    def log(lo, hi):
        return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    op = rng.choice(["cascade"] * 4 + ["stage1"] * 2 + ["suffix"] * 2 + ["merge"] + ["gateup"] * 3 + ["norm"] * 2)
    # query heads / kv heads: whole models and a tensor-parallel shard
    heads, kv_heads = rng.choice([(32, 8), (64, 8), (40, 8), (8, 1), (32, 8), (64, 8)])
    if op == "cascade":
        c = _cascade("", log(1, 256), heads, kv_heads, log(128, 32768), log(32, 1024), rng.choice([0, 0, 1]))
    elif op == "stage1" and rng.random() < 0.5:
        c = _stage1("", 1, log(1, 256), heads, kv_heads, log(128, 32768), True)
    elif op == "stage1":
        batch = log(2, 64)
        c = _stage1("", batch, rng.choice([1, 1, 2]), heads, kv_heads, log(128, min(16384, 131072 // batch)),
                    rng.random() < 0.5)
    elif op == "suffix":
        c = _suffix("", log(1, 256), heads, kv_heads, log(32, 1024), rng.choice([0, 1]))
    elif op == "merge":
        c = _merge("", log(1, 512), heads, rng.choice([1, 1, 2]), rng.choice([0, 1]))
    elif op == "gateup":
        k, inter, most = rng.choice([(4096, 14336, 4096), (4096, 14336, 4096), (8192, 28672, 1024), (8192, 3584, 4096)])
        c = _gateup("", log(1, most), k, inter)
    else:
        c = _norm("", log(1, 4096), rng.choice([2048, 4096, 5008, 5120]), rng.choice(["bf16", "bf16", "fp16"]),
                  rng.random() < 0.5)
    del c["name"]
    return c


# ---- sizes ------------------------------------------------------------------------
def _suffix_lens(case):
    """Suffix lengths of the batch, geometric and clipped; the same set for every seed."""
    rng = np.random.default_rng(case["batch"] * 8191 + case["suffix_mean"])
    return np.clip(rng.geometric(1.0 / case["suffix_mean"], size=case["batch"]), 1, MAX_SUFFIX).astype(np.int64)


def _kv_lens(case):
    """kv lengths of a stage-1 call's requests: all `kv`, or ragged in [kv / 4, kv]."""
    if case["uniform"]:
        return np.full(case["batch"], case["kv"], dtype=np.int64)
    rng = np.random.default_rng(case["batch"] * 8191 + case["kv"])
    return rng.integers(max(1, case["kv"] // 4), case["kv"] + 1, size=case["batch"]).astype(np.int64)


def _pages(lens):
    return (np.asarray(lens) + PAGE - 1) // PAGE


def work(case):
    op = case["op"]
    if op == "merge":
        rows = case["tokens"] * case["heads"]
        out = BF16 if case["out_code"] == 1 else F32
        return {"bytes": rows * (D * (F32 + BF16 + out) + 8 * F32 + F32), "flops": rows * D * 5}
    if op == "gateup":
        m, k, i = case["m"], case["k"], case["inter"]
        return {"bytes": BF16 * (m * k + 2 * i * k + m * i), "flops": 2 * m * k * 2 * i}
    if op == "norm":
        n = case["rows"] * case["k"]
        # both inputs and the residual out, the statistics, the normalised rows: the
        # residual need not be read back
        return {"bytes": 2 * n * 4 + 2 * case["k"] * (1 + case["beta"]) + F32 * case["rows"], "flops": 6 * n}
    h, kvh = case["heads"], case["kv_heads"]
    tok = kvh * D * BF16 * 2
    if op == "stage1":
        lens = _kv_lens(case)
        rows = case["batch"] * case["q_len"] * h
        return {"bytes": int(lens.sum()) * tok + rows * (D * (BF16 + F32) + 8 * F32)
                + int(_pages(lens).sum()) * I32 + case["batch"] * 2 * I64,
                "flops": 4 * D * h * case["q_len"] * int(lens.sum())}
    lens = _suffix_lens(case)
    rows = case["batch"] * h
    nbytes = int(lens.sum()) * tok + rows * (2 * D * BF16 + F32) + int(_pages(lens).sum()) * I32 + case["batch"] * I64
    flops = 4 * D * h * int(lens.sum())
    if op == "cascade":
        nbytes += case["prefix"] * tok + int(_pages(case["prefix"])) * I32 + I64
        flops += 4 * D * rows * case["prefix"]
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the distance from exact(), itself mostly the rounding of the
    outputs to 16 bits and, in stage 1, of the probabilities to bf16."""
    if case["op"] == "norm" and case["dtype"] == "fp16":
        return {"rel": 1.5e-3, "max": 1e-2}
    if case["op"] == "merge" and case["out_code"] == 2:
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 1e-2, "max": 8e-2}


# ---- inputs -----------------------------------------------------------------------
class _Gen:
    """Seeded device normals and host permutations."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)
        self.rng = np.random.default_rng(seed)

    def normal(self, *shape, dtype=torch.bfloat16, std=1.0):
        return torch.empty(*shape, device=DEV, dtype=dtype).normal_(0.0, std, generator=self.g)


def _dev(x, dtype):
    return torch.from_numpy(np.ascontiguousarray(x)).to(device=DEV, dtype=dtype)


def _tables(gen, lens):
    """Block table of the requests over scattered pages of one pool, and the pool's pages."""
    n = _pages(lens)
    phys = gen.rng.permutation(int(n.sum()))
    table = np.zeros((len(n), max(1, int(n.max()))), dtype=np.int32)
    at = 0
    for b, c in enumerate(n):
        table[b, :c] = phys[at:at + c]
        at += c
    return table, int(n.sum())


def prepare(case, seed):
    gen = _Gen(seed)
    op = case["op"]
    s = {"case": case}
    if op == "merge":
        t, h = case["tokens"], case["heads"]
        s["o1"] = gen.normal(t, h, D, dtype=torch.float32)
        s["o2"] = gen.normal(t, h, D)
        # log-sum-exps of a long shared prefix and of a shorter suffix
        l1 = gen.normal(t, h, dtype=torch.float32, std=0.5) + 9.0
        l2 = gen.normal(t, h, dtype=torch.float32, std=1.0) + 7.0
        if case["some_empty"]:
            empty = _dev(gen.rng.random(t) < 0.1, torch.bool)
            l2[empty] = -math.inf
            s["o2"][empty] = 0
        s["lse1"] = l1.reshape(-1, 1).expand(-1, 8).contiguous().reshape(-1)
        s["lse2"] = l2.reshape(-1)
        return s
    if op == "gateup":
        s["x"] = gen.normal(case["m"], case["k"])
        s["w"] = gen.normal(2 * case["inter"], case["k"], std=0.02)
        s["out"] = torch.empty(case["m"], case["inter"], device=DEV, dtype=torch.bfloat16)
        return s
    if op == "norm":
        dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float16
        s["x1"] = gen.normal(case["rows"], case["k"], dtype=dt)
        s["x2"] = gen.normal(case["rows"], case["k"], dtype=dt)
        s["gamma"] = (1.0 + gen.normal(case["k"], dtype=torch.float32, std=0.1)).to(dt)
        s["beta"] = gen.normal(case["k"], dtype=dt, std=0.1) if case["beta"] else None
        return s
    h, kvh = case["heads"], case["kv_heads"]
    if op == "stage1":
        lens = gen.rng.permutation(_kv_lens(case))
        table, blocks = _tables(gen, lens)
        s["q"] = gen.normal(case["batch"] * case["q_len"], h, D)
        s["k"], s["v"] = gen.normal(blocks, PAGE, kvh, D), gen.normal(blocks, PAGE, kvh, D)
        s["table"], s["lens"] = _dev(table, torch.int32), _dev(lens, torch.int64)
        s["q_lens"] = torch.full((case["batch"],), case["q_len"], dtype=torch.int64, device=DEV)
        return s
    lens = gen.rng.permutation(_suffix_lens(case))
    s["q"] = gen.normal(case["batch"], h, D)
    if op == "cascade" and case["layout"] == 0:
        # one pool for the shared prefix and the suffixes
        table, blocks = _tables(gen, np.concatenate([[case["prefix"]], lens]))
        s["table"] = _dev(table[1:, :max(1, int(_pages(lens).max()))], torch.int32)
        s["ptable"] = _dev(table[:1, :int(_pages(case["prefix"]))], torch.int32)
        s["k"], s["v"] = gen.normal(blocks, PAGE, kvh, D), gen.normal(blocks, PAGE, kvh, D)
        s["pk"], s["pv"] = s["k"], s["v"]
    else:
        table, blocks = _tables(gen, lens)
        s["table"] = _dev(table, torch.int32)
        shape = (blocks, kvh, PAGE, D) if case["layout"] else (blocks, PAGE, kvh, D)
        s["k"], s["v"] = gen.normal(*shape), gen.normal(*shape)
        if op == "cascade":
            ptable, pblocks = _tables(gen, [case["prefix"]])
            s["ptable"] = _dev(ptable, torch.int32)
            s["pk"], s["pv"] = gen.normal(pblocks, PAGE, kvh, D), gen.normal(pblocks, PAGE, kvh, D)
    s["lens"] = _dev(lens, torch.int64)
    if op == "cascade":
        s["plen"] = torch.tensor([case["prefix"]], dtype=torch.int64, device=DEV)
    return s


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "cascade":
        return torch.ops.npu.cascade_decode(s["q"], s["pk"], s["pv"], s["ptable"], s["plen"], s["k"], s["v"],
                                            s["table"], s["lens"], case["layout"])
    if op == "stage1":
        return torch.ops.npu.fa_fp32_stage1(s["q"], s["k"], s["v"], s["table"], s["q_lens"], s["lens"], case["q_len"])
    if op == "suffix":
        return torch.ops.npu.suffix_decode(s["q"], s["k"], s["v"], s["table"], s["lens"], case["layout"])
    if op == "merge":
        return torch.ops.npu.lse_merge(s["o1"], s["o2"], s["lse1"], s["lse2"], case["out_code"])
    if op == "gateup":
        return torch.ops.npu.f3_gateup_epilogue(s["x"], s["w"], None, s["out"], 1)[0]
    x_out, _, _ = torch.ops.npu.add_rms_norm_stats(s["x1"], s["x2"], None, None, EPS, 0)
    _, rstd, y = torch.ops.npu.add_rms_norm_stats(x_out, s["x2"], s["gamma"], s["beta"], EPS, 1)
    return x_out, rstd, y


# ---- the same in 64 bits ------------------------------------------------------------
def _attend(q, k, v):
    """q [kvh, rows, D], k and v [kvh, tokens, D] in fp64 -> O [kvh, rows, D], LSE [kvh, rows]."""
    o, lse = torch.empty_like(q), torch.empty(q.shape[:2], dtype=torch.float64, device=q.device)
    for g in range(q.shape[0]):
        sc = q[g] @ k[g].t().contiguous() * SCALE
        lse[g] = torch.logsumexp(sc, dim=-1)
        o[g] = torch.exp(sc - lse[g][:, None]) @ v[g]
    return o, lse


def _gather(pool, pages, n, layout=0):
    """The n tokens behind `pages` as fp64 [kvh, n, D]."""
    x = pool[pages.long()]
    x = x.permute(1, 0, 2, 3) if layout else x.permute(2, 0, 1, 3)
    return x.reshape(x.shape[0], -1, D)[:, :n].double().contiguous()


def _rows(q, kvh):
    """[T, H, D] -> fp64 [kvh, T * group, D]."""
    t, h, _ = q.shape
    return q.double().reshape(t, kvh, h // kvh, D).permute(1, 0, 2, 3).reshape(kvh, -1, D).contiguous()


def _unrows(x, t, h):
    """[kvh, T * group, ...] -> [T, H, ...]."""
    kvh = x.shape[0]
    x = x.reshape(kvh, t, h // kvh, *x.shape[2:])
    return x.transpose(0, 1).reshape(t, h, *x.shape[3:])


def exact(case, seed):
    s = prepare(case, seed)
    op = case["op"]
    if op == "merge":
        l1, l2 = s["lse1"].view(-1, 8)[:, 0].double(), s["lse2"].double()
        lse = torch.logaddexp(l1, l2)
        o1, o2 = s["o1"].double().view(-1, D), s["o2"].double().view(-1, D)
        o = o1 * torch.exp(l1 - lse)[:, None] + o2 * torch.exp(l2 - lse)[:, None]
        return o.view(s["o1"].shape)
    if op == "gateup":
        x, i = s["x"].double(), case["inter"]
        g, u = x @ s["w"][:i].double().t(), x @ s["w"][i:].double().t()
        return g * torch.sigmoid(g) * u
    if op == "norm":
        x = s["x1"].double() + s["x2"].double()
        rstd = torch.rsqrt(x.square().mean(dim=1, keepdim=True) + EPS)
        y = x * rstd * s["gamma"].double() + (0 if s["beta"] is None else s["beta"].double())
        pad = torch.zeros((case["rows"] + 7) // 8 * 8, 1, dtype=torch.float64, device=DEV)
        pad[:case["rows"]] = rstd
        return x, pad, y
    h, kvh = case["heads"], case["kv_heads"]
    lens = s["lens"].tolist()
    if op == "stage1":
        n, outs, lses = case["q_len"], [], []
        for b, ln in enumerate(lens):
            pg = s["table"][b, :(ln + PAGE - 1) // PAGE]
            o, lse = _attend(_rows(s["q"][b * n:(b + 1) * n], kvh), _gather(s["k"], pg, ln), _gather(s["v"], pg, ln))
            outs.append(_unrows(o, n, h))
            lses.append(_unrows(lse, n, h))
        return torch.cat(outs), torch.cat(lses).reshape(-1, 1).expand(-1, 8).reshape(-1)
    outs, lses = [], []
    for b, ln in enumerate(lens):
        pg = s["table"][b, :(ln + PAGE - 1) // PAGE]
        o, lse = _attend(_rows(s["q"][b:b + 1], kvh), _gather(s["k"], pg, ln, case["layout"]),
                         _gather(s["v"], pg, ln, case["layout"]))
        outs.append(_unrows(o, 1, h))
        lses.append(_unrows(lse, 1, h))
    o2, l2 = torch.cat(outs), torch.cat(lses)
    if op == "suffix":
        return o2, l2.reshape(-1)
    p = case["prefix"]
    o1, l1 = _attend(_rows(s["q"], kvh), _gather(s["pk"], s["ptable"][0], p), _gather(s["pv"], s["ptable"][0], p))
    o1, l1 = _unrows(o1, case["batch"], h), _unrows(l1, case["batch"], h)
    lse = torch.logaddexp(l1, l2)
    o = o1 * torch.exp(l1 - lse)[..., None] + o2 * torch.exp(l2 - lse)[..., None]
    return o, lse.reshape(-1)
