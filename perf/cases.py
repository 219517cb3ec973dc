"""The measured work of the library: what a program that serves quantized models has it do.

A case names an operation of the public binding (``uefi-gpu_amd/uq.py`` and the C
ABI behind it) and its sizes. Sizes come from the Qwen2.5-1.5B shape, the MoE
layer and the frontier MoE block that the benchmark and the tests run. Weights
and activations are the seeded synthetic ones of the benchmark (block scales
lognormal around 0.01, codes uniform, activations N(0, 1)).

Operations:

* ``matvec``  host x -> host y, one weight with int8 activations (``uq.matvec``)
* ``batch``   host x -> three host outputs, the q/k/v group (``uq.batch``)
* ``static``  device x -> device y of one weight (``uq_matvec_static``)
* ``mlp``     quantize, fused gate/up, quantize, down on device buffers
* ``linear``  fp32-activation reader, device (``uq_linear_dev``) or host (``uq.linear``)
* ``tables``  the linears of a frontier MoE block: router, then two job tables a token
* ``moe``     the MoE expert layer on device buffers, token by token
* ``prefill`` a prompt through the whole decoder, its logits read back
* ``decode``  greedy steps of the whole decoder after a prompt, the last logits read back
"""
import ctypes
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "uefi-gpu_amd"))

import uq  # noqa: E402

KINDS = {"F32": uq.KIND_F32, "BF16": uq.KIND_BF16, "Q8_0": uq.KIND_Q8_0, "Q4_K": uq.KIND_Q4_K, "Q3_K": uq.KIND_Q3_K,
         "Q6_K": uq.KIND_Q6_K, "IQ3_XXS": uq.KIND_IQ3_XXS, "IQ4_NL": uq.KIND_IQ4_NL, "IQ4_XS": uq.KIND_IQ4_XS}
# values and GGUF bytes of one block
BLOCK = {"F32": (1, 4), "BF16": (1, 2), "Q8_0": (32, 34), "Q4_K": (256, 144), "Q3_K": (256, 110), "Q6_K": (256, 210),
         "IQ3_XXS": (256, 98), "IQ4_NL": (32, 18), "IQ4_XS": (256, 136)}
INT8_KINDS = ("Q8_0", "Q4_K", "Q3_K")
READER_KINDS = ("F32", "BF16", "Q8_0", "Q6_K", "IQ3_XXS", "IQ4_NL", "IQ4_XS")
# the largest weight a drawn case may hold, in values and in bytes (the Q6_K head below)
MOST_VALUES, MOST_BYTES = 151936 * 2560, 151936 * 2560 // 256 * 210


def listed():
    return [
        # one k or v projection from host memory: the smallest call there is, all latency
        {"name": "matvec kv host", "op": "matvec", "kind": "Q8_0", "n": 1536, "m": 256},
        # the router of a frontier MoE block from host memory, a small call of the reader
        {"name": "linear router host", "op": "linear", "kind": "F32", "n": 2560, "m": 256, "host": True},
        # the feed-forward block of a decoder layer, token by token, in two weight formats
        {"name": "mlp q8_0", "op": "mlp", "kind": "Q8_0", "n": 1536, "hidden": 8960},
        {"name": "mlp q4_k", "op": "mlp", "kind": "Q4_K", "n": 1536, "hidden": 8960},
        # output heads: the largest matvecs of a decode step
        {"name": "head q8_0", "op": "static", "kind": "Q8_0", "n": 1536, "m": 151936},
        {"name": "head q3_k", "op": "static", "kind": "Q3_K", "n": 1536, "m": 151936},
        # fp32-activation reader: an ordinary linear with a ragged row count, and a head
        {"name": "linear iq4_xs", "op": "linear", "kind": "IQ4_XS", "n": 2560, "m": 3001, "host": False},
        {"name": "linear head q6_k", "op": "linear", "kind": "Q6_K", "n": 2560, "m": 151936, "host": False},
        # frontier MoE block: 10 routed IQ3_XXS / IQ4_NL experts and a shared Q8_0 expert a token
        {"name": "frontier moe tables", "op": "tables", "n": 2560, "ff": 640, "experts": 256, "top_k": 10, "tokens": 8},
        # MoE expert layer of a decode step
        {"name": "moe q3_k", "op": "moe", "kind": "Q3_K", "n": 2048, "ff": 768, "experts": 128, "top_k": 8, "tokens": 8},
        # whole calls on the Qwen2.5-1.5B shape: a prompt, and greedy decoding behind it
        {"name": "prefill 512", "op": "prefill", "layers": 28, "prompt": 512},
        {"name": "decode 512", "op": "decode", "layers": 28, "prompt": 512, "steps": 32},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return int(round(lo * (hi / lo) ** rng.random()))


def _cols(rng, kind, lo, hi):
    step = max(8, BLOCK[kind][0])
    return max(step, _log(rng, lo, hi) // step * step)


def _rows(rng, kind, n, lo, hi):
    return max(1, min(_log(rng, lo, hi), MOST_VALUES // n, MOST_BYTES // _row_bytes(kind, n)))


def draw(rng):
    op = rng.choice(["matvec", "batch", "static", "mlp", "linear", "linear", "linear", "tables", "moe", "prefill", "decode"])
    if op in ("matvec", "static"):
        kind = rng.choice(INT8_KINDS)
        n = _cols(rng, kind, 256, 16384)
        return {"op": op, "kind": kind, "n": n, "m": _rows(rng, kind, n, 64, 151936 if op == "static" else 16384)}
    if op == "batch":
        kind = rng.choice(INT8_KINDS)
        n = _cols(rng, kind, 512, 8192)
        kv = _rows(rng, kind, n, 64, 1024)
        return {"op": op, "kind": kind, "n": n, "m": n, "kv": kv}
    if op == "mlp":
        kind = rng.choice(INT8_KINDS)
        return {"op": op, "kind": kind, "n": _cols(rng, kind, 512, 4096), "hidden": _cols(rng, kind, 1024, 16384)}
    if op == "linear":
        kind = rng.choice(READER_KINDS)
        n = _cols(rng, kind, 256, 16384)
        host = rng.random() < 0.3
        return {"op": op, "kind": kind, "n": n, "m": _rows(rng, kind, n, 17, 16384 if host else 151936), "host": host}
    if op == "tables":
        return {"op": op, "n": 256 * rng.randint(2, 10), "ff": 32 * rng.randint(8, 24), "experts": rng.randint(16, 256),
                "top_k": rng.randint(2, 10), "tokens": rng.randint(1, 8)}
    if op == "moe":
        kind = rng.choice(INT8_KINDS)
        return {"op": op, "kind": kind, "n": 256 * rng.randint(2, 8), "ff": 256 * rng.randint(1, 3),
                "experts": rng.randint(16, 128), "top_k": rng.randint(2, 8), "tokens": rng.randint(1, 8)}
    layers = rng.choice([1, 2, rng.randint(3, 28)])
    if op == "prefill":
        return {"op": op, "layers": layers, "prompt": _log(rng, 8, 640)}
    return {"op": op, "layers": layers, "prompt": _log(rng, 8, 960), "steps": rng.randint(1, 32)}


# ---------------------------------------------------------------- inputs
def _row_bytes(kind, n):
    vals, size = BLOCK[kind]
    return n // vals * size


def _seed(seed, tag):
    return uq.tensor_seed(seed + 0x5EED, tag)


def _raw(kind, seed, tag, m, n):
    return uq.synth_quant(KINDS[kind], _seed(seed, tag), m, n)


def _x(seed, tag, n):
    return uq.synth_normal(_seed(seed, tag), n)


def _cfg(case):
    return dict(uq.QWEN25_15B, layers=case["layers"])


def _prompt(case, seed):
    return uq.synth_tokens(_seed(seed, "prompt"), case["prompt"], uq.QWEN25_15B["vocab"])


def _moe_cfg(case):
    return dict(dim=case["n"], ff=case["ff"], experts=case["experts"], top_k=case["top_k"],
                expert_kind=KINDS[case["kind"]], shared_kind=uq.KIND_Q8_0)


def _moe_inputs(case, seed):
    xs = _x(seed, "x", case["tokens"] * case["n"]).reshape(case["tokens"], case["n"])
    lg = _x(seed, "logits", case["tokens"] * case["experts"]).reshape(case["tokens"], case["experts"])
    return xs, lg


def _weights(case):
    """(tag, kind, rows, columns) of the case's plain weights."""
    op, n = case["op"], case["n"]
    if op == "batch":
        return [("q", case["kind"], case["m"], n), ("k", case["kind"], case["kv"], n), ("v", case["kind"], case["kv"], n)]
    if op == "mlp":
        h = case["hidden"]
        return [("gate", case["kind"], h, n), ("up", case["kind"], h, n), ("down", case["kind"], n, h)]
    return [("w", case["kind"], case["m"], n)]


def _experts(case, seed):
    """The routed expert ids of each token, drawn from the bank."""
    r = np.random.default_rng(_seed(seed, "ids"))
    return [[int(e) for e in r.choice(case["experts"], case["top_k"], replace=False)] for _ in range(case["tokens"])]


def _table_weights(case, seed):
    """(tag, kind, rows, columns) of the frontier block's weights that its tokens use."""
    n, ff = case["n"], case["ff"]
    out = [("router", "F32", case["experts"], n), ("sscale", "F32", 1, n), ("sgate", "Q8_0", ff, n),
           ("sup", "Q8_0", ff, n), ("sdown", "Q8_0", n, ff)]
    for e in sorted({e for ids in _experts(case, seed) for e in ids}):
        out += [("gate%d" % e, "IQ3_XXS", ff, n), ("up%d" % e, "IQ3_XXS", ff, n), ("down%d" % e, "IQ4_NL", n, ff)]
    return out


def _table_jobs(case, seed):
    """Per token its three tables: lists of (weight tag, input name, rows)."""
    n, ff, k = case["n"], case["ff"], case["top_k"]
    out = []
    for t, ids in enumerate(_experts(case, seed)):
        x = "x%d" % t
        first = [(p + str(e), x, ff) for e in ids for p in ("gate", "up")]
        first += [("sgate", x, ff), ("sup", x, ff), ("sscale", x, 1)]
        second = [("down%d" % e, "mid%d.%d" % (t, i), n) for i, e in enumerate(ids)] + [("sdown", "mid%d.%d" % (t, k), n)]
        out.append([[("router", x, case["experts"])], first, second])
    return out


def _table_input(case, seed, name):
    return _x(seed, name, case["ff"] if name.startswith("mid") else case["n"])


def _weight(kind, seed, tag, m, n):
    return uq.Weight(KINDS[kind], n, m, _raw(kind, seed, tag, m, n))


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def prepare(case, seed):
    uq.init(0)
    op = case["op"]
    s = {"case": case}
    if op in ("prefill", "decode"):
        s["model"] = uq.Qwen2Model(_cfg(case), uq.synth_qwen2(_cfg(case), _seed(seed, "model")))
        s["prompt"] = _prompt(case, seed)
        if op == "decode":
            s["first"] = s["model"].prefill(s["prompt"])
        return s
    if op == "moe":
        s["layer"] = uq.MoeLayer(_moe_cfg(case), *uq.synth_moe(_moe_cfg(case), _seed(seed, "moe")))
        s["x"], s["logits"] = (_dev(a) for a in _moe_inputs(case, seed))
        s["out"] = torch.empty_like(s["x"])
        torch.cuda.synchronize()
        return s
    if op == "tables":
        s["weights"] = {tag: _weight(kind, seed, tag, m, n) for tag, kind, m, n in _table_weights(case, seed)}
        tables = _table_jobs(case, seed)
        s["inputs"] = {x: _dev(_table_input(case, seed, x)) for x in sorted({j[1] for t in tables for b in t for j in b})}
        s["outs"], s["tables"] = [], []
        for batch in (b for t in tables for b in t):
            out = torch.empty(sum(m for _, _, m in batch), dtype=torch.float32, device="cuda")
            at = np.cumsum([0] + [m for _, _, m in batch])
            jobs = [uq.LinearJob(s["weights"][w].handle, s["inputs"][x].data_ptr(), out.data_ptr() + 4 * int(o))
                    for (w, x, _), o in zip(batch, at)]
            s["outs"].append(out)  # a table's outputs one behind the other, in job order
            s["tables"].append(((uq.LinearJob * len(jobs))(*jobs), len(jobs)))
        torch.cuda.synchronize()
        return s
    s["w"] = [_weight(kind, seed, tag, m, n) for tag, kind, m, n in _weights(case)]
    x = _x(seed, "x", case["n"])
    if op in ("matvec", "batch") or case.get("host"):
        s["x"] = x
        return s
    s["x"] = _dev(x)
    s["y"] = torch.empty(s["w"][-1].m, dtype=torch.float32, device="cuda")
    if op == "mlp":
        n, h = case["n"], case["hidden"]
        s["h"] = torch.empty(h, dtype=torch.float32, device="cuda")
        s["q"] = [torch.empty(v, dtype=torch.int8, device="cuda") for v in (n, h)]
        s["s"] = [torch.empty(v // 32, dtype=torch.float32, device="cuda") for v in (n, h)]
    torch.cuda.synchronize()
    return s


def _ok(rc):
    if rc != uq.OK:
        raise uq.UqError(rc, uq.lib().uq_last_error().decode(errors="replace"))


def run(s):
    case, L = s["case"], uq.lib()
    op = case["op"]
    if op == "matvec":
        return uq.matvec(s["w"][0], s["x"])
    if op == "batch":
        return uq.batch(s["w"], s["x"])
    if op == "static":
        _ok(L.uq_matvec_static(s["w"][0].handle, s["x"].data_ptr(), s["y"].data_ptr(), None))
        return s["y"]
    if op == "linear":
        if case["host"]:
            return uq.linear(s["w"][0], s["x"])
        _ok(L.uq_linear_dev(s["w"][0].handle, s["x"].data_ptr(), s["y"].data_ptr(), None))
        return s["y"]
    if op == "mlp":
        gate, up, down = (w.handle for w in s["w"])
        (q0, q1), (s0, s1) = s["q"], s["s"]
        _ok(L.uq_quant_act_dev(s["x"].data_ptr(), case["n"], q0.data_ptr(), s0.data_ptr(), None))
        _ok(L.uq_gateup_q_dev(gate, up, q0.data_ptr(), s0.data_ptr(), s["h"].data_ptr(), None))
        _ok(L.uq_quant_act_dev(s["h"].data_ptr(), case["hidden"], q1.data_ptr(), s1.data_ptr(), None))
        _ok(L.uq_matvec_q_dev(down, q1.data_ptr(), s1.data_ptr(), s["y"].data_ptr(), None))
        return {"h": s["h"], "y": s["y"]}
    if op == "tables":
        for jobs, count in s["tables"]:
            _ok(L.uq_linear_multi_dev(jobs, count, None))
        return s["outs"]
    if op == "moe":
        n, e = 4 * case["n"], 4 * case["experts"]
        x, lg, out = s["x"].data_ptr(), s["logits"].data_ptr(), s["out"].data_ptr()
        for t in range(case["tokens"]):
            s["layer"].ffn_dev(x + t * n, lg + t * e, out + t * n)
        return s["out"]
    if op == "prefill":
        first = s["model"].prefill(s["prompt"])
        return {"id": int(first), "logits": s["model"].logits()}
    ids, _ = s["model"].decode_run(s["first"], case["prompt"], case["steps"])
    return {"ids": ids.astype(np.int64), "logits": s["model"].logits()}


# ---------------------------------------------------------------- the work that a pass cannot do without
def _matrix(kind, m, n):
    return _row_bytes(kind, n) * m


def _layer_bytes(c):
    kv = c["kv_heads"] * c["head_dim"]
    rows = 2 * c["dim"] + 2 * kv + 2 * c["hidden"]
    return _matrix("Q8_0", rows, c["dim"]) + _matrix("Q8_0", c["dim"], c["hidden"])


def work(case):
    op = case["op"]
    if op in ("prefill", "decode"):
        c = _cfg(case)
        weights, head, kv = c["layers"] * _layer_bytes(c), _matrix("Q8_0", c["vocab"], c["dim"]), c["kv_heads"] * c["head_dim"]
        out = 4 * c["vocab"]
        values = weights // 34 * 32
        if op == "prefill":
            t = case["prompt"]
            attention = c["layers"] * 2 * c["heads"] * c["head_dim"] * t * (t + 1)
            return {"bytes": weights + head + t * _row_bytes("Q8_0", c["dim"]) + c["layers"] * t * kv * 4 + out,
                    "flops": 2 * values * t + attention + 2 * c["vocab"] * c["dim"]}
        steps, pos = case["steps"], case["prompt"]
        seen = sum(pos + i + 1 for i in range(steps))
        return {"bytes": steps * (weights + head + c["layers"] * kv * 4) + c["layers"] * seen * kv * 4 + out,
                "flops": steps * 2 * (values + c["vocab"] * c["dim"]) + c["layers"] * 4 * c["heads"] * c["head_dim"] * seen}
    if op == "moe":
        n, ff, t = case["n"], case["ff"], case["tokens"]
        one = 2 * _matrix(case["kind"], ff, n) + _matrix(case["kind"], n, ff)
        shared = 2 * _matrix("Q8_0", ff, n) + _matrix("Q8_0", n, ff)
        return {"bytes": t * (case["top_k"] * one + shared + 12 * n + 4 * case["experts"]),
                "flops": t * 6 * n * ff * (case["top_k"] + 1)}
    if op == "tables":
        n, ff, k = case["n"], case["ff"], case["top_k"]
        token = _matrix("F32", case["experts"] + 1, n) + k * (2 * _matrix("IQ3_XXS", ff, n) + _matrix("IQ4_NL", n, ff))
        token += 2 * _matrix("Q8_0", ff, n) + _matrix("Q8_0", n, ff)
        token += 4 * (n + case["experts"] + (2 * k + 2) * ff + 1 + (k + 1) * (ff + n))
        return {"bytes": case["tokens"] * token,
                "flops": case["tokens"] * 2 * n * (case["experts"] + 1 + 3 * (k + 1) * ff)}
    weights = _weights(case)
    total = sum(_matrix(kind, m, n) for _, kind, m, n in weights)
    if op == "mlp":
        io = 4 * (case["n"] + case["hidden"] + case["n"])
    else:
        io = 4 * (case["n"] + sum(m for _, _, m, _ in weights))
    return {"bytes": total + io, "flops": sum(2 * m * n for _, _, m, n in weights)}


# ---------------------------------------------------------------- 64-bit restatement
IQ4 = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)
# the IQ3_XXS grid of ggml (MIT licence, third_party/LICENSE.ggml): 256 entries of four values 8d + 4 (62 for d = 7)
IQ3 = (
    "000020004000110031007100020022001300240037005700101030100110211012105210031023101410451007100020"
    "202040201120022022201320332073201520752057201030703001302130523007303140734044407540374057401050"
    "705023502550536046600170417061703470167010013001010121011201320103012301430174010501001120111111"
    "021122111021302101212121122103212721003120310231133164316631104150410541025142516451175150612271"
    "047100022002110231020202220262021302240210123012501201122112121203123612761207120022202211227122"
    "022222227322042255221032013241320732473253423542305272521452475210723072617254721003010321031203"
    "320305035603270300132013021313134413641310233023012352232523272311333333034374432743005360532253"
    "555341636363366333730673400471045304730435047504471402247324042406246624703454344044154446445254"
    "345407545074017421740374210514050705001560156215551541252325272520353535014532457245274520551355"
    "056542752475420644066406460612161616712646260336633644465056255633663076127630075007700701072307"
    "2507621704172127542725270037513733370637124714470057205742570367")


def _f64(x):
    return torch.from_numpy(np.ascontiguousarray(x)).cuda().double()


def _half(b):
    return b.contiguous().view(torch.float16).double()


def _signed(b):
    return b.view(torch.int8).double()


def _values(kind, raw, m, n):
    """The weight's values [m][n] in 64 bits, from its GGUF bytes on the GPU."""
    vals, size = BLOCK[kind]
    b = raw.view(m * (n // vals), size)
    if kind == "F32":
        return b.contiguous().view(torch.float32).double().view(m, n)
    if kind == "BF16":
        return b.contiguous().view(torch.bfloat16).double().view(m, n)
    if kind == "Q8_0":
        return (_half(b[:, :2]) * _signed(b[:, 2:].contiguous())).view(m, n)
    book = torch.tensor(IQ4, dtype=torch.float64, device=raw.device)
    if kind == "IQ4_NL":
        q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1)
        return (_half(b[:, :2]) * book[q.long()]).view(m, n)
    w = b.int()
    if kind == "IQ4_XS":
        j = torch.arange(8, device=raw.device)
        high = (w[:, 2:3] | w[:, 3:4] << 8) >> (2 * j) & 3
        sc = (w[:, 4:8].repeat_interleave(2, 1) >> (4 * (j % 2)) & 15 | high << 4).double() - 32
        q = w[:, 8:].view(-1, 8, 16)
        q = torch.cat([q & 15, q >> 4], 2)
        return ((_half(b[:, :2]) * sc).unsqueeze(2) * book[q.long()]).reshape(m, n)
    if kind == "IQ3_XXS":
        level = torch.tensor([4, 12, 20, 28, 36, 44, 52, 62], dtype=torch.float64, device=raw.device)
        grid = level[torch.tensor([int(c) for c in IQ3], device=raw.device)].view(256, 4)
        q = grid[w[:, 2:66].long()].view(-1, 8, 4, 8)
        aux = b[:, 66:].contiguous().view(torch.int32).long() & 0xFFFFFFFF
        s7 = aux.unsqueeze(2) >> (7 * torch.arange(4, device=raw.device)) & 127
        bit = s7.unsqueeze(3) >> torch.arange(7, device=raw.device) & 1
        bit = torch.cat([bit, bit.sum(3, keepdim=True) & 1], 3)
        scale = _half(b[:, :2]) * (0.5 + (aux >> 28).double()) * 0.5
        return (scale.view(-1, 8, 1, 1) * q * (1 - 2 * bit)).reshape(m, n)
    if kind == "Q6_K":
        lo, hi = w[:, :128].view(-1, 2, 64), w[:, 128:192].view(-1, 2, 32)
        q = torch.stack([lo[..., :32] & 15, lo[..., 32:] & 15, lo[..., :32] >> 4, lo[..., 32:] >> 4], 2)
        q = q | torch.stack([hi >> s & 3 for s in (0, 2, 4, 6)], 2) << 4
        sc = _signed(b[:, 192:208].contiguous()).view(-1, 2, 4, 2)
        return (_half(b[:, 208:]).view(-1, 1, 1, 1) * sc.repeat_interleave(16, 3) * (q - 32).double()).reshape(m, n)
    if kind == "Q4_K":
        s = w[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, s[:, 8:] & 15 | s[:, :4] >> 6 << 4], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, s[:, 8:] >> 4 | s[:, 4:8] >> 6 << 4], 1).double()
        q = w[:, 16:].view(-1, 4, 32)
        q = torch.stack([q & 15, q >> 4], 2).view(-1, 8, 32).double()
        return ((_half(b[:, :2]) * sc).unsqueeze(2) * q - (_half(b[:, 2:4]) * mn).unsqueeze(2)).reshape(m, n)
    # Q3_K: high bits, low two bits, 16 six-bit scales, d
    lo, hi = w[:, 32:96].view(-1, 2, 32), w[:, :32]
    q = torch.stack([torch.stack([lo[:, h] >> (2 * j) & 3 | (hi >> (4 * h + j) & 1) << 2 for j in range(4)], 1) for h in range(2)], 1)
    s, k = w[:, 96:108], torch.arange(16, device=raw.device)
    low = torch.cat([s[:, :8] & 15, s[:, :8] >> 4], 1)
    sc = (low | (s[:, 8 + k % 4] >> (2 * (k // 4)) & 3) << 4).double() - 32
    q = (q - 4).view(-1, 16, 16).double()
    return (_half(b[:, 108:]).unsqueeze(2) * sc.unsqueeze(2) * q).reshape(m, n)


def _product(kind, raw, m, n, x):
    """W x [m] or W x for each row of x, in 64 bits, some rows of W at a time."""
    raw = torch.from_numpy(raw).cuda()
    rb, step = _row_bytes(kind, n), max(1, (1 << 25) // n)
    parts = [_values(kind, raw[r * rb:min(m, r + step) * rb], min(m, r + step) - r, n) @ x.T for r in range(0, m, step)]
    return torch.cat(parts).T.contiguous()


def _codes(x):
    """The int8 activations of the int8 path times their block scales: 32 values share amax / 127."""
    b = x.reshape(-1, 32)
    a = b.abs().amax(1, keepdim=True)
    q = torch.where(a > 0, b * (127 / a.clamp_min(1e-300)), b * 0).round().clamp(-127, 127)
    return (q * (a / 127)).view(x.shape)


def _silu(g):
    return g / (1 + torch.exp(-g))


class _Decoder:
    """The decoder of one or two layers in 64 bits, its K and V rounded to fp16 as the cache holds them."""

    def __init__(self, c, seed):
        self.c, self.t = c, uq.synth_qwen2(c, seed)
        self.K, self.V = ([torch.zeros(0, c["kv_heads"], c["head_dim"], dtype=torch.float64, device="cuda")] * c["layers"] for _ in "kv")

    def mat(self, name, x):
        _, n, rows, raw = self.t[name]
        return _product("Q8_0", raw, rows, n, x)

    def norm(self, x, name):
        return _codes(x / torch.sqrt((x * x).mean(1, keepdim=True) + self.c["eps"]) * _f64(self.t[name][3]))

    def rope(self, v, heads, pos):
        hd = self.c["head_dim"]
        i = torch.arange(hd // 2, dtype=torch.float64, device="cuda")
        ang = (pos.double().view(-1, 1) * self.c["theta"] ** (-2 * i / hd)).unsqueeze(1)
        v = v.view(-1, heads, hd)
        a, b = v[..., :hd // 2], v[..., hd // 2:]
        return torch.cat([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()], 2)

    def forward(self, tokens):
        c, t = self.c, len(tokens)
        hd, H, KV = c["head_dim"], c["heads"], c["kv_heads"]
        pos = torch.arange(self.K[0].shape[0], self.K[0].shape[0] + t, device="cuda")
        rb = _row_bytes("Q8_0", c["dim"])
        rows = self.t["token_embd.weight"][3].reshape(-1, rb)[np.asarray(tokens, np.int64)]
        x = _values("Q8_0", torch.from_numpy(np.ascontiguousarray(rows).reshape(-1)).cuda(), t, c["dim"])
        for l in range(c["layers"]):
            b = "blk.%d." % l
            xn = self.norm(x, b + "attn_norm.weight")
            q, k, v = (self.mat(b + "attn_%s.weight" % p, xn) + _f64(self.t[b + "attn_%s.bias" % p][3]) for p in "qkv")
            q, k = self.rope(q, H, pos), self.rope(k, KV, pos)
            self.K[l] = torch.cat([self.K[l], k.half().double()])
            self.V[l] = torch.cat([self.V[l], v.view(t, KV, hd).half().double()])
            ks, vs = (a.repeat_interleave(H // KV, 1).transpose(0, 1).contiguous() for a in (self.K[l], self.V[l]))
            s = q.transpose(0, 1) @ ks.transpose(1, 2).contiguous() / hd ** 0.5
            s = s.masked_fill(torch.arange(ks.shape[1], device="cuda") > pos.view(-1, 1), -torch.inf)
            att = (s.softmax(2) @ vs).transpose(0, 1).reshape(t, H * hd)
            x = x + self.mat(b + "attn_output.weight", _codes(att))
            xn = self.norm(x, b + "ffn_norm.weight")
            h = _silu(self.mat(b + "ffn_gate.weight", xn)) * self.mat(b + "ffn_up.weight", xn)
            x = x + self.mat(b + "ffn_down.weight", _codes(h))
        return self.mat("output.weight", self.norm(x[-1:], "output_norm.weight"))[0]


def exact(case, seed):
    """run()'s outputs for these inputs in 64 bits. The int8 path's activations are its int8 codes. None
    for a decoder of more than two layers: one code that rounds the other way moves all layers behind
    it, so that after a few layers no other order of summation gives these logits to better than some 1e-2."""
    op = case["op"]
    if op in ("prefill", "decode"):
        if case["layers"] > 2:
            return None
        d = _Decoder(_cfg(case), _seed(seed, "model"))
        logits = d.forward(_prompt(case, seed))
        if op == "prefill":
            return {"id": None, "logits": logits}
        for _ in range(case["steps"]):
            logits = d.forward([int(logits.argmax())])
        return {"ids": None, "logits": logits}
    if op == "tables":
        raws = {tag: (kind, _raw(kind, seed, tag, m, n), m, n) for tag, kind, m, n in _table_weights(case, seed)}
        product = lambda w, x: _product(*raws[w], _f64(_table_input(case, seed, x)).view(1, -1))[0]  # noqa: E731
        return [torch.cat([product(w, x) for w, x, _ in batch]) for token in _table_jobs(case, seed) for batch in token]
    if op == "moe":
        return _exact_moe(case, seed)
    x = _f64(_x(seed, "x", case["n"])).view(1, -1)
    if op in ("matvec", "batch", "static", "mlp"):
        x = _codes(x)
    outs = []
    for tag, kind, m, n in _weights(case):
        if tag == "down":
            x = _codes(_silu(outs[0]) * outs[1])
        outs.append(_product(kind, _raw(kind, seed, tag, m, n), m, n, x))
    if op == "mlp":
        return {"h": (_silu(outs[0]) * outs[1])[0], "y": outs[2][0]}
    return [o[0] for o in outs] if op == "batch" else outs[0][0]


def _exact_moe(case, seed):
    experts, shared, gate_inp = uq.synth_moe(_moe_cfg(case), _seed(seed, "moe"))
    xs, lg = (_f64(a) for a in _moe_inputs(case, seed))
    n, ff = case["n"], case["ff"]

    def expert(kind, raw, x):
        g, u = (_product(kind, r, ff, n, x) for r in raw[:2])
        return _product(kind, raw[2], n, ff, _codes(_silu(g) * u))[0]

    out = []
    for x, logit in zip(xs, lg):
        p = logit.softmax(0)
        w, ids = p.topk(case["top_k"])
        q = _codes(x).view(1, -1)
        y = torch.sigmoid(_f64(gate_inp) @ x) * expert("Q8_0", shared, q)
        for share, e in zip(w / w.sum(), ids):
            y = y + share * expert(case["kind"], experts[int(e)], q)
        out.append(y)
    return torch.stack(out)


def tolerance(case):
    op = case["op"]
    if op in ("prefill", "decode"):
        # a code that rounds the other way in one layer moves all that follow (see exact)
        return {"rel": 0.03, "max": 0.3, "differ": 0.01}
    if op in ("mlp", "moe"):
        # the hidden vector is rounded to int8 codes: one of them may round the other way
        return {"rel": 1e-3, "max": 0.02}
    # one sum of products an output, rounded to f32
    return {"rel": 1e-6, "max": 1e-5}
