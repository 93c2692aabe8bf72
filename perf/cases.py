"""The work this framework is measured on: its public entry points over the sizes, dtypes and
options that finetuning and prefill with it use.

A case names a path and its sizes:
  train    forward + backward of one attention layer through autograd (the drop-in's functional and
           registry forms, and the GPT-OSS `attention` with learned sink logits)
  prefill  forward only, without gradients
  packed   a padding-free batch, forward + backward (flash_swda_with_sink_varlen)
  padded   a padded batch as transformers hands it over, forward + backward
           (gpt_oss_attention_forward with a [B, L] mask)
  fp8      per-tensor e4m3 quantisation of q, k, v and the fp8 forward
W = 0 stands for a full causal layer (no window).
"""
from __future__ import annotations

import importlib
import math

import torch

fa = importlib.import_module("flashattention-gpt-oss-finetuning_amd")

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _case(name, path, B, Hq, Hkv, L, D, W, S, dtype, learned=False, lens="", do_std=1.0, fp8_pv=False):
    c = dict(path=path, B=B, Hq=Hq, Hkv=Hkv, L=L, D=D, W=W, S=S, dtype=dtype, learned=learned, lens=lens,
             do_std=do_std, fp8_pv=fp8_pv)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one short prompt through a GPT-OSS sliding layer: launches and host work are what counts
        _case("prefill_short", "prefill", 1, 64, 8, 257, 64, 128, 0, "bf16", learned=True),
        # the reference's default benchmark case (16 heads of 16 columns), through the registry form
        _case("reference_default", "train", 1, 16, 16, 4096, 16, 256, 4, "fp16"),
        # the headline: a GPT-OSS sliding layer at 4K context, positional sinks
        _case("sliding_4k", "train", 1, 64, 8, 4096, 64, 128, 4, "bf16"),
        # GPT-OSS's full causal layers: one short finetuning sample of odd length, the 4K context
        # of the headline, and the 8K of the compute-bound config
        _case("full_short_odd", "train", 1, 64, 8, 1001, 64, 0, 0, "bf16", learned=True),
        _case("full_4k", "train", 1, 64, 8, 4096, 64, 0, 0, "bf16", learned=True),
        _case("full_8k", "train", 1, 64, 8, 8192, 64, 0, 0, "bf16"),
        # long-context finetuning, sliding layer
        _case("sliding_32k", "train", 1, 64, 8, 32768, 64, 128, 4, "bf16", do_std=0.1),
        # a batch of wide heads with a larger sink block
        _case("wide_heads_batch", "train", 8, 32, 4, 2048, 128, 512, 16, "fp16"),
        # a padding-free finetuning batch of eight samples, sliding layer with learned sinks
        _case("packed_sliding", "packed", 8, 64, 8, 4096, 64, 128, 0, "bf16", learned=True,
              lens="4096,2048,1024,512,3000,1500,700,3504"),
        # a right-padded finetuning batch, full layer with learned sinks
        _case("padded_full", "padded", 4, 64, 8, 1536, 64, 0, 0, "bf16", learned=True, lens="1536,1187,640,933"),
        # the precision path: float32 tensors through the drop-in
        _case("fp32_sliding", "train", 1, 64, 8, 4096, 64, 128, 4, "fp32"),
        # prefill of a full layer with fp8 products, quantising the activations on the way
        _case("fp8_prefill", "fp8", 1, 64, 8, 8192, 64, 0, 0, "bf16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: lengths of 128 to 32768 rows (sliding) or 8192 (full), spread
    over their logarithm and mostly odd, the head layouts of the listed cases and of smaller models,
    windows from GPT-OSS's 128 to 1024, batches up to 8."""
    path = rng.choice(("train", "train", "train", "train", "prefill", "packed", "padded", "fp8", "fp32", "fp32"))
    while True:
        Hq, Hkv, D = rng.choice(((64, 8, 64), (64, 8, 64), (64, 8, 64), (32, 8, 64), (16, 16, 64), (32, 4, 128),
                                 (32, 8, 128), (16, 16, 16), (16, 8, 16), (16, 1, 32)))
        if path == "fp8" and D < 64:
            continue
        W = rng.choice((0, 0, 0, 128, 128, 256, 512, 1024))
        learned = rng.random() < 0.5
        S = 0 if learned or W == 0 or path in ("packed", "padded") else rng.choice((0, 4, 4, 16))
        dtype = "fp32" if path == "fp32" else "bf16" if path == "fp8" else rng.choice(("bf16", "bf16", "bf16", "fp16"))
        L = _log_int(rng, 128, 8192 if W == 0 else 32768)
        B = rng.choice((1, 1, 1, 2, 4, 8))
        lens = ""
        if path in ("packed", "padded"):
            B = rng.choice((2, 3, 4, 8))
            each = [max(1, int(L * rng.uniform(0.2, 1.0))) for _ in range(B)]
            each[rng.randrange(B)] = L
            lens = ",".join(map(str, each))
        c = _case("", "train" if path == "fp32" else path, B, Hq, Hkv, L, D, W, S, dtype, learned=learned, lens=lens,
                  fp8_pv=path == "fp8" and rng.random() < 0.5)
        w = work(c)
        # no dearer than the listed cases: full_8k, or fp32_sliding among the float32 ones
        if w["flops"] <= (3.2e10 if dtype == "fp32" else 1.9e12) and w["bytes"] <= 2.0e9:
            return c


def _lens(case):
    return [int(x) for x in case["lens"].split(",")] if case["lens"] else [case["L"]] * case["B"]


def _pairs(L, W, S):
    """Allowed (query, key) pairs of one head: row q sees min(q + 1, W) window keys and the sinks
    left of its window."""
    W = L if W == 0 else min(W, L)
    S = min(S, L)
    tri = lambda n, T: min(n, T) * (min(n, T) + 1) // 2 + (T - min(n, T)) * n
    return tri(W, L) + tri(S, L - W)


def work(case):
    """Every input read once and every output written once; 4 D operations per allowed pair and query
    head forward, 10 D backward."""
    lens, D, Hq, Hkv = _lens(case), case["D"], case["Hq"], case["Hkv"]
    eb = 4 if case["dtype"] == "fp32" else 2
    rows = sum(lens)
    out_rows = case["B"] * case["L"] if case["path"] == "padded" else rows
    pairs = sum(_pairs(n, case["W"], case["S"]) for n in lens) * Hq
    q, kv = Hq * D * eb, 2 * Hkv * D * eb
    nbytes = rows * (q + kv) + out_rows * q
    flops = 4 * D * pairs
    if case["path"] not in ("prefill", "fp8"):
        nbytes += rows * q + out_rows * (q + kv)  # dO; dQ, dK, dV
        flops += 10 * D * pairs
    return {"bytes": nbytes, "flops": flops}


def _inputs(case, seed):
    """q, k, v and dO ~ N(0, 1) (dO ~ N(0, do_std)), learned sink logits ~ N(0, 1): [B, H, L, D] views
    of [B, L, H, D] projections for the GPT-OSS paths, [total, H, D] packed rows, or [B, H, L, D]."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    B, Hq, Hkv, L, D = (case[x] for x in ("B", "Hq", "Hkv", "L", "D"))

    def make(H, std=1.0):
        if case["path"] == "packed":
            return (torch.randn(sum(_lens(case)), H, D, device="cuda", generator=g) * std).to(dt)
        if case["path"] == "padded" or case["learned"]:
            return (torch.randn(B, L, H, D, device="cuda", generator=g) * std).to(dt).transpose(1, 2)
        return (torch.randn(B, H, L, D, device="cuda", generator=g) * std).to(dt)

    q, k, v = make(Hq), make(Hkv), make(Hkv)
    do = make(Hq, case["do_std"])
    sinks = torch.randn(Hq, device="cuda", generator=g).to(dt) if case["learned"] else None
    return q, k, v, do, sinks


def prepare(case, seed):
    q, k, v, do, sinks = _inputs(case, seed)
    s = {"case": case, "q": q, "k": k, "v": v, "do": do, "sinks": sinks}
    path = case["path"]
    if path in ("train", "packed", "padded"):
        for n in ("q", "k", "v", "sinks"):
            if s[n] is not None:
                s[n].requires_grad_()
    if path == "packed":
        off = [0]
        for n in _lens(case):
            off.append(off[-1] + n)
        s["cu"] = torch.tensor(off, dtype=torch.int32, device="cuda")
    if path == "padded":
        # a right-padded batch: 1 where there is a token
        lens = torch.tensor(_lens(case), device="cuda")
        s["mask"] = (torch.arange(case["L"], device="cuda")[None, :] < lens[:, None]).to(torch.int64)
        s["do"] = do.transpose(1, 2)
    return s


def run(s):
    case, q, k, v, do, sinks = s["case"], s["q"], s["k"], s["v"], s["do"], s["sinks"]
    path, W, S, L = case["path"], case["W"], case["S"], case["L"]
    if path == "fp8":
        q8, qd = fa.quantize_fp8(q)
        k8, kd = fa.quantize_fp8(k)
        v8, vd = fa.quantize_fp8(v)
        return fa.flash_swda_with_sink_fp8(q8, k8, v8, W or None, S, descale=(qd, kd, vd), sinks=sinks,
                                           fp8_pv=case["fp8_pv"])
    if path == "prefill":
        with torch.no_grad():
            return fa.attention(q, k, v, W or None, S, sinks=sinks)
    if path == "packed":
        o = fa.flash_swda_with_sink_varlen(q, k, v, s["cu"], L, W or None, S, sinks=sinks)
    elif path == "padded":
        o, _ = fa.gpt_oss_attention_forward(None, q, k, v, s["mask"], sliding_window=W or None, s_aux=sinks)
    elif sinks is not None:
        o = fa.attention(q, k, v, W or None, S, sinks=sinks)
    elif case["D"] == 16:
        o = fa.swa_sink_attention(q, k, v, W or L, S)
    else:
        o = fa.flash_swda_with_sink(q, k, v, W or L, S)
    wrt = [q, k, v] + ([] if sinks is None else [sinks])
    return [o, *torch.autograd.grad(o, wrt, do)]


def tolerance(case):
    """Relative error of a correct implementation whose products take 16-bit operands (P and dS are
    rounded to them) or fp32 ones, about four times what the paths show against 64 bits."""
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    if case["path"] == "fp8":
        # e4m3 weights in P V, or bf16 ones on e4m3 values
        return {"rel": 0.03 if case["fp8_pv"] else 1e-2}
    return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 1.5e-3}


def _sequence(q, k, v, do, W, S, sinks):
    """One sequence in float64: q, do [Hq, L, D], k, v [Hkv, L, D] -> o, dq, dk, dv, dsinks (the
    gradients None without do).  Rows in chunks; a chunk's keys are its window's and the sinks."""
    Hq, L, D = q.shape
    Hkv = k.shape[0]
    G = Hq // Hkv
    W = L if W == 0 else min(W, L)
    S = min(S, L)
    scale = 1.0 / math.sqrt(D)
    o = torch.zeros(Hq, L, D, dtype=torch.float64, device=q.device)
    dq = torch.zeros_like(o) if do is not None else None
    dk = torch.zeros(Hkv, L, D, dtype=torch.float64, device=q.device) if do is not None else None
    dv = torch.zeros_like(dk) if do is not None else None
    dsk = torch.zeros(Hq, dtype=torch.float64, device=q.device) if sinks is not None and do is not None else None
    for h in range(Hkv):
        kh, vh = k[h].double(), v[h].double()
        for r0 in range(0, L, 1024):
            r1 = min(L, r0 + 1024)
            ws = max(0, r0 - W + 1)
            ns = min(S, ws)
            cols = torch.cat((torch.arange(ns, device=q.device), torch.arange(ws, r1, device=q.device)))
            rows = torch.arange(r0, r1, device=q.device)
            delta = rows[:, None] - cols[None, :]
            ok = (delta >= 0) & ((delta < W) | (cols[None, :] < S))
            ks, vs = kh[cols], vh[cols]
            kst, vst = ks.t().contiguous(), vs.t().contiguous()
            for hq in range(h * G, h * G + G):
                qh = q[hq, r0:r1].double()
                sc = (qh @ kst * scale).masked_fill_(~ok, float("-inf"))
                m = sc.amax(1, keepdim=True)
                if sinks is not None:
                    m = torch.maximum(m, sinks[hq].double())
                p = sc.sub_(m).exp_()
                den = p.sum(1, keepdim=True)
                if sinks is not None:
                    psink = torch.exp(sinks[hq].double() - m)
                    den = den + psink
                p /= den
                o[hq, r0:r1] = p @ vs
                if do is None:
                    continue
                doh = do[hq, r0:r1].double()
                row = (doh * o[hq, r0:r1]).sum(1, keepdim=True)
                dv[h].index_add_(0, cols, p.t().contiguous() @ doh)
                ds = p * (doh @ vst - row)
                dq[hq, r0:r1] = ds @ ks * scale
                dk[h].index_add_(0, cols, ds.t().contiguous() @ qh * scale)
                if dsk is not None:
                    dsk[hq] -= (psink / den * row).sum()
    return o, dq, dk, dv, dsk


def exact(case, seed):
    q, k, v, do, sinks = _inputs(case, seed)
    path, W, S, B = case["path"], case["W"], case["S"], case["B"]
    if path == "fp8":
        def dequantised(x):
            xf = x.float()
            d = float(xf.abs().max()) / 448.0
            return (xf / d).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).double() * d
        q, k, v = dequantised(q), dequantised(k), dequantised(v)
    grads = path not in ("fp8", "prefill")
    out = []
    off = 0
    for b, n in enumerate(_lens(case)):
        if path == "packed":
            one = lambda x: x[off:off + n].transpose(0, 1)
        else:
            one = lambda x: x[b, :, :n]
        out.append(_sequence(one(q), one(k), one(v), one(do) if grads else None, W, S, sinks))
        off += n

    def whole(i):  # the sequences' results in the layout of the tensors, zeros at padded rows
        if path == "packed":
            return torch.cat([r[i].transpose(0, 1) for r in out])
        H = out[0][i].shape[0]
        t = torch.zeros(B, H, case["L"], case["D"], dtype=torch.float64, device="cuda")
        for b, r in enumerate(out):
            t[b, :, :r[i].shape[1]] = r[i]
        return t

    o = whole(0)
    if path == "padded":
        o = o.transpose(1, 2)
    if not grads:
        return o
    return [o, whole(1), whole(2), whole(3)] + ([sum(r[4] for r in out)] if sinks is not None else [])
