"""What is timed of this framework: the calls a serving program makes per layer.

Every case is a dict of plain values; ``kind`` names the call:

  decode          paged_attention_decode over a float, int8 or fp8 pool, with
                  the reference's signature (lengths on the device only)
  decode_q4       paged_attention_decode_q4 over the 4-bit pool
  decode_turbo    paged_attention_decode_turbo over TurboQuant pages
  step            one layer of a decode step through PagedKVCacheManager: the
                  new token's K/V written, then attention over the pages
  hf_step         one layer of a Hugging Face decode step over a TurboQuantCache
                  layer (compressed pages and uncompressed residual, merged)
  prefill         kv_quant.quantize_pages: a prompt's K/V into an int8/fp8 pool
  prefill_turbo   tq_pages.quantize_pages: a prompt's K/V into TurboQuant pages
  codec           KVCacheCompressor: compress (packed) and decompress
  sparse          KVCacheCompressor.sparse_v_attend: scores, top-k, weighted sum

Lengths follow ``ctx`` ("fixed", "uniform" or "lognormal" between ``lo`` and
``hi``, ``pin`` one more sequence of that length) and ``lens_seed``; values,
page tables and rotations follow the seed given to ``prepare``.
"""
import math
import random

import torch

from vramancer_amd import kv_quant, tq_pages
from vramancer_amd.kv_quantizer import KVCacheCompressor
from vramancer_amd.paged_attention import PagedKVCacheManager, PagedKVConfig
from vramancer_amd.paged_attention_cuda import paged_attention_decode, paged_attention_decode_q4
from vramancer_amd.turboquant_cache import TurboQuantLayer, turbo_paged_attention

DEVICE = "cuda:0"
FLOAT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2, "int8": 1, "fp8": 1}


def listed():
    return [
        # the batch every layer of a 14B model decodes in full service: even
        # contexts, int8 cache
        dict(name="decode-int8-14b", kind="decode", dtype="int8", H=40, KH=8, D=128, PS=16, L=8, B=64,
             ctx="fixed", lo=4096, hi=4096, pin=0, lens_seed=0),
        # a 7B model's ragged batch over a bf16 cache
        dict(name="decode-bf16-7b", kind="decode", dtype="bf16", H=28, KH=4, D=128, PS=16, L=4, B=32,
             ctx="uniform", lo=1024, hi=8192, pin=0, lens_seed=0),
        # many users of very mixed lengths and one very long document, fp8 cache
        dict(name="decode-fp8-mixed", kind="decode", dtype="fp8", H=64, KH=8, D=128, PS=16, L=1, B=128,
             ctx="lognormal", lo=16, hi=131072, pin=131072, lens_seed=0),
        # one chat on its own: a single request, the manager's default dtype
        dict(name="decode-f16-single", kind="decode", dtype="f16", H=28, KH=4, D=128, PS=16, L=4, B=1,
             ctx="fixed", lo=1531, hi=1531, pin=0, lens_seed=0),
        # the 14B batch over the reference's 4-bit pool
        dict(name="decode-q4-14b", kind="decode_q4", dtype="q4", H=40, KH=8, D=128, PS=16, L=4, B=64,
             ctx="fixed", lo=4096, hi=4096, pin=0, lens_seed=0),
        # long contexts over TurboQuant pages, 3 bits per angle (the default)
        dict(name="decode-turbo3-long", kind="decode_turbo", bits=3, H=40, KH=8, D=128, PS=16, L=1, B=16,
             ctx="fixed", lo=32768, hi=32768, pin=0, lens_seed=0),
        # a small serving batch through the page manager: append, then attend
        dict(name="step-int8-serve", kind="step", dtype="int8", H=40, KH=8, D=128, PS=16, L=2, B=8,
             ctx="uniform", lo=200, hi=2000, pin=0, lens_seed=1),
        # Hugging Face generate() over the TurboQuant cache, head_dim 64, 4 bits
        dict(name="hf-turbo4-step", kind="hf_step", bits=4, H=16, KH=8, D=64, B=4, comp=8000, res=101),
        # four prompts of about 2000 tokens enter the int8 cache
        dict(name="prefill-int8", kind="prefill", dtype="int8", src="bf16", KH=8, D=128, PS=16, NP=512, tail=7),
        # the same prompts enter TurboQuant pages
        dict(name="prefill-turbo3", kind="prefill_turbo", bits=3, src="bf16", KH=8, D=128, PS=16, NP=512, tail=7),
        # K/V of 16 heads x 4096 tokens packed for storage, and unpacked again
        dict(name="codec-turbo3", kind="codec", bits=3, src="bf16", D=128, heads=16, tokens=4096),
        # sparse V: 40 query heads over a long compressed context, top 10 %
        dict(name="sparse-v-long", kind="sparse", bits=3, D=128, M=40, N=32768, ratio=0.1),
    ]


# ---------------------------------------------------------------------------
# Drawn cases
# ---------------------------------------------------------------------------

def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


HEADS = [(40, 8), (28, 4), (64, 8), (32, 8), (16, 8), (12, 12)]


def draw(rng):
    kind = rng.choices(["decode", "step", "decode_turbo", "decode_q4", "hf_step", "prefill", "prefill_turbo", "codec",
                        "sparse"], [36, 12, 10, 8, 8, 8, 8, 5, 5])[0]
    H, KH = rng.choice(HEADS)
    seed = rng.randrange(1 << 30)
    if kind in ("decode", "step", "decode_turbo", "decode_q4"):
        case = dict(kind=kind, H=H, KH=KH, PS=16, L=rng.randint(1, 4), pin=0, lens_seed=seed)
        case["B"] = _log_int(rng, 1, 32 if kind == "decode_turbo" else 128)
        case["ctx"] = rng.choice(["fixed", "uniform", "lognormal"])
        if kind == "decode":
            case["dtype"] = rng.choice(["bf16", "f16", "int8", "int8", "fp8", "fp8", "f32"])
            case["D"] = rng.choice([64, 80, 96, 128, 128, 128, 256] if case["dtype"] != "f32" else [64, 128])
            case["PS"] = rng.choice([16, 16, 16, 32])
            if case["dtype"] == "f32" or case["D"] == 256:
                case["PS"] = 16
            # at most about 300 MB of one layer's K/V
            per = 2 * KH * case["D"] * BYTES[case["dtype"]]
            cap = 300_000_000 // per
        elif kind == "step":
            case["dtype"] = rng.choice(["f16", "bf16", "int8", "int8"])
            case["D"] = rng.choice([64, 96, 128, 128])
            case["L"] = rng.randint(1, 2)
            case["B"] = _log_int(rng, 1, 64)
            cap = 60_000
        elif kind == "decode_turbo":
            case["bits"] = rng.choice([2, 3, 3, 4, 4])
            case["D"] = rng.choice([64, 96, 128, 128])
            case["L"] = 1
            cap = 2_000_000 // KH
        else:
            case["dtype"], case["D"], case["L"] = "q4", 128, 1
            cap = 150_000
        hi = min(131072, max(64, cap // case["B"]))
        top = _log_int(rng, 64, hi)
        case["lo"], case["hi"] = (top, top) if case["ctx"] == "fixed" else (max(1, top // 8), top)
        return case
    if kind == "hf_step":
        return dict(kind=kind, bits=rng.choice([3, 4]), H=H, KH=KH, D=rng.choice([64, 128]), B=rng.randint(1, 8),
                    comp=_log_int(rng, 256, 8192), res=rng.randint(1, 255))
    if kind in ("prefill", "prefill_turbo"):
        case = dict(kind=kind, src=rng.choice(["bf16", "f16", "f32"]), KH=KH, D=rng.choice([64, 96, 128, 128]), PS=16,
                    NP=_log_int(rng, 1, 1024), tail=rng.randint(1, 16))
        if kind == "prefill":
            case["dtype"] = rng.choice(["int8", "int8", "fp8"])
            case["PS"] = rng.choice([16, 16, 32])
        else:
            case["bits"] = rng.choice([2, 3, 4])
        return case
    if kind == "codec":
        return dict(kind=kind, bits=rng.choice([3, 4]), src=rng.choice(["bf16", "f16", "f32"]),
                    D=rng.choice([64, 96, 128, 128]), heads=rng.choice([1, 4, 8, 12, 16]), tokens=_log_int(rng, 17, 4096))
    return dict(kind="sparse", bits=rng.choice([3, 4]), D=rng.choice([64, 128]), M=rng.choice([12, 16, 28, 40]),
                N=_log_int(rng, 2048, 32768), ratio=rng.choice([0.1, 0.2]))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _lens(case):
    r = random.Random(case["lens_seed"])
    lo, hi = case["lo"], case["hi"]
    out = []
    for _ in range(case["B"]):
        if case["ctx"] == "fixed":
            n = hi
        elif case["ctx"] == "uniform":
            n = r.randint(lo, hi)
        else:
            n = int(min(hi, max(lo, round(r.lognormvariate(math.log(min(2048.0, math.sqrt(lo * hi) * 1.5)), 1.0)))))
        out.append(n)
    if case["pin"]:
        out.append(case["pin"])
    return out


def _gen(seed, device=DEVICE):
    return torch.Generator(device=device).manual_seed(int(seed))


def _rows(shape, gen, outliers=None, student=False, std=1.0):
    """K/V values: normal, with two large channels per head for the quantized
    caches, or Student-t with 3 degrees of freedom at unit variance."""
    x = torch.randn(shape, generator=gen, device=DEVICE)
    if student:
        chi2 = torch.zeros_like(x)
        for _ in range(3):
            chi2 += torch.randn(shape, generator=gen, device=DEVICE) ** 2
        x = x / chi2.sqrt()
    if outliers is not None:
        x[..., outliers] *= 20.0
    return x * std


def _table(lens, PS, seed):
    """Shuffled physical pages, a tenth of them spare."""
    pages = [(n + PS - 1) // PS for n in lens]
    P = max(1, math.ceil(sum(pages) * 1.1))
    perm = torch.randperm(P, generator=_gen(seed, "cpu")).to(torch.int32)
    table = torch.full((len(lens), max(1, max(pages))), -1, dtype=torch.int32)
    at = 0
    for b, n in enumerate(pages):
        table[b, :n] = perm[at:at + n]
        at += n
    return P, table.to(DEVICE)


def _q4(x):
    """Codes, scales and zeros of the 4-bit pool: per 32 dims a float16 scale
    and zero point, low nibble the even dim."""
    g = x.reshape(*x.shape[:-1], -1, 32)
    lo, hi = g.amin(-1), g.amax(-1)
    scale = ((hi - lo) / 15).clamp(min=1e-6).to(torch.float16)
    zero = (-lo / scale.float()).to(torch.float16)
    n = torch.clamp(torch.round(g / scale.float()[..., None] + zero.float()[..., None]), 0, 15)
    n = n.to(torch.uint8).reshape(x.shape)
    return n[..., 0::2] | (n[..., 1::2] << 4), scale, zero


CHUNK = 1024  # pages filled at a time


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("decode", "decode_q4", "decode_turbo"):
        lens = _lens(case)
        H, KH, D, PS, L = (case[k] for k in ("H", "KH", "D", "PS", "L"))
        P, s["table"] = _table(lens, PS, seed)
        s["lens"] = torch.tensor(lens, dtype=torch.int32, device=DEVICE)
        gen = _gen(seed + 1)
        s["q"] = torch.randn((len(lens), H, D), generator=gen, device=DEVICE)
        s["layer"] = layer = L // 2
        ids = torch.arange(P, dtype=torch.int32, device=DEVICE)
        if kind == "decode_turbo":
            torch.manual_seed(seed)
            s["comp"] = comp = KVCacheCompressor(D, case["bits"]).to(DEVICE)
            s["pool"] = tq_pages.allocate_pool(P, L, KH, comp, DEVICE, PS)
        elif kind == "decode_q4":
            s["pool"] = torch.zeros((P, L, 2, KH, PS, D // 2), dtype=torch.uint8, device=DEVICE)
            s["scales"] = torch.zeros((P, L, 2, KH, PS, D // 32), dtype=torch.float16, device=DEVICE)
            s["zeros"] = torch.zeros_like(s["scales"])
        elif case["dtype"] in FLOAT:
            s["pool"] = torch.zeros((P, L, 2, KH, PS, D), dtype=FLOAT[case["dtype"]], device=DEVICE)
            s["scales"] = None
        else:
            s["pool"], s["scales"] = kv_quant.allocate_pool(P, L, KH, D, case["dtype"], PS, DEVICE)
        big = [3, D // 2 + 1] if kind == "decode_q4" or case.get("dtype") == "int8" else None
        for a in range(0, P, CHUNK):
            e = min(P, a + CHUNK)
            k, v = (_rows((e - a, KH, PS, D), gen, big, student=kind == "decode_turbo",
                          std=0.5 if case.get("dtype") in ("bf16", "f16") else 1.0) for _ in range(2))
            if kind == "decode_turbo":
                tq_pages.quantize_pages(s["pool"], layer, ids[a:e], k.bfloat16(), v.bfloat16(), s["comp"],
                                        page_size=PS)
            elif kind == "decode_q4":
                for kv, x in ((0, k), (1, v)):
                    s["pool"][a:e, layer, kv], s["scales"][a:e, layer, kv], s["zeros"][a:e, layer, kv] = _q4(x)
            elif s["scales"] is not None:
                kv_quant.quantize_pages(s["pool"], s["scales"], layer, ids[a:e], k.bfloat16(), v.bfloat16())
            else:
                s["pool"][a:e, layer, 0], s["pool"][a:e, layer, 1] = k, v
        return s
    if kind == "step":
        lens = _lens(case)
        H, KH, D, PS, L, B = (case[k] for k in ("H", "KH", "D", "PS", "L", "B"))
        pages = sum(n // PS + 1 for n in lens)
        s["manager"] = m = PagedKVCacheManager(PagedKVConfig(
            page_size=PS, num_layers=L, num_kv_heads=KH, head_dim=D, max_pages=pages, device=DEVICE,
            dtype={"int8": "int8", "f16": "float16", "bf16": "bfloat16"}[case["dtype"]]))
        dtype = FLOAT.get(case["dtype"], torch.bfloat16)
        gen = _gen(seed + 1)
        s["rids"] = ["r%d" % b for b in range(B)]
        s["past"] = []
        for rid, n in zip(s["rids"], lens):
            kv = tuple(_rows((1, KH, n, D), gen, [3, D // 2 + 1]).to(dtype) for _ in range(2))
            s["past"].append(kv)
            m.from_hf_cache(rid, (kv,))
        s["ids"], s["slots"] = m.append_tokens(s["rids"])
        s["k"], s["v"] = (_rows((B, KH, D), gen, [3, D // 2 + 1]).to(dtype) for _ in range(2))
        s["q"] = torch.randn((B, H, D), generator=gen, device=DEVICE)
        return s
    if kind == "hf_step":
        H, KH, D, B = (case[k] for k in ("H", "KH", "D", "B"))
        torch.manual_seed(seed)
        comp = KVCacheCompressor(D, case["bits"]).to(DEVICE)
        s["layer"] = layer = TurboQuantLayer(comp, residual_length=256, paged_attention=True)
        gen = _gen(seed + 1)
        s["old"] = tuple(_rows((B, KH, case["comp"], D), gen, student=True).bfloat16() for _ in range(2))
        s["new"] = tuple(_rows((B, KH, case["res"], D), gen, student=True).bfloat16() for _ in range(2))
        layer.update(*s["old"])
        s["key"], s["value"] = layer.update(*s["new"])
        s["q"] = torch.randn((B, H, 1, D), generator=gen, device=DEVICE).bfloat16()
        return s
    if kind in ("prefill", "prefill_turbo"):
        KH, D, PS, NP = (case[k] for k in ("KH", "D", "PS", "NP"))
        gen = _gen(seed + 1)
        big = [3, D // 2 + 1] if kind == "prefill" else None
        s["k"], s["v"] = (_rows((NP, KH, PS, D), gen, big, student=big is None).to(FLOAT[case["src"]])
                          for _ in range(2))
        s["ids"] = torch.randperm(NP, generator=_gen(seed, "cpu")).to(torch.int32).to(DEVICE)
        s["valid"] = torch.full((NP,), PS, dtype=torch.int32, device=DEVICE)
        s["valid"][NP - 1] = case["tail"]
        if kind == "prefill":
            s["pool"], s["scales"] = kv_quant.allocate_pool(NP, 1, KH, D, case["dtype"], PS, DEVICE)
        else:
            torch.manual_seed(seed)
            s["comp"] = KVCacheCompressor(D, case["bits"]).to(DEVICE)
            s["pool"] = tq_pages.allocate_pool(NP, 1, KH, s["comp"], DEVICE, PS)
        return s
    torch.manual_seed(seed)
    s["comp"] = comp = KVCacheCompressor(case["D"], case["bits"]).to(DEVICE)
    gen = _gen(seed + 1)
    if kind == "codec":
        shape = (case["heads"], case["tokens"], case["D"])
        s["x"] = _rows(shape, gen, student=True).to(FLOAT[case["src"]])
        s["packed"] = comp.compress(_rows(shape, gen, student=True).to(FLOAT[case["src"]]))
        return s
    N, D = case["N"], case["D"]
    s["ck"] = comp.compress(_rows((N, D), gen, student=True).bfloat16(), pack=False)
    s["cv"] = comp.compress(_rows((N, D), gen, student=True).bfloat16(), pack=False)
    s["q"] = torch.randn((case["M"], D), generator=gen, device=DEVICE)
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        return paged_attention_decode(s["q"], s["pool"], s["table"], s["lens"], s["layer"], kv_scales=s["scales"])
    if kind == "decode_q4":
        return paged_attention_decode_q4(s["q"], s["pool"], s["scales"], s["zeros"], s["table"], s["lens"], s["layer"])
    if kind == "decode_turbo":
        return tq_pages.paged_attention_decode_turbo(s["q"], s["pool"], s["table"], s["lens"], s["layer"], s["comp"],
                                                     page_size=case["PS"])
    if kind == "step":
        m = s["manager"]
        m.write_kv_batch(0, s["ids"], s["slots"], s["k"], s["v"])
        return {"out": m.compute_attention_decode(s["q"], s["rids"], 0), "pool": m.gpu_pool}
    if kind == "hf_step":
        return turbo_paged_attention(None, s["q"], s["key"], s["value"], None)[0]
    if kind == "prefill":
        kv_quant.quantize_pages(s["pool"], s["scales"], 0, s["ids"], s["k"], s["v"], s["valid"])
        return {"pool": s["pool"], "scales": s["scales"]}
    if kind == "prefill_turbo":
        tq_pages.quantize_pages(s["pool"], 0, s["ids"], s["k"], s["v"], s["comp"], s["valid"], page_size=case["PS"])
        return s["pool"]
    if kind == "codec":
        c = s["comp"].compress(s["x"])
        return {"radius": c["radius"], "angles": c["angles_packed"], "signs": c["qjl_signs_packed"],
                "norms": c["qjl_norms"], "values": s["comp"].decompress(s["packed"])}
    return s["comp"].sparse_v_attend(s["q"], s["ck"], [s["cv"]], sparse_v_ratio=case["ratio"])


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def _turbo_row(D, bits, key):
    """Bytes of one compressed row: angles and radius, for keys also the sign
    bits and the residual norm."""
    pd = 1 << math.ceil(math.log2(max(D, 2)))
    return ((pd - 1) * bits + 7) // 8 + 2 + ((pd // 2 + 7) // 8 + 2 if key else 0), pd


def work(case):
    kind = case["kind"]
    if kind in ("decode", "decode_q4", "decode_turbo", "step"):
        lens = _lens(case)
        if kind == "step":
            lens = [n + 1 for n in lens]
        H, KH, D, PS = (case[k] for k in ("H", "KH", "D", "PS"))
        tokens, pages = sum(lens), sum((n + PS - 1) // PS for n in lens)
        if kind == "decode_turbo":
            per = _turbo_row(D, case["bits"], True)[0] + _turbo_row(D, case["bits"], False)[0]
            kv = tokens * KH * per
        elif kind == "decode_q4":
            kv = tokens * KH * 2 * (D // 2 + D // 32 * 4)
        else:
            kv = tokens * KH * 2 * D * BYTES[case["dtype"]]
            kv += {"int8": tokens * KH * 8, "fp8": pages * KH * 8}.get(case["dtype"], 0)
        move = kv + 8 * len(lens) * H * D + 4 * pages
        if kind == "step":
            move += len(lens) * KH * 2 * D * (2 + BYTES[case["dtype"]])
        return {"bytes": move, "flops": 4.0 * tokens * H * D}
    if kind == "hf_step":
        H, KH, D, B = (case[k] for k in ("H", "KH", "D", "B"))
        per = 2 * _turbo_row(D, case["bits"], False)[0]
        return {"bytes": B * KH * (case["comp"] * per + case["res"] * 4 * D) + 4 * B * H * D,
                "flops": 4.0 * B * (case["comp"] + case["res"]) * H * D}
    if kind in ("prefill", "prefill_turbo"):
        KH, D, PS = (case[k] for k in ("KH", "D", "PS"))
        rows = ((case["NP"] - 1) * PS + min(case["tail"], PS)) * KH
        esize = BYTES[case["src"]]
        if kind == "prefill":
            scales = rows * 8 if case["dtype"] == "int8" else case["NP"] * KH * 8
            return {"bytes": rows * 2 * D * (esize + 1) + scales, "flops": 4.0 * rows * D}
        k, pd = _turbo_row(D, case["bits"], True)
        v, _ = _turbo_row(D, case["bits"], False)
        # two rotations (pd log2 pd each), the angles, and the keys' projection
        return {"bytes": rows * (2 * D * esize + k + v), "flops": rows * (2.0 * pd * math.log2(pd) + pd * pd)}
    D = case["D"]
    row, pd = _turbo_row(D, case["bits"], True)
    if kind == "codec":
        rows = case["heads"] * case["tokens"]
        v, _ = _turbo_row(D, case["bits"], False)
        return {"bytes": rows * (D * BYTES[case["src"]] + row + v + 4 * D),
                "flops": rows * (2.0 * pd * math.log2(pd) + pd * pd)}
    # raw (one byte per angle and sign) keys; values' angles and radii
    M, N = case["M"], case["N"]
    k = max(1, math.ceil(case["ratio"] * N))
    return {"bytes": N * ((pd - 1) + pd // 2 + 4 + (pd - 1) + 2) + 8 * M * D,
            "flops": 2.0 * M * N * (pd + pd // 2) + 2.0 * M * k * D}


# ---------------------------------------------------------------------------
# Tolerances and 64-bit results
# ---------------------------------------------------------------------------

def tolerance(case):
    """About four times the error measured against ``exact``."""
    kind = case["kind"]
    if kind in ("prefill", "prefill_turbo"):
        return "exact"
    if kind == "hf_step":  # 1.7e-3: the output is rounded to bf16
        return {"rel": 8e-3}
    if kind == "codec":  # 1.1e-7 (decompressed values; the codes are whole numbers)
        return {"rel": 1e-6}
    if kind == "sparse":
        # 7.3e-7; a score at the edge of the top k may fall either side
        return {"rel": 1e-2}
    if kind == "decode_turbo":  # 2.1e-4: K and V as float16 parts
        return {"rel": 1e-3}
    if kind == "decode_q4":  # 1.5e-5
        return {"rel": 6e-5}
    if kind == "step":  # up to 7.4e-5: keys with large channels, hence large scores
        return {"rel": 3e-4}
    # 1e-6 (int8) to 8.1e-6 (fp8); f32 1.5e-7
    return {"rel": 1e-6 if case["dtype"] == "f32" else 3e-5}


def _attend(q, k, v, scale):
    """softmax(scale q k^T) v in float64: q [H, D], k / v [KH, n, D]."""
    H, KH = q.shape[0], k.shape[0]
    qg = q.double().reshape(KH, H // KH, -1)
    w = torch.softmax(torch.matmul(qg, k.transpose(1, 2).contiguous()) * scale, dim=-1)
    return torch.matmul(w, v).reshape(H, -1)


def _v_rows(raw):
    """V codes [..., PS, D] of a quantized pool, token-major: the pool tiles
    them as (t / 4, d % 16, d / 16, t % 4)."""
    *lead, PS, D = raw.shape
    return raw.reshape(*lead, PS // 4, 16, D // 16, 4).permute(
        *range(len(lead)), -4, -1, -2, -3).reshape(*lead, PS, D)


def _hadamard(pd):
    h = torch.ones((1, 1), dtype=torch.float64, device=DEVICE)
    while h.shape[0] < pd:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(pd)


def _polar(radius, angles, bits):
    """Rotated-space rows [..., pd] float64 of radii [...] and level-major bins."""
    pd = angles.shape[-1] + 1
    nb = 1 << bits
    r = radius.double()[..., None]
    level, at = int(math.log2(pd)) - 1, pd - 1
    while level >= 0:
        n = pd >> (level + 1)
        idx = angles[..., at - n:at].float()
        lo, hi = (-math.pi, math.pi) if level == 0 else (0.0, math.pi / 2)
        t = (lo + (idx + 0.5) * (hi - lo) / nb).double()
        r = torch.stack([r * torch.cos(t), r * torch.sin(t)], -1).reshape(*r.shape[:-1], 2 * n)
        at -= n
        level -= 1
    return r


def _unpack(packed, M, bits):
    """[N, bytes] -> [N, M]: `bits` bits a value, most significant first."""
    shifts = torch.arange(7, -1, -1, device=packed.device, dtype=torch.uint8)
    b = ((packed[..., None] >> shifts) & 1).reshape(packed.shape[0], -1)[:, :M * bits].reshape(-1, M, bits)
    return sum(b[..., i].to(torch.uint8) << (bits - 1 - i) for i in range(bits))


def _padded(x, pd):
    return torch.nn.functional.pad(x.double(), (0, pd - x.shape[-1]))


def exact(case, seed):
    kind = case["kind"]
    if kind == "prefill_turbo":  # whole numbers
        return None
    s = prepare(case, seed)
    if kind == "prefill":
        sc = torch.zeros(s["scales"].shape, dtype=torch.float64, device=DEVICE)
        live = torch.arange(case["PS"], device=DEVICE)[None, :] < s["valid"][:, None]
        for kv, x in ((0, s["k"]), (1, s["v"])):
            amax = x.double().abs().amax(-1) * live[:, None]  # [NP, KH, PS]
            sc[s["ids"].long(), 0, kv] = amax / 127 if case["dtype"] == "int8" else amax.amax(-1) / 448
        return {"pool": None, "scales": sc}
    if kind in ("decode", "decode_q4", "decode_turbo"):
        H, KH, D, PS = (case[k] for k in ("H", "KH", "D", "PS"))
        lens, scale = _lens(case), 1.0 / math.sqrt(D)
        out = torch.zeros((len(lens), H, D), dtype=torch.float64, device=DEVICE)
        for b, n in enumerate(lens):
            ids = s["table"][b, :(n + PS - 1) // PS].long()
            if kind == "decode_turbo":
                comp, pd, qd = s["comp"], s["comp"]._padded_dim, s["comp"].qjl_dim
                # the pool's codes, as its public reader gives them
                c = tq_pages.read_pages(s["pool"], s["layer"], ids, comp, PS)
                signs, jl = comp._hadamard_signs.double(), comp.jl_matrix.double()
                had = _hadamard(pd)
                qr = (_padded(s["q"][b], pd) * signs) @ had
                group = H // KH
                for h in range(KH):
                    f = {k: t[:, :, h].transpose(0, 1).reshape(2, ids.numel() * PS, *t.shape[4:])[:, :n]
                         for k, t in c.items()}
                    q = qr[h * group:(h + 1) * group]
                    raw = (q @ jl.T) @ (2.0 * f["qjl_signs"][0].double() - 1.0).T.contiguous()
                    corr = raw * (math.sqrt(math.pi / 2) / qd) * f["qjl_norms"][0].double()
                    sc = q @ _polar(f["radius"][0], f["angles"][0], case["bits"]).T.contiguous() + corr
                    o = torch.softmax(sc * scale, -1) @ _polar(f["radius"][1], f["angles"][1], case["bits"])
                    out[b, h * group:(h + 1) * group] = ((o @ had) * signs)[:, :D]
                continue
            if kind == "decode_q4":
                raw = s["pool"][ids, s["layer"]]
                x = torch.stack([raw & 15, raw >> 4], -1).reshape(*raw.shape[:-1], D // 32, 32).double()
                x = (x - s["zeros"][ids, s["layer"]].double()[..., None]) * s["scales"][ids, s["layer"]].double()[..., None]
                x = x.reshape(*raw.shape[:-1], D)
            elif s["scales"] is None:
                x = s["pool"][ids, s["layer"]].double()
            else:
                raw = s["pool"].view(torch.uint8)[ids, s["layer"]]
                x = torch.stack([raw[:, 0], _v_rows(raw[:, 1])], 1).view(s["pool"].dtype)
                sc = s["scales"][ids, s["layer"]].double()
                x = (x.float() if x.dtype != torch.int8 else x).double() * (
                    sc[..., None] if x.dtype == torch.int8 else sc[..., None, None])
            x = x.permute(1, 2, 0, 3, 4).reshape(2, KH, -1, D)[:, :, :n]
            out[b] = _attend(s["q"][b], x[0].contiguous(), x[1].contiguous(), scale)
        return out
    if kind == "step":
        D = case["D"]
        out = torch.zeros(s["q"].shape, dtype=torch.float64, device=DEVICE)
        for b, (k, v) in enumerate(s["past"]):
            x = [torch.cat([t[0], n[b][:, None]], 1).float() for t, n in ((k, s["k"]), (v, s["v"]))]
            if case["dtype"] == "int8":
                sc = [t.abs().amax(-1, keepdim=True) / 127 for t in x]
                x = [torch.clamp(torch.round(t / c), -127, 127).double() * c.double() for t, c in zip(x, sc)]
            out[b] = _attend(s["q"][b], x[0].double(), x[1].double(), 1.0 / math.sqrt(D))
        return {"out": out, "pool": None}
    if kind == "hf_step":
        B, H, _, D = s["q"].shape
        comp = s["layer"].compressor
        had, signs = _hadamard(comp._padded_dim), comp._hadamard_signs.double()
        out = torch.zeros((B, 1, H, D), dtype=torch.float64, device=DEVICE)
        for b in range(B):
            x = []
            for old, new in zip(s["old"], s["new"]):
                # the codes, by the public codec; decompressed here in 64 bits
                c = comp.compress(old[b], pack=False)
                dec = (_polar(c["radius"], torch.cat(c["angles"], -1), case["bits"]) @ had) * signs
                x.append(torch.cat([dec[:, :D].reshape(old[b].shape), new[b].double()], 1))
            out[b, 0] = _attend(s["q"][b, :, 0], x[0], x[1], 1.0 / math.sqrt(D))
        return out
    comp = s["comp"]
    pd = comp._padded_dim
    had, signs = _hadamard(pd), comp._hadamard_signs.double()
    if kind == "codec":
        c = s["packed"]
        dec = (_polar(c["radius"], _unpack(c["angles_packed"], pd - 1, case["bits"]), case["bits"]) @ had) * signs
        x = s["x"].reshape(-1, case["D"]).double()
        return {"radius": x.square().sum(-1).sqrt(), "angles": None, "signs": None, "norms": None,
                "values": dec[:, :case["D"]].reshape(s["x"].shape)}
    D, N = case["D"], case["N"]
    qr = (_padded(s["q"], pd) * signs) @ had
    ck, cv = s["ck"], s["cv"]
    raw = (qr @ comp.jl_matrix.double().T) @ (2.0 * ck["qjl_signs"].double() - 1.0).T.contiguous()
    corr = raw * (math.sqrt(math.pi / 2) / comp.qjl_dim) * ck["qjl_norms"].double().reshape(1, -1)
    sc = qr @ _polar(ck["radius"], torch.cat(ck["angles"], -1), case["bits"]).T.contiguous() + corr
    val = ((_polar(cv["radius"], torch.cat(cv["angles"], -1), case["bits"]) @ had) * signs)[:, :D]
    top, idx = torch.topk(sc / math.sqrt(D), min(N, max(1, math.ceil(case["ratio"] * N))), dim=-1)
    return torch.stack([torch.softmax(top[m], -1) @ val[idx[m]] for m in range(case["M"])])
