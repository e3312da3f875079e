"""The calls of the paged KV-cache path that are timed and compared between builds.

A case is one pass of what an attention layer asks of the library in one step,
through the Python entry points:

  "decode"   each sequence appends one token and attends its whole context
             (paged_decode_append);
  "prefill"  a step of prompt chunks, with or without single-token sequences
             beside them: the step's rows are appended, then attended causally
             (reshape_and_cache, paged_prefill);
  "rope"     the fused rotary embedding + append of a step's tokens;
  "copy"     the block copies of forked sequences.

The head layouts are those of the benchmark configurations and of the shape
suite (H query heads / Hkv kv heads / head_dim D): 14/2/64, 28/4/128, 32/8/128,
32/32/80, 32/32/96, 32/2/128 and 32/1/128.  Context and chunk lengths follow
from the case alone; the seed gives the contents and the block tables.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-cpp_amd", "python")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import vllm_kv_amd as vkv  # noqa: E402
from vllm_kv_amd import workloads  # noqa: E402

DEV = "cuda:0"
TORCH = {"f16": torch.float16, "f32": torch.float32, "fp8": torch.float16}   # queries and new rows
EB = {"f16": 2, "f32": 4, "fp8": 1}                                          # bytes of a cached element


# ------------------------------------------------------------------ the cases

def _decode(name, heads, kv_heads, dim, block, dtype, seqs, lo, hi, lens="uniform"):
    return {"name": name, "kind": "decode", "heads": heads, "kv_heads": kv_heads, "dim": dim, "block": block,
            "dtype": dtype, "seqs": seqs, "lo": lo, "hi": hi, "lens": lens}


def _prefill(name, heads, kv_heads, dim, block, dtype, prompts, chunk_lo, chunk_hi, prior_hi, decodes=0,
             ctx_lo=0, ctx_hi=0, listed=False):
    return {"name": name, "kind": "prefill", "heads": heads, "kv_heads": kv_heads, "dim": dim, "block": block,
            "dtype": dtype, "prompts": prompts, "chunk_lo": chunk_lo, "chunk_hi": chunk_hi, "prior_hi": prior_hi,
            "decodes": decodes, "ctx_lo": ctx_lo, "ctx_hi": ctx_hi, "listed": listed}


def listed():
    return [
        # a few interactive sequences of a small model: the smallest call, all latency
        _decode("step_4seq_d64", 14, 2, 64, 16, "f16", 4, 1, 512),
        # the same model serving a full batch
        _decode("step_128seq_d64", 14, 2, 64, 16, "f16", 128, 1, 2048),
        # the same model in the reference's own element type
        _decode("step_32seq_d64_f32", 14, 2, 64, 16, "f32", 32, 1, 4096),
        # an 8B-class model's decode step, the headline benchmark
        _decode("step_64seq_d128", 32, 8, 128, 16, "f16", 64, 512, 4096),
        # the same heads with a quantised cache: a large batch with a long tail of contexts
        _decode("step_256seq_d128_fp8", 32, 8, 128, 16, "fp8", 256, 128, 32768, "lognormal"),
        # multi-head attention at a head size that is no power of two
        _decode("step_32seq_d80_mha", 32, 32, 80, 16, "f16", 32, 128, 2048),
        # one user's prompt on the small model: what a single request waits for
        _prefill("prompt_1seq_d64", 14, 2, 64, 16, "f16", 1, 777, 777, 0),
        # the small model's server taking in chunks of several prompts
        _prefill("chunks_8seq_d64", 14, 2, 64, 16, "f16", 8, 100, 512, 2048),
        # a step of prompt chunks only on a 7B-class model, with the step's host-built work list
        _prefill("chunks_8seq_d128", 28, 4, 128, 32, "f16", 8, 512, 512, 2048, listed=True),
        # a mixed step over a quantised cache: chunks beside running sequences
        _prefill("mixed_128seq_d128_fp8", 28, 4, 128, 32, "fp8", 8, 512, 512, 2048, 120, 1024, 8192),
        # the rotary embedding and append of such a mixed step's tokens
        {"name": "rope_append_4216", "kind": "rope", "heads": 32, "kv_heads": 8, "dim": 128, "block": 16,
         "dtype": "f16", "tokens": 4216},
        # copy-on-write of 64 forked sequences' last blocks, every layer
        {"name": "fork_64", "kind": "copy", "kv_heads": 8, "dim": 128, "block": 64, "dtype": "f16", "layers": 32,
         "pairs": 64},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    u = rng.random()
    if u < 0.5:
        heads, kv_heads, dim, block, dtypes = rng.choice([
            (14, 2, 64, 16, ("f16", "f16", "f32", "fp8")), (28, 4, 128, 32, ("f16", "fp8")),
            (32, 8, 128, 16, ("f16", "f16", "fp8", "f32")), (32, 32, 80, 16, ("f16",)), (32, 32, 96, 16, ("f16",)),
            (32, 2, 128, 16, ("f16",)), (32, 1, 128, 16, ("f16",))])
        dtype = rng.choice(dtypes)
        seqs, hi = _log(rng, 1, 256), _log(rng, 64, 16384)
        lo = max(1, _log(rng, 1, hi))
        most = 1.5e9 / (2 * kv_heads * dim * EB[dtype])  # tokens
        while seqs * (lo + hi) / 2 > most:
            hi = hi * 2 // 3
            lo = min(lo, hi)
        return {k: v for k, v in _decode("", heads, kv_heads, dim, block, dtype, seqs, lo, hi).items() if k != "name"}
    if u < 0.88:
        heads, kv_heads, dim, block, dtypes = rng.choice([
            (14, 2, 64, 16, ("f16", "f16", "fp8")), (28, 4, 128, 32, ("f16", "fp8")),
            (32, 8, 128, 16, ("f16", "f16", "fp8"))])
        dtype = rng.choice(dtypes)
        prompts, hi = _log(rng, 1, 16), _log(rng, 16, 2048)
        lo = max(2, _log(rng, max(2, hi // 8), hi))
        prior = rng.choice([0, _log(rng, 64, 4096)])
        decodes = rng.choice([0, 0, _log(rng, 1, 120)])
        while prompts * hi * (prior / 2 + hi) * heads * dim * 4 > 5e10:
            prompts, prior, hi = max(1, prompts * 2 // 3), prior * 2 // 3, max(16, hi * 3 // 4)
            lo = min(lo, hi)
        ctx = _log(rng, 64, 4096) if decodes else 0
        c = _prefill("", heads, kv_heads, dim, block, dtype, prompts, lo, hi, prior, decodes, max(1, ctx // 8) if ctx else 0,
                     ctx, rng.random() < 0.5)
        return {k: v for k, v in c.items() if k != "name"}
    if u < 0.95:
        heads, kv_heads, dim, block = rng.choice([(14, 2, 64, 16), (28, 4, 128, 32), (32, 8, 128, 16)])
        return {"kind": "rope", "heads": heads, "kv_heads": kv_heads, "dim": dim, "block": block,
                "dtype": rng.choice(["f16", "f16", "fp8"]), "tokens": _log(rng, 1, 32768)}
    kv_heads, dim, block, layers = rng.choice([(2, 64, 16, 24), (4, 128, 32, 28), (8, 128, 16, 32), (8, 128, 64, 32)])
    return {"kind": "copy", "kv_heads": kv_heads, "dim": dim, "block": block, "dtype": rng.choice(["f16", "fp8"]),
            "layers": layers, "pairs": _log(rng, 1, 64)}


# ----------------------------------------------------------- lengths and inputs

def _lens(case):
    """(query tokens, keys) of every sequence of the step; prompts first."""
    if case["kind"] == "decode":
        rng = np.random.default_rng([case["seqs"], case["lo"], case["hi"]])
        if case["lens"] == "lognormal":
            keys = np.clip(np.round(rng.lognormal(7.6, 1.0, case["seqs"])), case["lo"], case["hi"])
        else:
            keys = rng.integers(case["lo"], case["hi"] + 1, case["seqs"])
        return np.ones(case["seqs"], np.int32), keys.astype(np.int32)
    rng = np.random.default_rng([case["prompts"], case["chunk_lo"], case["chunk_hi"], case["prior_hi"], case["decodes"]])
    q = rng.integers(case["chunk_lo"], case["chunk_hi"] + 1, case["prompts"])
    prior = rng.integers(0, case["prior_hi"] + 1, case["prompts"])
    one = rng.integers(case["ctx_lo"], case["ctx_hi"] + 1, case["decodes"]) if case["decodes"] else np.zeros(0, np.int64)
    return (np.concatenate([q, np.ones(case["decodes"])]).astype(np.int32),
            np.concatenate([prior + q, one]).astype(np.int32))


def _quantise(x):
    """e4m3 codes and fp32 scales of [..., D] rows: scale = amax / 448 (1 for a zero row)."""
    amax = x.abs().amax(-1)
    scale = torch.where(amax > 0, amax / torch.full_like(amax, 448.0), torch.ones_like(amax))
    return (x / scale[..., None]).to(torch.float8_e4m3fn).view(torch.uint8), scale


def _pool(gen, blocks, block, kv_heads, dim, dtype):
    """One of K and V as a pool [N, block, Hkv, D], with its scales for a quantised one."""
    shape = (blocks, block, kv_heads, dim)
    if dtype != "fp8":
        x = torch.empty(shape, dtype=TORCH[dtype], device=DEV)
        return x.normal_(generator=gen), None
    codes = torch.empty(shape, dtype=torch.uint8, device=DEV)
    scales = torch.empty(shape[:3], dtype=torch.float32, device=DEV)
    step = max(1, (1 << 27) // (block * kv_heads * dim))
    for b in range(0, blocks, step):
        x = torch.empty((min(step, blocks - b),) + shape[1:], dtype=torch.float32, device=DEV).normal_(generator=gen)
        far = torch.empty(x.shape, dtype=torch.float32, device=DEV).uniform_(generator=gen) < 0.01
        x = torch.where(far, x * 8.0, x)  # the outliers that activations have
        codes[b:b + step], scales[b:b + step] = _quantise(x)
    return codes, scales


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def prepare(case, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    rng = np.random.default_rng(seed)
    if case["kind"] == "copy":
        n, s = 4 * case["pairs"], {"case": case}
        shape = (case["layers"], n, case["block"], case["kv_heads"], case["dim"])
        if case["dtype"] == "fp8":
            pools = [torch.randint(0, 256, shape, dtype=torch.uint8, device=DEV, generator=gen) for _ in range(2)]
            pools += [torch.rand(shape[:4], device=DEV, generator=gen) for _ in range(2)]
        else:
            pools = [torch.empty(shape, dtype=TORCH[case["dtype"]], device=DEV).normal_(generator=gen) for _ in range(2)]
        ids = rng.permutation(n)[:2 * case["pairs"]].astype(np.int32)
        s.update(pools=pools, pairs=_dev(np.stack([ids[:case["pairs"]], ids[case["pairs"]:]], 1)))
        return s

    heads, kv_heads, dim, block, dtype = case["heads"], case["kv_heads"], case["dim"], case["block"], case["dtype"]
    if case["kind"] == "rope":
        tokens = case["tokens"]
        blocks = -(-tokens // block) + 1
        slots = rng.permutation(blocks * block)[:tokens].astype(np.int32)
    else:
        q_lens, keys = _lens(case)
        lay = workloads.make_layout(keys, block, rng)
        start = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
        tokens, blocks = int(start[-1]), lay.num_blocks
        seq = np.repeat(np.arange(len(q_lens)), q_lens)
        pos = keys[seq] - q_lens[seq] + np.arange(tokens) - start[seq]
        slots = lay.slots(pos, seq)

    def rows(h):
        return torch.empty((tokens, h, dim), dtype=TORCH[dtype], device=DEV).normal_(generator=gen)

    s = {"case": case, "q": rows(heads), "k": rows(kv_heads), "v": rows(kv_heads), "slots": _dev(slots)}
    s["kc"], s["ks"] = _pool(gen, blocks, block, kv_heads, dim, dtype)
    s["vc"], s["vs"] = _pool(gen, blocks, block, kv_heads, dim, dtype)
    if case["kind"] == "rope":
        s["table"] = _dev(vkv.rope_cos_sin_host(10000.0, dim, 4096))
        s["pos"] = _dev(rng.integers(0, 4096, tokens).astype(np.int32))
        return s
    s.update(out=torch.empty_like(s["q"]), tables=_dev(lay.block_tables), lens=_dev(keys), scale=dim ** -0.5)
    if case["kind"] == "prefill":
        s.update(start=_dev(start), most=int(q_lens.max()), multi=bool((q_lens > 1).all()), list=None)
        if case["listed"]:
            words = vkv.prefill_work_list(s["out"], s["q"], s["kc"], s["vc"], s["tables"], s["lens"], s["start"],
                                          s["most"], s["scale"], start, keys, s["ks"], s["vs"])
            s["list"] = _dev(words) if len(words) else None
    return s


# ------------------------------------------------------------------- one pass

def run(s):
    kind = s["case"]["kind"]
    if kind == "copy":
        vkv.copy_blocks(s["pools"], s["pairs"])
        return s["pools"]
    caches = [x for x in (s["kc"], s["vc"], s["ks"], s["vs"]) if x is not None]
    if kind == "rope":
        vkv.rope_reshape_and_cache(s["q"], s["k"], s["v"], s["table"], s["pos"], key_cache=s["kc"], value_cache=s["vc"],
                                   slot_mapping=s["slots"], key_scales=s["ks"], value_scales=s["vs"])
        return [s["q"]] + caches
    if kind == "decode":
        vkv.paged_decode_append(s["out"], s["q"], s["kc"], s["vc"], s["tables"], s["lens"], s["scale"], s["k"], s["v"],
                                s["slots"], s["ks"], s["vs"])
        return [s["out"]] + caches
    vkv.reshape_and_cache(s["k"], s["v"], s["kc"], s["vc"], s["slots"], s["ks"], s["vs"])
    vkv.paged_prefill(s["out"], s["q"], s["kc"], s["vc"], s["tables"], s["lens"], s["start"], s["most"], s["scale"],
                      s["ks"], s["vs"], multi_token_only=s["multi"], work_list=s["list"])
    return [s["out"]] + caches


# ----------------------------------------------------- least work, tolerance, 64 bits

def work(case):
    row = case["kv_heads"] * case["dim"] * EB[case["dtype"]] + (4 * case["kv_heads"] if case["dtype"] == "fp8" else 0)
    if case["kind"] == "copy":
        return {"bytes": 2 * 2 * case["pairs"] * case["layers"] * case["block"] * row, "flops": 0}
    io = 4 if case["dtype"] == "f32" else 2
    new, token = 2 * case["kv_heads"] * case["dim"] * io, case["heads"] * case["dim"] * io
    if case["kind"] == "rope":
        n = case["tokens"]
        return {"bytes": n * (2 * token + new + 2 * row + 8) + min(n, 4096) * case["dim"] * 4, "flops": 0}
    q_lens, keys = (x.astype(np.int64) for x in _lens(case))
    pairs = int((q_lens * (keys - q_lens) + q_lens * (q_lens + 1) // 2).sum())
    n = int(q_lens.sum())
    # K and V: the cached tokens read, the step's own read once as new rows and written
    return {"bytes": int(keys.sum() - n) * 2 * row + n * (new + 2 * row + 2 * token),
            "flops": 4 * case["dim"] * case["heads"] * pairs}


def tolerance(case):
    if case["kind"] == "copy":
        return "exact"
    return {"rel": 2e-5, "max": 1e-3} if case["dtype"] == "f32" else {"rel": 2e-3, "max": 0.05}


def exact(case, seed):
    s = prepare(case, seed)
    if case["kind"] == "copy":
        src, dst = s["pairs"][:, 0].long(), s["pairs"][:, 1].long()
        for x in s["pools"]:
            x[:, dst] = x[:, src]
        return s["pools"]
    fp8, dim = case["dtype"] == "fp8", case["dim"]
    q, k, v = s["q"].double(), s["k"].double(), s["v"].double()
    if case["kind"] == "rope":
        c, w = s["table"][s["pos"].long()].double().unbind(-1)
        c, w = c[:, None], w[:, None]
        q, k = (torch.cat([x[..., :dim // 2] * c - x[..., dim // 2:] * w, x[..., dim // 2:] * c + x[..., :dim // 2] * w], -1)
                for x in (q, k))
    caches, slots = [], s["slots"].long()
    for pool, scales, x in ((s["kc"], s["ks"], k), (s["vc"], s["vs"], v)):
        if fp8:
            # codes are whole values; the scales that belong to them are the rows' largest / 448
            codes, new = _quantise(x.float())
            pool.view(-1, *pool.shape[2:])[slots] = codes
            scales.view(-1, scales.shape[2])[slots] = new
        else:
            pool = pool.double() if case["kind"] == "rope" else pool  # rotated rows are computed, appended ones copied
            pool.view(-1, *pool.shape[2:])[slots] = x.to(pool.dtype)
        caches.append(None if fp8 else pool)
    scales = [] if not fp8 else [None, None] if case["kind"] == "rope" else [s["ks"], s["vs"]]
    if case["kind"] == "rope":
        return [q] + caches + scales

    q_lens, keys = _lens(case)
    group, at, out = case["heads"] // case["kv_heads"], 0, torch.empty_like(q)
    for i, (n, m) in enumerate(zip(q_lens.tolist(), keys.tolist())):
        used = s["tables"][i, :-(-m // case["block"])].long()
        kv = []
        for pool, sc in ((s["kc"], s["ks"]), (s["vc"], s["vs"])):
            x = pool[used].view(-1, *pool.shape[2:])[:m]
            x = x.view(torch.float8_e4m3fn).float().double() * sc[used].view(-1, sc.shape[2])[:m, :, None].double() if fp8 else x.double()
            kv.append(x.transpose(0, 1).contiguous())                               # [Hkv, keys, D]
        for h in range(case["kv_heads"]):
            x = q[at:at + n, h * group:(h + 1) * group].reshape(n * group, dim)
            logits = (x @ kv[0][h].t().contiguous()) * s["scale"]
            if n > 1:
                last = m - n + torch.arange(n, device=DEV).repeat_interleave(group)
                logits.masked_fill_(torch.arange(m, device=DEV)[None] > last[:, None], -math.inf)
            out[at:at + n, h * group:(h + 1) * group] = (torch.softmax(logits, -1) @ kv[1][h]).view(n, group, dim)
        at += n
    return [out] + caches + scales
