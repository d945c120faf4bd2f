"""Performance cases of the search & sampling library: what one decoding step, one speculative round or one beam
search of a program that uses the Python binding asks of it.  A case is a dict of plain values; `prepare` builds what
such a program holds before the call (context, logits on the GPU, histories, masks, output buffers it keeps), `run`
makes one pass through the public entry points.  Logits are bulk N(0, sigma^2) with eight peak tokens per row, as the
benchmark's configurations have them; sizes are the benchmark's, real vocabularies, and any size between them."""
import math

import numpy as np
import torch

import __graft_entry__

pkg = __graft_entry__.load_package()

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2}
MAX_LOGITS = 256 * 201088  # of the largest batch here

# The selection parameters requests of one batch arrive with: a chat default, nucleus only, greedy, a wide top-k,
# and a low-temperature top-k without a nucleus.
REQUEST_MENU = [(50, 0.9, 0.7), (0, 0.9, 1.0), (1, 0.0, 1.0), (200, 0.95, 1.0), (20, 1.0, 0.3)]


def listed():
    return [
        # A chat request decoded greedily, alone on the GPU: the smallest calls there are.
        {"name": "greedy_1x32064_f32", "op": "greedy", "rows": 1, "vocab": 32064, "dtype": "f32", "sigma": 2.0, "history": 512},
        # Greedy decoding of a large batch of bf16 logits (offline generation): one pass over the logits.
        {"name": "greedy_256x201088_bf16", "op": "greedy", "rows": 256, "vocab": 201088, "dtype": "bf16", "sigma": 3.0, "history": 0},
        # The everyday sampling step of a server: top-k with a nucleus inside it.
        {"name": "topk_64x128256_f32", "op": "sample", "rows": 64, "vocab": 128256, "dtype": "f32", "sigma": 3.0, "k": 50, "p": 0.9, "temperature": 0.7},
        # Nucleus sampling without top-k, the other default of chat servers.
        {"name": "topp_32x151936_bf16", "op": "sample", "rows": 32, "vocab": 151936, "dtype": "bf16", "sigma": 5.0, "k": 0, "p": 0.9, "temperature": 1.0},
        # Temperature only (k = 0, p = 1): samples from the whole vocabulary.
        {"name": "temperature_16x128256_f16", "op": "sample", "rows": 16, "vocab": 128256, "dtype": "f16", "sigma": 3.0, "k": 0, "p": 1.0, "temperature": 1.0},
        # A generator's step on its own engine: kept sets, draws in the engine's order, then EOS / append.
        {"name": "generate_4x151936_f16", "op": "generate", "rows": 4, "vocab": 151936, "dtype": "f16", "sigma": 3.0, "k": 50, "p": 0.9, "temperature": 0.8, "history": 256},
        # A batched sampler's step: every request has parameters and a logits row of its own; an odd vocabulary.
        {"name": "mixed_48x50257_f16", "op": "mixed", "rows": 48, "vocab": 50257, "dtype": "f16", "sigma": 3.0},
        # Structured output: a grammar mask, a repetition penalty and a nucleus over a large batch.
        {"name": "masked_256x201088_f32", "op": "masked", "rows": 256, "vocab": 201088, "dtype": "f32", "sigma": 3.0, "p": 0.95, "allowed": 0.05, "history": 1024},
        # Log-probabilities of a prompt's last tokens (prefill): hand-off out of the model's output, penalty, log-softmax.
        {"name": "logprobs_16x151936_f16", "op": "logprobs", "rows": 16, "seq": 8, "vocab": 151936, "dtype": "f16", "sigma": 3.0, "history": 128},
        # A whole short beam search as a transcription program runs it: scorer, reordered cache, hypotheses.
        {"name": "beam_search_2x4x51865_f16", "op": "beam_search", "batch": 2, "beams": 4, "vocab": 51865, "dtype": "f16", "sigma": 2.0, "steps": 12,
         "tensors": 8, "heads": 6, "seq": 448, "head_dim": 64},
        # One step of a large beam search: candidate selection and the reorder of a long cache.
        {"name": "beam_step_8x4x151936_f16", "op": "beam_step", "batch": 8, "beams": 4, "vocab": 151936, "dtype": "f16", "sigma": 2.0,
         "tensors": 32, "heads": 4, "seq": 2048, "head_dim": 128},
        # A speculative round: target selection of the verify rows, then accept / resample.
        {"name": "speculative_8x5x128256_bf16", "op": "speculative", "batch": 8, "draft": 5, "vocab": 128256, "dtype": "bf16", "sigma": 3.0, "k": 50, "p": 0.9,
         "temperature": 0.8, "history": 128},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: the kinds above, any number of rows, any vocabulary from 8000 to 201088, each element type."""
    op = rng.choice(["greedy", "greedy", "sample", "sample", "sample", "generate", "mixed", "masked", "logprobs", "beam_search", "beam_step", "speculative"])
    c = {"op": op, "vocab": _log(rng, 8000, 201088), "dtype": rng.choice(["f32", "f16", "bf16"]), "sigma": round(rng.uniform(2.0, 5.0), 2)}
    v = c["vocab"]
    if op == "greedy":
        c.update(rows=min(_log(rng, 1, 256), MAX_LOGITS // v), history=rng.choice([0, 0, _log(rng, 16, 2048)]))
    elif op == "sample":
        kind = rng.choice(["topk", "topk", "topp", "topp", "wide", "temperature"])
        k, p = {"topk": (_log(rng, 2, 64), round(rng.uniform(0.7, 1.0), 3)), "topp": (0, round(rng.uniform(0.7, 0.98), 3)),
                "wide": (_log(rng, 65, 2048), round(rng.uniform(0.7, 1.0), 3)), "temperature": (0, 1.0)}[kind]
        # the flattest rows of temperature-only and wide-nucleus batches are a few requests, not a full server batch
        rows = {"topk": 256, "topp": 64, "wide": 128, "temperature": 24}[kind]
        c.update(rows=_log(rng, 1, rows), k=k, p=p, temperature=round(rng.uniform(0.5, 1.2), 2))
    elif op == "generate":
        c.update(rows=_log(rng, 1, 64), k=_log(rng, 2, 64), p=round(rng.uniform(0.7, 1.0), 3), temperature=round(rng.uniform(0.5, 1.2), 2),
                 history=_log(rng, 16, 2048))
    elif op == "mixed":
        c.update(rows=_log(rng, 2, 128))
    elif op == "masked":
        # what grammars allow at a position: a handful of tokens up to a few thousand
        c.update(rows=_log(rng, 1, 256), p=round(rng.uniform(0.7, 0.98), 3), allowed=round(math.exp(rng.uniform(math.log(0.001), math.log(0.06))), 5),
                 history=_log(rng, 16, 1500))
    elif op == "logprobs":
        c.update(rows=_log(rng, 1, 64), seq=_log(rng, 1, 16), history=_log(rng, 16, 1024))
    elif op == "beam_search":
        c.update(batch=rng.randint(1, 3), beams=rng.randint(2, 6), steps=rng.randint(6, 16), tensors=2 * rng.randint(2, 4), heads=rng.randint(4, 8),
                 seq=_log(rng, 128, 448), head_dim=64)
    elif op == "beam_step":
        c.update(batch=rng.randint(1, 8), beams=rng.randint(2, 5), tensors=2 * rng.randint(4, 12), heads=rng.choice([2, 4, 8]), seq=_log(rng, 128, 1024), head_dim=128)
    else:
        c.update(batch=rng.randint(1, 16), draft=rng.randint(2, 8), k=_log(rng, 2, 64), p=round(rng.uniform(0.7, 1.0), 3),
                 temperature=round(rng.uniform(0.5, 1.2), 2), history=_log(rng, 16, 1024))
    return c


def _logits(g, rows, vocab, dtype, sigma):
    x = torch.randn(rows, vocab, generator=g, device="cuda") * sigma
    peaks = torch.randint(0, vocab, (rows, 8), generator=g, device="cuda")
    x.scatter_add_(1, peaks, torch.full((rows, 8), 10.0, device="cuda"))
    return x.to(DTYPES[dtype])


def _ids(g, rows, n, vocab):
    return torch.randint(0, vocab, (rows, n), generator=g, device="cuda", dtype=torch.int32)


def _uniforms(g, *shape, dtype=torch.float64):
    return torch.rand(*shape, generator=g, device="cuda", dtype=dtype)


def _rows(case):
    if "rows" in case:
        return case["rows"]
    return case["batch"] * (case["beams"] if "beams" in case else case["draft"] + 1)


def prepare(case, seed):
    op, v = case["op"], case["vocab"]
    rows = _rows(case)
    g = torch.Generator(device="cuda").manual_seed(seed)
    s = {"case": case, "ctx": pkg.SearchContext(rows, v)}
    xf = None
    if case.get("history") and op not in ("masked", "speculative"):
        xf = pkg.LogitsXform(history=_ids(g, rows, case["history"], v), repetition_penalty=1.1)
    if op == "logprobs":
        s["raw"] = _logits(g, rows * case["seq"], v, case["dtype"], case["sigma"]).view(rows, case["seq"], v)
        s["index"] = [(7 * r + seed) % case["seq"] for r in range(rows)]
        s["out"] = torch.empty((rows, v), dtype=torch.float32, device="cuda")
    elif op == "beam_search":
        s["logits"] = [_logits(g, rows, v, case["dtype"], case["sigma"]) for _ in range(case["steps"])]
        s["prompt"] = np.random.RandomState(seed % (1 << 32)).randint(0, v, (case["batch"], 4)).astype(np.int32)
    else:
        s["logits"] = _logits(g, rows, v, case["dtype"], case["sigma"])
    if op in ("beam_search", "beam_step"):
        shape = (rows, case["heads"], case["seq"], case["head_dim"])
        s["present"] = [torch.randint(-30000, 30000, shape, generator=g, device="cuda", dtype=torch.int16).view(torch.float16)
                        for _ in range(case["tensors"])]
        s["past"] = [torch.zeros_like(t) for t in s["present"]]
    if op == "beam_step":
        s["scores"] = -5.0 * _uniforms(g, rows, dtype=torch.float32)
        s["parents"] = torch.randint(0, case["beams"], (rows,), generator=g, device="cuda", dtype=torch.int32) + \
            torch.arange(case["batch"], device="cuda", dtype=torch.int32).repeat_interleave(case["beams"]) * case["beams"]
    if op == "mixed":
        s["params"] = [REQUEST_MENU[(r + seed) % len(REQUEST_MENU)] for r in range(rows)]
        s["logits"] = [row.clone() for row in s["logits"]]  # every request's logits lie on their own
    if op == "masked":
        words = (v - 1) // 32 + 1
        bits = torch.rand(rows, words * 32, generator=g, device="cuda") < case["allowed"]
        bits[:, v:] = False
        bits[:, 0] = True
        weights = 2 ** torch.arange(32, device="cuda", dtype=torch.int64)
        mask = torch.cat([(part.view(-1, words, 32).long() * weights).sum(-1) for part in bits.split(64)])
        mask = torch.where(mask >= 2 ** 31, mask - 2 ** 32, mask).int().contiguous()
        xf = pkg.LogitsXform(mask=mask, history=_ids(g, rows, case["history"], v), repetition_penalty=1.2,
                             mask_allowed_max=int(bits.sum(dim=1).max()))
    if op == "speculative":
        b, d, h = case["batch"], case["draft"], case["history"]
        # the draft model's logits resemble the target's; its kept sets and proposals are at hand when the round begins
        x = s["logits"].view(b, d + 1, v)[:, :d].float()
        draft = (x + 0.5 * torch.randn(b, d, v, generator=g, device="cuda")).view(b * d, v).to(DTYPES[case["dtype"]])
        tok, kc, ki, kp = s["ctx"].sample(draft, _uniforms(g, b * d), k=case["k"], p=case["p"], temperature=case["temperature"], kept_capacity=64)
        s["draft"] = (kc.view(b, d), ki.view(b, d, 64), kp.view(b, d, 64))
        s["proposal"] = tok.view(b, d)
        # every verify row sees its sequence's prefix and the proposals before it
        prefix = _ids(g, b, h, v)
        hist = torch.cat([prefix, s["proposal"]], dim=1).repeat_interleave(d + 1, dim=0).contiguous()
        lens = (h + torch.arange(d + 1, device="cuda", dtype=torch.int32)).repeat(b).contiguous()
        xf = pkg.LogitsXform(history=hist, history_lens=lens, repetition_penalty=1.1)
        s["accept_u"], s["sample_u"] = _uniforms(g, b, d, dtype=torch.float32), _uniforms(g, b, d + 1)
    s["xf"] = xf
    s["uniforms"] = _uniforms(g, rows)
    s["tokens"] = torch.zeros(rows, dtype=torch.int32, device="cuda")
    if op in ("greedy", "generate"):
        s["eos_seen"] = torch.zeros(rows, dtype=torch.int32, device="cuda")
        s["sequences"] = torch.zeros((rows, 2048), dtype=torch.int32, device="cuda")
        s["done"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    op = case["op"]
    if op == "greedy":
        ctx.argmax(s["logits"], xf=s["xf"], out=s["tokens"])
        ctx.greedy_tail(s["tokens"], s["eos_seen"], [2], 0, s["sequences"], 100, s["done"])
        return s["tokens"], s["eos_seen"], s["sequences"], s["done"]
    if op == "sample":
        return ctx.sample(s["logits"], s["uniforms"], k=case["k"], p=case["p"], temperature=case["temperature"], out=s["tokens"])
    if op == "generate":
        _, kc, ki, kp = ctx.sample(s["logits"], s["uniforms"], k=case["k"], p=case["p"], temperature=case["temperature"], xf=s["xf"], out=s["tokens"],
                                   kept_capacity=64)
        tokens, used = ctx.draw_in_order(kc, ki, kp, s["uniforms"])
        ctx.greedy_tail(tokens, s["eos_seen"], [2], 0, s["sequences"], 100, s["done"])
        return tokens, used, kc, ki, kp, s["eos_seen"], s["sequences"], s["done"]
    if op == "mixed":
        return ctx.sample(s["logits"], s["uniforms"], per_row=s["params"], out=s["tokens"])
    if op == "masked":
        return ctx.sample(s["logits"], s["uniforms"], k=0, p=case["p"], temperature=1.0, xf=s["xf"], out=s["tokens"])
    if op == "logprobs":
        out = ctx.logits_handoff(s["raw"], token_index=s["index"], out=s["out"])
        ctx.process_logits(out, s["xf"])
        return ctx.softmax(out, log=True)
    if op == "beam_step":
        scores, tokens, beams = ctx.beam_select(s["logits"], case["batch"], case["beams"], s["scores"])
        return scores, tokens, beams, ctx.kv_gather(s["present"], s["past"], s["parents"])
    if op == "beam_search":
        scorer = pkg.BeamScorer(ctx, case["batch"], case["beams"], 64, 0, [2], 1.0, True)
        scorer.set_prompt(s["prompt"])
        for logits in s["logits"]:
            scorer.search_step(logits)
            ctx.kv_gather(s["present"], s["past"], scorer.next_indices)
            if scorer.is_done():
                break
        best = [scorer.hypothesis(b, 0) for b in range(case["batch"])]
        scorer.close()
        return [np.array(t, np.int32) for t, _ in best], [float(x) for _, x in best], s["past"]
    b, d = case["batch"], case["draft"]
    _, kc, ki, kp = ctx.sample(s["logits"], s["uniforms"], k=case["k"], p=case["p"], temperature=case["temperature"], xf=s["xf"], out=s["tokens"],
                               kept_capacity=64)
    target = (kc.view(b, d + 1), ki.view(b, d + 1, 64), kp.view(b, d + 1, 64))
    accepted, final, draws = ctx.spec_verify_sparse(target, s["draft"], s["proposal"], s["accept_u"], s["sample_u"], mode=0)
    return accepted, final, draws, kc, ki, kp


def work(case):
    """Inputs read once, outputs written once; no matrix products, so a few operations per logit."""
    rows, v, elt = _rows(case), case["vocab"], BYTES[case["dtype"]]
    op, history = case["op"], case.get("history", 0)
    logits = rows * v
    b = logits * elt + rows * history * 4 + rows * 12
    if op == "masked":
        # a masked logit is not needed: the mask, the allowed logits (a sector of 32 bytes each, or every sector) and the history
        sector = 32 // elt
        b = rows * (v / 8 + v * elt * (1.0 - (1.0 - case["allowed"]) ** sector) + history * 4)
    elif op == "logprobs":
        b += logits * 4
    elif op in ("beam_search", "beam_step"):
        kv = case["tensors"] * rows * case["heads"] * case["seq"] * case["head_dim"] * 2
        b = (logits * elt + 2 * kv) * case.get("steps", 1)
    elif op in ("generate", "speculative"):
        b += rows * 64 * 8
    return {"bytes": float(b), "flops": 2.0 * logits * case.get("steps", 1)}


def tolerance(case):
    """Token ids, counts, flags and gathered bytes are the reference's to the bit; probabilities and scores are fp32."""
    return {"rel": 1e-5} if case["op"] in ("generate", "logprobs", "beam_search", "beam_step", "speculative") else "exact"
