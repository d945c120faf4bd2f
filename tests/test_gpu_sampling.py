"""GPU parity: argmax, logits processing and top-k / top-p sampling through the C ABI against the CPU
oracle on the same seeded inputs.  Bit-exact token ids and indices; probabilities compared bitwise
too (tolerance stated by the task: 1e-5 relative -- the kernels meet it with zero difference)."""
import os

import numpy as np
import pytest
import torch

from gpu_common import LOWEST, make_mask, pkg, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = pkg().SearchContext(256, 201088)
    yield c
    c.close()


def bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("rows,vocab", [(1, 32064), (3, 33), (4, 8192), (2, 8193), (5, 50257), (64, 128256), (3, 201088)])
def test_argmax_matches_oracle(ctx, orc, rows, vocab):
    say("argmax", rows, vocab)
    rng = np.random.default_rng(rows * 1000 + vocab)
    x = (rng.standard_normal((rows, vocab)) * 2).astype(np.float32)
    x[0] = np.round(x[0])  # ties
    got = ctx.argmax(torch.from_numpy(x).cuda()).cpu().numpy()
    assert np.array_equal(got, orc.argmax_batch(x))


def test_argmax_special_values(ctx, orc):
    say("argmax special")
    x = np.zeros((6, 1000), np.float32)
    x[0, :] = -np.inf
    x[1, 0] = np.nan
    x[1, 5] = 7
    x[2, 3] = np.nan
    x[2, 9] = 1
    x[3, 10] = -0.0
    x[3, :] *= -1  # all -0/+0
    x[4, :] = LOWEST
    x[5, 999] = np.inf
    got = ctx.argmax(torch.from_numpy(x).cuda()).cpu().numpy()
    assert np.array_equal(got, orc.argmax_batch(x))


@pytest.mark.parametrize("vocab", [40000, 131072, 201088])
def test_argmax_special_values_across_chunks(ctx, orc, vocab):
    """Rows of several 32768-id chunks: equal maxima in different chunks (the lowest id wins), a maximum in the last
    partial chunk, NaN at id 0 (wins outright), NaN elsewhere (never wins), rows without a finite value."""
    say("argmax special, chunks", vocab)
    rng = np.random.default_rng(vocab)
    x = (rng.standard_normal((10, vocab)) * 2).astype(np.float32)
    x[0, [vocab - 1, 33000, 5]] = 50.0
    x[1, [vocab - 1, 33000]] = 50.0
    x[2, vocab - 1] = 50.0
    x[3, 0] = np.nan
    x[3, 35000] = 60.0
    x[4, 35000] = np.nan
    x[4, 36000] = np.nan
    x[5, :] = -np.inf
    x[6, :] = np.nan
    x[7, :] = -np.inf
    x[7, 39999] = LOWEST
    x[8, :] = 3.0
    x[9, :] = np.nan
    x[9, 0] = 1.0
    x[9, 39000] = 1.0
    want = orc.argmax_batch(x)
    assert np.array_equal(ctx.argmax(torch.from_numpy(x).cuda()).cpu().numpy(), want)
    xf = pkg().LogitsXform(history=torch.from_numpy(np.tile(np.array([[5, 33000, 35000, 0]], np.int32), (10, 1))).cuda(),
                           repetition_penalty=1.3)
    proc = np.stack([orc.apply_repetition_penalty(x[r], np.array([5, 33000, 35000, 0], np.int32), 1.3) for r in range(10)])
    assert np.array_equal(ctx.argmax(torch.from_numpy(x).cuda(), xf=xf).cpu().numpy(), orc.argmax_batch(proc))
    with np.errstate(over="ignore"):  # lowest() becomes -inf in fp16
        h = x.astype(np.float16)
    assert np.array_equal(ctx.argmax(torch.from_numpy(h).cuda()).cpu().numpy(), orc.argmax_batch(orc.fp16_to_fp32(h)))


def test_argmax_of_rows_longer_than_the_chunked_path_holds(orc):
    """More than 16 chunks per row (vocabulary above 524288): the exact path answers; exactly 16: the chunked one."""
    say("argmax very long rows")
    rng = np.random.default_rng(77)
    for vocab in (524288, 524289 + 4096):
        ctx = pkg().SearchContext(2, vocab)
        x = (rng.standard_normal((2, vocab)) * 2).astype(np.float32)
        x[1, vocab - 1] = 40.0
        assert np.array_equal(ctx.argmax(torch.from_numpy(x).cuda()).cpu().numpy(), orc.argmax_batch(x))
        ctx.close()


def test_argmax_fp16(ctx, orc):
    say("argmax fp16")
    rng = np.random.default_rng(5)
    h = (rng.standard_normal((7, 151936)) * 2).astype(np.float16)
    got = ctx.argmax(torch.from_numpy(h).cuda()).cpu().numpy()
    assert np.array_equal(got, orc.argmax_batch(orc.fp16_to_fp32(h)))


def test_config1_greedy_with_repetition_penalty(ctx, orc):
    """Benchmark configuration 1: batch 1, vocab 32064, N(0,2^2) logits with a +8 spike, repetition penalty
    1.1 over 512 history ids, greedy argmax per step (16 of the 256 steps here)."""
    rng = np.random.default_rng(1)
    vocab = 32064
    for step in range(16):
        say("config1 step", step)
        x = (rng.standard_normal((1, vocab)) * 2).astype(np.float32)
        x[0, rng.integers(0, vocab)] += 8
        hist = rng.integers(0, vocab, (1, 512)).astype(np.int32)
        xf = pkg().LogitsXform(history=torch.from_numpy(hist).cuda(), repetition_penalty=1.1)
        got = ctx.argmax(torch.from_numpy(x).cuda(), xf=xf).cpu().numpy()
        want = orc.argmax(orc.apply_repetition_penalty(x[0], hist[0], 1.1))
        assert got[0] == want


@pytest.mark.parametrize("rows,vocab,dtype", [(2, 5000, np.float32), (3, 40000, np.float16), (40, 70001, np.float32),
                                              (33, 128256, np.float16)])
def test_argmax_with_fused_logits_processing(ctx, orc, rows, vocab, dtype):
    """Greedy selection with grammar mask, min-length and repetition penalty fused, on the
    single-workgroup-per-row kernel (small shapes) and the chunked kernel (large shapes)."""
    say("argmax fused", rows, vocab, dtype.__name__)
    rng = np.random.default_rng(rows + vocab)
    x = (rng.standard_normal((rows, vocab)) * 2).astype(dtype)
    x32 = orc.fp16_to_fp32(x) if dtype == np.float16 else x
    mask = make_mask(rng, rows, vocab, 0.5)
    hist = rng.integers(-2, vocab + 2, (rows, 300)).astype(np.int32)
    top = np.argmax(x32, axis=1)
    hist[:, 0] = top  # the raw maximum is penalised
    eos = [int(np.argsort(x32[0])[-2]), vocab - 1]
    xf = pkg().LogitsXform(mask=torch.from_numpy(mask.view(np.int32)).cuda(), history=torch.from_numpy(hist).cuda(),
                           repetition_penalty=1.7, eos_ids=eos, apply_min_length=True)
    got = ctx.argmax(torch.from_numpy(x).cuda(), xf=xf).cpu().numpy()
    proc = orc.apply_mask(x32, mask)
    for r in range(rows):
        row = orc.apply_min_length(proc[r], 0, 1, eos)
        row = orc.apply_repetition_penalty(row, hist[r], 1.7)
        assert got[r] == orc.argmax(row), r


@pytest.mark.parametrize("vocab", [33, 1000, 8192, 40000])
def test_process_logits_in_place(ctx, orc, vocab):
    say("process_logits", vocab)
    rng = np.random.default_rng(vocab)
    rows = 3
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    mask = make_mask(rng, rows, vocab, 0.3)
    hist = rng.integers(-2, vocab + 2, (rows, 100)).astype(np.int32)
    eos = [1, vocab - 1, vocab + 5]
    xf = pkg().LogitsXform(mask=torch.from_numpy(mask.view(np.int32)).cuda(), history=torch.from_numpy(hist).cuda(),
                           history_len=77, repetition_penalty=1.3, eos_ids=eos, apply_min_length=True)
    got = ctx.process_logits(torch.from_numpy(x).cuda(), xf).cpu().numpy()
    want = orc.apply_mask(x, mask)
    for r in range(rows):
        want[r] = orc.apply_min_length(want[r], 0, 1, eos)
        want[r] = orc.apply_repetition_penalty(want[r], hist[r, :77], 1.3)
    assert np.array_equal(bits(got), bits(want))
    assert np.isinf(got).any() or vocab < 100  # lowest()*1.3 overflows to -inf, as in the reference


def sample_and_check(ctx, orc, x, u, k, p, t, cap=64):
    rows = x.shape[0]
    tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=k, p=p, temperature=t,
                                 kept_capacity=cap)
    tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
    for r in range(rows):
        idx, probs = orc.sampled_categorical(x[r], k, p, t)
        assert kc[r] == len(idx), (r, kc[r], len(idx))
        n = min(len(idx), cap)
        assert np.array_equal(ki[r, :n], idx[:n]), r
        assert np.array_equal(bits(kp[r, :n]), bits(probs[:n])), r
        assert tok[r] == idx[orc.discrete_draw(probs, u[r])], r


@pytest.mark.parametrize("rows,vocab,k,p,t", [
    (4, 4099, 50, 0.9, 0.7), (3, 8192, 2, 0.0, 1.0), (2, 20000, 64, 0.5, 1.3), (5, 128256, 50, 0.9, 0.7),
    (2, 128256, 50, 1.0, 1.0), (3, 201088, 40, 0.95, 0.8), (2, 65, 64, 0.9, 1.0), (2, 300, 50, 0.9, 1.0),
])
def test_sample_topk_topp_small_k(ctx, orc, rows, vocab, k, p, t):
    say("sample topk", rows, vocab, k, p, t)
    rng = np.random.default_rng(vocab + k)
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    u = rng.random(rows)
    before = ctx.fallback_rows()
    sample_and_check(ctx, orc, x, u, k, p, t)
    assert ctx.fallback_rows() == before  # all rows stayed on the single-pass path


@pytest.mark.parametrize("vocab,k,p,t", [(128256, 50, 0.9, 0.7), (5000, 30, 0.0, 1.0), (201088, 0, 0.9, 1.0)])
def test_draw_on_cdf_boundaries(ctx, orc, vocab, k, p, t):
    """Uniform draws placed exactly on, just below and just above values of the cumulative distribution
    std::discrete_distribution builds (double quotients summed in sequence): the kernels' tree-order
    CDF cannot decide these and must fall back to the sequential construction."""
    say("cdf boundaries", vocab, k, p, t)
    rng = np.random.default_rng(vocab + k)
    base = (rng.standard_normal(vocab) * 3).astype(np.float32)
    idx, probs = orc.sampled_categorical(base, k, p, t)
    assert len(idx) >= 3
    total = 0.0
    for q in probs:  # libstdc++: sum in double, in order
        total += float(q)
    cp, run = [], 0.0
    for q in probs[:-1]:
        run += float(q) / total
        cp.append(run)
    picks = [0, len(cp) // 2, len(cp) - 1]
    us = []
    for j in picks:
        us += [cp[j], np.nextafter(cp[j], 0.0), np.nextafter(cp[j], 1.0)]
    us = np.array([v for v in us if 0.0 <= v < 1.0], np.float64)
    x = np.tile(base, (len(us), 1))
    sample_and_check(ctx, orc, x, us, k, p, t, cap=64)


def tokens_only(ctx, x, u, k, p, t):
    """A call that asks for the tokens alone (no kept sets): the route the benchmark times."""
    return ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(np.asarray(u, np.float64)).cuda(), k=k, p=p,
                      temperature=t).cpu().numpy()


@pytest.mark.parametrize("rows,vocab,k,p,t", [
    (64, 128256, 50, 0.9, 0.7), (32, 128256, 64, 0.95, 1.0), (16, 201088, 40, 0.5, 1.3), (8, 4099, 50, 0.0, 1.0),
    (8, 32064, 2, 0.9, 0.25), (8, 70001, 17, 1.0, 2.0), (4, 300, 50, 0.9, 1.0),
])
def test_token_only_calls_match_the_oracle(ctx, orc, rows, vocab, k, p, t):
    """Calls without kept-set outputs decide the nucleus cut and the draw from one fp64 prefix sum with guard
    bands; the tokens must be the ones the sequential arithmetic of the reference yields."""
    say("token only", rows, vocab, k, p, t)
    rng = np.random.default_rng(vocab * 7 + k)
    for rep in range(3):
        x = (rng.standard_normal((rows, vocab)) * (1.0 + 2.0 * rep)).astype(np.float32)
        if rep == 2:
            x = np.round(x * 4) / 4  # heavy ties
        u = rng.random(rows)
        got = tokens_only(ctx, x, u, k, p, t)
        assert np.array_equal(got, orc.sample_batch(x, k, p, t, u)), rep


@pytest.mark.parametrize("vocab,k,t", [(128256, 50, 0.7), (5000, 30, 1.0), (40000, 64, 1.5)])
def test_token_only_calls_on_the_edges_of_their_guard_bands(ctx, orc, vocab, k, t):
    """Token-only calls with draws placed on, just below and just above the values of the cumulative
    distribution, and with top-p masses placed on, just below and just above the fp32 cumulative probabilities
    of the reference's cut loop: none of these can be decided from the prefix sum in tree order, so the kernel
    must notice and run the sequential epilogue."""
    say("token only edges", vocab, k, t)
    rng = np.random.default_rng(vocab + k)
    base = (rng.standard_normal(vocab) * 3).astype(np.float32)
    # draws on the boundaries of the final distribution, for a cut in the middle and for no cut
    for p in (0.9, 0.0):
        idx, probs = orc.sampled_categorical(base, k, p, t)
        assert len(idx) >= 3
        total = 0.0
        for q in probs:
            total += float(q)
        cp, run = [], 0.0
        for q in probs[:-1]:
            run += float(q) / total
            cp.append(run)
        us = []
        for j in sorted({0, 1, len(cp) // 2, len(cp) - 1}):
            us += [cp[j], np.nextafter(cp[j], 0.0), np.nextafter(cp[j], 1.0)]
        us = np.array([v for v in us if 0.0 <= v < 1.0], np.float64)
        x = np.tile(base, (len(us), 1))
        assert np.array_equal(tokens_only(ctx, x, us, k, p, t), orc.sample_batch(x, k, p, t, us))
    # masses on the boundaries of the cut: the reference adds the fp32 probabilities in rank order
    _, pr = orc.sampled_categorical(base, k, 0.0, t)
    cum, run = [], np.float32(0.0)
    for q in pr:
        run = np.float32(run + q)
        cum.append(run)
    u = rng.random(8)
    x = np.tile(base, (len(u), 1))
    for j in sorted({0, 1, len(cum) // 3, len(cum) // 2, len(cum) - 2}):
        for mass in (cum[j], np.nextafter(cum[j], np.float32(0)), np.nextafter(cum[j], np.float32(1))):
            mass = float(mass)
            if not 0.0 < mass < 1.0:
                continue
            kept = len(orc.sampled_categorical(base, k, mass, t)[0])
            assert kept in (j + 1, j + 2), (j, mass, kept)  # the cut really falls where the mass was placed
            assert np.array_equal(tokens_only(ctx, x, u, k, mass, t), orc.sample_batch(x, k, mass, t, u)), (j, mass)


@pytest.mark.parametrize("vocab,sigma,p,dtype", [
    (128256, 5.0, 0.9, np.float32), (50257, 3.0, 0.9, np.float16), (151936, 4.0, 0.95, np.float32), (5000, 1.0, 0.6, np.float32),
    (65, 2.0, 0.9, np.float32), (64, 2.0, 0.9, np.float32), (20000, 2.0, 0.999999, np.float16), (32064, 0.0, 0.5, np.float32),
])
def test_token_only_nucleus_rows_on_the_edges_of_their_guard_bands(ctx, orc, vocab, sigma, p, dtype):
    """Nucleus rows whose token alone is asked for are drawn from one fp64 prefix sum unless the stop or the draw is too
    close to call: draws placed on, and within the guard bands beside, the reference's cumulative values (lists of a few
    tokens, of one window and of two), and masses on both sides of the ones at which the reference's search changes its
    mind -- also where it misses a stop, at the end of a batch of 16, 64, 256 ... elements."""
    say("token only nucleus", vocab, sigma, p, dtype)
    rng = np.random.default_rng(vocab + int(10 * p))
    base = (rng.standard_normal(vocab) * sigma).astype(dtype)
    kept = lambda mass: len(orc.sampled_categorical(base.astype(np.float32), 0, mass, 1.0)[0])
    _, probs = orc.sampled_categorical(base.astype(np.float32), 0, p, 1.0)
    cp = np.cumsum(np.asarray(probs, np.float64)) / np.sum(np.asarray(probs, np.float64))
    us = list(rng.random(16)) + [0.0, np.nextafter(1.0, 0.0)]
    for j in sorted({0, 1, len(cp) // 3, len(cp) // 2, len(cp) - 2} & set(range(len(cp)))):
        us += [cp[j], np.nextafter(cp[j], 0.0), np.nextafter(cp[j], 1.0), cp[j] - 1e-7, cp[j] + 1e-7, cp[j] - 3e-7, cp[j] + 3e-7]
    us = np.array([v for v in us if 0.0 <= v < 1.0], np.float64)
    x = np.tile(base, (len(us), 1))
    assert np.array_equal(tokens_only(ctx, x, us, 0, p, 1.0), orc.sample_batch(x.astype(np.float32), 0, p, 1.0, us))
    if vocab > 20000:
        return
    u = rng.random(6)
    x = np.tile(base, (len(u), 1))
    for count in (1, 15, 16, 63, 64, 256, 1024):
        low, high = np.float32(0.0), np.float32(1.0)  # the masses between which the search goes past `count` elements
        for _ in range(40):
            mid = np.float32((low + high) / 2)
            if mid in (low, high):
                break
            low, high = (mid, high) if kept(float(mid)) <= count else (low, mid)
        for mass in (low, high):
            if 0.0 < mass < 1.0:
                want = orc.sample_batch(x.astype(np.float32), 0, float(mass), 1.0, u)
                assert np.array_equal(tokens_only(ctx, x, u, 0, float(mass), 1.0), want), (count, mass)


@pytest.mark.parametrize("kind,vocab,p,t", [
    ("flat", 128256, 0.9, 1.0), ("flat", 40000, 0.97, 1.5), ("ties", 128256, 0.9, 1.0), ("ties", 50257, 0.6, 0.7), ("crowd", 128256, 0.5, 1.0),
    ("peaks", 151936, 0.9, 1.0), ("peaks", 4099, 0.95, 0.5), ("deep", 32064, 0.9995, 1.0), ("one", 151936, 0.3, 1.0), ("penalty", 50257, 0.9, 1.0),
])
def test_token_only_nucleus_rows_that_are_picked_instead_of_sorted(ctx, orc, kind, vocab, p, t):
    """Token-only nucleus rows whose token is picked from two buckets of a histogram: more candidates than a thread keeps in
    registers, ties by the dozen and by the ten thousand in the buckets of the stop and of the draw, nuclei that end with the
    first element below the candidates or after one element, exponentials down to nothing, processed logits."""
    say("picked", kind, vocab, p, t)
    rng = np.random.default_rng(vocab + int(100 * p))
    rows = 12
    x = rng.standard_normal((rows, vocab)).astype(np.float32)
    dtype, xf = torch.float32, {}
    if kind == "flat":
        x *= np.linspace(0.5, 2.5, rows, dtype=np.float32)[:, None]
    elif kind == "ties":
        x, dtype = 2.0 * x + 12.0, torch.bfloat16
    elif kind == "crowd":
        x = np.round(x)
    elif kind == "peaks":
        x[:, :20] += np.linspace(6.0, 30.0, rows, dtype=np.float32)[:, None]
    elif kind == "deep":
        x *= 6.0
    elif kind == "one":
        x[:, 77] += 40.0
    else:
        x *= 3.0
        xf = dict(history=rng.integers(0, vocab, (rows, 200)).astype(np.int32), penalty=1.2)
    xd = torch.from_numpy(np.ascontiguousarray(x, np.float32)).cuda().to(dtype)
    xw = xd.float().cpu().numpy()
    form = pkg().LogitsXform(history=torch.from_numpy(xf["history"]).cuda(), repetition_penalty=xf["penalty"]) if xf else None
    if xf:
        y = xd.clone()
        ctx.process_logits(y, form)
        xw = y.cpu().numpy()
    for rep in range(3):
        u = rng.random(rows)
        u[0], u[1] = 0.0, np.nextafter(1.0, 0.0)
        got = ctx.sample(xd, torch.from_numpy(u).cuda(), k=0, p=p, temperature=t, xf=form).cpu().numpy()
        assert np.array_equal(got, orc.sample_batch(xw, 0, p, t, u)), rep


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("dtype,shift,depth", [("f16", -33.0, None), ("f32", 0.0, 1419.6), ("f32", 0.0, 4258.7), ("f32", 3.0, 2839.1), ("f32", 3.0, 104.0)])
def test_picked_rows_whose_nucleus_ends_in_an_element_far_below(ctx, orc, dtype, shift, depth, masked):
    """Every third logit lies so far below the others that it weighs nothing, and the search goes on to the first of these:
    its exponential is a zero however far down it is (None: -inf; 1419.6 = 2048 ln 2 and 4258.7
    = 6144 ln 2, where an exponent that runs over into the sign gives about minus one, 2839.1 = 4096 ln 2, where it gives one)."""
    say("far below", dtype, shift, depth, masked)
    rng = np.random.default_rng(2839)
    rows, vocab, t, p = 128, 107, 0.4012862343238633, 0.99
    x = (rng.standard_normal((rows, vocab)) * 0.2 + shift).astype(np.float32)
    x[:, :4] = x.max(axis=1, keepdims=True)
    far = -np.inf if depth is None else x.max(axis=1, keepdims=True) - t * (depth + np.linspace(-12.0, 2.0, rows, dtype=np.float32)[:, None])
    x[:, 4::3] = far
    xd = torch.from_numpy(x).cuda().to({"f16": torch.float16, "f32": torch.float32}[dtype])
    xw, form = xd.float().cpu().numpy(), None
    if masked:
        words = np.zeros((rows, (vocab + 31) // 32), np.uint32)
        for i in range(vocab - 7):
            words[:, i >> 5] |= np.uint32(1 << (i & 31))
        form = pkg().LogitsXform(mask=torch.from_numpy(words.view(np.int32)).cuda(), mask_allowed_max=vocab - 7)
        xw[:, vocab - 7:] = np.finfo(np.float32).min
    for rep in range(3):
        u = rng.random(rows)
        u[: rows // 2] *= 0.12  # (among the ties at the top)
        got = ctx.sample(xd, torch.from_numpy(u).cuda(), k=0, p=p, temperature=t, xf=form).cpu().numpy()
        assert np.array_equal(got, orc.sample_batch(xw, 0, p, t, u)), rep


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("t", [1e-30, 1e-36, 2e-39, 1e-44])
@pytest.mark.parametrize("ties", [1, 5, 200])
def test_nucleus_rows_whose_factors_are_no_numbers_are_not_picked_from(ctx, orc, t, ties, masked):
    """1 / temperature is infinite below 2^-128, and so is the buckets' factor where the candidates lie next to nothing apart: the
    weights of the largest logits are NaN then and their first one is drawn, or they are alike."""
    say("no numbers", t, ties, masked)
    rng = np.random.default_rng(ties)
    rows, vocab = 24, 5000
    x = rng.standard_normal((rows, vocab)).astype(np.float32)
    x[:, 100:100 + ties] = 9.0
    x[rows // 2:] = np.where(x[rows // 2:] == 9.0, np.float32(0.0), np.float32(-1e-37))  # (a denormal or so between any two)
    xw, form = x, None
    if masked:
        words = np.zeros((rows, (vocab + 31) // 32), np.uint32)
        words[:, :20] = 0xffffffff
        form = pkg().LogitsXform(mask=torch.from_numpy(words.view(np.int32)).cuda(), mask_allowed_max=640)
        xw = x.copy()
        xw[:, 640:] = np.finfo(np.float32).min
    u = rng.random(rows)
    u[0], u[1] = 0.0, np.nextafter(1.0, 0.0)
    for p in (0.9, 1e-6):
        got = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=0, p=p, temperature=t, xf=form).cpu().numpy()
        assert np.array_equal(got, orc.sample_batch(xw, 0, p, t, u)), p


@pytest.mark.parametrize("way", ["fp32", "fp16", "long lists", "masked", "in several modes", "whole vocabulary"])
def test_rows_are_picked_from_and_given_back_where_the_draw_is_open(ctx, orc, way):
    """Draws in the middle of a token's share are picked; draws on the reference's cumulative values, which its own roundings decide, are
    given back, exactly these: a pick that nobody tries, or that nobody finishes, would give the same tokens."""
    say("picked and given back", way)
    rng = np.random.default_rng(len(way))
    vocab, t, p, dtype, form, per_row = 50257, 0.7, 0.9, torch.float32, None, None
    base = (rng.standard_normal(vocab) * (2.5 if way == "long lists" else 1.5)).astype(np.float32)
    base[rng.permutation(640)[:16]] = np.linspace(9.0, 8.0, 16, dtype=np.float32)
    if way == "fp16":
        dtype, base = torch.float16, base.astype(np.float16).astype(np.float32)
    if way == "whole vocabulary":
        p = 1.0
    want = base.copy()
    if way == "masked":
        words = np.zeros((vocab + 31) // 32, np.uint32)
        words[:20] = 0xffffffff
        want[640:] = np.finfo(np.float32).min
    _, probs = orc.sampled_categorical(want, 0, p, t)
    cp = np.cumsum(np.asarray(probs, np.float64)) / np.sum(np.asarray(probs, np.float64))
    on, inside = cp[:8], (cp[:8] + cp[1:9]) / 2
    u = np.concatenate([on, inside])
    if way == "masked":
        form = pkg().LogitsXform(mask=torch.from_numpy(np.tile(words, (len(u), 1)).view(np.int32)).cuda(), mask_allowed_max=640)
    if way == "in several modes":
        per_row = [(0, p, t)] * len(u) + [(200, 0.95, 1.0), (50, 0.9, 0.7)]
        u = np.concatenate([u, [0.3, 0.6]])
    x = torch.from_numpy(np.tile(base, (len(u), 1))).cuda().to(dtype)
    before = ctx.picks_given_back()
    got = ctx.sample(x, torch.from_numpy(u).cuda(), k=0, p=p, temperature=t, xf=form, per_row=per_row).cpu().numpy()
    assert ctx.picks_given_back() - before == len(on)
    n = len(on) + len(inside)
    assert np.array_equal(got[:n], orc.sample_batch(np.tile(want, (n, 1)), 0, p, t, u[:n]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [14, 15, 16, 62, 63, 64, 255, 1023])
def test_nuclei_that_end_with_a_batch_are_picked_from(ctx, orc, n, dtype):
    """n tokens of weight, and the search stops on the first of the others: where that is the last of one of the reference's batches
    (16, 64, 256 or 1024 elements) it is missed and the next one is kept as well, of which a pick knows how little it weighs."""
    say("batch end", n, dtype)
    rng = np.random.default_rng(n)
    rows, vocab, p = 64, 5000, 0.9
    x = (rng.random((rows, vocab)) - 25.0).astype(np.float32)
    for r in range(rows):
        x[r, rng.permutation(vocab)[:n]] = rng.random(n).astype(np.float32)
    xd = torch.from_numpy(x).cuda().to(dtype)
    xw = xd.float().cpu().numpy()
    assert len(orc.sampled_categorical(xw[0], 0, p, 1.0)[0]) == (n + 2 if n in (15, 63, 255, 1023) else n + 1)
    u = rng.random(rows)
    before = ctx.picks_given_back()
    got = ctx.sample(xd, torch.from_numpy(u).cuda(), k=0, p=p, temperature=1.0).cpu().numpy()
    assert ctx.picks_given_back() == before
    assert np.array_equal(got, orc.sample_batch(xw, 0, p, 1.0, u))
    u = 1.0 - 10.0 ** -rng.uniform(9.0, 16.0, rows)  # (on the last elements kept, or nearly)
    got = ctx.sample(xd, torch.from_numpy(u).cuda(), k=0, p=p, temperature=1.0).cpu().numpy()
    assert np.array_equal(got, orc.sample_batch(xw, 0, p, 1.0, u))


@pytest.mark.parametrize("n", [62, 63, 64, 127, 255, 1023, 4095])
def test_picked_rows_of_nearly_a_power_of_two_candidates(ctx, orc, n):
    """n candidates and, as the last element kept, the best one below them: one more than n in the counts."""
    say("power of two", n)
    rng = np.random.default_rng(n)
    rows, vocab = 64, n + 700
    for low in (-30.0, -9.0, -7.0):
        x = (rng.random((rows, vocab)) * 2.0 + low).astype(np.float32)
        for r in range(rows):
            x[r, rng.permutation(vocab)[:n]] = rng.random(n).astype(np.float32)
        xd = torch.from_numpy(x).cuda()
        for p in (0.9, 0.95, 0.99):
            u = rng.random(rows)
            u[0], u[1] = np.nextafter(1.0, 0.0), 1.0 - 1e-4
            got = ctx.sample(xd, torch.from_numpy(u).cuda(), k=0, p=p, temperature=1.0).cpu().numpy()
            assert np.array_equal(got, orc.sample_batch(x, 0, p, 1.0, u)), (low, p)


def test_results_written_straight_to_pinned_host_memory(ctx, orc):
    """The output pointers may name pinned host memory that the device can address (the reference mirrors its
    results through pinned memory, src/cuda/interface.cpp:51-60): the kernels store the tokens there themselves, no
    copy follows, and a host that has filled the buffer with -1 sees a step's tokens arrive without synchronising the
    stream.  Sampling, argmax and the EOS / append tail."""
    import time
    say("pinned outputs")
    rng = np.random.default_rng(404)
    rows, vocab = 64, 128256
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    u = rng.random(rows)
    xd, ud = torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda()
    torch.cuda.synchronize()
    out = torch.full((rows,), -1, dtype=torch.int32).pin_memory()
    view = out.numpy()

    def wait_for_tokens():
        t0 = time.perf_counter()
        while (view < 0).any():
            assert time.perf_counter() - t0 < 10.0, "tokens never arrived in pinned memory"

    ctx.sample(xd, ud, k=50, p=0.9, temperature=0.7, out=out)
    wait_for_tokens()  # no synchronisation: the kernel's own stores are what the host sees
    assert np.array_equal(view, orc.sample_batch(x, 50, 0.9, 0.7, u))
    torch.cuda.synchronize()
    view[:] = -1
    ctx.argmax(xd, out=out)
    wait_for_tokens()
    assert np.array_equal(view, orc.argmax_batch(x))
    torch.cuda.synchronize()
    # the tail of a greedy step with its tokens and its all-finished flag in pinned memory
    eos, pad, max_len, cur = [7, 9], 0, 8, 3
    tokens = torch.tensor([5, 7, 9, 11], dtype=torch.int32).pin_memory()
    done = torch.zeros(1, dtype=torch.int32).pin_memory()
    seen = torch.tensor([0, 0, 1, 1], dtype=torch.int32).cuda()
    seqs = torch.zeros((4, max_len), dtype=torch.int32).cuda()
    pkg().SearchContext.greedy_tail(ctx, tokens, seen, eos, pad, seqs, cur, done, allow_host=True)
    torch.cuda.synchronize()
    assert tokens.tolist() == [5, 7, pad, pad] and seen.cpu().tolist() == [0, 1, 1, 1] and done.item() == 0
    assert seqs[:, cur].cpu().tolist() == [5, 7, pad, pad]


def test_prepared_sample_calls_give_the_same_tokens(ctx, orc):
    """SearchContext.prepared_sample marshals a call once; issuing it -- repeatedly, on its stream, into pinned host
    memory or device memory, fp32 or fp16 rows -- gives the tokens of the same call made through `sample`."""
    say("prepared calls")
    rng = np.random.default_rng(405)
    rows, vocab = 64, 40000
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    u = rng.random(rows)
    xd, ud = torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda()
    want = orc.sample_batch(x, 50, 0.9, 0.7, u)
    out_dev = torch.full((rows,), -1, dtype=torch.int32, device="cuda")
    out_pin = torch.full((rows,), -1, dtype=torch.int32).pin_memory()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    calls = [ctx.prepared_sample(xd, ud, out_dev, k=50, p=0.9, temperature=0.7),
             ctx.prepared_sample(xd, ud, out_pin, k=50, p=0.9, temperature=0.7, stream=side)]
    for _ in range(3):
        out_dev.fill_(-1)
        out_pin.fill_(-1)
        torch.cuda.synchronize()
        for call in calls:  # (one after the other: calls on one context must not overlap, whatever their streams)
            call()
            torch.cuda.synchronize()
        assert np.array_equal(out_dev.cpu().numpy(), want)
        assert np.array_equal(out_pin.numpy(), want)
    xh = torch.from_numpy(x.astype(np.float16)).cuda()
    call16 = ctx.prepared_sample(xh, ud, out_dev, k=0, p=0.9, temperature=1.0)
    call16()
    torch.cuda.synchronize()
    assert np.array_equal(out_dev.cpu().numpy(), orc.sample_batch(xh.float().cpu().numpy(), 0, 0.9, 1.0, u))


def test_config2_topk_topp_batch64(ctx, orc):
    """Benchmark configuration 2 at full size: batch 64, vocab 128256, N(0,3^2) logits + 8 peaks/row at +10,
    T=0.7, k=50, p=0.9, shared uniforms; 4 of the 128 steps."""
    rng = np.random.default_rng(2)
    rows, vocab = 64, 128256
    for step in range(4):
        say("config2 step", step)
        x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
        for r in range(rows):
            x[r, rng.choice(vocab, 8, replace=False)] += 10
        u = rng.random(rows)
        tok = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=50, p=0.9, temperature=0.7)
        assert np.array_equal(tok.cpu().numpy(), orc.sample_batch(x, 50, 0.9, 0.7, u))


def test_sample_ties_and_degenerate_rows(ctx, orc):
    """Heavy ties (rounded logits, constant rows) push rows onto the exact general path; results must
    still equal the oracle's lowest-index tie rule."""
    say("sample ties")
    rng = np.random.default_rng(3)
    rows, vocab = 4, 20000
    x = np.round(rng.standard_normal((rows, vocab)) * 2).astype(np.float32)
    x[1, :] = 1.5
    x[2, :] = LOWEST
    x[2, 77] = 0.0
    u = rng.random(rows)
    sample_and_check(ctx, orc, x, u, 50, 0.9, 0.7)
    sample_and_check(ctx, orc, x, u, 10, 0.0, 1.0)


def test_sparse_mask_rows_with_heavy_ties(ctx, orc):
    """Nucleus rows under a sparse mask whose allowed logits are quantised (hundreds of ids per score, more than a
    bucket of the counting sort holds), constant, or carry a block of equal values at the top: the row leaves the
    bucket sort for the sorting network inside the same kernel; kept ids, probability bits and tokens equal the
    oracle's, with and without the promise about the mask."""
    say("sparse mask, heavy ties")
    rng = np.random.default_rng(77)
    rows, vocab = 5, 201088
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    x[0] = np.round(x[0] * 2) / 2
    x[1] = np.round(x[1])
    x[2, :] = np.float32(-1.25)
    x[3, : vocab // 3] = np.float32(9.5)
    mask = make_mask(rng, rows, vocab, 0.05)
    allowed = np.unpackbits(mask.view(np.uint8), axis=1, bitorder="little")[:, :vocab].astype(bool)
    hist = rng.integers(0, vocab, (rows, 300)).astype(np.int32)
    u = rng.random(rows)
    xf = pkg().LogitsXform(mask=torch.from_numpy(mask.view(np.int32)).cuda(), history=torch.from_numpy(hist).cuda(),
                           repetition_penalty=1.3)
    proc = orc.apply_mask(x, mask)
    cap = 16384
    for promise in (0, int(allowed.sum(axis=1).max())):
        xf.c.mask_allowed_max = promise
        tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=0, p=0.9, temperature=1.0,
                                     xf=xf, kept_capacity=cap)
        tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
        for r in range(rows):
            idx, probs = orc.sampled_categorical(orc.apply_repetition_penalty(proc[r], hist[r], 1.3), 0, 0.9, 1.0)
            n = min(len(idx), cap)
            assert kc[r] == len(idx), (promise, r, kc[r], len(idx))
            assert np.array_equal(ki[r, :n], idx[:n]), (promise, r)
            assert np.array_equal(bits(kp[r, :n]), bits(probs[:n])), (promise, r)
            assert tok[r] == idx[orc.discrete_draw(probs, u[r])], (promise, r)


def test_grammar_rows_with_15_63_or_255_allowed_ids_stay_off_the_exact_path(ctx, orc):
    """A grammar that lets 15, 63 or 255 ids through, all of them inside the nucleus: the search only stops on the
    first masked id, which is the 16th, 64th, 256th element, and the reference notices such a stop one element later
    (src/sampling_distribution.h:166-181): the kept set ends with two masked ids.  The sparse-mask kernel knows the
    second one (and the elements behind the first in general); kept sets and tokens equal the oracle's, with and
    without a repetition penalty over ids that include masked ones, and no row takes the exact path."""
    say("grammar rows whose list ends on a batch end")
    rng = np.random.default_rng(1563)
    vocab = 201088
    words = (vocab - 1) // 32 + 1
    sizes = [15, 63, 255, 15, 63, 14, 16]
    rows = len(sizes)
    x = (rng.standard_normal((rows, vocab)) * 2).astype(np.float32)
    bits_ = np.zeros((rows, words * 32), bool)
    for r, n in enumerate(sizes):
        ids = rng.choice(vocab, n, replace=False)
        if r == 3:
            ids[0] = 1  # id 0 is masked: the first masked id is 0, the second 2
            ids[1] = 3
        bits_[r, ids] = True
        x[r, ids] = (5.0 + 0.1 * rng.standard_normal(n)).astype(np.float32)  # near-equal: the nucleus needs all of them
    mask = np.ascontiguousarray(np.packbits(bits_.reshape(rows, words, 32), axis=-1, bitorder="little").view(np.uint32).reshape(rows, words))
    proc = orc.apply_mask(x, mask)
    u = rng.random(rows)
    u[1] = 0.99999999
    hist = rng.integers(0, 40, (rows, 24)).astype(np.int32)  # low ids: masked ones among them, 0 and 2 included
    for penalty in (None, 1.3):
        for promise in (0, 256):
            xf = pkg().LogitsXform(mask=torch.from_numpy(mask.view(np.int32)).cuda(),
                                   history=torch.from_numpy(hist).cuda() if penalty else None,
                                   repetition_penalty=penalty or 1.0, mask_allowed_max=promise)
            before = ctx.fallback_rows()
            tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=0, p=0.9, temperature=1.0,
                                         xf=xf, kept_capacity=512)
            took_exact = ctx.fallback_rows() - before
            tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
            for r in range(rows):
                want = orc.apply_repetition_penalty(proc[r], hist[r], penalty) if penalty else proc[r]
                idx, probs = orc.sampled_categorical(want, 0, 0.9, 1.0)
                assert kc[r] == len(idx), (penalty, promise, r, kc[r], len(idx))
                assert np.array_equal(ki[r, :len(idx)], idx), (penalty, promise, r)
                assert np.array_equal(bits(kp[r, :len(idx)]), bits(probs)), (penalty, promise, r)
                assert tok[r] == idx[orc.discrete_draw(probs, u[r])], (penalty, promise, r)
            if penalty is None:
                assert [int(k) for k in kc] == [17, 65, 257, 17, 65, 15, 17], kc
            assert took_exact == 0, (penalty, promise, took_exact)


@pytest.mark.parametrize("sigma,p,t", [(4.0, 0.95, 1.0), (1.0, 0.9, 1.0), (5.0, 0.9, 1.0), (3.0, 0.5, 0.7)])
def test_nucleus_rows_with_lists_near_and_beyond_the_sort(ctx, orc, sigma, p, t):
    """Unmasked nucleus rows of 128256 ids whose chunks list a few thousand to tens of thousands of keys: nuclei that
    fit the finish kernel's sort with room to spare, that fill it almost completely, and that exceed it (sorted in
    rounds).  Kept counts, the first kept ids with their probability bits, and tokens equal the
    oracle's."""
    say("nucleus near the sort's capacity", sigma, p, t)
    rng = np.random.default_rng(int(sigma * 10 + p * 100))
    rows, vocab = 6, 128256
    x = (rng.standard_normal((rows, vocab)) * sigma).astype(np.float32)
    x[1] += np.float32(0.7)
    x[2, : vocab // 2] -= np.float32(2.0)  # one half of the row lower: chunk thresholds differ
    u = rng.random(rows)
    cap = 4096
    tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=0, p=p, temperature=t,
                                 kept_capacity=cap)
    tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
    for r in range(rows):
        idx, probs = orc.sampled_categorical(x[r], 0, p, t)
        n = min(len(idx), cap)
        assert kc[r] == len(idx), (r, kc[r], len(idx))
        assert np.array_equal(ki[r, :n], idx[:n]), r
        assert np.array_equal(bits(kp[r, :n]), bits(probs[:n])), r
        assert tok[r] == idx[orc.discrete_draw(probs, u[r])], r


def test_nucleus_whose_stop_falls_on_a_batch_end_stays_off_the_exact_path(ctx, orc):
    """Peaked rows whose nucleus search stops on the 16th, 64th or 256th element: the reference notices such a stop
    only one element later (src/sampling_distribution.h:166-181), so the kept set has 17, 65, 257 tokens, and a
    candidate list trimmed right behind the stop would be one element short.  The finish kernel then takes the next
    run of buckets along; the rows are finished on the fast path with the oracle's kept sets and tokens."""
    say("nucleus stop on a batch end, peaked rows")
    rng = np.random.default_rng(1664)
    vocab, p, t = 128256, 0.9, 1.0
    # (tokens at the top, depth of the element the search stops on, elements behind it and their depth); in the last
    # three rows the stop's element already lies below the candidates' threshold: the list ends with it, and the
    # element behind it is in no list at all
    shapes = [(15, 11.5, 50, 11.6), (63, 10.0, 30, 10.2), (255, 8.8, 30, 9.3), (15, 11.5, 0, 0.0),
              (15, 12.5, 3, 13.0), (63, 11.0, 3, 11.5), (15, 12.5, 0, 0.0)]
    x = (rng.standard_normal((len(shapes), vocab)) - 15.0).astype(np.float32)
    for r, (n_top, stop_depth, n_after, after_depth) in enumerate(shapes):
        ids = rng.choice(32768, n_top + 1 + n_after, replace=False)  # all in the first chunk
        x[r, ids[:n_top]] = 20.0
        x[r, ids[n_top]] = np.float32(20.0 - stop_depth)
        x[r, ids[n_top + 1:]] = (20.0 - after_depth - 0.01 * rng.random(n_after)).astype(np.float32)
    u = rng.random(len(shapes))
    u[0] = 0.9999999  # the draw reaches the element behind the stop
    before = ctx.fallback_rows()
    tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=0, p=p, temperature=t,
                                 kept_capacity=512)
    took_exact = ctx.fallback_rows() - before
    tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
    for r, (n_top, _, _, _) in enumerate(shapes):
        idx, probs = orc.sampled_categorical(x[r], 0, p, t)
        assert len(idx) == n_top + 2, (r, len(idx))  # the stop's element and the one behind it
        assert kc[r] == len(idx), (r, kc[r], len(idx))
        assert np.array_equal(ki[r, :len(idx)], idx), r
        assert np.array_equal(bits(kp[r, :len(idx)]), bits(probs)), r
        assert tok[r] == idx[orc.discrete_draw(probs, u[r])], r
    assert took_exact == 0, took_exact
    # the same rows as fp16
    x16 = x.astype(np.float16)
    before = ctx.fallback_rows()
    tok16 = ctx.sample(torch.from_numpy(x16).cuda(), torch.from_numpy(u).cuda(), k=0, p=p, temperature=t).cpu().numpy()
    assert np.array_equal(tok16, orc.sample_batch(x16.astype(np.float32), 0, p, t, u))
    assert ctx.fallback_rows() == before


@pytest.mark.parametrize("sigma,p,t,wide_rows", [(3.0, 0.95, 1.0, 6), (2.0, 0.9, 1.0, 5), (4.0, 0.99, 1.5, 5), (1.0, 0.9, 1.0, 5)])
def test_nucleus_rows_wider_than_the_sort(ctx, orc, sigma, p, t, wide_rows):
    """Unmasked nucleus rows of 128256 ids whose nuclei hold 30000 to 90000 tokens, several times what the finish
    kernel sorts at once: it sorts them in rounds into global memory.  One row is quantised to steps of 1/64 (dozens of
    equal scores per step: buckets beyond the usual ranking), one to steps of 1/4 (thousands: those rows are the exact
    path's).  Every kept id and probability bit, to the nucleus' last element, and the tokens equal the oracle's;
    the rows without heavy ties stay off the exact path."""
    say("nucleus wider than the sort", sigma, p, t)
    rng = np.random.default_rng(int(sigma * 10 + p * 1000))
    rows, vocab = 7, 128256
    x = (rng.standard_normal((rows, vocab)) * sigma).astype(np.float32)
    x[1] += np.float32(0.7)
    x[2, : vocab // 2] -= np.float32(1.0)  # one half of the row lower: chunk thresholds differ
    x[3, 1000:1040] = np.nan
    x[4, 5] = 40.0  # one token far above the rest
    x[5] = (np.round(x[5] * 64) / 64).astype(np.float32)
    x[6] = (np.round(x[6] * 4) / 4).astype(np.float32)
    u = rng.random(rows)
    u[0] = 0.999999  # a draw from the nucleus' far end
    before = ctx.fallback_rows()
    tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=0, p=p, temperature=t,
                                 kept_capacity=vocab)
    took_exact = ctx.fallback_rows() - before
    tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
    for r in range(rows):
        idx, probs = orc.sampled_categorical(x[r], 0, p, t)
        n = len(idx)
        assert kc[r] == n, (r, kc[r], n)
        assert np.array_equal(ki[r, :n], idx), r
        assert np.array_equal(bits(kp[r, :n]), bits(probs)), r
        assert tok[r] == idx[orc.discrete_draw(probs, u[r])], r
    assert took_exact <= rows - wide_rows, took_exact


@pytest.mark.parametrize("k", [100, 512, 2048, 6000])
def test_large_k_rows_with_ties_nans_and_clustered_best_tokens(ctx, orc, k):
    """Top-k rows with 64 < k <= 8192 at 128256 ids: fewer numbers than k (NaNs fill the rest), a score shared by
    thousands of ids at the k-th place, the best tokens all in one chunk or in one thread's run of ids, one chunk
    without a number.  Kept sets, probability bits and tokens equal the oracle's."""
    say("large k, ties and NaNs", k)
    rng = np.random.default_rng(k)
    rows, vocab = 6, 128256
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    x[0, :] = np.nan
    x[0, rng.integers(0, vocab, k // 2)] = rng.standard_normal(k // 2).astype(np.float32)
    x[1] = np.round(x[1])
    x[2, 40000:40000 + 3 * k] = 30.0 + rng.standard_normal(3 * k).astype(np.float32)
    x[3, 70000:70032] = 50.0
    x[4, 32768:65536] = np.nan
    u = rng.random(rows)
    tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=k, p=0.9, temperature=0.8,
                                 kept_capacity=2048)
    tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
    for r in range(rows):
        idx, probs = orc.sampled_categorical(x[r], k, 0.9, 0.8)
        n = min(len(idx), 2048)
        assert kc[r] == len(idx), (r, kc[r], len(idx))
        assert np.array_equal(ki[r, :n], idx[:n]), r
        assert np.array_equal(bits(kp[r, :n]), bits(probs[:n])), r
        assert tok[r] == idx[orc.discrete_draw(probs, u[r])], r


@pytest.mark.parametrize("vocab,k", [(128256, 50), (70000, 64), (40000, 2), (128256, 1)])
def test_rows_that_tie_at_their_kth_score_are_selected_not_sorted(ctx, orc, vocab, k):
    """Rows whose k best cannot be told from a chunk's bound -- all ids masked to lowest() but a few, NaNs needed to
    fill the k, one score shared by thousands of ids, a few large values in one thread's run of ids -- leave the
    single-pass path inside the streaming kernel; there the k best are selected exactly (the keys above the k-th
    score, then the first ties in id order) and the tokens, kept ids and probabilities equal the oracle's."""
    say("sample selection", vocab, k)
    rng = np.random.default_rng(vocab + k)
    rows = 6
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    x[0, :] = LOWEST
    x[0, rng.integers(0, vocab, 5)] = [0.0, 1.0, -1.0, 0.5, 0.25]
    x[1, :] = np.nan
    x[1, rng.integers(0, vocab, 20)] = rng.standard_normal(20).astype(np.float32)
    x[2, :] = 1.5
    x[3, : vocab // 2] = 7.0   # above everything else: half the row ties for every place
    x[4, 1000:1200] = 40.0 + rng.standard_normal(200).astype(np.float32)  # the best 200 in consecutive ids
    u = rng.random(rows)
    before = ctx.fallback_rows()
    if k == 1:
        got = ctx.argmax(torch.from_numpy(x).cuda()).cpu().numpy()
        assert np.array_equal(got, orc.argmax_batch(x))
    else:
        sample_and_check(ctx, orc, x, u, k, 0.9, 0.7)
        sample_and_check(ctx, orc, x, u, k, 0.0, 1.0)
        assert ctx.fallback_rows() > before  # (rows 0 and 1 at least cannot stay on the single-pass path)


@pytest.mark.parametrize("vocab", [2, 70, 5000, 40000])
def test_sample_rows_without_finite_logits(ctx, orc, vocab):
    """A row of -inf logits (everything masked, then a penalty above 1 applied to lowest()) has NaN
    weights; the reference's draw then lands on position 0 of its kept list whatever the uniform is."""
    say("sample all -inf", vocab)
    x = np.full((2, vocab), -np.inf, np.float32)
    x[1, vocab // 2] = 0.0
    u = np.array([0.73, 0.41])
    for k, p in ((0, 0.9), (1, 0.0), (5, 0.5), (50, 0.0), (200, 0.9)):
        tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=k, p=p, temperature=0.8,
                                     kept_capacity=64)
        for r in range(2):
            idx, probs = orc.sampled_categorical(x[r], k, p, 0.8)
            assert kc[r].item() == len(idx), (k, p, r)
            assert tok[r].item() == idx[orc.discrete_draw(probs, u[r])], (k, p, r)
        assert tok[0].item() == 0 and tok[1].item() == vocab // 2


def test_sample_large_k_general_path(ctx, orc):
    say("sample k=200")
    rng = np.random.default_rng(4)
    x = (rng.standard_normal((2, 5000)) * 3).astype(np.float32)
    u = rng.random(2)
    sample_and_check(ctx, orc, x, u, 200, 0.95, 0.9, cap=256)
    sample_and_check(ctx, orc, x, u, 6000, 0.0, 1.0, cap=64)  # k > vocab clamps


@pytest.mark.parametrize("vocab,k,p,t,quantum", [
    (128256, 65, 0.9, 0.7, 0.0), (128256, 100, 1.0, 1.0, 0.0), (128256, 512, 0.95, 1.3, 0.0), (201088, 300, 0.0, 0.8, 0.0),
    (128256, 513, 0.95, 1.3, 0.0),  # from here four offers per thread bound the chunk
    (128256, 2048, 0.9, 1.0, 0.0), (201088, 2048, 0.0, 1.0, 0.0), (128256, 1500, 0.99, 0.8, 0.25), (5000, 2048, 0.9, 1.0, 0.0),
    (128256, 2049, 0.95, 1.3, 0.0), (128256, 8192, 0.9, 1.0, 0.0), (201088, 5000, 0.0, 0.9, 0.0), (70000, 6000, 0.95, 1.1, 0.5),
    (128256, 8193, 0.95, 1.3, 0.0),  # beyond the limit of this route: the full-sort path
    (33000, 100, 0.9, 1.0, 0.0),    # the short last chunk holds fewer than k threads' worth of elements
    (40000, 500, 0.99, 1.0, 0.25),  # ties across the cut
    (700, 500, 0.9, 1.0, 0.0),      # k close to the vocabulary
])
def test_sample_large_k_through_the_candidate_lists(ctx, orc, vocab, k, p, t, quantum):
    """Top-k rows with 64 < k <= 8192 are streamed like nucleus rows (candidates = elements at or above
    the k-th best of the per-thread offers of their chunk: the maxima up to k = 512, beyond that the maxima of
    the quarters or eighths of every thread's elements) and finished by the sorting kernel, not by the full-sort
    path; kept sets, probabilities and tokens equal the oracle's."""
    say("sample large k", vocab, k, p, t, quantum)
    rng = np.random.default_rng(vocab + k)
    rows = 5
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    if quantum:
        x = (np.round(x / quantum) * quantum).astype(np.float32)
    x[1, :] = np.float32(0.5)            # a constant row: heavy ties, the exact path is allowed here
    x[2, rng.integers(0, vocab, 50)] = -np.inf
    u = rng.random(rows)
    before = ctx.fallback_rows()
    tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=k, p=p, temperature=t,
                                 kept_capacity=2048)
    tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
    for r in range(rows):
        idx, probs = orc.sampled_categorical(x[r], k, p, t)
        n = min(len(idx), 2048)
        assert kc[r] == len(idx), r
        assert np.array_equal(ki[r, :n], idx[:n]), r
        assert np.array_equal(bits(kp[r, :n]), bits(probs[:n])), r
        assert tok[r] == idx[orc.discrete_draw(probs, u[r])], r
    if k <= 8192 and not quantum:
        assert ctx.fallback_rows() - before <= 1  # at most the constant row


@pytest.mark.parametrize("rows,vocab,p,t", [(3, 5000, 0.9, 1.0), (2, 128256, 0.95, 0.7), (2, 40, 0.6, 1.0),
                                            (2, 64, 0.9, 1.0), (2, 65, 0.9, 1.0), (3, 3000, 0.0, 1.0),
                                            (2, 3000, 0.3, 2.0)])
def test_sample_nucleus(ctx, orc, rows, vocab, p, t):
    say("sample nucleus", rows, vocab, p, t)
    rng = np.random.default_rng(vocab + int(p * 100))
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    u = rng.random(rows)
    sample_and_check(ctx, orc, x, u, 0, p, t, cap=128)


@pytest.mark.parametrize("vocab,sigma,p,fast", [(128256, 4.0, 0.95, True), (201088, 5.0, 0.9, True), (128256, 2.0, 0.95, False),
                                                (40000, 4.0, 0.999, False)])
def test_nucleus_with_more_candidates_than_the_sort_holds(ctx, orc, vocab, sigma, p, fast):
    """Unmasked rows: nearly the whole vocabulary lies within the candidate depth of the maximum.  The finish
    kernel then keeps the best ~16000 by raising its threshold; when they contain the nucleus (peaked rows)
    the row stays on the fast path, otherwise the exact path takes it.  Results equal the oracle's either way."""
    say("nucleus trim", vocab, sigma, p)
    rng = np.random.default_rng(int(vocab + sigma * 10))
    rows = 4
    x = (rng.standard_normal((rows, vocab)) * sigma).astype(np.float32)
    x[3] = (np.round(x[3] * 2) / 2).astype(np.float32)  # ties at the raised threshold
    u = rng.random(rows)
    before = ctx.fallback_rows()
    tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=0, p=p, temperature=1.0,
                                 kept_capacity=4096)
    tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
    for r in range(rows):
        idx, probs = orc.sampled_categorical(x[r], 0, p, 1.0)
        assert kc[r] == len(idx), (r, kc[r], len(idx))
        n = min(len(idx), 4096)
        assert np.array_equal(ki[r, :n], idx[:n]), r
        assert np.array_equal(bits(kp[r, :n]), bits(probs[:n])), r
        assert tok[r] == idx[orc.discrete_draw(probs, u[r])], r
    took_exact = ctx.fallback_rows() - before
    assert took_exact == 0 if fast else took_exact > 0, took_exact


@pytest.mark.parametrize("vocab", [32, 128, 130, 512, 2048, 8192, 32768, 131072])
def test_nucleus_stop_on_last_element_of_a_sort_batch(ctx, orc, vocab):
    """Constant rows with p = 0.5 meet the tail-bound stop at element vocab/2; where that is the end of one of
    the reference's sort batches (16, 64, 256, ...) the stop is only noticed one element later
    (src/sampling_distribution.h:166-181), so vocab/2 + 1 tokens are kept."""
    say("nucleus batch end", vocab)
    rng = np.random.default_rng(vocab)
    x = np.full((3, vocab), -0.5, np.float32)
    x[1, :] = 0.0
    x[2, vocab // 2:] = -0.5000001  # a second, slightly lower level
    u = rng.random(3)
    sample_and_check(ctx, orc, x, u, 0, 0.5, 1.0, cap=256)
    idx, _ = orc.sampled_categorical(x[0], 0, 0.5, 1.0)
    quirk = vocab > 64 and vocab // 2 in (16, 64, 256, 1024, 4096, 16384, 65536)
    assert len(idx) == vocab // 2 + (1 if quirk else 0)


@pytest.mark.parametrize("frac,quantum", [(0.004, 0.0), (0.012, 0.0), (0.03, 0.0), (0.012, 0.5), (0.03, 0.5),
                                           (0.06, 0.25)])
def test_nucleus_candidate_counts_and_ties(ctx, orc, frac, quantum):
    """Masked nucleus rows whose candidate lists fall in every size class of the finish kernel's sort
    (about 800 to 12000 keys); a quantum > 0 rounds the logits to a coarse grid so that hundreds of
    candidates tie and the sort must fall back from score buckets to the sorting network."""
    say("nucleus sizes", frac, quantum)
    rng = np.random.default_rng(int(frac * 1000) + int(quantum * 8))
    rows, vocab = 3, 201088
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    if quantum:
        x = (np.round(x / quantum) * quantum).astype(np.float32)
    mask = make_mask(rng, rows, vocab, frac)
    u = rng.random(rows)
    xf = pkg().LogitsXform(mask=torch.from_numpy(mask.view(np.int32)).cuda())
    tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=0, p=0.95,
                                 temperature=1.0, xf=xf, kept_capacity=16384)
    tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
    proc = orc.apply_mask(x, mask)
    for r in range(rows):
        idx, probs = orc.sampled_categorical(proc[r], 0, 0.95, 1.0)
        assert kc[r] == len(idx)
        assert np.array_equal(ki[r, :len(idx)], idx)
        assert np.array_equal(bits(kp[r, :len(idx)]), bits(probs))
        assert tok[r] == idx[orc.discrete_draw(probs, u[r])]


def test_config5_constrained_nucleus(ctx, orc):
    """Benchmark configuration 5 shape (8 of 256 rows per step, 2 steps): vocab 201088, 5 % grammar mask,
    T=1.0, top-p 0.95, repetition penalty 1.2 over 1024 ids."""
    rng = np.random.default_rng(5)
    rows, vocab = 8, 201088
    for step in range(2):
        say("config5 step", step)
        x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
        mask = make_mask(rng, rows, vocab, 0.05)
        hist = rng.integers(0, vocab, (rows, 1024)).astype(np.int32)
        u = rng.random(rows)
        xf = pkg().LogitsXform(mask=torch.from_numpy(mask.view(np.int32)).cuda(),
                               history=torch.from_numpy(hist).cuda(), repetition_penalty=1.2)
        tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=0, p=0.95,
                                     temperature=1.0, xf=xf, kept_capacity=16384)
        tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
        proc = orc.apply_mask(x, mask)
        for r in range(rows):
            row = orc.apply_repetition_penalty(proc[r], hist[r], 1.2)
            idx, probs = orc.sampled_categorical(row, 0, 0.95, 1.0)
            assert kc[r] == len(idx) and len(idx) > 1000
            assert np.array_equal(ki[r, :len(idx)], idx)
            assert np.array_equal(bits(kp[r, :len(idx)]), bits(probs))
            assert tok[r] == idx[orc.discrete_draw(probs, u[r])]


@pytest.mark.parametrize("vocab,hist_len,span,k,p", [
    (40000, 2200, 40000, 50, 0.9),    # a history longer than two ids per thread, spread over two chunks
    (40000, 2200, 40000, 0, 0.9),
    (70001, 8000, 2500, 40, 1.0),     # more distinct history ids in one chunk than its list holds: exact path
    (70001, 8000, 2500, 0, 0.95),
    (33000, 300, 232, 8, 0.0),        # the short last chunk holds history ids
    (33000, 300, 232, 0, 0.8),
])
def test_sample_long_and_dense_histories(ctx, orc, vocab, hist_len, span, k, p):
    """History ids are processed apart from the other logits (a list per 32768-id chunk): long histories,
    duplicates, ids outside the vocabulary, lists that overflow, ids in a short last chunk."""
    say("sample histories", vocab, hist_len, span, k, p)
    rng = np.random.default_rng(hist_len + span + k)
    rows = 3
    scale = 2.0 if k else 6.0           # nucleus rows stay peaked, so that their candidates fit the fast path
    x = (rng.standard_normal((rows, vocab)) * scale).astype(np.float32)
    hist = (vocab - span + rng.integers(0, span, (rows, hist_len))).astype(np.int32)
    hist[:, :40] = hist[:, 40:80]       # duplicates
    hist[0, 5] = vocab + 3              # beyond the vocabulary: ignored
    hist[1, 7] = -2                     # negative: ignored
    x[:, hist[2, 100:110]] = 4.6 * scale  # penalised ids among the best of their rows
    mask = make_mask(rng, rows, vocab, 0.7)
    u = rng.random(rows)
    before = ctx.fallback_rows()
    for pen in (1.3, 0.75):
        xf = pkg().LogitsXform(mask=torch.from_numpy(mask.view(np.int32)).cuda(), history=torch.from_numpy(hist).cuda(),
                               repetition_penalty=pen)
        tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=k, p=p, temperature=0.9,
                                     xf=xf, kept_capacity=4096)
        tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
        proc = orc.apply_mask(x, mask)
        for r in range(rows):
            valid = hist[r][(hist[r] >= 0) & (hist[r] < vocab)]
            row = orc.apply_repetition_penalty(proc[r], valid, pen)
            idx, probs = orc.sampled_categorical(row, k, p, 0.9)
            assert kc[r] == len(idx), (r, pen)
            n = min(len(idx), 4096)
            assert np.array_equal(ki[r, :n], idx[:n]), (r, pen)
            assert np.array_equal(bits(kp[r, :n]), bits(probs[:n])), (r, pen)
            assert tok[r] == idx[orc.discrete_draw(probs, u[r])], (r, pen)
    took_exact = ctx.fallback_rows() - before
    assert (took_exact > 0) == (span == 2500), took_exact  # only the overflowing lists go to the exact path


@pytest.mark.parametrize("vocab", [40001, 40002, 40003, 65539, 98305, 98308])
def test_logits_processing_on_rows_of_any_alignment_and_end(ctx, orc, vocab):
    """The kernels with logits processing request a chunk's fp32 logits as sixteen 128-bit loads per thread whatever
    the row's alignment and end (a quad that straddles the end is read as the row's last four elements and put right
    afterwards): rows that start on every 4-byte offset of a 16-byte line, vocabularies that end one, two and three
    elements into a quad, a last chunk of a single element, history ids and masked ids on the row's last elements.
    Argmax, top-k, k = 300 and nucleus rows against the oracle."""
    say("rows of any alignment", vocab)
    rng = np.random.default_rng(vocab)
    rows = 6
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    x[0, vocab - 1] = 30.0   # the row's best on its last element ...
    x[1, vocab - 2] = 30.0   # ... on the one before, penalised below
    x[2, vocab - 3] = 30.0   # ... masked below
    hist = rng.integers(0, vocab, (rows, 200)).astype(np.int32)
    hist[:, 0] = vocab - 2
    hist[:, 1] = vocab - 1
    mask = make_mask(rng, rows, vocab, 0.8)
    words = mask.reshape(rows, -1)
    words[2, (vocab - 3) >> 5] &= ~np.uint32(1 << ((vocab - 3) & 31))
    u = rng.random(rows)
    xf = pkg().LogitsXform(mask=torch.from_numpy(mask.view(np.int32)).cuda(), history=torch.from_numpy(hist).cuda(),
                           repetition_penalty=1.6)
    xd = torch.from_numpy(x).cuda()
    proc = orc.apply_mask(x, mask)
    want = [orc.apply_repetition_penalty(proc[r], hist[r], 1.6) for r in range(rows)]
    got = ctx.argmax(xd, xf=xf).cpu().numpy()
    for r in range(rows):
        assert got[r] == orc.argmax(want[r]), r
    for k, p, t in ((50, 0.9, 0.7), (300, 0.95, 1.0), (0, 0.9, 1.0)):
        tok, kc, ki, kp = ctx.sample(xd, torch.from_numpy(u).cuda(), k=k, p=p, temperature=t, xf=xf, kept_capacity=2048)
        tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
        for r in range(rows):
            idx, probs = orc.sampled_categorical(want[r], k, p, t)
            n = min(len(idx), 2048)
            assert kc[r] == len(idx), (k, r)
            assert np.array_equal(ki[r, :n], idx[:n]), (k, r)
            assert np.array_equal(bits(kp[r, :n]), bits(probs[:n])), (k, r)
            assert tok[r] == idx[orc.discrete_draw(probs, u[r])], (k, r)


@pytest.mark.parametrize("rows,vocab", [(1, 8191), (300, 8193), (3, 16383), (5, 16385), (2, 32770), (40, 33000), (9, 49161), (130, 50257),
                                        (16, 131072), (4, 131073), (90, 98400), (50, 99839), (50, 99840), (50, 101375), (50, 101376), (1, 262144), (2, 262145),
                                        (1, 524288)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_chunks_of_every_size(orc, rows, vocab, dtype):
    """Rows of top-k and argmax calls are cut into chunks of 8192, 16384 or 32768 logits, or evenly where the last one would be short, by
    the number of workgroups: vocabularies on both sides of every chunk size and of the most lists a row's finishing workgroup merges,
    batches on both sides of a workgroup per CU; a row's best on a chunk's first and last ids, masked ids and history ids among them."""
    say("chunks", rows, vocab, dtype)
    rng = np.random.default_rng(vocab * 7 + rows)
    checked = sorted({0, 1 % rows, rows // 2, rows - 1})
    c = pkg().SearchContext(rows, vocab)
    try:
        x = (torch.randn(rows, vocab, generator=torch.Generator().manual_seed(vocab)) * 3).to(dtype)
        for r in checked:
            for e in rng.choice([8191, 8192, 16383, 16384, 32767, 32768, vocab - 1, vocab - 2, (vocab - 1) // 64 * 64], 4):
                x[r, min(int(e), vocab - 1)] = 14.0 + float(rng.integers(0, 3))
        xd, u = x.cuda(), rng.random(rows)
        ud = torch.from_numpy(u).cuda()
        hist = rng.integers(0, vocab, (rows, 70)).astype(np.int32)
        hist[:, 0], hist[:, 1] = vocab - 1, min(8192, vocab - 2)
        mask = make_mask(rng, rows, vocab, 0.7)
        xf = pkg().LogitsXform(mask=torch.from_numpy(mask.view(np.int32)).cuda(), history=torch.from_numpy(hist).cuda(), repetition_penalty=1.3)
        for processed in (False, True):
            want = {r: x[r].float().numpy() for r in checked}
            if processed:
                want = {r: orc.apply_repetition_penalty(orc.apply_mask(want[r][None], mask[r:r + 1])[0], hist[r], 1.3) for r in checked}
            got = c.argmax(xd, xf=xf if processed else None).cpu().numpy()
            for r in checked:
                assert got[r] == orc.argmax(want[r]), (processed, r)
            for k in (2, 50, 64):
                tok, kc, ki, kp = c.sample(xd, ud, k=k, p=0.9, temperature=0.8, xf=xf if processed else None, kept_capacity=64)
                tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
                for r in checked:
                    idx, probs = orc.sampled_categorical(want[r], k, 0.9, 0.8)
                    n = len(idx)
                    assert kc[r] == n and np.array_equal(ki[r, :n], idx), (processed, k, r)
                    assert np.array_equal(bits(kp[r, :n]), bits(probs)), (processed, k, r)
                    assert tok[r] == idx[orc.discrete_draw(probs, u[r])], (processed, k, r)
        if vocab > 8192:
            assert c.fallback_rows() == 0  # no chunk is too short for its bound
    finally:
        c.close()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("processed", [False, True])
def test_batches_of_more_workgroups_than_cus(orc, dtype, processed):
    """Nucleus and large-k rows and rows in several modes are streamed by kernels of their own where there are more workgroups than CUs, and
    where some k takes every element for an offer: 40 rows of seven chunks."""
    say("many workgroups", dtype, processed)
    rows, vocab, cap = 40, 201088, 4096
    rng = np.random.default_rng(31)
    x = (torch.randn(rows, vocab, generator=torch.Generator().manual_seed(32)) * 5).to(dtype)
    hist = rng.integers(0, vocab, (rows, 90)).astype(np.int32)
    u = rng.random(rows)
    xf = pkg().LogitsXform(history=torch.from_numpy(hist).cuda(), repetition_penalty=1.2) if processed else None
    c = pkg().SearchContext(rows, vocab)
    checked = (0, 17, 39)
    try:
        want = {r: x[r].float().numpy() for r in checked}
        if processed:
            want = {r: orc.apply_repetition_penalty(want[r], hist[r], 1.2) for r in checked}
        xd, ud = x.cuda(), torch.from_numpy(u).cuda()
        several = [(0, 0.8, 1.0), (50, 0.9, 0.7), (300, 0.95, 1.0), (1000, 0.9, 1.0), (1, 0.0, 1.0)]
        calls = [[one] * rows for one in ((0, 0.8, 1.0), (1000, 0.9, 1.0), (2048, 0.0, 1.0), (3000, 0.9, 1.0))]
        calls += [[several[r % 5] for r in range(rows)], [several[r % 5] if r != 17 else (2500, 0.95, 1.0) for r in range(rows)]]
        for params in calls:
            tok, kc, ki, kp = c.sample(xd, ud, per_row=params, xf=xf, kept_capacity=cap)
            tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
            for r in checked:
                idx, probs = orc.sampled_categorical(want[r], *params[r])
                n = min(len(idx), cap)
                assert kc[r] == len(idx) and np.array_equal(ki[r, :n], idx[:n]), (params[r], r)
                assert np.array_equal(bits(kp[r, :n]), bits(probs[:n])), (params[r], r)
                assert tok[r] == idx[orc.discrete_draw(probs, u[r])], (params[r], r)
    finally:
        c.close()


@pytest.mark.parametrize("hist_len", [1500, 2500, 3400, 5000])
def test_sparse_mask_rows_with_thousands_of_distinct_history_ids(orc, hist_len):
    """Nucleus rows under a sparse grammar mask whose history holds more distinct ids than the sparse-mask kernel's
    threads take on as processed candidates (two each): such rows must leave that kernel, not lose ids.  Half of
    the history ids are allowed and strong, so that every one of them is inside the nucleus."""
    say("sparse mask, long history", hist_len)
    rng = np.random.default_rng(hist_len)
    rows, vocab = 2, 201088
    c = pkg().SearchContext(rows, vocab)
    try:
        x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
        mask = make_mask(rng, rows, vocab, 0.04)
        hist = np.stack([rng.choice(vocab, hist_len, replace=False) for _ in range(rows)]).astype(np.int32)
        for r in range(rows):
            ids = hist[r, :hist_len // 2]
            np.bitwise_or.at(mask.reshape(rows, -1)[r], ids >> 5, np.uint32(1) << (ids & 31).astype(np.uint32))
            x[r, ids] += 6.0
        u = rng.random(rows)
        xf = pkg().LogitsXform(mask=torch.from_numpy(mask.view(np.int32)).cuda(), history=torch.from_numpy(hist).cuda(),
                               repetition_penalty=1.2)
        tok, kc, ki, kp = c.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=0, p=0.95, temperature=1.0,
                                   xf=xf, kept_capacity=16384)
        tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
        proc = orc.apply_mask(x, mask)
        for r in range(rows):
            row = orc.apply_repetition_penalty(proc[r], hist[r], 1.2)
            idx, probs = orc.sampled_categorical(row, 0, 0.95, 1.0)
            assert kc[r] == len(idx), r
            assert np.array_equal(ki[r, :len(idx)], idx), r
            assert np.array_equal(bits(kp[r, :len(idx)]), bits(probs)), r
            assert tok[r] == idx[orc.discrete_draw(probs, u[r])], r
    finally:
        c.close()


@pytest.mark.parametrize("vocab", [5000, 70001])
def test_nucleus_with_minus_infinity_below_the_threshold(ctx, orc, vocab):
    """Rows whose elements outside the candidate range are all -inf: the element after the nucleus, which a
    stop on a sort-batch end keeps, is then a -inf one (probability 0) with the lowest id."""
    say("nucleus -inf tail", vocab)
    rng = np.random.default_rng(vocab)
    rows = 4
    x = np.full((rows, vocab), -np.inf, np.float32)
    for r, n in enumerate([16, 64, 15, 256]):   # 16, 64, 256: the nucleus ends on a batch end when p is near 1
        ids = rng.choice(vocab, n, replace=False)
        x[r, ids] = rng.standard_normal(n).astype(np.float32)
    u = rng.random(rows)
    for p in (0.9999999, 0.5):
        tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=0, p=p, temperature=1.0,
                                     kept_capacity=1024)
        tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
        for r in range(rows):
            idx, probs = orc.sampled_categorical(x[r], 0, p, 1.0)
            assert kc[r] == len(idx), (r, p, kc[r], len(idx))
            assert np.array_equal(ki[r, :len(idx)], idx), (r, p)
            assert np.array_equal(bits(kp[r, :len(idx)]), bits(probs)), (r, p)
            assert tok[r] == idx[orc.discrete_draw(probs, u[r])], (r, p)


@pytest.mark.parametrize("rows,vocab", [(6, 30000), (64, 40000), (70, 9000)])
def test_sample_heterogeneous_rows(ctx, orc, rows, vocab):
    """BatchedSampler semantics: per-row (k, p, T), greedy = (1, 0, 1).  Up to 64 rows the parameters
    travel inside the kernel arguments, above that through a table on the device: both sides of that edge."""
    say("sample heterogeneous", rows, vocab)
    rng = np.random.default_rng(6)
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    u = rng.random(rows)
    kinds = [(1, 0.0, 1.0), (50, 0.9, 0.7), (0, 0.9, 1.0), (8, 1.0, 1.5), (-1, 0.5, 0.8), (100, 0.0, 1.0)]
    params = [kinds[(r * 5 + r // 6) % 6] for r in range(rows)]
    params[0] = kinds[0]
    tok = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), per_row=params).cpu().numpy()
    for r, (k, p, t) in enumerate(params):
        assert tok[r] == orc.sample_row(x[r], k, p, t, u[r]), r
    assert tok[0] == orc.argmax(x[0])


@pytest.mark.parametrize("seed", range(int(os.environ.get("MI355X_RANDOM_FIRST", "0")),
                                        int(os.environ.get("MI355X_RANDOM_FIRST", "0")) +
                                        int(os.environ.get("MI355X_RANDOM_CASES", "300"))))
def test_sample_randomised_shapes_and_parameters(ctx, orc, seed):
    """Differential test over random shapes (vocabularies around the 32768-logit chunk edges included),
    per-row (k, p, T) mixes, logit scales, coarse grids (ties), grammar masks, repetition penalties and
    min-length masking: tokens of every row and the kept sets of uniform-parameter cases must equal
    the oracle's."""
    rng = np.random.default_rng(1000 + seed)
    edges = [1, 2, 63, 64, 65, 255, 4097, 32767, 32768, 32769, 65536, 65537, 98304, 131071, 131073, 196608, 201088]
    vocab = int(rng.choice(edges)) if seed % 2 else int(rng.integers(2, 140000))
    rows = int(rng.integers(1, 7))
    scale = float(rng.choice([0.05, 1.0, 3.0, 30.0]))
    x = (rng.standard_normal((rows, vocab)) * scale).astype(np.float32)
    if seed % 3 == 0:
        x = (np.round(x * 2) / 2).astype(np.float32)  # heavy ties
    if seed % 5 == 0:
        x[0, :] = 1.25  # a constant row
    # the logits as fp32, fp16 or bf16 (the oracle sees the widened values)
    kind = ("f32", "f16", "bf16")[seed % 7 % 3]
    if kind == "f16":
        with np.errstate(over="ignore"):
            x_dev = torch.from_numpy(x.astype(np.float16)).cuda()
        x = x_dev.float().cpu().numpy()
    elif kind == "bf16":
        x_dev = torch.from_numpy(x).to(torch.bfloat16).cuda()
        x = x_dev.float().cpu().numpy()
    else:
        x_dev = torch.from_numpy(x).cuda()
    say("sample random", seed, rows, vocab, scale, kind)
    xf, proc = None, x
    if seed % 4 in (1, 2):
        mask = make_mask(rng, rows, vocab, float(rng.choice([0.02, 0.5, 0.98])))
        hist_len = int(rng.integers(1, 200)) if seed % 9 else int(rng.integers(1500, 6000))  # now and then a long one
        hist = rng.integers(0, vocab, (rows, hist_len)).astype(np.int32)
        pen = float(rng.choice([1.0, 1.3, 0.8]))
        eos = [int(rng.integers(0, vocab))]
        allowed = int(np.unpackbits(mask.view(np.uint8)).reshape(rows, -1).sum(axis=1).max())
        promise = int(rng.choice([0, allowed, 3]))  # none, the true bound, a broken promise (still exact)
        xf = pkg().LogitsXform(mask=torch.from_numpy(mask.view(np.int32)).cuda(), history=torch.from_numpy(hist).cuda(),
                               repetition_penalty=pen, eos_ids=eos, apply_min_length=bool(seed % 8 == 1),
                               mask_allowed_max=promise)
        proc = orc.apply_mask(x, mask)
        proc = np.stack([orc.apply_repetition_penalty(orc.apply_min_length(proc[r], 0, 1 if seed % 8 == 1 else 0, eos),
                                                       hist[r], pen) for r in range(rows)])
    u = rng.random(rows)

    def params():
        k = int(rng.choice([0, 1, 2, 5, 40, 50, 64, 65, 200, 513, 2048, 2049, vocab, vocab + 7]))
        p = float(rng.choice([0.0, 0.1, 0.5, 0.9, 0.999, 1.0]))
        return k, p, float(rng.uniform(0.3, 2.0))

    if seed % 2:  # heterogeneous rows
        per_row = [params() for _ in range(rows)]
        tok = ctx.sample(x_dev, torch.from_numpy(u).cuda(), per_row=per_row, xf=xf).cpu().numpy()
        for r, (k, p, t) in enumerate(per_row):
            assert tok[r] == orc.sample_row(proc[r], k, p, t, u[r]), (r, k, p, t)
    else:
        k, p, t = params()
        cap = 256
        tok, kc, ki, kp = ctx.sample(x_dev, torch.from_numpy(u).cuda(), k=k, p=p, temperature=t,
                                     xf=xf, kept_capacity=cap)
        tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
        for r in range(rows):
            idx, probs = orc.sampled_categorical(proc[r], k, p, t)
            n = min(len(idx), cap)
            assert kc[r] == len(idx), (r, k, p, t)
            assert np.array_equal(ki[r, :n], idx[:n]), (r, k, p, t)
            assert np.array_equal(bits(kp[r, :n]), bits(probs[:n])), (r, k, p, t)
            assert tok[r] == idx[orc.discrete_draw(probs, u[r])], (r, k, p, t)


@pytest.mark.parametrize("k", [50, 57, 64])
def test_topk_with_clustered_best_tokens_stays_on_the_fast_path(ctx, orc, k):
    """The per-chunk bound pools the best eight per-thread maxima of every wave; rows whose best tokens
    sit next to each other (one wave holds most of them) or whose k is close to 64 let many more than k
    elements past it.  The kernel then takes the exact bound and lists again: results equal the oracle's
    and no row needs the full-sort path."""
    say("clustered top-k", k)
    rng = np.random.default_rng(900 + k)
    rows, vocab = 12, 128256
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    for r in range(rows // 2):
        start = int(rng.integers(0, vocab - 1024)) // 256 * 256
        if r % 2:   # 24 neighbouring ids hold the row's best tokens (six threads with four of them each)
            x[r, start:start + 24] = 14.0 + rng.standard_normal(24).astype(np.float32)
        else:       # 60 of the best tokens at every fourth id of one 256-id strip: one each in 60 threads of one wave
            x[r, start:start + 240:4] = 14.0 + rng.standard_normal(60).astype(np.float32)
    u = rng.random(rows)
    before = ctx.fallback_rows()
    tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=k, p=0.95, temperature=0.8,
                                 kept_capacity=64)
    tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
    for r in range(rows):
        idx, probs = orc.sampled_categorical(x[r], k, 0.95, 0.8)
        assert kc[r] == len(idx), r
        assert np.array_equal(ki[r, :len(idx)], idx), r
        assert np.array_equal(bits(kp[r, :len(idx)]), bits(probs)), r
        assert tok[r] == idx[orc.discrete_draw(probs, u[r])], r
    assert ctx.fallback_rows() == before


def test_wait_that_gives_up_hands_rows_to_the_exact_path(orc):
    """Failure handling of the top-k hand-over between workgroups, forced from the host: with a poll limit
    of 0 a finishing workgroup gives up on every list that has not arrived yet.  Its row must come out of
    the exact path unchanged, the context must report the event, and every later call must still be right
    (all its top-k rows then take the exact path)."""
    say("poll limit 0")
    rng = np.random.default_rng(77)
    rows, vocab = 128, 201088  # seven workgroups per row, far more workgroups than the GPU runs at once
    c = pkg().SearchContext(rows, vocab)
    try:
        x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
        u = rng.random(rows)
        want = np.array([orc.sample_row(x[r], 50, 0.9, 0.7, u[r]) for r in range(rows)], np.int32)
        xd, ud = torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda()
        assert np.array_equal(c.sample(xd, ud, k=50, p=0.9, temperature=0.7).cpu().numpy(), want)
        assert not c.wait_gave_up() and c.fallback_rows() == 0
        c.set_poll_limit(0)
        assert np.array_equal(c.sample(xd, ud, k=50, p=0.9, temperature=0.7).cpu().numpy(), want)
        assert c.wait_gave_up()
        assert 0 < c.fallback_rows() <= rows
        c.set_poll_limit(1 << 21)
        before = c.fallback_rows()
        assert np.array_equal(c.sample(xd, ud, k=50, p=0.9, temperature=0.7).cpu().numpy(), want)
        assert c.fallback_rows() - before == rows  # the fast path stays off for this context
        tk, ts = c.topk_scores(xd[:4], 8)
        for r in range(4):
            order = np.lexsort((np.arange(vocab), -x[r].astype(np.float64)))[:8]
            assert np.array_equal(tk[r].cpu().numpy(), order.astype(np.int32))
    finally:
        c.close()


def test_argument_errors(ctx):
    x = torch.zeros((2, 100), device="cuda")
    u = torch.zeros(2, dtype=torch.float64, device="cuda")
    with pytest.raises(RuntimeError, match="temperature"):
        ctx.sample(x, u, k=5, p=0.5, temperature=0.0)
    big = torch.zeros((257, 10), device="cuda")
    with pytest.raises(RuntimeError, match="capacity"):
        ctx.argmax(big)


@pytest.mark.parametrize("vocab,ngram,hist_len", [(1000, 2, 60), (40000, 3, 300), (70001, 1, 17), (300, 4, 2), (5000, 2, 1500)])
def test_no_repeat_ngram_ban(ctx, orc, vocab, ngram, hist_len):
    """ApplyNoRepeatNgramToLogits after mask, min-length and penalty (LogitsPenaltyProcessor::Apply order):
    in-place processing, greedy argmax and sampling all see the banned ids as lowest()."""
    say("no-repeat ngram", vocab, ngram, hist_len)
    rng = np.random.default_rng(vocab + ngram)
    rows = 4
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    hist = rng.integers(0, 6, (rows, hist_len)).astype(np.int32)  # six distinct ids: every n-gram repeats
    hist[1, :] = rng.integers(0, vocab, hist_len)  # a row whose n-grams hardly ever repeat
    x[:, :6] += 8.0  # the banned ids would otherwise win
    mask = make_mask(rng, rows, vocab, 0.9)
    eos = [3, vocab - 1]
    for pen in (1.0, 1.3):
        xf = pkg().LogitsXform(mask=torch.from_numpy(mask.view(np.int32)).cuda(), history=torch.from_numpy(hist).cuda(),
                               repetition_penalty=pen, eos_ids=eos, apply_min_length=True, no_repeat_ngram_size=ngram)
        want = orc.apply_mask(x, mask)
        for r in range(rows):
            w = orc.apply_min_length(want[r], 0, 1, eos)
            w = orc.apply_repetition_penalty(w, hist[r], pen)
            want[r] = orc.apply_no_repeat_ngram(w, hist[r], ngram)
        got = ctx.process_logits(torch.from_numpy(x.copy()).cuda(), xf).cpu().numpy()
        assert np.array_equal(bits(got), bits(want))
        if hist_len >= ngram:
            assert (want[0] != orc.apply_repetition_penalty(orc.apply_min_length(orc.apply_mask(x, mask)[0], 0, 1, eos),
                                                             hist[0], pen)).any()  # something was banned
        tok = ctx.argmax(torch.from_numpy(x).cuda(), xf=xf).cpu().numpy()
        assert np.array_equal(tok, orc.argmax_batch(want))
        u = rng.random(rows)
        for k, p in ((40, 0.9), (0, 0.8)):
            tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=k, p=p, temperature=0.9,
                                         xf=xf, kept_capacity=64)
            for r in range(rows):
                idx, probs = orc.sampled_categorical(want[r], k, p, 0.9)
                n = min(len(idx), 64)
                assert kc[r].item() == len(idx)
                assert np.array_equal(ki[r, :n].cpu().numpy(), idx[:n])
                assert np.array_equal(bits(kp[r, :n].cpu().numpy()), bits(probs[:n]))
                assert tok[r].item() == idx[orc.discrete_draw(probs, u[r])]


@pytest.mark.parametrize("vocab,K,seed_len,greedy", [(32064, 8, 40, False), (32064, 8, 40, True), (5000, 3, 2, False),
                                                     (140000, 5, 700, False)])
def test_target_selection_of_verify_rows(ctx, orc, vocab, K, seed_len, greedy):
    """ComputeTargetTokenSelection for the K+1 verify rows of one sequence (src/speculative_sampling.h:59-79,
    src/speculative_decoding_strategy.cpp:632-656): row i is processed with current_length = seed + i and
    the prefix seed tokens + the first i proposal tokens -- one shared history buffer, per-row lengths --
    then reduced to the greedy token or the kept (ids, probabilities)."""
    say("target selection", vocab, K, seed_len, greedy)
    rng = np.random.default_rng(vocab + K + seed_len)
    rows = K + 1
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    seq = rng.integers(0, 8, seed_len + K).astype(np.int32)  # few distinct ids: n-grams repeat
    x[:, :8] += 6.0
    eos = [5, 7]
    min_len = seed_len + 3  # the first rows are still too short for EOS
    lens = (seed_len + np.arange(rows)).astype(np.int32)
    xf = pkg().LogitsXform(history=torch.from_numpy(seq[None, :]).cuda(), shared_history=True,
                           history_lens=torch.from_numpy(lens).cuda(), repetition_penalty=1.2, eos_ids=eos,
                           min_length=min_len, no_repeat_ngram_size=2)
    k, p, t = 50, 0.9, 0.8
    u = rng.random(rows)
    if greedy:
        tok = ctx.argmax(torch.from_numpy(x).cuda(), xf=xf).cpu().numpy()
    else:
        tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=k, p=p, temperature=t,
                                     xf=xf, kept_capacity=64)
        tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
    for i in range(rows):
        g, idx, probs = orc.target_selection(x[i], int(lens[i]), seq[:lens[i]], greedy, k, p, t, rep_pen=1.2,
                                             min_len=min_len, ngram=2, eos=eos)
        if greedy:
            assert tok[i] == g, i
        else:
            assert kc[i] == len(idx), i
            assert np.array_equal(ki[i, :len(idx)], idx), i
            assert np.array_equal(bits(kp[i, :len(idx)]), bits(probs)), i
            assert tok[i] == idx[orc.discrete_draw(probs, u[i])], i


@pytest.mark.parametrize("batch", [1, 7, 300])
def test_greedy_tail_eos_pad_append(ctx, batch):
    """CheckForEOSAndPad + AppendNextTokensToSequences against the CPU search's PadIfAlreadyEOS / SetNextToken /
    AppendNextTokensToSequences loop (src/search.cpp:194-201,256-296) over a whole generation."""
    say("greedy tail", batch)
    rng = np.random.default_rng(batch)
    max_length, eos, pad = 12, [3, 9], 1
    seq = np.zeros((batch, max_length), np.int32)
    seen = np.zeros(batch, bool)
    d_seq = torch.zeros((batch, max_length), dtype=torch.int32, device="cuda")
    d_seen = torch.zeros(batch, dtype=torch.int32, device="cuda")
    d_done = torch.zeros(1, dtype=torch.int32, device="cuda")
    length, done = 0, False
    while not done and length < max_length:
        tokens = rng.integers(0, 12 if length > 3 else 40, batch).astype(np.int32)
        d_tok = torch.from_numpy(tokens).cuda()
        ctx.greedy_tail(d_tok, d_seen, eos, pad, d_seq, length, d_done)
        want = np.where(seen, pad, tokens)
        seen |= np.isin(want, eos) & ~seen
        done = bool(seen.all())
        assert np.array_equal(d_tok.cpu().numpy(), want)
        assert np.array_equal(d_seen.cpu().numpy().astype(bool), seen)
        assert bool(d_done.item()) == done
        if not done:  # the CPU search appends only while some row is alive; the device writes the column anyway
            seq[:, length] = want
            length += 1
            assert np.array_equal(d_seq.cpu().numpy()[:, :length], seq[:, :length])
    assert done or length == max_length
    before = d_seq.clone()
    ctx.greedy_tail(torch.zeros(batch, dtype=torch.int32, device="cuda"), d_seen, eos, pad, d_seq, max_length, d_done)
    assert torch.equal(before, d_seq)  # nothing is written beyond max_length


@pytest.mark.parametrize("vocab,frac,penalty,p", [
    (201088, 0.05, 1.2, 0.95),     # the sparse-mask kernel finishes the rows
    (201088, 0.0005, 1.2, 0.95),   # a hundred allowed ids
    (201088, 0.079, 0.8, 0.9),     # close to what the sort buffer holds; a penalty below one lifts masked history ids
    (201088, 0.0816, 1.2, 0.9),    # around the capacity: some rows fit, some are left to the dense kernels
    (201088, 0.5, 1.2, 0.95),      # dense: every row declined
    (70001, 0.05, 1.3, 0.999),     # the nucleus takes nearly every allowed id
    (70001, 0.02, 1.0, 0.3),       # no penalty: no history bitmap
    (4099, 0.3, 1.1, 0.95),
])
def test_nucleus_rows_under_sparse_and_dense_masks(ctx, orc, vocab, frac, penalty, p):
    """Rows in nucleus mode with a grammar mask of any density, min-length EOS masking, a history with ids that
    are masked, ids that are allowed, repeats and out-of-range ids; a few allowed logits are -inf, NaN or
    lowest().  Kept ids, probability bits and tokens equal the oracle's."""
    say("nucleus under mask", vocab, frac, penalty, p)
    rng = np.random.default_rng(int(vocab * 1000 + frac * 1e6))
    rows = 6
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    mask = make_mask(rng, rows, vocab, frac)
    allowed = np.unpackbits(mask.view(np.uint8), axis=1, bitorder="little")[:, :vocab].astype(bool)
    for r in range(rows):
        ids = np.flatnonzero(allowed[r])
        if len(ids) > 8:  # special values among the allowed logits
            x[r, ids[1]] = -np.inf
            x[r, ids[3]] = np.nan if r % 2 else LOWEST
            x[r, ids[5]] = x[r, ids[6]]  # a tie
    hist = rng.integers(0, vocab, (rows, 200)).astype(np.int32)
    hist[:, 7] = hist[:, 3]  # a repeat
    hist[:, 9] = -1
    for r in range(rows):
        ids = np.flatnonzero(allowed[r])
        hist[r, 0] = ids[0]                      # allowed ids in the history
        hist[r, 1] = ids[len(ids) // 2]
        hist[r, 2] = np.flatnonzero(~allowed[r])[0] if (~allowed[r]).any() else 0  # the first masked id is in the history
    eos = [int(np.flatnonzero(allowed[0])[0]), 2]
    u = rng.random(rows)
    xf = pkg().LogitsXform(mask=torch.from_numpy(mask.view(np.int32)).cuda(), history=torch.from_numpy(hist).cuda(),
                           repetition_penalty=penalty, eos_ids=eos, apply_min_length=True)
    cap = 20000
    proc = orc.apply_mask(x, mask)
    want = []
    for r in range(rows):
        row = proc[r].copy()
        row[eos] = LOWEST
        row = orc.apply_repetition_penalty(row, hist[r][(hist[r] >= 0)], penalty)
        want.append(orc.sampled_categorical(row, 0, p, 0.9))
    # without a promise about the mask, with the true bound on the allowed ids per row, and with a promise
    # that the rows break (they are still sampled correctly, by the exact path)
    for promise in (0, int(allowed.sum(axis=1).max()), 3):
        xf.c.mask_allowed_max = promise
        tok, kc, ki, kp = ctx.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k=0, p=p, temperature=0.9,
                                     xf=xf, kept_capacity=cap)
        tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
        for r in range(rows):
            idx, probs = want[r]
            n = min(len(idx), cap)
            assert kc[r] == len(idx), (promise, r, kc[r], len(idx))
            assert np.array_equal(ki[r, :n], idx[:n]), (promise, r)
            assert np.array_equal(bits(kp[r, :n]), bits(probs[:n])), (promise, r)
            assert tok[r] == idx[orc.discrete_draw(probs, u[r])], (promise, r)


def exact_path_rows(name, rng, vocab):
    if name == "gaussian":
        return (rng.standard_normal((2, vocab)) * 3).astype(np.float32)
    if name == "constant":
        return np.full((2, vocab), 1.5, np.float32)
    if name == "rounded":  # thirteen distinct scores: every digit of the sort's first level overflows
        return np.round(rng.standard_normal((2, vocab)) * 2).astype(np.float32)
    if name == "peaked":  # nearly every score inside a sliver of the row's range
        x = (5.0 + rng.random((2, vocab)) * 1e-3).astype(np.float32)
        x[:, rng.integers(0, vocab, 6)] = [100.0, -100.0, 50.0, 7.0, 5.0005, -3.0]
        return x
    if name == "mostly_lowest":  # what a grammar mask leaves behind
        x = (rng.standard_normal((2, vocab)) * 3).astype(np.float32)
        x[rng.random((2, vocab)) < 0.95] = LOWEST
        return x
    if name == "specials":
        x = (rng.standard_normal((2, vocab)) * 3).astype(np.float32)
        x[0, rng.integers(0, vocab, 9)] = [np.inf, -np.inf, np.nan, -np.inf, np.inf, 0.0, -0.0, LOWEST, np.nan]
        x[1, rng.integers(0, vocab, 4)] = [-np.inf, -np.inf, LOWEST, LOWEST]
        return x
    raise KeyError(name)


@pytest.mark.parametrize("vocab", [65, 511, 513, 4100, 10239, 10241, 16384, 70001, 128256, 201088])
@pytest.mark.parametrize("name", ["gaussian", "constant", "rounded", "peaked", "mostly_lowest", "specials"])
def test_exact_path_orders_whole_rows(ctx, orc, name, vocab):
    """k above the candidate-list bound (8192) and sampling from the whole vocabulary (k = 0, p = 1) take the exact
    path, which sorts the entire row; the kept ids are that order, checked to the last element."""
    say("exact path", name, vocab)
    rng = np.random.default_rng(vocab + len(name))
    x = exact_path_rows(name, rng, vocab)
    u = rng.random(2)
    before = ctx.fallback_rows()
    sample_and_check(ctx, orc, x, u, vocab, 0.0, 0.9, cap=vocab)
    sample_and_check(ctx, orc, x, u, 0, 1.0, 1.1, cap=vocab)
    if vocab > 2048:
        sample_and_check(ctx, orc, x, u, 2049, 0.97, 1.0, cap=2049)
    # k <= 8192 goes through the candidate lists, which hand rows with ties or NaNs at their bound to the exact path too
    assert ctx.fallback_rows() - before >= (4 if vocab > 8192 else 2)


def test_exact_path_sixteen_bit_rows(ctx, orc):
    """fp16 rows hold a few thousand distinct scores: long runs of ties through the exact path's sort."""
    say("exact path fp16")
    rng = np.random.default_rng(16)
    x16 = (rng.standard_normal((2, 128256)) * 3).astype(np.float16)
    u = rng.random(2)
    tok, kc, ki, kp = ctx.sample(torch.from_numpy(x16).cuda(), torch.from_numpy(u).cuda(), k=0, p=1.0, temperature=1.0,
                                 kept_capacity=128256)
    x = x16.astype(np.float32)
    for r in range(2):
        idx, probs = orc.sampled_categorical(x[r], 0, 1.0, 1.0)
        assert kc[r].item() == len(idx)
        assert np.array_equal(ki[r, :len(idx)].cpu().numpy(), idx), r
        assert np.array_equal(bits(kp[r, :len(idx)].cpu().numpy()), bits(probs)), r
        assert tok[r].item() == idx[orc.discrete_draw(probs, u[r])], r


@pytest.mark.parametrize("rows,cap", [(1, 8), (9, 64), (70, 300), (5, 20000)])
def test_draw_in_order_follows_one_engine(ctx, orc, rows, cap):
    """mi355x_draw_in_order: rows take the prepared canonical doubles in the order one std::mt19937 would serve them:
    a row with a single kept token and a finished row consume none, every other row the next one."""
    say("draw_in_order", rows, cap)
    rng = np.random.default_rng(rows * 7 + cap)
    counts = rng.integers(1, cap + 1, rows).astype(np.int32)
    counts[rng.random(rows) < 0.3] = 1
    skip = (rng.random(rows) < 0.25).astype(np.int32)
    ids = rng.integers(0, 1 << 20, (rows, cap)).astype(np.int32)
    probs = rng.random((rows, cap)).astype(np.float32)
    for r in range(rows):
        probs[r, :counts[r]] /= probs[r, :counts[r]].sum(dtype=np.float32)
    pool = rng.random(rows)
    for use_skip in (True, False):
        tok, used = ctx.draw_in_order(torch.from_numpy(counts).cuda(), torch.from_numpy(ids).cuda(),
                                      torch.from_numpy(probs).cuda(), torch.from_numpy(pool).cuda(),
                                      torch.from_numpy(skip).cuda() if use_skip else None)
        tok = tok.cpu().numpy()
        d = 0
        for r in range(rows):
            if (use_skip and skip[r]) or counts[r] < 2:
                assert tok[r] == ids[r, 0], r
                continue
            assert tok[r] == ids[r, orc.discrete_draw(probs[r, :counts[r]], pool[d])], (r, d)
            d += 1
        assert used.item() == d
    # a kept-set size beyond the capacity of the lists breaks the contract: the call says so instead of counting
    broken = counts.copy()
    broken[rows // 2] = cap + 3
    _, used = ctx.draw_in_order(torch.from_numpy(broken).cuda(), torch.from_numpy(ids).cuda(),
                                torch.from_numpy(probs).cuda(), torch.from_numpy(pool).cuda(), None)
    assert used.item() == -1


@pytest.mark.parametrize("rows,cap", [(1, 1), (2, 2), (63, 63), (64, 64), (65, 64), (130, 64), (200, 3), (70, 65)])
def test_draw_in_order_at_the_edges_of_a_wave_per_row(ctx, orc, rows, cap):
    """Lists of up to 64 entries are drawn from by a wave per row, batches around a wave's lanes and beyond; one entry more
    takes a workgroup per row."""
    test_draw_in_order_follows_one_engine(ctx, orc, rows, cap)


@pytest.mark.parametrize("vocab", [4095, 4096, 8191, 8193, 12289, 50257, 128256])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_whole_vocabulary_rows_spread_over_the_gpu(ctx, orc, vocab, dtype):
    """Temperature-only sampling (k = 0, p >= 1): token-only calls, whose ties stay unordered until the draw, on rows
    that end on and beside the edges of chunks and tiles; kept sets of a few entries; a batch of scattered rows of
    which only some sample from the whole vocabulary; rows the spread path declines (a maximum of -1e38 or infinity)
    and rows whose buckets it cuts (one score for all, runs of ties) among the others."""
    say("whole vocabulary", vocab, dtype)
    rng = np.random.default_rng(vocab)
    rows = 11
    x = (rng.standard_normal((rows, vocab)) * np.linspace(0.5, 5.0, rows)[:, None]).astype(np.float32)
    x[1, : vocab // 2] = np.round(x[1, : vocab // 2])  # runs of ties longer than a bucket holds
    x[2, :] = 0.25
    x[3, :] = -1e38
    x[4, 7] = 90.0      # one token far above the rest
    x[5, 11:400] = np.nan
    x[6, vocab - 1] = np.inf
    x[7, ::3] = -np.inf
    xd = torch.from_numpy(x).cuda().to(dtype)
    xw = x if dtype == torch.float32 else ctx.logits_handoff(xd.view(rows, 1, vocab)).cpu().numpy()
    u = rng.random(rows)
    u[0], u[8], u[9] = 0.0, 0.9999999999, 1e-12
    ud = torch.from_numpy(u).cuda()
    for p, t in ((1.0, 1.0), (1.0, 0.3), (2.0, 1.5)):
        want = orc.sample_batch(xw, 0, p, t, u)
        assert np.array_equal(ctx.sample(xd, ud, k=0, p=p, temperature=t).cpu().numpy(), want), (p, t)
        tok, kc, ki, kp = [v.cpu().numpy() for v in ctx.sample(xd, ud, k=1, p=p, temperature=t, kept_capacity=300)]
        assert np.array_equal(tok, want), (p, t)
        for r in range(rows):
            idx, probs = orc.sampled_categorical(xw[r], 1, p, t)
            n = min(len(idx), 300)
            assert kc[r] == len(idx) and np.array_equal(ki[r, :n], idx[:n]) and np.array_equal(bits(kp[r, :n]), bits(probs[:n])), (p, t, r)
            assert (ki[r, n:] == -1).all() and (kp[r, n:] == 0).all()
    params = [[(0, 1.0, 0.8), (20, 0.9, 1.0), (0, 0.7, 1.0)][r % 3] for r in range(rows)]
    got = ctx.sample([row.clone() for row in xd], ud, per_row=params).cpu().numpy()
    assert np.array_equal(got, [orc.sample_row(xw[r], *params[r], u[r]) for r in range(rows)])


@pytest.mark.parametrize("vocab,sigma,t,dtype", [
    (9001, 3.0, 1.0, np.float32), (50257, 2.0, 1.0, np.float16), (128256, 5.0, 0.7, np.float32), (40960, 0.5, 2.0, np.float32), (8192, 12.0, 0.5, np.float16),
])
def test_whole_vocabulary_draws_on_the_edges_of_their_guard_bands(ctx, orc, vocab, sigma, t, dtype):
    """Temperature-only rows whose token alone is asked for are picked from the masses of a histogram's buckets unless a
    cumulative value lies too close to the draw: draws placed on the reference's cumulative values and within and beyond the
    band beside them, at the first and the last elements that have any weight, and on both ends."""
    say("whole vocabulary edges", vocab, sigma, t, dtype)
    rng = np.random.default_rng(vocab)
    base = (rng.standard_normal(vocab) * sigma).astype(dtype)
    _, probs = orc.sampled_categorical(base.astype(np.float32), 0, 1.0, t)
    cp = np.cumsum(np.asarray(probs, np.float64)) / np.sum(np.asarray(probs, np.float64))
    us = list(rng.random(12)) + [0.0, 1e-300, np.nextafter(1.0, 0.0), 1.0 - 1e-9]
    for j in sorted({0, 1, len(cp) // 50, len(cp) // 5, len(cp) // 2, len(cp) - 2}):
        us += [cp[j], np.nextafter(cp[j], 0.0), np.nextafter(cp[j], 1.0), cp[j] - 1e-8, cp[j] + 1e-8, cp[j] - 2e-7, cp[j] + 2e-7]
    us = np.array([v for v in us if 0.0 <= v < 1.0], np.float64)
    x = np.tile(base, (len(us), 1))
    assert np.array_equal(tokens_only(ctx, x, us, 0, 1.0, t), orc.sample_batch(x.astype(np.float32), 0, 1.0, t, us))


@pytest.mark.parametrize("vocab,sigma,t", [(4097, 2.0, 1.0), (4160, 0.5, 1.0), (50257, 3.0, 1.0), (128256, 2.0, 0.8)])
def test_whole_vocabulary_draws_that_replay_the_sums(ctx, orc, vocab, sigma, t):
    """Draws on the reference's cumulative values, at the first, at both ends of a wave's 64 and at the last ones, and beside them at
    distances inside, at the edge of and beyond the band (2.25 n + 512) 2^-53, within which the reference's own sums are replayed."""
    say("replayed draws", vocab)
    rng = np.random.default_rng(vocab)
    base = (rng.standard_normal(vocab) * sigma).astype(np.float32)
    _, probs = orc.sampled_categorical(base, 0, 1.0, t)
    w = np.asarray(probs, np.float64)
    cp = np.cumsum(w / np.cumsum(w)[-1])
    band = (2.25 * len(cp) + 512) * 2.0 ** -53
    us = []
    for j in sorted({0, 1, 63, 64, 127, len(cp) // 3, len(cp) // 2 | 63, len(cp) - 66, len(cp) - 3, len(cp) - 2}):
        us += [cp[j], np.nextafter(cp[j], 0.0), np.nextafter(cp[j], 1.0)] + [cp[j] + s * f * band for s in (-1, 1) for f in (0.1, 0.99, 1.01, 8.0)]
    us = np.array([v for v in us if 0.0 <= v < 1.0], np.float64)
    x = np.tile(base, (len(us), 1))
    assert np.array_equal(tokens_only(ctx, x, us, 0, 1.0, t), orc.sample_batch(x, 0, 1.0, t, us))


@pytest.mark.parametrize("rows,vocab,dtype", [(1, 4099, torch.float32), (9, 50257, torch.float16), (40, 20011, torch.bfloat16), (300, 4099, torch.float32)])
def test_rows_given_back_by_the_pick_are_sorted_and_finished(orc, rows, vocab, dtype):
    """Temperature-only rows that the pick gives back, their draws on cumulative values: one of them, some among others, all, and more
    than there are workgroups at once; eagerly and from a graph that is replayed with eager calls between."""
    say("rows given back", rows, vocab, dtype)
    ctx = pkg().SearchContext(rows, vocab)
    rng = np.random.default_rng(rows)
    x = (2.0 * rng.standard_normal((rows, vocab))).astype(np.float32)
    if rows == 40:
        x[4, :] = -1e38
        x[5, 11] = np.inf
    xd = torch.from_numpy(x).cuda().to(dtype)
    xw = xd.float().cpu().numpy()
    u = rng.random(rows)
    open_draws = [r for r in range(0, rows, 1 if rows in (1, 300) else 3) if r not in (4, 5)]
    for r in open_draws:
        _, probs = orc.sampled_categorical(xw[r], 0, 1.0, 0.9)
        cp = np.cumsum(np.asarray(probs, np.float64))
        u[r] = cp[int(rng.integers(len(cp) // 100, len(cp) // 2))] / cp[-1]
    ud = torch.from_numpy(u).cuda()
    want = orc.sample_batch(xw, 0, 1.0, 0.9, u)
    back = len(open_draws) + (2 if rows == 40 else 0)  # (a row of maxima that are not ordinary numbers is given back as well)

    def given_back(step):
        before = ctx.picks_given_back()
        step()
        return ctx.picks_given_back() - before

    for _ in range(3):
        got = []
        assert given_back(lambda: got.append(ctx.sample(xd, ud, k=0, p=1.0, temperature=0.9).cpu().numpy())) >= back
        assert np.array_equal(got[0], want)
    out = torch.zeros(rows, dtype=torch.int32, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ctx.sample(xd, ud, k=0, p=1.0, temperature=0.9, out=out)
    for _ in range(3):
        out.zero_()
        assert given_back(graph.replay) >= back
        assert np.array_equal(out.cpu().numpy(), want)
        assert np.array_equal(ctx.sample(xd, ud, k=0, p=1.0, temperature=0.9).cpu().numpy(), want)
    ctx.close()


@pytest.mark.parametrize("rows,vocab,dtype", [(1, 4099, torch.bfloat16), (9, 50257, torch.float32), (40, 20011, torch.float16), (300, 4099, torch.float32)])
def test_rows_given_back_by_the_pick_whose_waits_give_up(orc, rows, vocab, dtype):
    """The tiles of a row that the pick gives back wait for the row's chunks; a wait that gives up -- forced with a poll limit of 0 -- leaves
    the row to the exact path, with the same token, and the next call is as before."""
    say("waits of rows given back", rows, vocab, dtype)
    ctx = pkg().SearchContext(rows, vocab)
    rng = np.random.default_rng(vocab)
    xd = torch.from_numpy((2.0 * rng.standard_normal((rows, vocab))).astype(np.float32)).cuda().to(dtype)
    xw = xd.float().cpu().numpy()
    u = rng.random(rows)
    for r in range(rows):
        _, probs = orc.sampled_categorical(xw[r], 0, 1.0, 0.9)
        cp = np.cumsum(np.asarray(probs, np.float64))
        u[r] = cp[int(rng.integers(len(cp) // 100, len(cp) // 2))] / cp[-1]
    ud = torch.from_numpy(u).cuda()
    want = orc.sample_batch(xw, 0, 1.0, 0.9, u)
    for limit in (1 << 21, 0, 1 << 21):
        ctx.set_poll_limit(limit)
        before, back = ctx.sum_waits_gave_up(), ctx.picks_given_back()
        for _ in range(3):
            assert np.array_equal(ctx.sample(xd, ud, k=0, p=1.0, temperature=0.9).cpu().numpy(), want), limit
        assert ctx.picks_given_back() - back >= 3 * rows
        assert (ctx.sum_waits_gave_up() > before) == (limit == 0)
    ctx.close()


@pytest.mark.parametrize("rows,vocab,dtype", [(24, 50257, torch.float16), (100, 4099, torch.float32), (60, 20011, torch.bfloat16)])
def test_whole_vocabulary_rows_of_p_one_and_above_among_others(orc, rows, vocab, dtype):
    """Rows of p = 1 that are picked or given back, rows of p above one (all of them given back), a row whose maximum is not finite, and rows
    of other modes between them, in one call: more than one row of each kind, by the argument table and (100 rows) by the device's."""
    say("p of one and above", rows, vocab, dtype)
    ctx = pkg().SearchContext(rows, vocab)
    rng = np.random.default_rng(rows)
    x = (2.0 * rng.standard_normal((rows, vocab))).astype(np.float32)
    if dtype != torch.float16:  # (whose values all are ordinary)
        x[6] = -1e38
    xd = torch.from_numpy(x).cuda().to(dtype)
    xw = xd.float().cpu().numpy()
    kinds = [(0, 1.0, 0.9), (50, 0.9, 0.7), (1, 2.0, 1.1), (0, 1.0, 0.9), (0, 0.9, 1.0), (200, 0.95, 1.0), (0, 1.0, 0.4), (0, 1.5, 0.8)]
    params = [kinds[r % len(kinds)] for r in range(rows)]
    u = rng.random(rows)
    for r in range(3, rows, len(kinds)):  # the open draws
        _, probs = orc.sampled_categorical(xw[r], *params[r])
        cp = np.cumsum(np.asarray(probs, np.float64))
        u[r] = cp[int(rng.integers(len(cp) // 100, len(cp) // 2))] / cp[-1]
    want = np.array([orc.sample_batch(xw[r:r + 1], *params[r], u[r:r + 1])[0] for r in range(rows)])
    ud = torch.from_numpy(u).cuda()
    for _ in range(3):
        before = ctx.picks_given_back()
        assert np.array_equal(ctx.sample(xd, ud, per_row=params).cpu().numpy(), want)
        assert ctx.picks_given_back() - before >= sum(p > 1.0 for _, p, _ in params) + len(range(3, rows, len(kinds)))
    above = [(k, 1.5 if p == 1.0 else p, t) for k, p, t in params]  # (no row to pick from: no pick)
    want = np.array([orc.sample_batch(xw[r:r + 1], *above[r], u[r:r + 1])[0] for r in range(rows)])
    assert np.array_equal(ctx.sample(xd, ud, per_row=above).cpu().numpy(), want)
    ctx.close()


@pytest.mark.parametrize("rows,vocab", [(64, 128256), (256, 32064)])
def test_batches_of_which_every_row_is_given_back_are_spread_over_the_gpu(rows, vocab):
    """A NaN in every row sends all of them past the pick: the step takes about as long as where the kept set is asked for and no pick is
    tried.  Sorted and finished by one workgroup a CU the rows took 1.75 times as long."""
    say("time of batches given back", rows, vocab)
    ctx = pkg().SearchContext(rows, vocab)
    g = torch.Generator(device="cuda").manual_seed(vocab)
    x = torch.randn(rows, vocab, generator=g, device="cuda") * 3
    x[:, 7] = float("nan")
    u = torch.rand(rows, generator=g, device="cuda", dtype=torch.float64)
    best = {}
    for kept in (0, 8):
        for _ in range(8):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(8):
                ctx.sample(x, u, k=0, p=1.0, temperature=1.0, kept_capacity=kept)
            end.record()
            end.synchronize()
            best[kept] = min(best.get(kept, 1e9), start.elapsed_time(end))
    ctx.close()
    assert best[0] < 1.4 * best[8], best


def crowded_rows(name, rng, rows, vocab):
    """Rows of which many ids share a score, or lie so close together that a bucket of the row's histogram (a 2048th of
    about thirty temperatures) holds more of them than a tile takes whole: (logits, element type, temperatures)."""
    x = rng.standard_normal((rows, vocab)).astype(np.float32)
    if name == "far_from_zero":  # bf16 has a value per 0.0625 around 12
        return 2.0 * x + 12.0, torch.bfloat16, (1.0, 0.4)
    if name == "far_below_zero":  # and one per 0.25 around -33, as GPT-2's logits lie
        return 2.0 * x - 33.0, torch.bfloat16, (1.0, 2.5)
    if name == "narrow":
        return 0.02 * x, torch.float16, (1.0, 5.0)
    if name == "flat":  # temperatures past the spread of the scores
        return x, torch.float32, (1.0, 6.0, 40.0)
    if name == "narrow_below_a_peak":
        x[:, 17] = 250.0
        x[:, vocab - 1] = -300.0
        return x, torch.float32, (20.0,)
    if name == "one_score":
        return np.full_like(x, -0.0), torch.float32, (1.0,)
    if name == "two_scores":
        return np.where(x > 0.3, np.float32(1.0), np.float32(1.001)), torch.float32, (1.0,)
    if name == "neighbouring_scores":  # a few hundred scores an ulp apart, in one bucket with everything else
        return np.nextafter(np.float32(1.0), np.float32(2.0)) + (rng.integers(0, 300, (rows, vocab)) * 2.0 ** -23).astype(np.float32), torch.float32, (1.0,)
    raise KeyError(name)


@pytest.mark.parametrize("vocab", [4099, 20011, 50257, 128256])
@pytest.mark.parametrize("name", ["far_from_zero", "far_below_zero", "narrow", "flat", "narrow_below_a_peak", "one_score", "two_scores",
                                  "neighbouring_scores"])
def test_whole_vocabulary_rows_with_crowded_buckets(ctx, orc, name, vocab):
    """Temperature-only sampling of rows whose histogram has buckets larger than a tile: tokens without the order of
    ties, and kept sets in their order.  (A bucket of more than 32768 scores, the bulk of a longer row below a peak, is
    given back to the exact path.)"""
    say("crowded buckets", name, vocab)
    rng = np.random.default_rng(vocab)
    rows = 5
    x, dtype, temperatures = crowded_rows(name, rng, rows, vocab)
    xd = torch.from_numpy(np.ascontiguousarray(x)).cuda().to(dtype)
    xw = xd.float().cpu().numpy()
    u = rng.random(rows)
    u[0], u[1] = 0.0, 0.999999
    ud = torch.from_numpy(u).cuda()
    for t in temperatures:
        want = orc.sample_batch(xw, 0, 1.0, t, u)
        assert np.array_equal(ctx.sample(xd, ud, k=0, p=1.0, temperature=t).cpu().numpy(), want), t
        tok, kc, ki, kp = [v.cpu().numpy() for v in ctx.sample(xd[:2], ud, k=0, p=1.0, temperature=t, kept_capacity=vocab)]
        assert np.array_equal(tok, want[:2]), t
        for r in range(2):
            idx, probs = orc.sampled_categorical(xw[r], 0, 1.0, t)
            n = len(idx)
            assert kc[r] == n and np.array_equal(ki[r, :n], idx) and np.array_equal(bits(kp[r, :n]), bits(probs)), (t, r)


@pytest.mark.parametrize("vocab,shift", [(128256, 12.0), (50257, -33.0)])
def test_rows_far_from_zero_are_spread_over_the_gpu_too(ctx, vocab, shift):
    """bf16 rows whose bulk lies where the type has few values cost a temperature-only step about what rows around zero
    do (one workgroup per row took 17 to 30 times as much)."""
    say("time of rows far from zero", vocab, shift)
    g = torch.Generator(device="cuda").manual_seed(vocab)
    u = torch.rand(8, generator=g, device="cuda", dtype=torch.float64)
    best = {}
    for mean in (0.0, shift):
        x = (torch.randn(8, vocab, generator=g, device="cuda") * 2 + mean).to(torch.bfloat16)
        for _ in range(6):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(8):
                ctx.sample(x, u, k=0, p=1.0, temperature=1.0)
            end.record()
            end.synchronize()
            best[mean] = min(best.get(mean, 1e9), start.elapsed_time(end))
    assert best[shift] < 3 * best[0.0], best
