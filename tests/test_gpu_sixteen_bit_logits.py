"""fp16 / bf16 logits read directly by the sampling, top-k-scores and argmax entry points: results must equal
the oracle run on the rows widened with the CPU path's conversions (Logits::Get casts before the search sees
the scores, src/models/logits.cpp:72-76; FastFloat16ToFloat32 / BFloat16ToFloat32, src/models/utils.cpp:84-109).
Token ids, kept ids and probability bits are compared exactly."""
import numpy as np
import pytest
import torch

from gpu_common import make_mask, pkg, say

pytestmark = pytest.mark.gpu

KIND = {torch.float16: 0, torch.bfloat16: 1}


@pytest.fixture(scope="module")
def ctx():
    c = pkg().SearchContext(96, 201088)
    yield c
    c.close()


def bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


def to_bits16(t):
    return t.view(torch.int16).cpu().numpy().view(np.uint16)


def widened(orc, t):
    return orc.cast(to_bits16(t), KIND[t.dtype], np.float32)


def check_sample(ctx, orc, x16, u, per_row, xf=None, proc=None, cap=1024):
    rows = x16.shape[0]
    tok, kc, ki, kp = ctx.sample(x16, torch.from_numpy(u).cuda(), per_row=per_row, xf=xf, kept_capacity=cap)
    tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
    wide = widened(orc, x16) if proc is None else proc
    for r in range(rows):
        k, p, t = per_row[r]
        idx, probs = orc.sampled_categorical(wide[r], k, p, t)
        n = min(len(idx), cap)
        assert kc[r] == len(idx), (r, per_row[r], kc[r], len(idx))
        assert np.array_equal(ki[r, :n], idx[:n]), (r, per_row[r])
        assert np.array_equal(bits(kp[r, :n]), bits(probs[:n])), (r, per_row[r])
        assert tok[r] == idx[orc.discrete_draw(probs, u[r])], (r, per_row[r])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,vocab", [(64, 128256), (5, 40000 + 13), (3, 33000), (4, 70), (2, 201088)])
def test_sample_reads_sixteen_bit_rows(ctx, orc, dtype, rows, vocab):
    """Every selection mode on fp16 / bf16 rows, aligned and unaligned row starts, short last chunks."""
    say("sample 16-bit", dtype, rows, vocab)
    g = torch.Generator(device="cuda").manual_seed(vocab + rows)
    x = (torch.randn(rows, vocab, generator=g, device="cuda") * 3).to(dtype)
    rng = np.random.default_rng(vocab)
    u = rng.random(rows)
    menu = [(50, 0.9, 0.7), (1, 0.0, 1.0), (0, 0.9, 1.0), (64, 0.0, 1.3), (100, 0.95, 1.0), (0, 0.5, 0.6), (8, 1.0, 2.0),
            (600, 0.9, 1.0)]
    per_row = [menu[(r * 3 + r // 8) % len(menu)] for r in range(rows)]
    check_sample(ctx, orc, x, u, per_row)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_sixteen_bit_ties_are_broken_by_lowest_id(ctx, orc, dtype):
    """Sixteen-bit rows are full of equal values: the kept sets must follow score descending, id ascending."""
    say("sample 16-bit ties", dtype)
    rows, vocab = 6, 50000
    g = torch.Generator(device="cuda").manual_seed(4)
    x = torch.round(torch.randn(rows, vocab, generator=g, device="cuda") * 2).to(dtype)  # a few dozen distinct values
    u = np.random.default_rng(1).random(rows)
    check_sample(ctx, orc, x, u, [(50, 0.9, 0.7), (10, 0.0, 1.0), (64, 0.5, 1.0), (2, 0.0, 1.0), (1, 0.0, 1.0), (40, 1.0, 1.0)])


def test_every_fp16_pattern_through_the_streaming_loads(ctx, orc):
    """All 65536 fp16 bit patterns in one row (exponent field 31 decodes as an ordinary exponent, subnormals are
    exact): the 64 best ids and their widened scores from mi355x_topk_scores equal a sort of the widened row."""
    say("topk_scores over all fp16 patterns")
    pat = np.arange(65536, dtype=np.uint16)
    rng = np.random.default_rng(9)
    rows = np.stack([pat, rng.permutation(pat), pat[::-1].copy()])
    x = torch.from_numpy(rows.view(np.int16)).cuda().view(torch.float16)
    tok, sc = ctx.topk_scores(x, 64)
    wide = orc.cast(rows, 0, np.float32)
    for r in range(3):
        order = np.lexsort((np.arange(65536), -wide[r].astype(np.float64)))[:64]
        assert np.array_equal(tok[r].cpu().numpy(), order)
        assert np.array_equal(bits(sc[r].cpu().numpy()), bits(wide[r][order]))
    assert wide[0].max() == np.float32(131008.0)  # 0x7fff decoded as 65536 * (1 + 1023/1024)
    # and the sampler keeps exactly the ids whose widened value is largest
    u = np.array([0.3, 0.6, 0.9])
    check_sample(ctx, orc, x, u, [(64, 0.0, 30000.0), (20, 0.0, 5000.0), (50, 0.9, 20000.0)])


def test_every_bf16_pattern_through_the_streaming_loads(ctx, orc):
    """All 65536 bf16 patterns, NaNs and infinities included: NaNs order below every number, +inf wins."""
    say("topk_scores over all bf16 patterns")
    pat = np.arange(65536, dtype=np.uint16)
    rows = np.stack([pat, np.random.default_rng(2).permutation(pat)])
    x = torch.from_numpy(rows.view(np.int16)).cuda().view(torch.bfloat16)
    tok, sc = ctx.topk_scores(x, 64)
    wide = orc.cast(rows, 1, np.float32)
    for r in range(2):
        key = np.where(np.isnan(wide[r]), -np.inf, wide[r].astype(np.float64))
        nan_last = np.isnan(wide[r]).astype(np.int64)
        order = np.lexsort((np.arange(65536), -key, nan_last))[:64]
        assert np.array_equal(tok[r].cpu().numpy(), order)
        assert np.array_equal(bits(sc[r].cpu().numpy()), bits(wide[r][order]))
    assert np.isinf(wide[0][tok[0, 0].item()])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_sixteen_bit_rows_with_logits_processing(ctx, orc, dtype):
    """Grammar mask, min-length EOS masking and repetition penalty applied to the widened values."""
    say("sample 16-bit xform", dtype)
    rows, vocab = 6, 70001
    g = torch.Generator(device="cuda").manual_seed(11)
    x = (torch.randn(rows, vocab, generator=g, device="cuda") * 3).to(dtype)
    rng = np.random.default_rng(12)
    mask = make_mask(rng, rows, vocab, 0.3)
    hist = rng.integers(0, vocab, (rows, 300)).astype(np.int32)
    hist[:, 0] = x.float().argmax(dim=1).cpu().numpy()
    eos = [5, 70000]
    u = rng.random(rows)
    xf = pkg().LogitsXform(mask=torch.from_numpy(mask.view(np.int32)).cuda(), history=torch.from_numpy(hist).cuda(),
                           repetition_penalty=1.3, eos_ids=eos, apply_min_length=True)
    proc = orc.apply_mask(widened(orc, x), mask)
    for r in range(rows):
        proc[r, eos] = np.finfo(np.float32).min
        proc[r] = orc.apply_repetition_penalty(proc[r], hist[r], 1.3)
    check_sample(ctx, orc, x, u, [(50, 0.9, 0.7), (0, 0.9, 1.0), (1, 0.0, 1.0), (100, 0.0, 1.0), (0, 0.3, 0.5), (64, 0.95, 1.0)],
                 xf=xf, proc=proc, cap=4096)
    am = ctx.argmax(x, xf).cpu().numpy()
    assert np.array_equal(am, orc.argmax_batch(proc))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("vocab", [40001, 40002, 40003, 40004, 40005, 40006, 40007, 98305])
def test_sixteen_bit_rows_with_logits_processing_that_end_inside_a_group_of_eight(ctx, orc, dtype, vocab):
    """The kernels with logits processing read a sixteen-bit chunk as eight 128-bit loads per thread whatever the
    row's end; the group of eight that straddles it is fetched once more element by element.  Vocabularies that end
    one to seven elements into a group (and a last chunk of one element), the row's best tokens on its last
    elements, some of them penalised or masked."""
    say("16-bit xform row ends", dtype, vocab)
    rows = 5
    g = torch.Generator(device="cuda").manual_seed(vocab)
    x = (torch.randn(rows, vocab, generator=g, device="cuda") * 3).to(dtype)
    x[0, vocab - 1] = 30.0
    x[1, vocab - 2] = 30.0
    x[2, vocab - 3] = 30.0
    x[3, vocab - 1] = 29.0
    x[3, vocab - 5] = 30.0
    rng = np.random.default_rng(vocab)
    mask = make_mask(rng, rows, vocab, 0.8)
    mask[2, (vocab - 3) >> 5] &= ~np.uint32(1 << ((vocab - 3) & 31))
    hist = rng.integers(0, vocab, (rows, 120)).astype(np.int32)
    hist[:, 0] = vocab - 2
    hist[:, 1] = vocab - 1
    u = rng.random(rows)
    xf = pkg().LogitsXform(mask=torch.from_numpy(mask.view(np.int32)).cuda(), history=torch.from_numpy(hist).cuda(),
                           repetition_penalty=1.5)
    proc = orc.apply_mask(widened(orc, x), mask)
    for r in range(rows):
        proc[r] = orc.apply_repetition_penalty(proc[r], hist[r], 1.5)
    check_sample(ctx, orc, x, u, [(50, 0.9, 0.7), (0, 0.9, 1.0), (1, 0.0, 1.0), (300, 0.95, 1.0), (8, 0.0, 1.0)], xf=xf, proc=proc,
                 cap=4096)
    assert np.array_equal(ctx.argmax(x, xf).cpu().numpy(), orc.argmax_batch(proc))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_argmax_sixteen_bit_rows(ctx, orc, dtype):
    say("argmax 16-bit", dtype)
    g = torch.Generator(device="cuda").manual_seed(21)
    x = (torch.randn(7, 151936, generator=g, device="cuda") * 2).to(dtype)
    assert np.array_equal(ctx.argmax(x).cpu().numpy(), orc.argmax_batch(widened(orc, x)))
    y = x[:, 3:100003]  # rows that start off a 16-byte boundary
    assert np.array_equal(ctx.argmax(y).cpu().numpy(), orc.argmax_batch(widened(orc, y.contiguous())))
    for width in (1, 7, 64):  # rows too short for the streaming kernel take the small kernels
        z = x[:, 5:5 + width].contiguous()
        assert np.array_equal(ctx.argmax(z).cpu().numpy(), orc.argmax_batch(widened(orc, z))), width
    # the entry point without a context: the chunked kernel (rows x chunks >= 256) and the row kernel
    for rows, vocab in ((40, 70001), (3, 5000)):
        w = (torch.randn(rows, vocab, generator=g, device="cuda") * 2).to(dtype)
        out = torch.empty(rows, dtype=torch.int32, device="cuda")
        assert np.array_equal(pkg().argmax_static(w, out).cpu().numpy(), orc.argmax_batch(widened(orc, w))), (rows, vocab)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("vocab", [50257, 51865, 98311])
def test_rows_that_start_on_every_offset_of_a_16_byte_line(ctx, orc, dtype, vocab):
    """Odd vocabularies put every row on a start of its own inside a 16-byte line, and a view can start anywhere: the
    streaming kernels read such rows with the same 128-bit loads as aligned ones.  Nine rows cut out of one buffer
    at element offsets 0 .. 8, argmax and every selection mode, against the oracle on the same elements."""
    say("row starts", dtype, vocab)
    g = torch.Generator(device="cuda").manual_seed(vocab)
    rows = 9
    big = (torch.randn(rows, vocab + 16, generator=g, device="cuda") * 3).to(dtype)
    views = [big[r, r:r + vocab] for r in range(rows)]
    dense = torch.stack(views).contiguous()  # rows vocab elements apart: starts differ row by row, too
    wide = dense.cpu().numpy() if dtype == torch.float32 else widened(orc, dense)
    assert np.array_equal(ctx.argmax(dense).cpu().numpy(), orc.argmax_batch(wide))
    rng = np.random.default_rng(vocab)
    u = rng.random(rows)
    for k, p, t in ((50, 0.9, 0.7), (0, 0.9, 1.0), (300, 0.95, 1.0)):
        for x in (dense, views):  # rows a stride apart, and rows scattered over memory with starts of their own
            tok, kc, ki, kp = ctx.sample(x, torch.from_numpy(u).cuda(), k=k, p=p, temperature=t, kept_capacity=4096)
            tok, kc, ki, kp = tok.cpu().numpy(), kc.cpu().numpy(), ki.cpu().numpy(), kp.cpu().numpy()
            for r in range(rows):
                idx, probs = orc.sampled_categorical(wide[r], k, p, t)
                n = min(len(idx), 4096)
                assert kc[r] == len(idx), (k, r)
                assert np.array_equal(ki[r, :n], idx[:n]), (k, r)
                assert np.array_equal(bits(kp[r, :n]), bits(probs[:n])), (k, r)
                assert tok[r] == idx[orc.discrete_draw(probs, u[r])], (k, r)


def test_config2_shape_in_fp16_equals_fp32_on_the_widened_rows(ctx, orc):
    """Benchmark configuration 2 with fp16 logits: identical tokens to the fp32 entry point fed the widened rows."""
    say("config2 fp16")
    rows, vocab = 64, 128256
    g = torch.Generator(device="cuda").manual_seed(2)
    x = torch.randn(rows, vocab, generator=g, device="cuda") * 3
    x.scatter_add_(1, torch.randint(0, vocab, (rows, 8), generator=g, device="cuda"), torch.full((rows, 8), 10.0, device="cuda"))
    h = x.half()
    u = torch.rand(rows, generator=g, device="cuda", dtype=torch.float64)
    a = ctx.sample(h, u, k=50, p=0.9, temperature=0.7)
    b = ctx.sample(torch.from_numpy(widened(orc, h)).cuda(), u, k=50, p=0.9, temperature=0.7)
    assert torch.equal(a, b)
    assert np.array_equal(a.cpu().numpy(), orc.sample_batch(widened(orc, h), 50, 0.9, 0.7, u.cpu().numpy()))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_rows_scattered_over_memory(ctx, orc, dtype):
    """mi355x_sample_scattered: 70 rows (two launches of at most 64) that live in separate allocations, at odd
    offsets and in reverse order, give what mi355x_sample gives on the same rows packed into one matrix."""
    say("scattered rows", dtype)
    rows, vocab = 70, 50001
    g = torch.Generator(device="cuda").manual_seed(70)
    backing = [(torch.randn(vocab + 11, generator=g, device="cuda") * 3).to(dtype) for _ in range(rows)]
    row_list = [backing[rows - 1 - r][(r % 5):(r % 5) + vocab] for r in range(rows)]
    packed = torch.stack(row_list).contiguous()
    rng = np.random.default_rng(7)
    u = torch.from_numpy(rng.random(rows)).cuda()
    menu = [(50, 0.9, 0.7), (1, 0.0, 1.0), (0, 0.9, 1.0), (100, 0.95, 1.0), (64, 0.0, 1.2)]
    per_row = [menu[(r * 2 + r // 9) % len(menu)] for r in range(rows)]
    mask = make_mask(rng, rows, vocab, 0.5)
    hist = rng.integers(0, vocab, (rows, 40)).astype(np.int32)
    xf = pkg().LogitsXform(mask=torch.from_numpy(mask.view(np.int32)).cuda(), history=torch.from_numpy(hist).cuda(),
                           repetition_penalty=1.25)
    for use_xf in (None, xf):
        a = ctx.sample(row_list, u, per_row=per_row, xf=use_xf, kept_capacity=128)
        b = ctx.sample(packed, u, per_row=per_row, xf=use_xf, kept_capacity=128)
        for got, want in zip(a, b):
            assert torch.equal(got, want)
    # uniform parameters, no per-row table from the caller
    assert torch.equal(ctx.sample(row_list, u, k=50, p=0.9, temperature=0.7), ctx.sample(packed, u, k=50, p=0.9, temperature=0.7))
    if dtype == torch.float32:
        want = [orc.sample_row(packed[r].cpu().numpy(), *per_row[r], u[r].item()) for r in range(rows)]
        assert ctx.sample(row_list, u, per_row=per_row).cpu().tolist() == want


def test_captured_calls_with_host_tables_use_up_staging_slots():
    """Per-row parameters of more than 64 rows and the KV pointer tables are copied from the caller's host arrays into
    pinned staging memory of the context; a call captured into a graph keeps its slot for good, so a context
    serves a bounded number of such captured calls (56) and says so when they are used up."""
    say("staging slots under capture")
    c = pkg().SearchContext(80, 4099)
    rows, vocab = 70, 4099
    x = torch.randn(rows, vocab, device="cuda")
    u = torch.rand(rows, device="cuda", dtype=torch.float64)
    out = torch.empty(rows, dtype=torch.int32, device="cuda")
    per_row = [(50, 0.9, 0.7)] * rows
    present = [torch.randn(4, 64, device="cuda") for _ in range(2)]
    past = [torch.zeros_like(p) for p in present]
    idx = torch.tensor([1, 1, 0, 3], dtype=torch.int32, device="cuda")
    eager = c.sample(x, u, per_row=per_row).clone()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            c.sample(x, u, per_row=per_row, out=out)
            for _ in range(55):
                c.kv_gather(present, past, idx)
            with pytest.raises(RuntimeError, match="staged 56"):
                c.kv_gather(present, past, idx)
        out.zero_()
        graph.replay()
        side.synchronize()
    assert torch.equal(out, eager)
    for t, src in zip(past, present):
        assert torch.equal(t, src[idx.long()])
    # eager calls are not affected: they go through the ring
    for _ in range(20):
        c.kv_gather(present, past, idx)
    torch.cuda.synchronize()
    c.close()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("k,p,temp", [(0, 0.9, 1.0), (0, 0.97, 0.7), (0, 0.9, 1e6), (300, 0.0, 1.0), (1000, 0.95, 2.0)])
def test_draws_that_fall_into_runs_of_ties(ctx, orc, dtype, k, p, temp):
    """Token-only calls keep ties of sixteen-bit logits unordered until the draw falls into a run of them: runs of two
    to thousands of equal scores, runs that the kept set ends inside, rows of few distinct values, a temperature at
    which different scores share an exponential, and buckets that hold many keys of several scores."""
    say("ties", dtype, k, p, temp)
    rng = np.random.default_rng(int(k + 100 * p))
    rows, vocab = 12, 60013
    x = (rng.standard_normal((rows, vocab)) * 2).astype(np.float32)
    x[1:4] += 16.0                                           # coarse steps: hundreds of ties per value
    x[4, rng.integers(0, vocab, 500)] = 12.0                 # the best score itself is a run
    x[5, rng.integers(0, vocab, 3000)] = 14.0
    x[6] = np.round(x[6] * 2) / 2 + 8.0                      # a dozen distinct values
    x[7, rng.integers(0, vocab, 6000)] = 0.001 * rng.standard_normal(6000)  # many scores close to zero
    x[7, 9] = 6.0
    x[8, :2] = 20.0
    x16 = torch.from_numpy(x).cuda().to(dtype)
    wide = widened(orc, x16)
    for rep in range(3):
        u = rng.random(rows)
        got = ctx.sample(x16, torch.from_numpy(u).cuda(), k=k, p=p, temperature=temp).cpu().numpy()
        assert np.array_equal(got, orc.sample_batch(wide, k, p, temp, u)), rep


def rows_with_one_run(rng, rows, vocab, run, dtype):
    """`run` ids of every row share the best score, the first and the last id among them; the rest lies far below."""
    x = (rng.standard_normal((rows, vocab)) - 25.0).astype(np.float32)
    for r in range(rows):
        ids = rng.permutation(vocab - 2)[: run - 2] + 1
        x[r, ids] = x[r, 0] = x[r, vocab - 1] = 5.0
    return torch.from_numpy(x).cuda().to(dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("vocab,run", [(40001, 2), (40001, 64), (128256, 65), (128256, 1025), (70001, 5000), (524288, 9000), (128256, 16000)])
def test_the_token_of_a_run_of_ties(orc, vocab, run, dtype):
    """A nucleus whose entries share one score, token only: the run is not ordered before the draw, the id of the drawn
    rank is found among its ids afterwards -- pair by pair for short runs, by a selection for long ones."""
    say("run of ties", vocab, run, dtype)
    rng = np.random.default_rng(run)
    rows = 6
    c = pkg().SearchContext(rows, vocab)
    x = rows_with_one_run(rng, rows, vocab, run, dtype)
    u = np.array([0.0, 1.0 - 2.0 ** -53, 0.5 / run, 0.5, 0.25, 0.999])
    got = c.sample(x, torch.from_numpy(u).cuda(), k=0, p=0.9, temperature=1.0).cpu().numpy()
    assert np.array_equal(got, orc.sample_batch(x.float().cpu().numpy(), 0, 0.9, 1.0, u))
    c.close()


def test_long_runs_of_ties_take_linear_time():
    """A run of 16000 ties costs a step no more than a few times what the sort of as many distinct entries does (fp32
    rows); a compare per pair of ties made it sixty times as much."""
    say("time of a run of ties")
    rng = np.random.default_rng(1)
    c = pkg().SearchContext(8, 128256)
    u = torch.from_numpy(rng.random(8)).cuda()
    best = {}
    for dtype in (torch.float32, torch.float16):
        x = rows_with_one_run(rng, 8, 128256, 16000, dtype)
        for _ in range(6):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(4):
                c.sample(x, u, k=0, p=0.9, temperature=1.0)
            end.record()
            end.synchronize()
            best[dtype] = min(best.get(dtype, 1e9), start.elapsed_time(end))
    assert best[torch.float16] < 5 * best[torch.float32], best
    c.close()
