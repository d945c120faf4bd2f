// Host side of the C ABI declared in include/mi355x_search.h: argument validation, workspace
// management and kernel launches.  No computation happens here, and there is no CPU fallback: every
// entry point either launches the HIP kernels or fails.
#include <hip/hip_runtime.h>
#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <cmath>
#include <cstring>
#include <cstdlib>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <type_traits>
#include <vector>
#include "api_internal.h"

namespace {

thread_local std::string g_error;

}  // namespace

int ms_vfail(int code, const char* fmt, va_list ap) {
  char buf[512];
  vsnprintf(buf, sizeof(buf), fmt, ap);
  g_error = buf;
  return code;
}

namespace {

int Fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  ms_vfail(code, fmt, ap);
  va_end(ap);
  return code;
}

#define HIP_TRY(expr)                                                                       \
  do {                                                                                      \
    hipError_t e_ = (expr);                                                                 \
    if (e_ != hipSuccess) return Fail(MI355X_E_HIP, "%s: %s", #expr, hipGetErrorString(e_)); \
  } while (0)

int NextPow2(int v) {
  int p = 64;
  while (p < v) p <<= 1;
  return p;
}

}  // namespace

// What a context shares with its beam scorers, which may be destroyed after it and may belong to different threads:
// pinned host memory, held until the last of them is gone.
//  - A word per scorer, which the step that finishes the last batch entry sets, so that asking whether a search is done
//    takes no copy.  Scorers past kWords at a time have no word.
//  - An area where small results and states go between host and device, by calls that hold its mutex and wait for
//    their copy before they return.
struct ScorerHost {
  static constexpr int kWords = 64;
  static constexpr size_t kReadbackBytes = 256 * 1024;
  char* readback{};
  std::mutex readback_mutex;
  int* words{};
  std::atomic<uint64_t> used{};  // bit i: word i is taken
  ~ScorerHost() {
    if (readback) (void)hipHostFree(readback);
  }
  hipError_t Allocate() {
    void* pinned = nullptr;
    const hipError_t e = hipHostMalloc(&pinned, kReadbackBytes + kWords * sizeof(int), hipHostMallocDefault);
    if (e != hipSuccess) return e;
    readback = static_cast<char*>(pinned);
    words = reinterpret_cast<int*>(readback + kReadbackBytes);
    return hipSuccess;
  }
  int TakeWord() {  // -1: none left
    uint64_t seen = used.load();
    while (~seen != 0 && !used.compare_exchange_weak(seen, seen | (seen + 1))) {
    }
    return ~seen != 0 ? __builtin_ctzll(~seen) : -1;
  }
  void GiveBackWord(int word) { used.fetch_and(~(uint64_t{1} << word)); }
};

struct mi355x_search_ctx {
  int device{};
  int max_rows{}, max_vocab{}, max_chunks{};
  size_t bytes{};
  std::vector<void*> allocs;
  ms::u64* cand_small{};
  size_t cand_lists{};  // lists of kSmallCap slots
  uint32_t* chunk_cnt{};
  uint32_t* chunk_max{};
  uint32_t* chunk_thr{};
  ms::u64* chunk_next{};
  uint32_t* row_arrive{};
  ms::u64* row_best{};
  ms::u64* big{};
  ms::u64* big2{};
  size_t big_stride{};
  uint32_t* fallback_rows{};
  uint32_t* row_done{};
  int poll_limit{ms::kDefaultPollLimit};
  uint32_t* ban{};  // [max_rows, mask words]: ids banned by the no-repeat-n-gram rule
  mi355x_sample_params* params_dev{};
  float* beam_row_scores{};
  ms::u64* seg_cand{};  // [max_rows][max_segs][kBeamMaxCand] beam-search candidates per segment
  int max_segs{};
  uint32_t* seg_max{};
  double* seg_sum{};
  int4* seg_step{};
  int4* sub_step{};
  int* sub_se{};
  float* row_max{};
  float* row_sum{};
  ms::WideRow* wide_rows{};
  uint32_t* wide_tile_start{};
  uint2* wide_cut_bucket{};
  uint32_t* wide_rest{};
  int32_t* beam_row_tokens{};
  // Pinned host staging for the per-row parameters of more than 64 rows, which come in a caller's HOST array and do
  // not fit the kernel arguments: the call copies the array into a slot here and records a copy from the slot to the
  // device table.  Slots of the ring are reused once the copy that read them
  // is done (an event per slot); a call on a capturing stream gets a slot of its own that is never reused, so the
  // copy node of its graph reads the same bytes at every replay.
  static constexpr int kStageRing = 8, kStageCaptured = 56;
  char* stage{};
  size_t stage_slot_bytes{};
  std::shared_ptr<ScorerHost> scorer_host;
  hipEvent_t stage_event[kStageRing]{};
  bool stage_pending[kStageRing]{};
  int stage_next{}, stage_captured{};

  template <typename T>
  hipError_t Alloc(T** p, size_t count, bool zero) {
    void* q = nullptr;
    const size_t n = count * sizeof(T);
    hipError_t e = hipMalloc(&q, n ? n : 16);
    if (e != hipSuccess) return e;
    allocs.push_back(q);
    bytes += n;
    if (zero) {
      e = hipMemset(q, 0, n ? n : 16);
      if (e != hipSuccess) return e;
    }
    *p = static_cast<T*>(q);
    return hipSuccess;
  }
};

namespace {

int CheckRows(const mi355x_search_ctx* ctx, int rows, int vocab) {
  if (!ctx) return Fail(MI355X_E_INVALID, "null context");
  if (rows <= 0 || vocab <= 0) return Fail(MI355X_E_INVALID, "rows (%d) and vocab (%d) must be positive", rows, vocab);
  if (rows > ctx->max_rows || vocab > ctx->max_vocab)
    return Fail(MI355X_E_CAPACITY, "rows=%d vocab=%d exceed the context's capacity (%d, %d)", rows, vocab,
                ctx->max_rows, ctx->max_vocab);
  return MI355X_OK;
}

// Validates the caller's logits-processing request and turns it into the kernels' form.  With a
// no-repeat-n-gram size it also launches the kernel that writes the rows' banned-id bitmaps into
// the context's workspace.
int MakeXform(mi355x_search_ctx* ctx, const mi355x_logits_xform* in, int rows, int vocab, hipStream_t stream,
              ms::Xform* out) {
  return ms_make_xform(ctx, in, rows, vocab, stream, out);
}

}  // namespace

// `ctx` may be null (an entry point without a context): the n-gram rule, whose bitmaps live in a
// context's workspace, is then refused.
int ms_make_xform(mi355x_search_ctx* ctx, const mi355x_logits_xform* in, int rows, int vocab, hipStream_t stream,
                  ms::Xform* out) {
  std::memset(out, 0, sizeof(*out));
  out->penalty = 1.0f;
  if (!in) return MI355X_OK;
  out->mask = in->mask;
  out->history = in->history;
  out->history_stride = in->history_stride;
  out->history_len = in->history_len;
  out->history_lens = in->history ? in->history_lens : nullptr;
  out->min_length = in->min_length;
  out->penalty = in->repetition_penalty;
  if (in->history && !in->history_lens && in->history_stride != 0 && in->history_len > in->history_stride)
    return Fail(MI355X_E_INVALID, "history_len (%d) exceeds history_stride (%d)", in->history_len, in->history_stride);
  if (in->history_len < 0 || in->history_stride < 0) return Fail(MI355X_E_INVALID, "negative history_len or history_stride");
  if (in->history_lens && !in->history) return Fail(MI355X_E_INVALID, "history_lens given without history");
  if (in->apply_min_length || (in->history_lens && in->min_length > 0)) {
    if (in->n_eos < 0 || in->n_eos > MI355X_MAX_EOS)
      return Fail(MI355X_E_INVALID, "n_eos (%d) out of range [0, %d]", in->n_eos, MI355X_MAX_EOS);
    out->n_eos = in->n_eos;
    for (int i = 0; i < in->n_eos; ++i) out->eos[i] = in->eos_ids[i];
  }
  if (in->no_repeat_ngram_size > 0) {
    if (!in->history) return Fail(MI355X_E_INVALID, "no_repeat_ngram_size needs a history");
    if (!ctx) return Fail(MI355X_E_UNSUPPORTED, "no_repeat_ngram_size needs a context (its bitmaps live in the workspace)");
    if (out->history_lens || out->history_len >= in->no_repeat_ngram_size) {
      HIP_TRY(ms_launch_ngram_ban(out, rows, vocab, in->no_repeat_ngram_size, ctx->ban, stream));
      out->ban = ctx->ban;
    }
  }
  return MI355X_OK;
}

// small_k: every row is one of top-k (k <= 64) or argmax.
void PlanStream(const mi355x_search_ctx* ctx, ms::SampleArgs* a, bool small_k) {
  const bool sixteen_bit = a->dtype == MI355X_F16 || a->dtype == MI355X_BF16;
  const ms::StreamPlan plan =
      ms::plan_stream({a->rows, a->vocab, small_k, a->emit_topk == ms::kEmitArgmax, sixteen_bit, a->xf.active()}, ctx->cand_lists);
  a->chunk_room = plan.room;
  a->chunk_elems = plan.elems;
  a->chunks = plan.chunks;
  a->rows_first = plan.rows_first ? 1 : 0;
}

extern "C" {

const char* mi355x_search_last_error(void) { return g_error.c_str(); }

int mi355x_search_create(int device, int max_rows, int max_vocab, mi355x_search_ctx** out) {
  if (!out) return Fail(MI355X_E_INVALID, "null output pointer");
  *out = nullptr;
  if (max_rows <= 0 || max_vocab <= 0) return Fail(MI355X_E_INVALID, "max_rows and max_vocab must be positive");
  int count = 0;
  HIP_TRY(hipGetDeviceCount(&count));
  if (device < 0 || device >= count) return Fail(MI355X_E_INVALID, "device %d out of range (%d visible)", device, count);
  HIP_TRY(hipSetDevice(device));
  hipDeviceProp_t prop;
  HIP_TRY(hipGetDeviceProperties(&prop, device));
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return Fail(MI355X_E_UNSUPPORTED, "kernels are built for gfx950 only; device %d is %s", device, prop.gcnArchName);
  auto* c = new (std::nothrow) mi355x_search_ctx;
  if (!c) return Fail(MI355X_E_INVALID, "out of host memory");
  c->device = device;
  c->max_rows = max_rows;
  c->max_vocab = max_vocab;
  c->max_chunks = (max_vocab + ms::kChunk - 1) / ms::kChunk;
  const size_t rc = static_cast<size_t>(max_rows) * c->max_chunks;
  c->big_stride = static_cast<size_t>(NextPow2(max_vocab));
  if (c->big_stride < static_cast<size_t>(c->max_chunks) * ms::kChunk) c->big_stride = static_cast<size_t>(c->max_chunks) * ms::kChunk;
  if (c->big_stride < static_cast<size_t>(ms::kSChunk)) c->big_stride = ms::kSChunk;
  hipError_t e = hipSuccess;
  auto ok = [&](hipError_t r) {
    if (e == hipSuccess) e = r;
  };
  c->cand_lists = ms::stream_lists(max_rows, max_vocab);
  ok(c->Alloc(&c->cand_small, c->cand_lists * ms::kSmallCap, true));  // all-zero between launches
  ok(c->Alloc(&c->chunk_cnt, rc, true));
  ok(c->Alloc(&c->chunk_max, rc, true));
  ok(c->Alloc(&c->chunk_thr, rc, true));
  ok(c->Alloc(&c->chunk_next, rc, true));
  ok(c->Alloc(&c->row_arrive, static_cast<size_t>(max_rows), true));
  ok(c->Alloc(&c->row_best, static_cast<size_t>(max_rows), true));
  ok(c->Alloc(&c->big, static_cast<size_t>(max_rows) * c->big_stride, false));
  ok(c->Alloc(&c->big2, static_cast<size_t>(max_rows) * c->big_stride, false));
  ok(c->Alloc(&c->row_done, static_cast<size_t>(max_rows), true));
  ok(c->Alloc(&c->fallback_rows, 4, true));  // [0] rows finished by the exact path, [1] a wait gave up, [2] exact-sum segments and tiles whose wait gave up, [3] rows given back by a pick
  ok(c->Alloc(&c->ban, static_cast<size_t>(max_rows) * ((max_vocab - 1) / 32 + 1), false));
  ok(c->Alloc(&c->params_dev, static_cast<size_t>(max_rows), false));
  ok(c->Alloc(&c->beam_row_scores, static_cast<size_t>(max_rows) * ms::kBeamMaxCand, false));
  ok(c->Alloc(&c->beam_row_tokens, static_cast<size_t>(max_rows) * ms::kBeamMaxCand, false));
  // (segments of the exact sums; the tiles of rows sampled from the whole vocabulary are shorter and share the arrays)
  c->max_segs = (max_vocab + ms::kWideTile - 1) / ms::kWideTile;
  static_assert(ms::kWideTile <= ms::kSegElems, "room for either");
  ok(c->Alloc(&c->wide_rows, static_cast<size_t>(max_rows), false));
  const size_t tile_starts = static_cast<size_t>(max_rows) * (c->max_segs + 1);
  ok(c->Alloc(&c->wide_tile_start, tile_starts, false));
  ok(c->Alloc(&c->wide_rest, 2 + static_cast<size_t>(max_rows) * (2 + ms::kRestStride), false));
  ok(c->Alloc(&c->wide_cut_bucket, static_cast<size_t>(max_rows) * (c->max_segs + 1), false));
  ok(c->Alloc(&c->seg_max, static_cast<size_t>(max_rows) * c->max_segs, false));
  ok(c->Alloc(&c->seg_sum, static_cast<size_t>(max_rows) * c->max_segs, false));
  // "not written yet" everywhere (all bits set): the state the exact-sum kernels expect and leave behind
  if (c->seg_sum) ok(hipMemset(c->seg_sum, 0xff, static_cast<size_t>(max_rows) * c->max_segs * sizeof(double)));
  ok(c->Alloc(&c->seg_cand, static_cast<size_t>(max_rows) * c->max_segs * ms::kBeamMaxCand, false));
  ok(c->Alloc(&c->seg_step, static_cast<size_t>(max_rows) * c->max_segs, false));
  ok(c->Alloc(&c->sub_step, static_cast<size_t>(max_rows) * c->max_segs * ms::kSegSubs, false));
  ok(c->Alloc(&c->sub_se, static_cast<size_t>(max_rows) * c->max_segs * ms::kSegSubs, false));
  ok(c->Alloc(&c->row_max, static_cast<size_t>(max_rows), false));
  ok(c->Alloc(&c->row_sum, static_cast<size_t>(max_rows), false));
  c->stage_slot_bytes = (static_cast<size_t>(max_rows) * sizeof(mi355x_sample_params) + 255) & ~static_cast<size_t>(255);
  if (e == hipSuccess) {
    void* pinned = nullptr;
    const size_t slots = c->stage_slot_bytes * (mi355x_search_ctx::kStageRing + mi355x_search_ctx::kStageCaptured);
    e = hipHostMalloc(&pinned, slots, hipHostMallocDefault);
    c->stage = static_cast<char*>(pinned);
  }
  if (e == hipSuccess) {
    c->scorer_host = std::make_shared<ScorerHost>();
    e = c->scorer_host->Allocate();
  }
  for (int i = 0; i < mi355x_search_ctx::kStageRing && e == hipSuccess; ++i)
    e = hipEventCreateWithFlags(&c->stage_event[i], hipEventDisableTiming);
  if (e == hipSuccess) e = ms_sample_init();
  if (e == hipSuccess) e = ms_static_scratch_setup();  // set-up of mi355x_argmax_static on this device
  // the fills above ran on the null stream: done before a caller's stream, which need not wait for it, uses them
  if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
  if (e != hipSuccess) {
    mi355x_search_destroy(c);
    return Fail(MI355X_E_HIP, "workspace allocation failed: %s", hipGetErrorString(e));
  }
  *out = c;
  return MI355X_OK;
}

void mi355x_search_destroy(mi355x_search_ctx* ctx) {
  if (!ctx) return;
  (void)hipSetDevice(ctx->device);
  for (void* p : ctx->allocs) (void)hipFree(p);
  for (hipEvent_t ev : ctx->stage_event)
    if (ev) (void)hipEventDestroy(ev);
  if (ctx->stage) (void)hipHostFree(ctx->stage);
  delete ctx;
}

size_t mi355x_search_workspace_bytes(const mi355x_search_ctx* ctx) { return ctx ? ctx->bytes : 0; }

int mi355x_search_abi_version(void) { return MI355X_ABI_VERSION; }

int mi355x_process_logits(mi355x_search_ctx* ctx, void* stream, float* logits, int64_t row_stride, int rows,
                          int vocab, const mi355x_logits_xform* xf) {
  if (int r = CheckRows(ctx, rows, vocab)) return r;
  if (!logits) return Fail(MI355X_E_INVALID, "null logits");
  if (row_stride < vocab) return Fail(MI355X_E_INVALID, "row_stride (%lld) smaller than vocab (%d)", (long long)row_stride, vocab);
  ms::Xform x;
  if (int r = MakeXform(ctx, xf, rows, vocab, static_cast<hipStream_t>(stream), &x)) return r;
  if (!x.active()) return MI355X_OK;
  HIP_TRY(ms_launch_process_logits(logits, row_stride, rows, vocab, &x, static_cast<hipStream_t>(stream)));
  return MI355X_OK;
}

int mi355x_argmax(mi355x_search_ctx* ctx, void* stream, const void* logits, int dtype, int64_t row_stride,
                  int rows, int vocab, const mi355x_logits_xform* xf, int32_t* out_tokens) {
  if (int r = CheckRows(ctx, rows, vocab)) return r;
  if (!logits || !out_tokens) return Fail(MI355X_E_INVALID, "null logits or output");
  if (dtype != MI355X_F32 && dtype != MI355X_F16 && dtype != MI355X_BF16)
    return Fail(MI355X_E_UNSUPPORTED, "dtype %d not supported", dtype);
  if (row_stride < vocab) return Fail(MI355X_E_INVALID, "row_stride smaller than vocab");
  // rows of more than 64 logits go through the fused selection kernel (k = 1, ids only), whatever their type
  const bool fused = vocab > 64 && vocab <= ms::kStreamMaxVocab;
  if (fused) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    ms::SampleArgs f{};
    if (int r = MakeXform(ctx, xf, rows, vocab, s, &f.xf)) return r;
    f.logits = logits;
    f.dtype = dtype;
    f.row_stride = row_stride;
    f.rows = rows;
    f.vocab = vocab;
    f.uniform = mi355x_sample_params{1, 0.0f, 1.0f};
    f.out_tokens = out_tokens;
    f.emit_topk = ms::kEmitArgmax;
    PlanStream(ctx, &f, true);
    f.cand_small = ctx->cand_small;
    f.chunk_cnt = ctx->chunk_cnt;
    f.chunk_max = ctx->chunk_max;
    f.chunk_thr = ctx->chunk_thr;
    f.chunk_next = ctx->chunk_next;
    f.big = ctx->big;
    f.big_stride = ctx->big_stride;
    f.fallback_rows = ctx->fallback_rows;
    f.poll_limit = ctx->poll_limit;
    HIP_TRY(ms_launch_sample(&f, nullptr, true, false, false, s, nullptr));
    return MI355X_OK;
  }
  ms::ArgmaxArgs a{};
  if (int r = MakeXform(ctx, xf, rows, vocab, static_cast<hipStream_t>(stream), &a.xf)) return r;
  a.logits = logits;
  a.row_stride = row_stride;
  a.rows = rows;
  a.vocab = vocab;
  a.chunks = (vocab + ms::kChunk - 1) / ms::kChunk;
  a.out_tokens = out_tokens;
  a.row_best = ctx->row_best;
  a.row_arrive = ctx->row_arrive;
  HIP_TRY(ms_launch_argmax(&a, dtype, static_cast<hipStream_t>(stream)));
  return MI355X_OK;
}

int mi355x_sample(mi355x_search_ctx* ctx, void* stream, const float* logits, int64_t row_stride, int rows,
                  int vocab, const mi355x_logits_xform* xf, mi355x_sample_params params,
                  const mi355x_sample_params* per_row_params, const double* uniforms, int32_t* out_tokens,
                  int32_t* kept_count, int32_t* kept_ids, float* kept_probs, int kept_capacity) {
  return mi355x_sample_typed(ctx, stream, logits, MI355X_F32, row_stride, rows, vocab, xf, params, per_row_params,
                             uniforms, out_tokens, kept_count, kept_ids, kept_probs, kept_capacity);
}

namespace {

// True while `s` records into a graph: an entry point that reads a caller's HOST array with an asynchronous copy
// would leave a node that reads that array again at every replay.
bool Capturing(hipStream_t s) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(s, &status) == hipSuccess && status != hipStreamCaptureStatusNone;
}

// A captured call that takes a table from a caller's host array counts against the context's bound on such calls,
// whether its table needs a permanent staging slot or travels inside the kernel arguments.
int TakeCapturedSlot(mi355x_search_ctx* ctx, int* slot) {
  if (ctx->stage_captured == mi355x_search_ctx::kStageCaptured)
    return Fail(MI355X_E_UNSUPPORTED, "this context has staged %d host tables for graph capture, all it provides for",
                mi355x_search_ctx::kStageCaptured);
  *slot = mi355x_search_ctx::kStageRing + ctx->stage_captured++;
  return MI355X_OK;
}

// Records a copy of `bytes` bytes of the caller's host array `src` to the device table `dst` on stream s, through a
// pinned staging slot of the context (see mi355x_search_ctx::stage).
int StageToDevice(mi355x_search_ctx* ctx, hipStream_t s, void* dst, const void* src, size_t bytes) {
  if (bytes > ctx->stage_slot_bytes) return Fail(MI355X_E_CAPACITY, "a host table of %zu bytes exceeds the staging slot", bytes);
  const bool capturing = Capturing(s);
  int slot;
  if (capturing) {
    if (int rc = TakeCapturedSlot(ctx, &slot)) return rc;
  } else {
    slot = ctx->stage_next;
    ctx->stage_next = (slot + 1) % mi355x_search_ctx::kStageRing;
    if (ctx->stage_pending[slot]) HIP_TRY(hipEventSynchronize(ctx->stage_event[slot]));
  }
  char* pinned = ctx->stage + static_cast<size_t>(slot) * ctx->stage_slot_bytes;
  std::memcpy(pinned, src, bytes);
  HIP_TRY(hipMemcpyAsync(dst, pinned, bytes, hipMemcpyHostToDevice, s));
  if (!capturing) {
    HIP_TRY(hipEventRecord(ctx->stage_event[slot], s));
    ctx->stage_pending[slot] = true;
  }
  return MI355X_OK;
}

// One launch set of the sampling path.  Rows lie row_stride elements apart from `logits`, or -- row_ptrs not
// null, at most kInlineParamRows rows -- start at the device pointers row_ptrs[0 .. rows).
int SampleImpl(mi355x_search_ctx* ctx, hipStream_t s, const void* logits, const void* const* row_ptrs, int dtype,
               int64_t row_stride, int rows, int vocab, const mi355x_logits_xform* xf, mi355x_sample_params params,
               const mi355x_sample_params* per_row_params, const double* uniforms, int32_t* out_tokens,
               int32_t* kept_count, int32_t* kept_ids, float* kept_probs, int kept_capacity, bool kept_pad) {
  ms::SampleArgs a{};
  if (int r = MakeXform(ctx, xf, rows, vocab, s, &a.xf)) return r;
  bool any_nucleus = false, any_other = false, any_large_k = false, any_exact = false, any_wide = false, any_pick = false;
  ms::InlineParams table{};
  bool use_table = false;
  // Sampling from the whole vocabulary is spread over the GPU wherever its kernels can take the row as it lies: no
  // logits processing, a row long enough to cut up, no more tiles than the finishing workgroup holds.
  const int tiles = (vocab + ms::kWideTile - 1) / ms::kWideTile;
  const bool wide_fits = vocab >= ms::kWideMinVocab && tiles <= ms::kWideMaxTiles && vocab <= ms::kStreamMaxVocab && !a.xf.active();
  auto check = [&](const mi355x_sample_params& p) -> int {
    if (!(p.temperature > 0.0f)) return Fail(MI355X_E_INVALID, "temperature must be positive (got %g)", p.temperature);
    // the kernels' own rule (row_mode) decides; these flags only have to cover it
    const int kk = p.k < vocab ? p.k : vocab;
    const bool fits = vocab > 64 && vocab <= ms::kStreamMaxVocab;
    const bool whole = p.k <= 1 && !(p.p < 1.0f);  // no top-k and no nucleus: the whole vocabulary
    const bool nucleus = p.k <= 1 && !whole, large_k = p.k > 1 && kk > 64 && kk <= ms::kLargeKMax;
    if (nucleus && vocab > 64) any_nucleus = true;
    if (large_k && vocab > 64) any_large_k = true;
    if (large_k && kk > 4 * ms::kLargeKOneOffer) a.all_offers = 1;
    if (whole && wide_fits) {
      any_wide = true;
      any_pick |= p.p == 1.0f;  // (a pick gives back what lies above one: p = 1.5, 256 x 32064 fp32 279 us with a pick, 151 without)
    } else if (vocab > 64 && (!fits || whole || (p.k > 1 && kk > ms::kLargeKMax))) any_exact = true;
    else if (!((nucleus || large_k) && fits)) any_other = true;
    return MI355X_OK;
  };
  if (per_row_params) {
    for (int r = 0; r < rows; ++r)
      if (int rc = check(per_row_params[r])) return rc;
  } else {
    if (int rc = check(params)) return rc;
  }
  if (row_ptrs || (per_row_params && rows <= ms::kInlineParamRows)) {
    for (int r = 0; r < rows; ++r) {
      table.row[r] = per_row_params ? per_row_params[r] : params;
      table.row_ptr[r] = row_ptrs ? row_ptrs[r] : nullptr;
    }
    use_table = true;
  } else if (per_row_params) {
    if (int rc = StageToDevice(ctx, s, ctx->params_dev, per_row_params, sizeof(mi355x_sample_params) * rows)) return rc;
    a.per_row = ctx->params_dev;
  }
  a.logits = row_ptrs ? row_ptrs[0] : logits;
  a.dtype = dtype;
  a.row_stride = row_stride;
  a.rows = rows;
  a.vocab = vocab;
  a.uniform = params;
  a.uniforms = uniforms;
  a.out_tokens = out_tokens;
  a.kept_count = kept_count;
  a.kept_ids = kept_ids;
  a.kept_probs = kept_probs;
  a.kept_capacity = kept_capacity;
  a.kept_pad = kept_pad ? 1 : 0;
  a.cand_small = ctx->cand_small;
  a.chunk_cnt = ctx->chunk_cnt;
  a.chunk_max = ctx->chunk_max;
  a.chunk_thr = ctx->chunk_thr;
  a.chunk_next = ctx->chunk_next;
  a.big = ctx->big;
  a.big2 = ctx->big2;
  a.big_stride = ctx->big_stride;
  a.fallback_rows = ctx->fallback_rows;
  a.poll_limit = ctx->poll_limit;
  a.row_done = ctx->row_done;
  PlanStream(ctx, &a, !any_nucleus && !any_large_k);
  a.exact_kernel = (any_exact ? ms::kExactRows : 0) | (any_wide ? ms::kWideRows : 0);
  const ms::WideArgs wide{(vocab + ms::kWideChunk - 1) / ms::kWideChunk, tiles, ctx->wide_rows, ctx->wide_tile_start, ctx->wide_cut_bucket, ctx->seg_sum,
                          ctx->seg_step, ctx->sub_step, ctx->sub_se, ctx->chunk_next, any_pick && kept_ids == nullptr && kept_count == nullptr,
                          {ctx->wide_rest, ctx->wide_rest + 1, ctx->wide_rest + 2, ctx->wide_rest + 2 + ctx->max_rows, ctx->wide_rest + 2 + 2 * static_cast<size_t>(ctx->max_rows)}};
  // a caller that bounds the number of allowed ids per row lets the sparse-mask kernel work alone
  if (xf && xf->mask && xf->mask_allowed_max > 0) {
    const int hist = a.xf.history_lens ? a.xf.history_stride : a.xf.history_len;
    const int64_t listed = static_cast<int64_t>(xf->mask_allowed_max) + (a.xf.use_penalty() ? hist : 0) + 2;
    a.sparse_only = listed <= ms::kNucleusCap && hist <= 2048 ? static_cast<int>(listed) : 0;  // (what the kernel can list; beyond, all three kernels)
  }
  HIP_TRY(ms_launch_sample(&a, use_table ? &table : nullptr, any_other, any_nucleus, any_large_k, s, &wide));
  return MI355X_OK;
}

int CheckSampleArgs(int dtype, const double* uniforms, const int32_t* out_tokens, const int32_t* kept_ids,
                    const float* kept_probs, int kept_capacity) {
  if (!uniforms || !out_tokens) return Fail(MI355X_E_INVALID, "null logits, uniforms or output");
  if (dtype != MI355X_F32 && dtype != MI355X_F16 && dtype != MI355X_BF16)
    return Fail(MI355X_E_UNSUPPORTED, "dtype %d not supported", dtype);
  if ((kept_ids || kept_probs) && kept_capacity <= 0) return Fail(MI355X_E_INVALID, "kept_capacity must be positive");
  if (kept_probs && !kept_ids) return Fail(MI355X_E_INVALID, "kept_probs requires kept_ids");
  return MI355X_OK;
}

int SampleRows(mi355x_search_ctx* ctx, void* stream, const void* logits, int dtype, int64_t row_stride, int rows, int vocab,
               const mi355x_logits_xform* xf, mi355x_sample_params params, const mi355x_sample_params* per_row_params,
               const double* uniforms, int32_t* out_tokens, int32_t* kept_count, int32_t* kept_ids, float* kept_probs,
               int kept_capacity, bool kept_pad) {
  if (int r = CheckRows(ctx, rows, vocab)) return r;
  if (!logits) return Fail(MI355X_E_INVALID, "null logits, uniforms or output");
  if (int r = CheckSampleArgs(dtype, uniforms, out_tokens, kept_ids, kept_probs, kept_capacity)) return r;
  if (row_stride < vocab) return Fail(MI355X_E_INVALID, "row_stride smaller than vocab");
  return SampleImpl(ctx, static_cast<hipStream_t>(stream), logits, nullptr, dtype, row_stride, rows, vocab, xf, params,
                    per_row_params, uniforms, out_tokens, kept_count, kept_ids, kept_probs, kept_capacity, kept_pad);
}

int SampleScattered(mi355x_search_ctx* ctx, void* stream, const void* const* row_ptrs, int dtype, int rows, int vocab,
                    const mi355x_logits_xform* xf, mi355x_sample_params params, const mi355x_sample_params* per_row_params,
                    const double* uniforms, int32_t* out_tokens, int32_t* kept_count, int32_t* kept_ids, float* kept_probs,
                    int kept_capacity, bool kept_pad) {
  if (int r = CheckRows(ctx, rows, vocab)) return r;
  if (!row_ptrs) return Fail(MI355X_E_INVALID, "null row pointer array");
  for (int r = 0; r < rows; ++r)
    if (!row_ptrs[r]) return Fail(MI355X_E_INVALID, "row %d has a null pointer", r);
  if (int r = CheckSampleArgs(dtype, uniforms, out_tokens, kept_ids, kept_probs, kept_capacity)) return r;
  const int words = (vocab - 1) / 32 + 1;
  // the row pointers travel inside the kernel arguments, kInlineParamRows rows per launch
  for (int r0 = 0; r0 < rows; r0 += ms::kInlineParamRows) {
    const int n = rows - r0 < ms::kInlineParamRows ? rows - r0 : ms::kInlineParamRows;
    mi355x_logits_xform part;
    if (xf) {
      part = *xf;
      if (part.mask) part.mask += static_cast<size_t>(r0) * words;
      if (part.history) part.history += static_cast<size_t>(r0) * part.history_stride;
      if (part.history_lens) part.history_lens += r0;
    }
    if (int rc = SampleImpl(ctx, static_cast<hipStream_t>(stream), nullptr, row_ptrs + r0, dtype, vocab, n, vocab,
                            xf ? &part : nullptr, params, per_row_params ? per_row_params + r0 : nullptr, uniforms + r0,
                            out_tokens + r0, kept_count ? kept_count + r0 : nullptr,
                            kept_ids ? kept_ids + static_cast<size_t>(r0) * kept_capacity : nullptr,
                            kept_probs ? kept_probs + static_cast<size_t>(r0) * kept_capacity : nullptr, kept_capacity, kept_pad))
      return rc;
  }
  return MI355X_OK;
}

}  // namespace

int mi355x_sample_typed(mi355x_search_ctx* ctx, void* stream, const void* logits, int dtype, int64_t row_stride,
                        int rows, int vocab, const mi355x_logits_xform* xf, mi355x_sample_params params,
                        const mi355x_sample_params* per_row_params, const double* uniforms, int32_t* out_tokens,
                        int32_t* kept_count, int32_t* kept_ids, float* kept_probs, int kept_capacity) {
  return SampleRows(ctx, stream, logits, dtype, row_stride, rows, vocab, xf, params, per_row_params, uniforms, out_tokens,
                    kept_count, kept_ids, kept_probs, kept_capacity, false);
}

int mi355x_sample_scattered(mi355x_search_ctx* ctx, void* stream, const void* const* row_ptrs, int dtype, int rows,
                            int vocab, const mi355x_logits_xform* xf, mi355x_sample_params params,
                            const mi355x_sample_params* per_row_params, const double* uniforms, int32_t* out_tokens,
                            int32_t* kept_count, int32_t* kept_ids, float* kept_probs, int kept_capacity) {
  return SampleScattered(ctx, stream, row_ptrs, dtype, rows, vocab, xf, params, per_row_params, uniforms, out_tokens, kept_count,
                         kept_ids, kept_probs, kept_capacity, false);
}

// mi355x_sample_typed, or mi355x_sample_scattered where row_ptrs is given, whose kept ids and probabilities are padded
// with -1 and 0 up to the capacity (the Python binding's form: a fill of each by launches of their own costs two).
int ms_sample_padded(mi355x_search_ctx* ctx, void* stream, const void* logits, const void* const* row_ptrs, int dtype,
                     int64_t row_stride, int rows, int vocab, const mi355x_logits_xform* xf, mi355x_sample_params params,
                     const mi355x_sample_params* per_row_params, const double* uniforms, int32_t* out_tokens, int32_t* kept_count,
                     int32_t* kept_ids, float* kept_probs, int kept_capacity) {
  if (row_ptrs)
    return SampleScattered(ctx, stream, row_ptrs, dtype, rows, vocab, xf, params, per_row_params, uniforms, out_tokens, kept_count,
                           kept_ids, kept_probs, kept_capacity, true);
  return SampleRows(ctx, stream, logits, dtype, row_stride, rows, vocab, xf, params, per_row_params, uniforms, out_tokens, kept_count,
                    kept_ids, kept_probs, kept_capacity, true);
}

// Copies 32-bit words between buffers of one device, behind the work of `stream`, and waits for it: what the Python
// binding hands out as the scorer's state is complete when the caller has it, on any stream.
int ms_copy_words_and_wait(void* stream, void* dst, const void* src, size_t words) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (Capturing(s))
    return Fail(MI355X_E_UNSUPPORTED, "a copy of a scorer's state is complete on return: it cannot be recorded into a graph");
  if (words != 0) HIP_TRY(ms_launch_copy_words(static_cast<const uint32_t*>(src), static_cast<uint32_t*>(dst), words, s));
  HIP_TRY(hipStreamSynchronize(s));
  return MI355X_OK;
}

int mi355x_topk_scores(mi355x_search_ctx* ctx, void* stream, const void* logits, int dtype, int64_t row_stride,
                       int rows, int vocab, int k, int32_t* out_tokens, float* out_scores) {
  if (int r = CheckRows(ctx, rows, vocab)) return r;
  if (!logits || !out_tokens || !out_scores) return Fail(MI355X_E_INVALID, "null logits or output");
  if (dtype != MI355X_F32 && dtype != MI355X_F16 && dtype != MI355X_BF16)
    return Fail(MI355X_E_UNSUPPORTED, "dtype %d not supported", dtype);
  if (k < 1 || k > vocab) return Fail(MI355X_E_INVALID, "k (%d) must be in [1, vocab]", k);
  if (row_stride < vocab) return Fail(MI355X_E_INVALID, "row_stride smaller than vocab");
  hipStream_t s = static_cast<hipStream_t>(stream);
  // sixteen-bit rows are read as they are and widened in registers (DeviceInterface::TopKScores makes an fp32
  // copy first, src/cuda/interface.cpp:440-451); the scores returned are the widened values
  ms::SampleArgs a{};
  if (int r = MakeXform(ctx, nullptr, rows, vocab, s, &a.xf)) return r;
  a.logits = logits;
  a.dtype = dtype;
  a.row_stride = row_stride;
  a.rows = rows;
  a.vocab = vocab;
  a.uniform = mi355x_sample_params{k, 0.0f, 1.0f};
  a.out_tokens = out_tokens;
  a.out_scores = out_scores;
  a.emit_topk = 1;
  a.cand_small = ctx->cand_small;
  a.chunk_cnt = ctx->chunk_cnt;
  a.chunk_max = ctx->chunk_max;
  a.chunk_thr = ctx->chunk_thr;
  a.chunk_next = ctx->chunk_next;
  a.big = ctx->big;
  a.big2 = ctx->big2;
  a.big_stride = ctx->big_stride;
  a.fallback_rows = ctx->fallback_rows;
  a.poll_limit = ctx->poll_limit;
  // up to 64: the fused kernel's sorted candidate lists; up to kLargeKMax: the candidate lists of the large-k
  // sampling route with an epilogue that emits instead of drawing; beyond (and for rows of more chunks than a
  // finishing workgroup ranks): the exact path's whole-row sort.  The kernels' own rule (row_mode) decides.
  const bool fits = vocab > 64 && vocab <= ms::kStreamMaxVocab;
  const bool large_k = fits && k > 64 && k <= ms::kLargeKMax;
  const bool exact = vocab > 64 && (!fits || k > ms::kLargeKMax);
  a.exact_kernel = exact ? ms::kExactRows : 0;
  a.all_offers = k > 4 * ms::kLargeKOneOffer ? 1 : 0;
  PlanStream(ctx, &a, !large_k);
  HIP_TRY(ms_launch_sample(&a, nullptr, !large_k && !exact, false, large_k, s, nullptr));
  return MI355X_OK;
}

// Fills the argument block of the multi-workgroup sequential sum when the shape calls for it and the
// context's workspace covers it.
static bool FillSeqSum(mi355x_search_ctx* ctx, const void* x, int64_t row_stride, int rows, int vocab, float inv_temp,
                       ms::SeqSumArgs* q) {
  const int segs = (vocab + ms::kSegElems - 1) / ms::kSegElems;
  if (vocab < ms::kSeqSumMinVocab || rows > ctx->max_rows || vocab > ctx->max_vocab || segs > ms::kMaxSegs) return false;
  q->x = x;
  q->row_stride = row_stride;
  q->rows = rows;
  q->vocab = vocab;
  q->segs = segs;
  q->inv_temp = inv_temp;
  q->seg_max = ctx->seg_max;
  q->seg_sum = ctx->seg_sum;
  q->seg_step = ctx->seg_step;
  q->sub_step = ctx->sub_step;
  q->sub_se = ctx->sub_se;
  q->out_max = ctx->row_max;
  q->out_sum = ctx->row_sum;
  q->poll_limit = ctx->poll_limit;
  q->gave_up = ctx->fallback_rows + 2;
  return true;
}

int mi355x_softmax(mi355x_search_ctx* ctx, void* stream, float* scores, int64_t row_stride, int rows, int vocab,
                   float temperature, int log_softmax) {
  if (!ctx) return Fail(MI355X_E_INVALID, "null context");
  if (!scores || rows <= 0 || vocab <= 0) return Fail(MI355X_E_INVALID, "null scores or non-positive size");
  if (row_stride < vocab) return Fail(MI355X_E_INVALID, "row_stride smaller than vocab");
  if (!(temperature > 0.0f)) return Fail(MI355X_E_INVALID, "temperature must be positive (got %g)", temperature);
  hipStream_t s = static_cast<hipStream_t>(stream);
  ms::SeqSumArgs q{};
  if (FillSeqSum(ctx, scores, row_stride, rows, vocab, 1.0f / temperature, &q)) {
    // long rows: the exact sum is spread over the whole GPU, then an element-wise pass finishes
    HIP_TRY(ms_launch_seqsum(&q, MI355X_F32, s));
    HIP_TRY(ms_launch_softmax_apply(scores, row_stride, &q, log_softmax, s));
  } else {
    HIP_TRY(ms_launch_softmax(scores, row_stride, rows, vocab, temperature, log_softmax, s));
  }
  return MI355X_OK;
}

namespace {
// mi355x_beam_select; with `step`, the launch that finishes the selection also does the scorer step where the
// path taken has such a launch (*fused says whether it did).
int BeamSelectImpl(mi355x_search_ctx* ctx, void* stream, const void* logits, int dtype, int64_t row_stride,
                   int batch, int beams, int vocab, const float* beam_scores, float* out_scores,
                   int32_t* out_tokens, int32_t* out_beam_indices, const ms::ScorerStep* step, bool* fused) {
  if (batch <= 0 || beams <= 0) return Fail(MI355X_E_INVALID, "batch and beams must be positive");
  if (beams > ms::kBeamMaxCand / 2) return Fail(MI355X_E_UNSUPPORTED, "beams (%d) above the supported %d", beams, ms::kBeamMaxCand / 2);
  if (int r = CheckRows(ctx, batch * beams, vocab)) return r;
  if (!logits || !beam_scores || !out_scores || !out_tokens || !out_beam_indices)
    return Fail(MI355X_E_INVALID, "null argument");
  if (dtype != MI355X_F32 && dtype != MI355X_F16 && dtype != MI355X_BF16)
    return Fail(MI355X_E_UNSUPPORTED, "dtype %d not supported", dtype);
  if (row_stride < vocab) return Fail(MI355X_E_INVALID, "row_stride smaller than vocab");
  if (static_cast<long long>(beams) * vocab < 2LL * beams)
    return Fail(MI355X_E_INVALID, "beam search requires num_beams * vocab_size (%lld) >= 2 * num_beams (%d)",
                static_cast<long long>(beams) * vocab, 2 * beams);
  if (static_cast<unsigned long long>(beams) * static_cast<unsigned long long>(vocab) > 0xffffffffull)
    return Fail(MI355X_E_UNSUPPORTED, "beams * vocab exceeds 2^32");
  ms::BeamArgs a{};
  a.logits = logits;
  a.row_stride = row_stride;
  a.batch = batch;
  a.beams = beams;
  a.vocab = vocab;
  a.beam_scores = beam_scores;
  a.row_scores = ctx->beam_row_scores;
  a.row_tokens = ctx->beam_row_tokens;
  a.out_scores = out_scores;
  a.out_tokens = out_tokens;
  a.out_beams = out_beam_indices;
  ms::SeqSumArgs q{};
  if (FillSeqSum(ctx, logits, row_stride, batch * beams, vocab, 1.0f, &q)) {
    a.row_max = q.out_max;
    a.row_sum = q.out_sum;
    if (static_cast<long long>(beams) * q.segs * 2 * beams <= ms::kBeamFinCap) {
      // long rows: the segments list their best logits inside the launch that sums their exponentials, the
      // exact sums follow, and one workgroup per batch entry scores the listed candidates
      a.seg_cand = ctx->seg_cand;
      a.seg_max = q.seg_max;
      a.segs = q.segs;
      HIP_TRY(ms_launch_seqsum_max(&q, dtype, static_cast<hipStream_t>(stream)));
      HIP_TRY(ms_launch_beam_exp_step(&q, &a, dtype, static_cast<hipStream_t>(stream)));
      HIP_TRY(ms_launch_seqsum_walk(&q, dtype, static_cast<hipStream_t>(stream)));
      HIP_TRY(ms_launch_beam_finish(&a, dtype, step, static_cast<hipStream_t>(stream)));
      if (fused) *fused = step != nullptr;
      return MI355X_OK;
    }
    HIP_TRY(ms_launch_seqsum(&q, dtype, static_cast<hipStream_t>(stream)));
  }
  HIP_TRY(ms_launch_beam_select(&a, dtype, static_cast<hipStream_t>(stream)));
  return MI355X_OK;
}
}  // namespace

int mi355x_beam_select(mi355x_search_ctx* ctx, void* stream, const void* logits, int dtype, int64_t row_stride,
                       int batch, int beams, int vocab, const float* beam_scores, float* out_scores,
                       int32_t* out_tokens, int32_t* out_beam_indices) {
  return BeamSelectImpl(ctx, stream, logits, dtype, row_stride, batch, beams, vocab, beam_scores, out_scores, out_tokens,
                        out_beam_indices, nullptr, nullptr);
}

int mi355x_spec_verify_sparse(mi355x_search_ctx* ctx, void* stream, const int32_t* target_count,
                              const int32_t* target_ids, const float* target_probs, int target_capacity,
                              const int32_t* draft_count, const int32_t* draft_ids, const float* draft_probs,
                              int draft_capacity, const int32_t* proposal, const float* accept_u,
                              const double* sample_u, int batch, int K, int mode, int32_t* accepted_len,
                              int32_t* final_token, int32_t* engine_draws) {
  if (!ctx || !target_count || !target_ids || !proposal || !accepted_len || !final_token || !engine_draws)
    return Fail(MI355X_E_INVALID, "null argument");
  if (mode < 0 || mode > 2) return Fail(MI355X_E_INVALID, "mode (%d) must be 0, 1 or 2", mode);
  if (batch <= 0 || K < 1 || K > 64) return Fail(MI355X_E_INVALID, "batch (%d) must be positive and K (%d) in [1, 64]", batch, K);
  if (target_capacity <= 0) return Fail(MI355X_E_INVALID, "target_capacity must be positive");
  if (mode != 2 && (!target_probs || !sample_u)) return Fail(MI355X_E_INVALID, "null target_probs or sample_u");
  if (mode == 0 && (!draft_count || !draft_ids || !draft_probs || !accept_u || draft_capacity <= 0))
    return Fail(MI355X_E_INVALID, "mode 0 needs the draft distributions and accept_u");
  if (batch > ctx->max_rows) return Fail(MI355X_E_CAPACITY, "batch=%d exceeds the context's capacity (%d)", batch, ctx->max_rows);
  if (static_cast<size_t>(target_capacity) > 2 * ctx->big_stride)
    return Fail(MI355X_E_CAPACITY, "target_capacity=%d exceeds the context's workspace (%zu)", target_capacity, 2 * ctx->big_stride);
  ms::SpecSparseArgs a{};
  a.t_count = target_count;
  a.t_ids = target_ids;
  a.t_probs = target_probs;
  a.t_cap = target_capacity;
  a.d_count = draft_count;
  a.d_ids = draft_ids;
  a.d_probs = draft_probs;
  a.d_cap = draft_capacity;
  a.proposal = proposal;
  a.accept_u = accept_u;
  a.sample_u = sample_u;
  a.K = K;
  a.mode = mode;
  a.residual = reinterpret_cast<float*>(ctx->big);
  a.residual_stride = 2 * ctx->big_stride;
  a.accepted_len = accepted_len;
  a.final_token = final_token;
  a.engine_draws = engine_draws;
  HIP_TRY(ms_launch_spec_verify_sparse(&a, batch, static_cast<hipStream_t>(stream)));
  return MI355X_OK;
}

int mi355x_draw_in_order(mi355x_search_ctx* ctx, void* stream, const int32_t* kept_count, const int32_t* kept_ids,
                         const float* kept_probs, int kept_capacity, int rows, const int32_t* skip_rows,
                         const double* uniform_pool, int32_t* out_tokens, int32_t* draws_used) {
  if (!ctx || !kept_count || !kept_ids || !kept_probs || !uniform_pool || !out_tokens)
    return Fail(MI355X_E_INVALID, "null argument");
  if (rows <= 0 || kept_capacity <= 0) return Fail(MI355X_E_INVALID, "rows and kept_capacity must be positive");
  HIP_TRY(ms_launch_draw_in_order(kept_count, kept_ids, kept_probs, kept_capacity, rows, skip_rows, uniform_pool, out_tokens,
                                  draws_used, static_cast<hipStream_t>(stream)));
  return MI355X_OK;
}

int mi355x_greedy_tail(mi355x_search_ctx* ctx, void* stream, int32_t* next_tokens, int32_t* eos_seen, int batch,
                       const int32_t* eos_ids, int n_eos, int32_t pad_token_id, int32_t* sequences, int max_length,
                       int current_length, int32_t* done) {
  if (!ctx || !next_tokens || !eos_seen || !sequences || !done) return Fail(MI355X_E_INVALID, "null argument");
  if (batch <= 0 || max_length <= 0 || current_length < 0)
    return Fail(MI355X_E_INVALID, "batch (%d) and max_length (%d) must be positive, current_length (%d) not negative",
                batch, max_length, current_length);
  if (n_eos < 0 || n_eos > MI355X_MAX_EOS || (n_eos > 0 && !eos_ids))
    return Fail(MI355X_E_INVALID, "n_eos (%d) out of range [0, %d] or null eos_ids", n_eos, MI355X_MAX_EOS);
  HIP_TRY(ms_launch_greedy_tail(next_tokens, eos_seen, batch, eos_ids, n_eos, pad_token_id, sequences, max_length,
                                current_length, done, static_cast<hipStream_t>(stream)));
  return MI355X_OK;
}

int mi355x_cast(mi355x_search_ctx* ctx, void* stream, const void* in, int in_dtype, void* out, int out_dtype,
                size_t count) {
  if (!ctx || !in || !out) return Fail(MI355X_E_INVALID, "null argument");
  if (in_dtype == out_dtype) return Fail(MI355X_E_INVALID, "Cast - input and output types are the same");
  int kind = -1;
  if (in_dtype == MI355X_F16 && out_dtype == MI355X_F32) kind = 0;
  else if (in_dtype == MI355X_BF16 && out_dtype == MI355X_F32) kind = 1;
  else if (in_dtype == MI355X_F32 && out_dtype == MI355X_F16) kind = 2;
  else if (in_dtype == MI355X_F32 && out_dtype == MI355X_BF16) kind = 3;
  else if (in_dtype == MI355X_I32 && out_dtype == MI355X_I64) kind = 4;
  if (kind < 0) return Fail(MI355X_E_UNSUPPORTED, "cast from type %d to type %d is not implemented", in_dtype, out_dtype);
  if (count == 0) return MI355X_OK;
  HIP_TRY(ms_launch_cast(in, out, count, kind, static_cast<hipStream_t>(stream)));
  return MI355X_OK;
}

int mi355x_logits_handoff(mi355x_search_ctx* ctx, void* stream, const void* raw, int dtype, int rows, int seq_len,
                          int vocab, const int32_t* token_index, float* out, int64_t out_stride) {
  if (!ctx || !raw || !out) return Fail(MI355X_E_INVALID, "null argument");
  if (rows <= 0 || seq_len <= 0 || vocab <= 0) return Fail(MI355X_E_INVALID, "non-positive size");
  if (out_stride < vocab) return Fail(MI355X_E_INVALID, "out_stride smaller than vocab");
  if (rows > 65535) return Fail(MI355X_E_CAPACITY, "too many rows (%d)", rows);
  const int kind = dtype == MI355X_F16 ? 0 : dtype == MI355X_BF16 ? 1 : dtype == MI355X_F32 ? 2 : -1;
  if (kind < 0) return Fail(MI355X_E_UNSUPPORTED, "dtype %d not supported", dtype);
  if (token_index) {
    if (rows > ctx->max_rows) return Fail(MI355X_E_CAPACITY, "rows (%d) exceed the context's %d", rows, ctx->max_rows);
    for (int r = 0; r < rows; ++r)
      if (token_index[r] < 0 || token_index[r] >= seq_len)
        return Fail(MI355X_E_INVALID, "token_index[%d] = %d outside [0, %d)", r, token_index[r], seq_len);
  }
  if (int slot; token_index && Capturing(static_cast<hipStream_t>(stream)))
    if (int rc = TakeCapturedSlot(ctx, &slot)) return rc;
  // the positions travel inside the kernel arguments, kTokenIndexRows rows per launch
  const int per_launch = token_index ? ms::kTokenIndexRows : rows;
  const size_t row_bytes = static_cast<size_t>(seq_len) * vocab * (kind == 2 ? 4 : 2);
  for (int r0 = 0; r0 < rows; r0 += per_launch) {
    const int n = rows - r0 < per_launch ? rows - r0 : per_launch;
    ms::TokenIndex index;
    if (token_index) std::copy_n(token_index + r0, n, index.token);
    HIP_TRY(ms_launch_logits_handoff(&index, token_index ? 1 : 0, static_cast<const char*>(raw) + static_cast<size_t>(r0) * row_bytes, kind, n,
                                     seq_len, vocab, out + static_cast<size_t>(r0) * out_stride, out_stride, static_cast<hipStream_t>(stream)));
  }
  return MI355X_OK;
}

int mi355x_kv_gather(mi355x_search_ctx* ctx, void* stream, const void* const* present, void* const* past,
                     int n_tensors, const int32_t* beam_indices, int rows, size_t block_bytes) {
  if (!ctx || !present || !past || !beam_indices) return Fail(MI355X_E_INVALID, "null argument");
  if (n_tensors <= 0 || rows <= 0 || block_bytes == 0) return Fail(MI355X_E_INVALID, "non-positive size");
  if (n_tensors > 2048 || rows > 65535)
    return Fail(MI355X_E_CAPACITY, "too many tensors (%d) or rows (%d)", n_tensors, rows);
  // Widest power-of-two access (at most 16 bytes) that every block of every tensor is aligned to.
  uintptr_t align = static_cast<uintptr_t>(block_bytes);
  for (int t = 0; t < n_tensors; ++t) {
    if (!present[t] || !past[t]) return Fail(MI355X_E_INVALID, "null tensor pointer at %d", t);
    align |= reinterpret_cast<uintptr_t>(present[t]) | reinterpret_cast<uintptr_t>(past[t]);
  }
  int width = 16;
  while (align & static_cast<uintptr_t>(width - 1)) width >>= 1;
  if (int slot; Capturing(static_cast<hipStream_t>(stream)))
    if (int rc = TakeCapturedSlot(ctx, &slot)) return rc;
  // the addresses travel inside the kernel arguments, kKvTensors tensors per launch
  for (int t0 = 0; t0 < n_tensors; t0 += ms::kKvTensors) {
    const int n = n_tensors - t0 < ms::kKvTensors ? n_tensors - t0 : ms::kKvTensors;
    ms::KvTensors tensors;
    std::copy_n(present + t0, n, tensors.present);
    std::copy_n(past + t0, n, tensors.past);
    HIP_TRY(ms_launch_kv_gather(&tensors, n, beam_indices, rows, block_bytes, width, static_cast<hipStream_t>(stream)));
  }
  return MI355X_OK;
}

int mi355x_spec_verify(mi355x_search_ctx* ctx, void* stream, const float* p_target, const float* p_draft,
                       const int32_t* draft_tokens, const float* accept_u, const double* sample_u, int batch, int K,
                       int vocab, int32_t* accepted_len, int32_t* final_token) {
  if (!ctx || !p_target || !p_draft || !draft_tokens || !accept_u || !sample_u || !accepted_len || !final_token)
    return Fail(MI355X_E_INVALID, "null argument");
  if (batch <= 0 || K <= 0 || vocab < 2) return Fail(MI355X_E_INVALID, "batch, K must be positive and vocab >= 2");
  HIP_TRY(ms_launch_spec_verify(p_target, p_draft, draft_tokens, accept_u, sample_u, batch, K, vocab, accepted_len,
                                final_token, static_cast<hipStream_t>(stream)));
  return MI355X_OK;
}

int mi355x_search_fallback_rows(mi355x_search_ctx* ctx, void* stream, unsigned* rows) {
  if (!ctx || !rows) return Fail(MI355X_E_INVALID, "null argument");
  HIP_TRY(hipMemcpyAsync(rows, ctx->fallback_rows, sizeof(unsigned), hipMemcpyDeviceToHost,
                         static_cast<hipStream_t>(stream)));
  HIP_TRY(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
  return MI355X_OK;
}

int mi355x_search_wait_gave_up(mi355x_search_ctx* ctx, void* stream, int* gave_up) {
  if (!ctx || !gave_up) return Fail(MI355X_E_INVALID, "null argument");
  unsigned word = 0;
  HIP_TRY(hipMemcpyAsync(&word, ctx->fallback_rows + 1, sizeof(unsigned), hipMemcpyDeviceToHost,
                         static_cast<hipStream_t>(stream)));
  HIP_TRY(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
  *gave_up = word != 0u;
  return MI355X_OK;
}

int mi355x_search_sum_waits_gave_up(mi355x_search_ctx* ctx, void* stream, unsigned* segments) {
  if (!ctx || !segments) return Fail(MI355X_E_INVALID, "null argument");
  HIP_TRY(hipMemcpyAsync(segments, ctx->fallback_rows + 2, sizeof(unsigned), hipMemcpyDeviceToHost,
                         static_cast<hipStream_t>(stream)));
  HIP_TRY(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
  return MI355X_OK;
}

// How many rows whose token was to be picked (token_pick.h) have been given back to the way that orders them, modulo 2^32.
int ms_picks_given_back(mi355x_search_ctx* ctx, void* stream, unsigned* rows) {
  if (!ctx || !rows) return Fail(MI355X_E_INVALID, "null argument");
  HIP_TRY(hipMemcpyAsync(rows, ctx->fallback_rows + 3, sizeof(unsigned), hipMemcpyDeviceToHost, static_cast<hipStream_t>(stream)));
  HIP_TRY(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
  return MI355X_OK;
}

int mi355x_search_set_poll_limit(mi355x_search_ctx* ctx, int polls) {
  if (!ctx) return Fail(MI355X_E_INVALID, "null context");
  if (polls < 0) return Fail(MI355X_E_INVALID, "negative poll limit");
  ctx->poll_limit = polls;
  return MI355X_OK;
}

// ---- device-resident beam scorer ---------------------------------------------------------------------
struct mi355x_beam_scorer {
  mi355x_search_ctx* ctx{};
  ms::ScorerState st{};
  char* memory{};  // everything below, one allocation: creating eighteen of them and clearing each took 0.25 ms
  int32_t* seq[2]{};
  int cur{};
  int length{};
  bool finalized{};
  float* cand_scores{};    // [batch, 2*beams]: the candidates of mi355x_beam_search_step
  int32_t* cand_tokens{};
  int32_t* cand_beams{};
  // The hypotheses' lists as the device holds them after the finalisation, read back together by the first
  // mi355x_beam_scorer_hypothesis (and again after a further step): used counts, lengths, slots, scores -- and, where
  // they fit the readback area next to them, the tokens.
  size_t lists_bytes{}, tokens_bytes{};
  std::vector<char> lists;  // empty: not read back
  std::shared_ptr<ScorerHost> host;  // (only the search steps use `ctx` itself after the creation: it may be gone before the others)
  int done_word{-1};  // which of its words st.all_done is (-1: none, the count is read back)
};

int mi355x_beam_scorer_create(mi355x_search_ctx* ctx, int batch, int beams, int max_length, int pad_token_id,
                              const int32_t* eos_ids, int n_eos, float length_penalty, int early_stopping,
                              mi355x_beam_scorer** out) {
  if (!ctx || !out) return Fail(MI355X_E_INVALID, "null argument");
  *out = nullptr;
  if (batch <= 0 || beams <= 1 || max_length <= 0) return Fail(MI355X_E_INVALID, "batch, max_length must be positive and beams > 1");
  if (beams > ms::kBeamMaxCand / 2) return Fail(MI355X_E_UNSUPPORTED, "beams (%d) above the supported %d", beams, ms::kBeamMaxCand / 2);
  if (n_eos < 0 || n_eos > MI355X_MAX_EOS || (n_eos > 0 && !eos_ids)) return Fail(MI355X_E_INVALID, "bad eos list");
  HIP_TRY(hipSetDevice(ctx->device));
  auto* s = new (std::nothrow) mi355x_beam_scorer;
  if (!s) return Fail(MI355X_E_INVALID, "out of host memory");
  s->ctx = ctx;
  const size_t bb = static_cast<size_t>(batch) * beams, ranks = static_cast<size_t>(batch) * (beams + 1);
  ms::ScorerState& st = s->st;
  st.batch = batch;
  st.beams = beams;
  st.max_length = max_length;
  st.pad = pad_token_id;
  st.early_stopping = early_stopping != 0;
  st.n_eos = n_eos;
  for (int i = 0; i < n_eos; ++i) st.eos[i] = eos_ids[i];
  // Placed twice: to learn the size, and once there is memory.  The small arrays that start with something else than
  // zeros or are read back together come first.
  size_t at = 0, head_bytes = 0;
  float* pow_table = nullptr;
  auto place = [&](auto** p, size_t count) {
    at = (at + 255) & ~static_cast<size_t>(255);
    *p = reinterpret_cast<std::remove_reference_t<decltype(*p)>>(s->memory + at);
    at += count * sizeof(**p);
  };
  auto layout = [&] {
    at = 0;
    place(&st.hyp_used, batch);
    place(&st.hyp_len, bb);
    place(&st.hyp_slot, ranks);
    place(&st.hyp_score, bb);
    s->lists_bytes = at;
    place(&st.next_scores, bb);
    place(&st.not_done, 1);
    place(&pow_table, static_cast<size_t>(max_length) + 1);
    head_bytes = at;
    place(&st.hyp_tokens, ranks * max_length);
    s->tokens_bytes = ranks * max_length * sizeof(int32_t);
    place(&st.next_tokens, bb);
    place(&st.next_indices, bb);
    place(&st.done, batch);
    place(&st.pending, batch);
    place(&st.arrive, 1);
    place(&s->seq[0], bb * max_length);
    place(&s->seq[1], bb * max_length);
    place(&s->cand_scores, 2 * bb);
    place(&s->cand_tokens, 2 * bb);
    place(&s->cand_beams, 2 * bb);
  };
  layout();
  void* memory = nullptr;
  hipError_t e = hipMalloc(&memory, at);
  if (e == hipSuccess) {
    s->memory = static_cast<char*>(memory);
    layout();
    st.pow_table = pow_table;
    // initial beam scores 0, -1e9, -1e9, ... per batch entry (src/beam_search_scorer.cpp:76-81); rank -> row
    // identity; pow(length, length_penalty) from the host libm, the function the reference calls (pow(x, 1) is x).
    std::vector<char> head(head_bytes, 0);
    auto host = [&](auto* device) { return reinterpret_cast<std::remove_const_t<std::remove_pointer_t<decltype(device)>>*>(head.data() + (reinterpret_cast<const char*>(device) - s->memory)); };
    for (size_t i = 0; i < bb; ++i) host(st.next_scores)[i] = i % beams ? -1e9f : 0.0f;
    for (size_t i = 0; i < ranks; ++i) host(st.hyp_slot)[i] = static_cast<int>(i % (beams + 1));
    for (int l = 0; l <= max_length; ++l) host(pow_table)[l] = length_penalty == 1.0f ? static_cast<float>(l) : std::pow(static_cast<float>(l), length_penalty);
    *host(st.not_done) = batch;
    s->host = ctx->scorer_host;
    s->done_word = s->host->TakeWord();
    if (s->done_word >= 0) {
      st.all_done = s->host->words + s->done_word;
      *st.all_done = 0;
    }
    std::lock_guard<std::mutex> hold(s->host->readback_mutex);
    e = hipMemsetAsync(s->memory + head_bytes, 0, at - head_bytes, nullptr);
    const char* from = head.data();
    if (head_bytes <= ScorerHost::kReadbackBytes) from = static_cast<const char*>(std::memcpy(s->host->readback, head.data(), head_bytes));
    if (e == hipSuccess) e = hipMemcpyAsync(s->memory, from, head_bytes, hipMemcpyHostToDevice, nullptr);
    if (e == hipSuccess) e = hipStreamSynchronize(nullptr);  // the state is there before any stream uses it
  }
  if (e != hipSuccess) {
    mi355x_beam_scorer_destroy(s);
    return Fail(MI355X_E_HIP, "beam scorer allocation failed: %s", hipGetErrorString(e));
  }
  *out = s;
  return MI355X_OK;
}

void mi355x_beam_scorer_destroy(mi355x_beam_scorer* s) {
  if (!s) return;
  if (s->memory) (void)hipFree(s->memory);  // (waits for the steps under way: no launch sets the word after this)
  if (s->done_word >= 0) s->host->GiveBackWord(s->done_word);
  delete s;
}

int mi355x_beam_scorer_set_prompt(mi355x_beam_scorer* s, void* stream, const int32_t* tokens, int prompt_len) {
  if (!s || !tokens) return Fail(MI355X_E_INVALID, "null argument");
  if (prompt_len < 0 || prompt_len > s->st.max_length) return Fail(MI355X_E_INVALID, "User-defined tokens exceed max_length.");
  const int bb = s->st.batch * s->st.beams;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (Capturing(st))
    return Fail(MI355X_E_UNSUPPORTED, "the prompt is in place on return and sets the scorer's length: a graph replay would do neither");
  if (static_cast<size_t>(s->st.batch) * prompt_len <= ms::kPromptTokens) {  // inside the kernel arguments
    ms::PromptTokens prompt;
    std::copy_n(tokens, static_cast<size_t>(s->st.batch) * prompt_len, prompt.token);
    HIP_TRY(ms_launch_scorer_prompt(&prompt, prompt_len, s->st.beams, bb, s->st.max_length, s->seq[s->cur], st));
  } else {
    std::vector<int32_t> host(static_cast<size_t>(bb) * s->st.max_length, 0);
    for (int i = 0; i < bb; ++i)
      std::memcpy(host.data() + static_cast<size_t>(i) * s->st.max_length,
                  tokens + static_cast<size_t>(i / s->st.beams) * prompt_len, sizeof(int32_t) * prompt_len);
    HIP_TRY(hipMemcpyAsync(s->seq[s->cur], host.data(), host.size() * sizeof(int32_t), hipMemcpyHostToDevice, st));
    HIP_TRY(hipStreamSynchronize(st));  // `host` goes out of scope
  }
  HIP_TRY(hipStreamSynchronize(st));  // steps and readers on any stream find the prompt
  s->length = prompt_len;
  return MI355X_OK;
}

int mi355x_beam_scorer_step(mi355x_beam_scorer* s, void* stream, const float* cand_scores, const int32_t* cand_tokens,
                            const int32_t* cand_beam_indices) {
  if (!s || !cand_scores || !cand_tokens || !cand_beam_indices) return Fail(MI355X_E_INVALID, "null argument");
  if (s->length >= s->st.max_length) return Fail(MI355X_E_INVALID, "sequence already at max_length (%d)", s->st.max_length);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (Capturing(st))
    return Fail(MI355X_E_UNSUPPORTED, "a scorer step carries the sequence length and buffer of this very step: a graph replay would repeat it");
  HIP_TRY(ms_launch_scorer_step(&s->st, s->seq[s->cur], s->seq[1 - s->cur], s->length, cand_scores, cand_tokens,
                                cand_beam_indices, st));
  s->cur = 1 - s->cur;
  s->length += 1;
  s->lists.clear();
  return MI355X_OK;
}

int mi355x_beam_search_step(mi355x_beam_scorer* s, void* stream, const void* logits, int dtype, int64_t row_stride,
                            int vocab) {
  if (!s) return Fail(MI355X_E_INVALID, "null argument");
  if (s->length >= s->st.max_length) return Fail(MI355X_E_INVALID, "sequence already at max_length (%d)", s->st.max_length);
  if (Capturing(static_cast<hipStream_t>(stream)))
    return Fail(MI355X_E_UNSUPPORTED, "a search step carries the sequence length and buffer of this very step: a graph replay would repeat it");
  ms::ScorerStep step{s->st, s->seq[s->cur], s->seq[1 - s->cur], s->length};
  bool fused = false;
  if (int r = BeamSelectImpl(s->ctx, stream, logits, dtype, row_stride, s->st.batch, s->st.beams, vocab, s->st.next_scores,
                             s->cand_scores, s->cand_tokens, s->cand_beams, &step, &fused))
    return r;
  if (!fused) return mi355x_beam_scorer_step(s, stream, s->cand_scores, s->cand_tokens, s->cand_beams);
  s->cur = 1 - s->cur;
  s->length += 1;
  s->lists.clear();
  return MI355X_OK;
}

const float* mi355x_beam_scorer_next_scores(const mi355x_beam_scorer* s) { return s ? s->st.next_scores : nullptr; }
const int32_t* mi355x_beam_scorer_next_tokens(const mi355x_beam_scorer* s) { return s ? s->st.next_tokens : nullptr; }
const int32_t* mi355x_beam_scorer_next_indices(const mi355x_beam_scorer* s) { return s ? s->st.next_indices : nullptr; }
const int32_t* mi355x_beam_scorer_sequences(const mi355x_beam_scorer* s, int* length) {
  if (!s) return nullptr;
  if (length) *length = s->length;
  return s->seq[s->cur];
}

int mi355x_beam_scorer_is_done(mi355x_beam_scorer* s, void* stream, int* done) {
  if (!s || !done) return Fail(MI355X_E_INVALID, "null argument");
  hipStream_t st = static_cast<hipStream_t>(stream);
  bool all_done = false;
  if (s->st.all_done) {
    HIP_TRY(hipStreamSynchronize(st));
    all_done = *static_cast<volatile int*>(s->st.all_done) != 0;
  } else {
    std::lock_guard<std::mutex> hold(s->host->readback_mutex);
    int* const nd = reinterpret_cast<int*>(s->host->readback);
    HIP_TRY(hipMemcpyAsync(nd, s->st.not_done, sizeof(int), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    all_done = *nd == 0;
  }
  *done = all_done || (s->length == s->st.max_length);  // BeamSearch_Cpu::IsDone, src/search.cpp:345-352
  return MI355X_OK;
}

int mi355x_beam_scorer_hypothesis(mi355x_beam_scorer* s, void* stream, int batch, int index, int32_t* out, int capacity,
                                  int* length, float* score) {
  if (!s || !out || !length) return Fail(MI355X_E_INVALID, "null argument");
  if (batch < 0 || batch >= s->st.batch) return Fail(MI355X_E_INVALID, "batch index out of range");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (!s->finalized) {
    HIP_TRY(ms_launch_scorer_finalize(&s->st, s->seq[s->cur], s->length, st));
    s->finalized = true;
  }
  const int nb = s->st.beams;
  const bool tokens_too = s->lists_bytes + s->tokens_bytes <= ScorerHost::kReadbackBytes;
  char* const area = s->host->readback;
  if (s->lists.empty()) {
    const bool fits = s->lists_bytes <= ScorerHost::kReadbackBytes;
    std::lock_guard<std::mutex> hold(s->host->readback_mutex);
    std::vector<char> lists(s->lists_bytes + (tokens_too ? s->tokens_bytes : 0));
    HIP_TRY(hipMemcpyAsync(fits ? area : lists.data(), s->memory, s->lists_bytes, hipMemcpyDeviceToHost, st));
    if (tokens_too) HIP_TRY(hipMemcpyAsync(area + s->lists_bytes, s->st.hyp_tokens, s->tokens_bytes, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    if (fits) std::memcpy(lists.data(), area, lists.size());
    s->lists = std::move(lists);
  }
  auto host = [&](auto* device) { return reinterpret_cast<decltype(device)>(s->lists.data() + (reinterpret_cast<char*>(device) - s->memory)); };
  if (index < 0 || index >= host(s->st.hyp_used)[batch]) return Fail(MI355X_E_INVALID, "GetHypothesis index out of bounds");
  const int len = host(s->st.hyp_len)[batch * nb + index], slot = host(s->st.hyp_slot)[batch * (nb + 1) + index];
  const int n = len < capacity ? len : capacity;
  const size_t first = (static_cast<size_t>(batch) * (nb + 1) + slot) * s->st.max_length;
  if (tokens_too) {
    std::memcpy(out, s->lists.data() + s->lists_bytes + first * sizeof(int32_t), sizeof(int32_t) * n);
  } else {
    HIP_TRY(hipMemcpyAsync(out, s->st.hyp_tokens + first, sizeof(int32_t) * n, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
  }
  *length = len;
  if (score) *score = host(s->st.hyp_score)[batch * nb + index];
  return MI355X_OK;
}

}  // extern "C"
