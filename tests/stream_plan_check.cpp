// The plans of stream_plan.h for every vocabulary that streams and many batch sizes: a workgroup's chunk fits its kernel, no chunk
// is empty, the candidate lists fit the context's and the lists of a row the workgroup that merges them.
#include <cstdio>
#include <initializer_list>
#include "../onnxruntime-genai_amd/csrc/stream_plan.h"

static int failures = 0;

static void check(const ms::StreamCall& call) {
  const size_t lists = ms::stream_lists(static_cast<int>(call.rows), call.vocab);  // (of the smallest context that takes the call)
  const ms::StreamPlan p = ms::plan_stream(call, lists);
  const char* wrong = nullptr;
  if (p.room != ms::kSChunk && p.room != ms::kSChunk / 2 && p.room != ms::kSChunk / 4) wrong = "no kernel has that room";
  else if (p.elems <= 0 || p.elems > p.room || p.elems % 64 != 0) wrong = "a chunk does not fit its kernel, or its bitmap words are shared";
  else if (p.chunks < 1 || static_cast<long long>(p.chunks) * p.elems < call.vocab) wrong = "logits of no chunk";
  else if (static_cast<long long>(p.chunks - 1) * p.elems >= call.vocab) wrong = "an empty chunk";
  else if (static_cast<size_t>(call.rows) * static_cast<size_t>(p.chunks) > lists) wrong = "more lists than the context has";
  else if (call.vocab <= ms::kStreamMaxVocab && p.chunks > (call.argmax ? ms::kArgmaxMaxChunks : ms::kStreamMaxChunks)) wrong = "more lists than a row may have";
  else if (!call.small_k && (p.room != ms::kSChunk || p.elems != ms::kSChunk || p.rows_first)) wrong = "kernels of other rows have one chunk size and order";
  else if (call.small_k && !call.argmax && p.chunks > 1 && call.vocab - (p.chunks - 1) * p.elems < (call.sixteen_bit ? 8 : 4) * 384)
    wrong = "a last chunk of few lanes";
  else if (call.small_k && !call.argmax && call.vocab - (p.chunks - 1) * p.room >= (call.sixteen_bit ? 8 : 4) * 384 && p.elems != p.room)
    wrong = "no chunk is whole, though the last one has lanes enough";
  else if (call.small_k && !call.argmax && p.room < ms::kSChunk && p.chunks % 4 == 0 && call.rows * p.chunks > 2 * ms::kCus && !p.rows_first)
    wrong = "the workgroups that finish many rows are on two of the eight XCDs, or on one";
  if (wrong && ++failures <= 20)
    std::printf("%lld x %d small_k %d argmax %d sixteen_bit %d processed %d: %s (room %d, elems %d, chunks %d)\n", call.rows, call.vocab, call.small_k,
                call.argmax, call.sixteen_bit, call.processed, wrong, p.room, p.elems, p.chunks);
}

int main() {
  auto kinds = [](long long rows, int vocab) {
    check({rows, vocab, false, false, false, false});
    for (int flags = 0; flags < 8; ++flags) check({rows, vocab, true, (flags & 1) != 0, (flags & 2) != 0, (flags & 4) != 0});
  };
  for (int vocab = 1; vocab <= ms::kStreamMaxVocab; ++vocab)
    for (long long rows : {1, 4, 16, 63, 256, 1000}) kinds(rows, vocab);
  for (int vocab : {1, 65, 8192, 8193, 32064, 50257, 65536, 128256, 131072, 151936, 201088, 262144, 524288, 524289, 1048576, 3000001})
    for (long long rows = 1; rows <= 1100; ++rows) kinds(rows, vocab);
  std::printf("%d failures\n", failures);
  return failures != 0;
}
