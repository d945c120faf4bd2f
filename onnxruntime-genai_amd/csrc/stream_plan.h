// How the rows of a call are cut into chunks, a workgroup of a streaming kernel each (sample_stream.h).  Host arithmetic
// alone, so that its bounds can be checked without a GPU (tests/stream_plan_check.cpp).
#pragma once
#include <cstddef>

namespace ms {

constexpr int kCus = 256;             // of the GPU
constexpr int kSChunk = 32768;        // logits per workgroup of the streaming kernels; those of top-k and argmax rows also come for 16384 and 8192
constexpr int kStreamMaxChunks = 16;  // whose lists a finishing workgroup merges ...
constexpr int kArgmaxMaxChunks = 64;  // ... or whose best elements, a lane each
constexpr int kEvenLanes = 384;       // a top-k row whose last chunk has elements for fewer lanes (4, or 8 of sixteen bits, each) is cut evenly
constexpr int kStreamMaxVocab = kStreamMaxChunks * kSChunk;  // longer rows take the exact path

struct StreamPlan {
  int room;         // logits the workgroup of the kernel has room for
  int elems;        // logits of a chunk but the last
  int chunks;
  bool rows_first;  // workgroups are numbered chunk by chunk, the rows of one chunk side by side
};

// What of a call the plan depends on.
struct StreamCall {
  long long rows;
  int vocab;
  bool small_k;      // every row is one of top-k (k <= 64) or argmax; all others have chunks of kSChunk
  bool argmax;
  bool sixteen_bit;  // the logits
  bool processed;    // by penalties, masks and the like on the way
};

// Lists of candidates that a context has room for: at least rows x chunks of any plan it makes.
inline size_t stream_lists(int max_rows, int max_vocab) {
  const size_t halves = static_cast<size_t>(max_rows) * ((static_cast<size_t>(max_vocab) + kSChunk / 2 - 1) / (kSChunk / 2));
  return halves < static_cast<size_t>(kCus) ? static_cast<size_t>(kCus) : halves;
}

// A workgroup spends some ten vector instructions on every logit it has room for and a fixed time on selecting and
// handing over, so chunks are short while the GPU has a CU for each of them (8192, then 16384 logits) and long beyond:
// twice the workgroups select twice as often.  us, chunks of 32768 -> as chosen, 1 / 8 / 32 rows: argmax of 128256 fp32
// logits 5.2 -> 4.0, 5.5 -> 4.3, 6.3 -> 5.6, with a penalty over 256 ids 7.5 -> 5.4, 7.7 -> 5.7, 8.2 -> 7.2; top-k of 32064 with the
// penalty 11.1 -> 8.3, 11.2 -> 8.7, 11.7 -> 9.0; of 151936 fp16 9.1 -> 8.3, 9.7 -> 8.7, 10.2 (as before).  The lines:
//  * Top-k lists are merged four at a time by a wave, more through LDS: 7 of 8192 instead of 4 of 16384 logits, 1 x 50257 fp32 7.1 -> 7.7.
//  * More workgroups than CUs, sixteen-bit top-k rows: 16384, whose kernel takes half the registers, so that two fit a CU
//    (256 x 201088 55.2 -> 42.4, 64 x 151936 16.6 -> 14.6, with a penalty over 128 ids 69.5 -> 53.6 and 20.7 -> 18.9), but 32768 while that is
//    a workgroup per CU (64 x 128256 10.3 against 11.3, with the penalty 12.6 against 13.5).
//  * Argmax of more workgroups than CUs: 16384 up to two per CU (64 x 50257 fp16 7.2 -> 5.3) and where those of 32768 do not all run at
//    once either (256 x 201088 fp16 23.8 -> 22.5, bf16 22.7 -> 22.4, fp32 with a penalty 40.1 -> 37.5; 200 x 151936 bf16, whose 1000 of 32768 fill the
//    GPU just twice, 14.8 -> 15.3); in between some shapes gain and others lose (64 x 151936 fp16 0.91, 128 x 128256 fp16 1.13).  Sixteen-bit
//    rows with logits processing lose (256 x 128256 22.5 -> 25.9).
//  * Numbered row by row, rows of an even number of chunks have their finishing workgroups on every other XCD, those of four on two, of
//    eight on one: many workgroups are numbered chunk by chunk (256 x 128256 fp16 36.1 -> 28.4, fp32 27.7 -> 26.8); few start and end in order with
//    their rows side by side (64 x 128256 fp32 11.5, against 12.1).  Short chunks of top-k rows, four or eight (or twelve, or sixteen) a row, from
//    two workgroups per CU on: 100 x 128256 fp16 19.2 -> 17.0, with a penalty 25.7 -> 22.2, 130 x 65536 15.3 -> 13.7, 200 x 50257 18.8 -> 16.7; with ten or
//    thirteen chunks a row they stay (60 x 151936 14.8 against 15.0, with a penalty 18.7 against 19.3).
//  * A last chunk of few logits has them in few lanes, whose maxima bound nothing: rows are cut evenly then (64 x 50257 fp16 in chunks
//    of 16384 24.2 -> 9.0, 64 x 33000 in chunks of 32768 23.5 -> 9.5).  The line is at 384 lanes, six of a workgroup's eight waves.  Top-50 of
//    50 x 98304 and a last chunk of 258 lanes, whose fifth wave has two of them, as it is and evenly: fp32 29.5 and 13.4 us, fp16 32.2 and 13.7;
//    of 300 to 512 lanes 12.8 and 13.5, 13.0 and 13.6, since no chunk of an even cut is whole (64 x 100000 fp32 with a penalty, 424 lanes,
//    13.2 and 14.0).  Argmax rows, which need no bound, are cut evenly for a last chunk of under a quarter (50 x 98304 and 1700 more 7.3 and 7.0).
inline StreamPlan plan_stream(const StreamCall& call, size_t lists) {
  const long long rows = call.rows;
  auto chunks_of = [&](int room) { return static_cast<int>((static_cast<long long>(call.vocab) + room - 1) / room); };
  const int whole = kSChunk, half = kSChunk / 2, quarter = kSChunk / 4;
  const int wholes = chunks_of(whole), halves = chunks_of(half), quarters = chunks_of(quarter);
  if (!call.small_k) return StreamPlan{whole, whole, wholes, false};
  const int most = call.argmax ? kArgmaxMaxChunks : kStreamMaxChunks;
  const bool quarters_merge = quarters <= most && (call.argmax || quarters <= 4 || halves > 4);
  // beyond a workgroup per CU: half chunks or whole ones
  const bool many_halves = call.argmax ? !(call.sixteen_bit && call.processed) && ((rows * halves <= 2 * kCus && wholes > 1) || rows * wholes > 2 * kCus)
                                       : call.sixteen_bit && rows * wholes > kCus;
  int room = whole;
  if (quarters == 1 || (quarters_merge && rows * quarters <= kCus)) room = quarter;
  else if (halves == 1 || (halves <= most && (rows * halves <= kCus || many_halves))) room = half;
  if (static_cast<size_t>(rows) * static_cast<size_t>(chunks_of(room)) > lists) room = whole;
  StreamPlan plan{room, room, chunks_of(room), false};
  long long in_order = 4 * kCus - 1;  // workgroups that are numbered row by row
  if (call.argmax) in_order = room < whole ? kCus : 2 * kCus;
  else if (room < whole && plan.chunks % 4 == 0) in_order = 2 * kCus;
  plan.rows_first = rows * plan.chunks > in_order;
  const int last = call.vocab - (plan.chunks - 1) * room;
  const int short_of = call.argmax ? room / 4 : (call.sixteen_bit ? 8 : 4) * kEvenLanes;
  if (last < short_of) plan.elems = ((call.vocab + plan.chunks - 1) / plan.chunks + 63) & ~63;
  return plan;
}

}  // namespace ms
