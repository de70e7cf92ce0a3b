// The 𝚒 runtime C ABI (include/i.h): component handles and combinators.
// Reference behaviour: core/src/lib.rs:61-121, 289-351.
#include "../../../include/i.h"

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <algorithm>
#include <map>
#include <memory>
#include <condition_variable>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "../../../include/i_hip.h"
#include "../backend_hip/program.h"
#include "../runtime/hip_rt.h"
#include "../runtime/host_copy.h"
#include "../runtime/static_scratch.h"
#include "error.h"
#include "handles.h"

struct i_program {
  ihipc::Program* inner = nullptr;
  ~i_program() { delete inner; }
};

namespace {

i_component* wrap(ic::Component c) { return new i_component{std::make_shared<const ic::Component>(std::move(c))}; }

i_component* combine(const i_component* left, const i_component* right, ic::Component::Kind kind) {
  if (!left) {
    icore::set_error("null left component");
    return nullptr;
  }
  if (!right) {
    icore::set_error("null right component");
    return nullptr;
  }
  ic::Component c;
  c.kind = kind;
  c.a = left->inner;  // component trees are immutable, so sharing is a clone
  c.b = right->inner;
  return wrap(std::move(c));
}

// Strict UTF-8 check, matching CStr::to_str in the reference's read_str.
bool valid_utf8(const char* s) {
  const unsigned char* p = reinterpret_cast<const unsigned char*>(s);
  while (*p) {
    int n = *p < 0x80 ? 0 : (*p >> 5) == 0x6 ? 1 : (*p >> 4) == 0xE ? 2 : (*p >> 3) == 0x1E ? 3 : -1;
    if (n < 0) return false;
    if (n == 1 && *p < 0xC2) return false;
    ++p;
    for (int i = 0; i < n; ++i, ++p)
      if ((*p & 0xC0) != 0x80) return false;
  }
  return true;
}

int fail(const std::string& message) {
  icore::set_error(message);
  return -1;
}

// Shapes of the host operands, cut to the ranks the program reads.
std::vector<std::vector<size_t>> host_shapes(const ihipc::Program& p, const i_tensor* inputs, size_t input_count) {
  std::vector<std::vector<size_t>> out;
  for (size_t i = 0; i < input_count; ++i)
    out.emplace_back(inputs[i].shape ? std::vector<size_t>(inputs[i].shape, inputs[i].shape + inputs[i].rank) : std::vector<size_t>());
  return out;
}

// Device memory for the operands of host calls: one block per device that the library keeps from call to call
// (a host call returns after the GPU has finished, so the block is free again), as large as the largest call needed,
// at most ILANG_HIP_STAGING_MB (default 1024; 0: every operand is allocated, copied and freed on its own).  Calls
// whose operands are less than 64 MiB go through a page-locked host mirror of the block as well (run_mirrored).  Larger
// operands cross in page-locked chunks that several host threads fill and empty while
// the chunk before is in flight (runtime/host_copy.h).  A call that finds the block in use by another thread, or
// needs more, allocates as before.
struct Staging {
  void* base = nullptr;
  size_t capacity = 0;
  void* pinned = nullptr;  // a page-locked host mirror of the first pinned_bytes of the block
  size_t pinned_bytes = 0;
  std::vector<hipEvent_t> events;  // kept with it
  std::mutex busy;

  // a mirror of at least `bytes` (a power of two, 8 MiB and more), made larger if need be; false: there is none to be had
  bool mirror(size_t bytes) {
    if (pinned_bytes >= bytes) return true;
    size_t size = size_t(8) << 20;
    while (size < bytes) size *= 2;
    if (pinned) (void)hipHostFree(pinned);
    pinned = nullptr;
    pinned_bytes = 0;
    if (hipHostMalloc(&pinned, size, hipHostMallocDefault) != hipSuccess) {
      pinned = nullptr;
      (void)hipGetLastError();
      return false;
    }
    pinned_bytes = size;
    return true;
  }
  bool event(size_t n, hipEvent_t* e) {
    while (events.size() <= n) {
      hipEvent_t made = nullptr;
      if (hipEventCreateWithFlags(&made, hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
      events.push_back(made);
    }
    *e = events[n];
    return true;
  }
};
constexpr size_t kMirroredBytes = size_t(64) << 20;  // calls of less go through the mirror

struct StagingTable {
  std::mutex mu;
  std::map<int, std::unique_ptr<Staging>> blocks;
};
StagingTable& staging_table() {
  static StagingTable* table = new StagingTable();
  return *table;
}
Staging* staging_of_current_device() {
  StagingTable& t = staging_table();
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return nullptr;
  std::lock_guard<std::mutex> lock(t.mu);
  auto& block = t.blocks[device];
  if (!block) block = std::make_unique<Staging>();
  return block.get();
}

// Frees the blocks that no call is using at this moment; returns the bytes released (device and page-locked).
size_t release_staging_blocks() {
  size_t released = 0;
  StagingTable& t = staging_table();
  std::lock_guard<std::mutex> lock(t.mu);
  for (auto& [device, block] : t.blocks) {
    std::unique_lock<std::mutex> idle(block->busy, std::try_to_lock);
    if (!idle.owns_lock()) continue;
    if (block->base) {
      ihip::dev_free(block->base);
      released += block->capacity;
    }
    if (block->pinned) {
      (void)hipHostFree(block->pinned);
      released += block->pinned_bytes;
    }
    for (hipEvent_t e : block->events) (void)hipEventDestroy(e);
    block->events.clear();
    block->base = block->pinned = nullptr;
    block->capacity = block->pinned_bytes = 0;
  }
  return released;
}

size_t staging_limit() {
  static const size_t limit = [] {
    const char* mb = std::getenv("ILANG_HIP_STAGING_MB");
    return (mb ? (size_t)std::max(0, std::atoi(mb)) : size_t(1024)) << 20;
  }();
  return limit;
}

// The two streams beside the call's own that a call in slices uses: `which` 0 carries the uploads, 1 the downloads
// (one each per device, created on first use and kept; not synchronised with the default stream, on which the
// kernels run); nullptr when there is none to be had.  Any further stream of a process, whoever creates it and whether or not it
// is ever used or destroyed, costs products that pad their operands 2 to 3 % on a stream that was used before it (bf16 2047 x
// 3001 x 777 28.2 -> 28.8 us, f32 1023 x 1501 x 699 33.6 -> 34.5; other calls nothing); the slices give host calls of 17 to 34 MB 10
// to 20 % (8 x 2 heads of 2048 x 64 1040 -> 825 us), so they stay.
hipStream_t side_stream_of_current_device(int which) {
  static std::mutex mu;
  static std::map<int, hipStream_t>* streams = new std::map<int, hipStream_t>();
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return nullptr;
  std::lock_guard<std::mutex> lock(mu);
  auto it = streams->find(2 * device + which);
  if (it != streams->end()) return it->second;
  hipStream_t made = nullptr;
  if (hipStreamCreateWithFlags(&made, hipStreamNonBlocking) != hipSuccess) {
    (void)hipGetLastError();
    made = nullptr;
  }
  (*streams)[2 * device + which] = made;
  return made;
}

// Calls in slices write rows of the outputs while later rows of the inputs are still to be read.  Does an output lie in
// memory that an input, or another output, has as well?  (An output that starts where an input of as long rows starts is
// fine, as for a call in place: a slice writes only rows that it has read.)
bool slices_collide(const i_tensor* inputs, const std::vector<ihipc::DeviceTensor>& in, const std::vector<char>& sliced,
                    const std::vector<ihipc::DeviceTensor>& out, const std::vector<float*>& out_ptrs) {
  struct Range {
    uintptr_t from, to;
  };
  auto range_of = [](const void* data, const ihipc::DeviceTensor& t) {
    size_t bytes = 4;
    for (size_t d : t.shape) bytes *= d;
    const uintptr_t from = reinterpret_cast<uintptr_t>(data);
    return Range{from, from + bytes};
  };
  auto meet = [](Range a, Range b) { return a.from < b.to && b.from < a.to && a.from != a.to && b.from != b.to; };
  for (size_t o = 0; o < out.size(); ++o) {
    const Range to = range_of(out_ptrs[o], out[o]);
    for (size_t i = 0; i < in.size(); ++i) {
      const Range from = range_of(inputs[i].data, in[i]);
      const bool same_rows = sliced[i] && to.from == from.from && to.to == from.to;  // (and as many: the leading extents are equal)
      if (!same_rows && meet(to, from)) return true;
    }
    for (size_t other = 0; other < o; ++other)
      if (meet(to, range_of(out_ptrs[other], out[other]))) return true;
  }
  return false;
}

// A call in slices (large operands of a program that only maps over its leading index, ihipc::row_sliceable): the
// inputs that every slice needs whole are uploaded first; then, slice after slice, the rows of the other inputs go
// up on the upload stream and the program is enqueued on `stream` behind them for just those rows, so the kernels
// of one slice run while the next is on the link; a second host thread brings the rows of the outputs down on the
// download stream as soon as their slice has run, beside the uploads of the slices after it (the link carries both
// directions at once).  Returns false when the call is not taken in slices (nothing has been enqueued then); true
// with the outputs in host memory, or with *err set.
constexpr size_t kSlicedCallBytes = size_t(64) << 20;  // what crosses the link in slices, at least
constexpr size_t kSliceBytes = size_t(32) << 20;       // ... and per slice, about
bool run_host_in_slices(ihipc::Program& p, const i_tensor* inputs, const std::vector<ihipc::DeviceTensor>& in,
                        const std::vector<ihipc::DeviceTensor>& out, const std::vector<float*>& out_ptrs, hipStream_t stream,
                        std::string* err) {
  std::vector<char> sliced;
  if (!ihipc::row_sliceable(p, &sliced) || sliced.size() != in.size() || out.empty() || out[0].shape.empty()) return false;
  const size_t rows = out[0].shape[0];
  auto row_bytes = [](const ihipc::DeviceTensor& t) {
    size_t n = 4;
    for (size_t d = 1; d < t.shape.size(); ++d) n *= t.shape[d];
    return n;
  };
  size_t moving = 0, whole = 0;
  for (size_t i = 0; i < in.size(); ++i) {
    if (sliced[i] && (in[i].shape.empty() || in[i].shape[0] != rows)) return false;
    (sliced[i] ? moving : whole) += row_bytes(in[i]) * (in[i].shape.empty() ? 1 : in[i].shape[0]);
  }
  for (size_t o = 0; o < out.size(); ++o) {
    if (out[o].shape.empty() || out[o].shape[0] != rows || !out_ptrs[o]) return false;
    moving += row_bytes(out[o]) * rows;
  }
  if (rows < 2 || moving < kSlicedCallBytes || moving < whole || slices_collide(inputs, in, sliced, out, out_ptrs)) return false;
  const size_t wanted = std::min<size_t>(std::min<size_t>(8, rows), std::max<size_t>(2, moving / kSliceBytes));
  const size_t each = (rows + wanted - 1) / wanted, slices = (rows + each - 1) / each;
  hipStream_t up = side_stream_of_current_device(0), down = side_stream_of_current_device(1);
  int device = 0;
  if (!up || !down || hipGetDevice(&device) != hipSuccess) return false;
  std::vector<hipEvent_t> landed(slices, nullptr), done(slices, nullptr);
  auto destroy_events = [&] {
    for (hipEvent_t e : landed)
      if (e) (void)hipEventDestroy(e);
    for (hipEvent_t e : done)
      if (e) (void)hipEventDestroy(e);
  };
  for (size_t s = 0; s < slices; ++s)
    if (hipEventCreateWithFlags(&landed[s], hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&done[s], hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      destroy_events();
      return false;
    }
  // the downloads: slice s once the main thread says that it has been enqueued (or that nothing more will be)
  std::mutex mu;
  std::condition_variable changed;
  size_t enqueued = 0;
  bool stop = false;
  std::string down_err;
  auto bring_down_slices = [&] {
    (void)hipSetDevice(device);
    for (size_t s = 0; s < slices; ++s) {
      {
        std::unique_lock<std::mutex> lock(mu);
        changed.wait(lock, [&] { return enqueued > s || stop; });
        if (enqueued <= s) return;
      }
      if (hipStreamWaitEvent(down, done[s], 0) != hipSuccess) {
        down_err = "hipStreamWaitEvent failed";
        return;
      }
      const size_t r0 = s * each, r1 = std::min(rows, r0 + each);
      for (size_t o = 0; o < out.size(); ++o) {
        const size_t at = r0 * row_bytes(out[o]), bytes = (r1 - r0) * row_bytes(out[o]);
        if (ihip::Err e = ihip::download_pipelined(reinterpret_cast<char*>(out_ptrs[o]) + at, static_cast<const char*>(out[o].data) + at, bytes, down);
            !e.empty()) {
          down_err = e;
          return;
        }
      }
    }
  };
  auto bring_down = [&] {
    try {
      bring_down_slices();
    } catch (const std::exception& e) {  // (nothing may leave a thread's function)
      down_err = e.what();
    }
  };
  std::thread helper;
  try {
    helper = std::thread(bring_down);
  } catch (const std::exception&) {
    destroy_events();
    return false;
  }
  auto finish = [&](const std::string& what, bool all_enqueued) {
    {
      std::lock_guard<std::mutex> lock(mu);
      stop = !all_enqueued;
      if (all_enqueued) enqueued = slices;
    }
    changed.notify_all();
    helper.join();
    *err = !what.empty() ? what : down_err;
    if (!err->empty()) {
      (void)hipStreamSynchronize(up);
      (void)hipStreamSynchronize(down);
      (void)ihip::sync(stream);
    }
    destroy_events();
    return true;
  };
  // (the device copies may still be read by the kernels of the call before this one on `stream`: the kept block
  // is handed from call to call only after a wait for `stream`, so nothing is in flight there)
  for (size_t i = 0; i < in.size(); ++i)
    if (!sliced[i]) {
      const size_t bytes = row_bytes(in[i]) * (in[i].shape.empty() ? 1 : in[i].shape[0]);
      if (ihip::Err e = ihip::upload_pipelined(in[i].data, inputs[i].data, bytes, up); !e.empty()) return finish(e, false);
    }
  for (size_t s = 0; s < slices; ++s) {
    const size_t r0 = s * each, r1 = std::min(rows, r0 + each);
    std::vector<ihipc::DeviceTensor> in_s(in), out_s(out);
    for (size_t i = 0; i < in.size(); ++i) {
      if (!sliced[i]) continue;
      const size_t at = r0 * row_bytes(in[i]), bytes = (r1 - r0) * row_bytes(in[i]);
      in_s[i].data = static_cast<char*>(in[i].data) + at;
      in_s[i].shape[0] = r1 - r0;
      if (ihip::Err e = ihip::upload_pipelined(in_s[i].data, static_cast<const char*>(static_cast<const void*>(inputs[i].data)) + at, bytes, up);
          !e.empty())
        return finish(e, false);
    }
    for (size_t o = 0; o < out.size(); ++o) {
      out_s[o].data = static_cast<char*>(out[o].data) + r0 * row_bytes(out[o]);
      out_s[o].shape[0] = r1 - r0;
    }
    if (hipEventRecord(landed[s], up) != hipSuccess || hipStreamWaitEvent(stream, landed[s], 0) != hipSuccess)
      return finish("hipStreamWaitEvent failed", false);
    std::string e;
    try {
      e = ihipc::execute(p, in_s, out_s, stream);
    } catch (const std::exception& ex) {
      e = ex.what();
    }
    if (e.empty() && hipEventRecord(done[s], stream) != hipSuccess) e = "hipEventRecord failed";
    if (!e.empty()) return finish(e, false);
    {
      std::lock_guard<std::mutex> lock(mu);
      enqueued = s + 1;
    }
    changed.notify_all();
  }
  ihipc::append_to_report(p, "host: operands in " + std::to_string(slices) + " slices of " + std::to_string(each) +
                                 " rows, the kernels above are those of the last slice\n");
  return finish({}, true);
}

// A call whose operands lie in the kept block with a page-locked mirror of it.  Several host threads gather the inputs in
// the mirror a MiB at a time, and every 2 to 8 MiB that are there start across while the next are gathered; the outputs come
// back in pieces of 2 MiB and more.  A program that only maps over its leading index runs in slices of about 8 MiB from 6 on, as above: the
// kernels of a slice, and its outputs on their way down, run beside the uploads of those after it.  One thread drives
// all of it: what has come down is copied out between two slices.  Attention of 8 x 2
// heads of 2048 x 64 (33 MB) 1170 -> 840 us a call, 5 x 7 of 777 x 72 1530 -> 760, 2 x 8 of 412 x 64 340 -> 300, 2 x 3 of 398 x 32
// 160 -> 105; the link alone takes 610, 570, 123 and 22.
constexpr size_t kMirrorPiece = size_t(1) << 20, kMirroredSlicedBytes = size_t(6) << 20, kMirroredSliceBytes = size_t(8) << 20;
std::string run_mirrored(ihipc::Program& p, const i_tensor* inputs, const std::vector<ihipc::DeviceTensor>& in,
                         const std::vector<ihipc::DeviceTensor>& out, const std::vector<float*>& out_ptrs, size_t call_bytes, Staging& block,
                         hipStream_t stream) {
  char* const base = static_cast<char*>(block.base);
  char* const mirror = static_cast<char*>(block.pinned);
  auto elements = [](const ihipc::DeviceTensor& t) {
    size_t n = 1;
    for (size_t d : t.shape) n *= d;
    return n;
  };
  // slices of the leading index, if the program allows it and there is enough to move
  std::vector<char> sliced;
  size_t rows = out.empty() || out[0].shape.empty() ? 0 : out[0].shape[0], moving = 0, whole = 0;
  bool in_slices = rows >= 2 && call_bytes >= kMirroredSlicedBytes && ihipc::row_sliceable(p, &sliced) && sliced.size() == in.size();
  for (size_t i = 0; in_slices && i < in.size(); ++i) {
    in_slices = !sliced[i] || (!in[i].shape.empty() && in[i].shape[0] == rows);
    (sliced[i] ? moving : whole) += 4 * elements(in[i]);
  }
  for (size_t o = 0; in_slices && o < out.size(); ++o) {
    in_slices = !out[o].shape.empty() && out[o].shape[0] == rows && (out_ptrs[o] || elements(out[o]) == 0);
    moving += 4 * elements(out[o]);
  }
  in_slices = in_slices && !slices_collide(inputs, in, sliced, out, out_ptrs);
  hipStream_t up = stream, down = stream;
  if (in_slices && moving >= kMirroredSlicedBytes && moving >= whole) {
    up = side_stream_of_current_device(0);
    down = side_stream_of_current_device(1);
  }
  in_slices = in_slices && up && down && up != stream;
  if (!in_slices) up = down = stream;
  const size_t wanted = in_slices ? std::min<size_t>(std::min<size_t>(8, rows), std::max<size_t>(2, moving / kMirroredSliceBytes)) : 1;
  const size_t each = in_slices ? (rows + wanted - 1) / wanted : 0, slices = in_slices ? (rows + each - 1) / each : 1;

  // (transfers of whole operands end on a multiple of 256 bytes, which every operand has room for: 120 and 200 bytes cost a call of
  // 32 us one more)
  auto rounded = [in_slices](size_t end) { return in_slices ? end : (end + 255) / 256 * 256; };
  // ---- up: the pieces in the order in which they cross, and how many there are up to the end of each slice
  std::vector<ihip::CopyPiece> gathered;
  std::vector<size_t> gathered_until;
  auto offset = [&](const ihipc::DeviceTensor& t) { return (size_t)(static_cast<char*>(t.data) - base); };
  auto gather = [&](const void* data, size_t at, size_t bytes) {  // into bytes of the mirror from `at` on
    for (size_t done = 0; done < bytes; done += kMirrorPiece)
      gathered.push_back({mirror + at + done, static_cast<const char*>(data) + done, std::min(bytes - done, kMirrorPiece)});
  };
  for (size_t i = 0; i < in.size(); ++i)
    if (!in_slices || !sliced[i]) gather(inputs[i].data, offset(in[i]), 4 * elements(in[i]));
  for (size_t s = 0; s < slices; ++s) {
    const size_t r0 = s * each, r1 = std::min(rows, r0 + each);
    for (size_t i = 0; in_slices && i < in.size(); ++i)
      if (sliced[i]) {
        const size_t row = 4 * elements(in[i]) / rows;
        gather(reinterpret_cast<const char*>(inputs[i].data) + r0 * row, offset(in[i]) + r0 * row, (r1 - r0) * row);
      }
    gathered_until.push_back(gathered.size());
  }
  ihip::CopyAhead ahead(gathered);
  // Sends the pieces before `until`, as soon as they are there; small neighbours go together.  9 us of every transfer are its
  // own, so a run of pieces that lie together goes in equal transfers of about 8 MiB, behind two shorter ones for the sake of an early
  // start (row sums of 60 MB in slices of 8.6: 1425 us with 4, 4 and 0.6 MiB a slice).
  size_t sent = 0, transfers = 0;
  auto send = [&](size_t until) -> ihip::Err {
    auto at = [&](size_t n) { return (size_t)(static_cast<char*>(gathered[n].dst) - mirror); };
    auto end = [&](size_t n) { return at(n) + gathered[n].bytes; };
    while (sent < until) {
      size_t last = sent;  // of the run (operands start on the next 256 bytes after the one before)
      while (last + 1 < until && at(last + 1) >= end(last) && at(last + 1) - end(last) < 256) ++last;
      const size_t lo = at(sent), run = end(last) - lo, about = (transfers < 2 ? size_t(2) << transfers : 8) * kMirrorPiece;
      const size_t least = run / std::max<size_t>(1, (run + about / 2) / about);
      size_t hi = lo;
      for (; sent <= last && hi - lo < least; ++sent) {
        ahead.wait(sent);
        hi = end(sent);
      }
      ++transfers;
      if (ihip::Err e = ihip::h2d(base + lo, mirror + lo, rounded(hi) - lo, up); !e.empty()) return e;
    }
    return {};
  };
  // ---- down: pieces on their way, copied out in order.  Small neighbours cross together here too.
  struct Piece {
    size_t at, bytes;
    char* to;
    bool first;          // of its transfer: copying it out waits for that
    hipEvent_t landed;   // nullptr: the last transfer of all, awaited with the stream
  };
  std::vector<Piece> pieces;
  size_t copied = 0, events = 2 * slices, enqueued = 0;  // pieces that are copied out; events in use; pieces that are on their way
  size_t unmarked = SIZE_MAX;                            // the first piece of the last transfer, as long as no event follows that
  bool waited = false;                                   // for the stream, with nothing enqueued after
  auto mark = [&]() -> ihip::Err {
    if (unmarked == SIZE_MAX) return {};
    if (!block.event(events++, &pieces[unmarked].landed)) return "no event for a transfer";
    if (ihip::Err e = ihip::check(hipEventRecord(pieces[unmarked].landed, down), "hipEventRecord"); !e.empty()) return e;
    unmarked = SIZE_MAX;
    return {};
  };
  auto enqueue = [&]() -> ihip::Err {  // the pieces that are not on their way yet, in one transfer
    if (enqueued == pieces.size()) return {};
    if (ihip::Err e = mark(); !e.empty()) return e;
    Piece& first = pieces[enqueued];
    const size_t end = rounded(pieces.back().at + pieces.back().bytes);
    first.first = true;
    if (ihip::Err e = ihip::d2h(mirror + first.at, base + first.at, end - first.at, down); !e.empty()) return e;
    unmarked = enqueued;
    enqueued = pieces.size();
    return {};
  };
  auto bring = [&](size_t at, size_t bytes, char* to) -> ihip::Err {
    const size_t step = std::max(2 * kMirrorPiece, (bytes / 4 + 4095) / 4096 * 4096);
    for (size_t done = 0; done < bytes; done += step) {
      const size_t here = at + done, size = std::min(step, bytes - done);
      if (enqueued < pieces.size()) {
        const size_t end = pieces.back().at + pieces.back().bytes;  // (outputs, too, start on the next 256 bytes after the one before)
        if (in_slices || here < end || here - end >= 256 || here + size - pieces[enqueued].at > 2 * kMirrorPiece)
          if (ihip::Err e = enqueue(); !e.empty()) return e;
      }
      pieces.push_back({here, size, to + done, false, nullptr});
    }
    return {};
  };
  auto copy_out = [&](size_t until) -> ihip::Err {
    for (; copied < until; ++copied) {
      const Piece& piece = pieces[copied];
      if (piece.first && !waited) {
        if (ihip::Err e = piece.landed ? ihip::check(hipEventSynchronize(piece.landed), "hipEventSynchronize") : ihip::sync(down); !e.empty()) return e;
        waited = !piece.landed;
      }
      ihip::copy_by_threads(piece.to, mirror + piece.at, piece.bytes);
    }
    return {};
  };

  auto run = [&]() -> ihip::Err {
    std::vector<size_t> pieces_at;  // how many there were before each slice
    for (size_t s = 0; s < slices; ++s) {
      const size_t r0 = s * each, r1 = std::min(rows, r0 + each);
      std::vector<ihipc::DeviceTensor> in_cut, out_cut;
      if (in_slices) {
        in_cut = in;
        out_cut = out;
      }
      const std::vector<ihipc::DeviceTensor>&in_s = in_slices ? in_cut : in, &out_s = in_slices ? out_cut : out;
      auto cut = [&](ihipc::DeviceTensor& t) {  // rows r0 .. r1; returns the byte offset of the first
        const size_t skip = 4 * elements(t) / rows * r0;
        t.data = static_cast<char*>(t.data) + skip;
        t.shape[0] = r1 - r0;
        return skip;
      };
      std::vector<size_t> out_skip(out.size(), 0);
      for (size_t i = 0; in_slices && i < in.size(); ++i) {
        if (sliced[i]) (void)cut(in_cut[i]);
      }
      for (size_t o = 0; in_slices && o < out.size(); ++o) out_skip[o] = cut(out_cut[o]);
      if (ihip::Err e = send(gathered_until[s]); !e.empty()) return e;
      hipEvent_t landed = nullptr, ran = nullptr;
      if (in_slices) {
        if (!block.event(2 * s, &landed) || !block.event(2 * s + 1, &ran)) return "no event for a slice";
        if (ihip::Err e = ihip::check(hipEventRecord(landed, up), "hipEventRecord"); !e.empty()) return e;
        if (ihip::Err e = ihip::check(hipStreamWaitEvent(stream, landed, 0), "hipStreamWaitEvent"); !e.empty()) return e;
      }
      if (ihip::Err e = ihipc::execute(p, in_s, out_s, stream); !e.empty()) return e;
      if (in_slices) {
        if (ihip::Err e = ihip::check(hipEventRecord(ran, stream), "hipEventRecord"); !e.empty()) return e;
        if (ihip::Err e = ihip::check(hipStreamWaitEvent(down, ran, 0), "hipStreamWaitEvent"); !e.empty()) return e;
      }
      pieces_at.push_back(pieces.size());
      for (size_t o = 0; o < out.size(); ++o) {
        if (elements(out[o]) == 0) continue;
        if (!out_ptrs[o]) return "output " + std::to_string(o) + " has no data";
        if (ihip::Err e = bring(offset(out_s[o]), 4 * elements(out_s[o]), reinterpret_cast<char*>(out_ptrs[o]) + out_skip[o]); !e.empty()) return e;
      }
      if (ihip::Err e = enqueue(); !e.empty()) return e;
      if (in_slices)
        if (ihip::Err e = mark(); !e.empty()) return e;
      // (two slices back: down by now, unless the kernels are what takes the time, and then nothing waits for this thread)
      if (s >= 2)
        if (ihip::Err e = copy_out(pieces_at[s - 1]); !e.empty()) return e;
    }
    return copy_out(pieces.size());
  };
  std::string err;
  try {
    err = run();
  } catch (const std::exception& e) {
    err = e.what();
  }
  if (in_slices && !err.empty()) {  // (nothing may still be using the kept block)
    (void)hipStreamSynchronize(up);
    (void)hipStreamSynchronize(down);
  }
  if (!waited || !err.empty()) {
    const ihip::Err sync_err = ihip::sync(stream);
    if (err.empty()) err = sync_err;
  }
  if (in_slices && err.empty())
    ihipc::append_to_report(p, "host: operands in " + std::to_string(slices) + " slices of " + std::to_string(each) +
                                   " rows, the kernels above are those of the last slice\n");
  return err;
}

// Host entry: upload f32 operands, run, download, wait.  Mirrors the
// blocking behaviour of the reference's exec (core/src/lib.rs:200-225).
std::string run_host(ihipc::Program& p, const i_tensor* inputs, size_t input_count, const std::vector<float*>& out_ptrs) {
  const auto in_shapes = host_shapes(p, inputs, input_count);
  std::vector<std::vector<size_t>> out_shapes;
  if (std::string e = ihipc::output_shapes(p, in_shapes, &out_shapes); !e.empty()) return e;
  std::vector<void*> owned;
  hipStream_t stream = nullptr;
  bool staged = false;
  auto cleanup = [&] {
    if (staged) (void)ihip::sync(stream);  // (an early return: nothing may still be using the kept block)
    for (void* ptr : owned) ihip::dev_free(ptr);
  };
  // the operands' device copies: carved from the kept block when it is free and large enough (or can be made so)
  auto bytes_of = [](const std::vector<size_t>& shape) {
    size_t n = 4;
    for (size_t d : shape) n *= d;
    return (std::max<size_t>(n, 4) + 255) / 256 * 256;
  };
  size_t wanted = 0;
  for (size_t i = 0; i < input_count; ++i) wanted += bytes_of(in_shapes[i]);
  for (const auto& shape : out_shapes) wanted += bytes_of(shape);
  std::unique_lock<std::mutex> staging_lock;
  char* carve = nullptr;
  Staging* mirrored = nullptr;  // host data passes through the page-locked mirror of the kept block
  if (wanted <= staging_limit()) {
    if (Staging* block = staging_of_current_device()) {
      staging_lock = std::unique_lock<std::mutex>(block->busy, std::try_to_lock);
      if (staging_lock.owns_lock()) {
        if (block->capacity < wanted) {
          ihip::dev_free(block->base);
          block->base = nullptr;
          block->capacity = 0;
          if (ihip::dev_alloc(&block->base, wanted).empty()) block->capacity = wanted;
        }
        if (block->capacity >= wanted) {
          carve = static_cast<char*>(block->base);
          staged = true;
          if (wanted < kMirroredBytes && block->mirror(wanted)) mirrored = block;
        }
      }
    }
  }
  auto device_copy = [&](void** ptr, const std::vector<size_t>& shape) -> ihip::Err {
    if (carve) {
      *ptr = carve;
      carve += bytes_of(shape);
      return {};
    }
    size_t n = 1;
    for (size_t d : shape) n *= d;
    if (ihip::Err e = ihip::dev_alloc(ptr, n * 4); !e.empty()) return e;
    owned.push_back(*ptr);
    return {};
  };
  std::vector<ihipc::DeviceTensor> in, out;
  for (size_t i = 0; i < input_count; ++i) {
    size_t n = 1;
    for (size_t d : in_shapes[i]) n *= d;
    ihipc::DeviceTensor t;
    t.shape = in_shapes[i];
    if (n && !inputs[i].data) {
      cleanup();
      return "input " + std::to_string(i) + " has no data";
    }
    if (ihip::Err e = device_copy(&t.data, in_shapes[i]); !e.empty()) {
      cleanup();
      return e;
    }
    in.push_back(std::move(t));
  }
  for (size_t o = 0; o < out_shapes.size(); ++o) {
    size_t n = 1;
    for (size_t d : out_shapes[o]) n *= d;
    ihipc::DeviceTensor t;
    t.shape = out_shapes[o];
    if (ihip::Err e = device_copy(&t.data, out_shapes[o]); !e.empty()) {
      cleanup();
      return e;
    }
    out.push_back(std::move(t));
  }
  std::string err;
  if (mirrored) {
    try {
      err = run_mirrored(p, inputs, in, out, out_ptrs, wanted, *mirrored, stream);
    } catch (const std::exception& e) {  // (out of memory before anything was enqueued)
      err = e.what();
    }
    cleanup();
    return err;
  }
  // large operands: in slices when the program allows it, else one after the other and then the program
  const bool in_slices = run_host_in_slices(p, inputs, in, out, out_ptrs, stream, &err);  // (outputs included)
  if (!in_slices) {
    for (size_t i = 0; err.empty() && i < input_count; ++i) {
      size_t n = 1;
      for (size_t d : in_shapes[i]) n *= d;
      err = ihip::upload_pipelined(in[i].data, inputs[i].data, n * 4, stream);
    }
    try {
      if (err.empty()) err = ihipc::execute(p, in, out, stream);
    } catch (const std::exception& e) {
      err = e.what();
    }
  }
  for (size_t o = 0; !in_slices && err.empty() && o < out.size(); ++o) {
    size_t n = 1;
    for (size_t d : out_shapes[o]) n *= d;
    if (n && !out_ptrs[o]) err = "output " + std::to_string(o) + " has no data";
    else err = ihip::download_pipelined(out_ptrs[o], out[o].data, n * 4, stream);
  }
  const ihip::Err sync_err = ihip::sync(stream);
  if (err.empty()) err = sync_err;
  cleanup();
  return err;
}

// Argument checks shared by the device entry points; fills `in` / `out` and returns true, or sets the error.
bool device_call_ok(const i_program* program, const i_device_tensor* inputs, size_t input_count,
                    const i_device_tensor* outputs, size_t output_count, std::vector<ihipc::DeviceTensor>* in,
                    std::vector<ihipc::DeviceTensor>* out) {
  if (!program) return fail("null program"), false;
  if (input_count > 0 && !inputs) return fail("null inputs"), false;
  if (output_count != ihipc::output_count(*program->inner)) return fail("wrong output count"), false;
  if (output_count > 0 && !outputs) return fail("null outputs"), false;
  auto convert = [](const i_device_tensor* t, size_t n, std::vector<ihipc::DeviceTensor>* dst) -> bool {
    for (size_t i = 0; i < n; ++i) {
      if (t[i].dtype != I_DTYPE_F32 && t[i].dtype != I_DTYPE_BF16) return false;
      ihipc::DeviceTensor d;
      d.data = t[i].data;
      d.dtype = t[i].dtype == I_DTYPE_BF16 ? ihipc::DType::BF16 : ihipc::DType::F32;
      if (t[i].rank > 0 && !t[i].shape) return false;
      d.shape.assign(t[i].shape, t[i].shape + t[i].rank);
      dst->push_back(std::move(d));
    }
    return true;
  };
  if (!convert(inputs, input_count, in) || !convert(outputs, output_count, out))
    return fail("bad device tensor (dtype or shape)"), false;
  return true;
}

}  // namespace

#pragma GCC visibility push(default)
extern "C" {

i_component* i_parse(const char* src) {
  if (!src || !valid_utf8(src)) {
    icore::set_error("null source");
    return nullptr;
  }
  try {
    ic::Component c;
    c.kind = ic::Component::Leaf;
    c.expr = ic::parse_expr(src);
    return wrap(std::move(c));
  } catch (const ic::CompileError& e) {
    icore::set_error(e.debug_string());
  } catch (const std::exception& e) {
    icore::set_error(e.what());
  }
  return nullptr;
}

i_component* i_identity(void) { return wrap(ic::Component{}); }

i_component* i_chain(const i_component* l, const i_component* r) { return combine(l, r, ic::Component::Chain); }
i_component* i_compose(const i_component* l, const i_component* r) { return combine(l, r, ic::Component::Compose); }
i_component* i_fanout(const i_component* l, const i_component* r) { return combine(l, r, ic::Component::Fanout); }
i_component* i_pair(const i_component* l, const i_component* r) { return combine(l, r, ic::Component::Pair); }

i_component* i_swap(const i_component* component) {
  if (!component) {
    icore::set_error("null component");
    return nullptr;
  }
  ic::Component c;
  c.kind = ic::Component::Swap;
  c.a = component->inner;
  return wrap(std::move(c));
}

char* i_code(const i_component* component) {
  if (!component) {
    icore::set_error("null component");
    return nullptr;
  }
  try {
    const std::string text = ihipc::program_code(*component->inner);
    if (text.find('\0') != std::string::npos) {
      icore::set_error("source contains interior NUL");
      return nullptr;
    }
    char* out = static_cast<char*>(std::malloc(text.size() + 1));
    if (!out) {
      icore::set_error("out of memory");
      return nullptr;
    }
    std::memcpy(out, text.c_str(), text.size() + 1);
    return out;
  } catch (const ic::CompileError& e) {
    icore::set_error(e.debug_string());
  } catch (const std::exception& e) {
    icore::set_error(e.what());
  }
  return nullptr;
}

i_program* i_compile(const i_component* component) {
  if (!component) {
    icore::set_error("null component");
    return nullptr;
  }
  try {
    ihipc::Program* inner = nullptr;
    const std::string err = ihipc::compile_program(*component->inner, &inner);
    if (!err.empty()) {
      icore::set_error(err);
      return nullptr;
    }
    auto* program = new i_program;
    program->inner = inner;
    return program;
  } catch (const ic::CompileError& e) {
    icore::set_error(e.debug_string());
  } catch (const std::exception& e) {
    icore::set_error(e.what());
  }
  return nullptr;
}

size_t i_output_count(const i_program* program) {
  if (!program) {
    icore::set_error("null program");
    return 0;
  }
  return ihipc::output_count(*program->inner);
}

int i_output_ranks(const i_program* program, size_t* ranks) {
  if (!program) return fail("null program");
  if (!ranks) return fail("null ranks");
  const auto r = ihipc::output_ranks(*program->inner);
  for (size_t i = 0; i < r.size(); ++i) ranks[i] = r[i];
  return 0;
}

int i_output_shapes(const i_program* program, const i_tensor* inputs, size_t input_count, size_t** shapes) {
  if (!program) return fail("null program");
  if (input_count > 0 && !inputs) return fail("null inputs");
  if (!shapes) return fail("null shapes");
  std::vector<std::vector<size_t>> out;
  const std::string err = ihipc::output_shapes(*program->inner, host_shapes(*program->inner, inputs, input_count), &out);
  if (!err.empty()) return fail(err);
  for (size_t o = 0; o < out.size(); ++o)
    for (size_t d = 0; d < out[o].size(); ++d) shapes[o][d] = out[o][d];
  return 0;
}

int i_exec_into(const i_program* program, const i_tensor* inputs, size_t input_count, i_tensor_mut* outputs,
                size_t output_count) {
  if (!program) return fail("null program");
  if (input_count > 0 && !inputs) return fail("null inputs");
  if (output_count != ihipc::output_count(*program->inner)) return fail("wrong output count");
  if (output_count > 0 && !outputs) return fail("null outputs");
  // An output whose extents the caller states is checked against what the program writes: a smaller buffer would be
  // overrun on the host.  (The reference takes the caller's word, core/src/lib.rs:200-225; a tensor without a shape
  // array is taken on trust here too.)
  {
    std::vector<std::vector<size_t>> written;
    if (std::string e = ihipc::output_shapes(*program->inner, host_shapes(*program->inner, inputs, input_count), &written); !e.empty())
      return fail(e);
    for (size_t o = 0; o < output_count && o < written.size(); ++o) {
      if (!outputs[o].shape) continue;
      bool same = outputs[o].rank == written[o].size();
      for (size_t d = 0; same && d < written[o].size(); ++d) same = outputs[o].shape[d] == written[o][d];
      if (!same) {
        auto text = [](const size_t* dims, size_t rank) {
          std::string t = "[";
          for (size_t d = 0; d < rank; ++d) t += (d ? ", " : "") + std::to_string(dims[d]);
          return t + "]";
        };
        return fail("output " + std::to_string(o) + " has shape " + text(outputs[o].shape, outputs[o].rank) + ", the program writes " +
                    text(written[o].data(), written[o].size()));
      }
    }
  }
  std::vector<float*> out_ptrs;
  for (size_t o = 0; o < output_count; ++o) out_ptrs.push_back(outputs[o].data);
  const std::string err = run_host(*program->inner, inputs, input_count, out_ptrs);
  return err.empty() ? 0 : fail(err);
}

i_outputs i_exec(const i_program* program, const i_tensor* inputs, size_t input_count) {
  i_outputs none{nullptr, 0};
  if (!program) {
    icore::set_error("null program");
    return none;
  }
  if (input_count > 0 && !inputs) {
    icore::set_error("null inputs");
    return none;
  }
  ihipc::Program& p = *program->inner;
  std::vector<std::vector<size_t>> shapes;
  if (std::string err = ihipc::output_shapes(p, host_shapes(p, inputs, input_count), &shapes); !err.empty()) {
    icore::set_error(err);
    return none;
  }
  const size_t count = shapes.size();
  auto* tensors = static_cast<i_owned_tensor*>(std::calloc(count ? count : 1, sizeof(i_owned_tensor)));
  std::vector<float*> out_ptrs;
  bool ok = tensors != nullptr;
  for (size_t o = 0; ok && o < count; ++o) {
    size_t len = 1;
    for (size_t d : shapes[o]) len *= d;
    tensors[o].rank = shapes[o].size();
    tensors[o].len = len;
    tensors[o].data = static_cast<float*>(std::calloc(len ? len : 1, sizeof(float)));  // zero-filled, as the reference
    tensors[o].shape = static_cast<size_t*>(std::calloc(shapes[o].size() ? shapes[o].size() : 1, sizeof(size_t)));
    ok = tensors[o].data && tensors[o].shape;
    if (ok) std::copy(shapes[o].begin(), shapes[o].end(), tensors[o].shape);
    out_ptrs.push_back(tensors[o].data);
  }
  i_outputs result{tensors, count};
  std::string err = ok ? run_host(p, inputs, input_count, out_ptrs) : std::string("out of memory");
  if (!err.empty()) {
    i_outputs_free(result);
    icore::set_error(err);
    return none;
  }
  return result;
}

int i_exec_into_device(const i_program* program, const i_device_tensor* inputs, size_t input_count,
                       const i_device_tensor* outputs, size_t output_count, void* stream) {
  std::vector<ihipc::DeviceTensor> in, out;
  if (!device_call_ok(program, inputs, input_count, outputs, output_count, &in, &out)) return -1;
  try {
    const std::string err = ihipc::execute(*program->inner, in, out, static_cast<hipStream_t>(stream));
    return err.empty() ? 0 : fail(err);
  } catch (const std::exception& e) {
    return fail(e.what());
  }
}

int i_exec_into_device_noalloc(const i_program* program, const i_device_tensor* inputs, size_t input_count,
                               const i_device_tensor* outputs, size_t output_count, void* stream) {
  std::vector<ihipc::DeviceTensor> in, out;
  if (!device_call_ok(program, inputs, input_count, outputs, output_count, &in, &out)) return -1;
  try {
    // set-up, once per device: the address of this device's copy of the static workspace
    void* base = nullptr;
    if (ihip::Err e = ihip::static_scratch(&base); !e.empty()) return fail(e);
    // size the temporaries first, so that a program that does not fit is refused before anything is enqueued
    // (with the temporaries of split loops first; when that is too much, without them: the loops then run whole)
    size_t need = 0;
    bool refuse_optional = false;
    if (std::string e = ihipc::workspace_bytes(*program->inner, in, out, &need); !e.empty()) return fail(e);
    if (need > ihip::kStaticScratchBytes) {
      refuse_optional = true;
      if (std::string e = ihipc::workspace_bytes(*program->inner, in, out, &need, true); !e.empty()) return fail(e);
    }
    if (need > ihip::kStaticScratchBytes)
      return fail("program needs " + std::to_string(need) + " bytes of temporaries for these operands, the static workspace holds " +
                  std::to_string(ihip::kStaticScratchBytes) + " (use i_exec_into_device)");
    ihipc::Workspace ws{base, ihip::kStaticScratchBytes, 0, refuse_optional};
    const std::string err = ihipc::execute(*program->inner, in, out, static_cast<hipStream_t>(stream), &ws);
    return err.empty() ? 0 : fail(err);
  } catch (const std::exception& e) {
    return fail(e.what());
  }
}

size_t i_hip_release_cached_memory(void) {
  size_t released = ihipc::release_stream_blocks();
  released += release_staging_blocks();
  released += ihip::release_copy_chunks();
  released += ihip::trim_temp_pool();
  return released;
}

int i_hip_program_option(i_program* program, const char* name, int value) {
  if (!program) return fail("null program");
  if (!name) return fail("null option name");
  const std::string err = ihipc::set_option(*program->inner, name, value);
  return err.empty() ? 0 : fail(err);
}

int i_hip_program_clock_probe(i_program* program, void* ticks) {
  if (!program) return fail("null program");
  const std::string err = ihipc::set_clock_probe(*program->inner, ticks);
  return err.empty() ? 0 : fail(err);
}

int i_hip_program_row_slices(const i_program* program, unsigned char* sliced, size_t capacity) {
  if (!program) {
    icore::set_error("null program");
    return -1;
  }
  std::vector<char> flags;
  if (!ihipc::row_sliceable(*program->inner, &flags)) return 0;
  if (sliced && capacity < flags.size()) {
    icore::set_error("the program has " + std::to_string(flags.size()) + " inputs");
    return -1;
  }
  for (size_t i = 0; sliced && i < flags.size(); ++i) sliced[i] = flags[i] ? 1 : 0;
  return (int)flags.size();
}

char* i_hip_program_report(const i_program* program) {
  if (!program) {
    icore::set_error("null program");
    return nullptr;
  }
  const std::string text = ihipc::last_report(*program->inner);
  char* out = static_cast<char*>(std::malloc(text.size() + 1));
  if (!out) {
    icore::set_error("out of memory");
    return nullptr;
  }
  std::memcpy(out, text.c_str(), text.size() + 1);
  return out;
}

void i_component_free(i_component* component) { delete component; }

void i_program_free(i_program* program) { delete program; }

void i_outputs_free(i_outputs outputs) {
  if (!outputs.tensors) return;
  for (size_t i = 0; i < outputs.count; ++i) {
    std::free(outputs.tensors[i].data);
    std::free(outputs.tensors[i].shape);
  }
  std::free(outputs.tensors);
}

void i_string_free(char* s) { std::free(s); }

const char* i_error(void) { return icore::last_error(); }

}  // extern "C"
#pragma GCC visibility pop
