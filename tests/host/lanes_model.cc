// The two lanes of a program on modelled hardware queues (CPU only; built by tests/test_lanes_model.py with context.cc, lanes.hip
// and the HIP calls below in the place of the runtime).
//
// Streams are dealt out to four hardware queues, the least loaded first; a queue runs what its streams hold in the order it
// was submitted, waits for events included.  Every launch takes the time its argument says, so the moment each one starts
// is known as soon as it is submitted.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <string>
#include <vector>

#include "../../sirius_amd/csrc/context.h"

// ---------------------------------------------------------------------------------------------- the modelled runtime
namespace {
constexpr int kQueues = 4;
struct Stream {
  int queue;
};
struct Event {
  double done = 0.0;   // when the last record of it is reached; one that was never recorded holds nobody up
};
struct Span {
  double start, end;
};
struct Launch {        // the argument of every launch
  int id;
  double duration;
};
std::mutex g_mu;
double g_time[kQueues];
int g_load[kQueues];
std::vector<Span> g_spans;
int g_streams_alive = 0, g_events_alive = 0;

Stream* as_stream(hipStream_t s) { return reinterpret_cast<Stream*>(s); }
Event* as_event(hipEvent_t e) { return reinterpret_cast<Event*>(e); }

// another thread captures a graph in global mode: calls that may disturb a capture are refused unless the calling thread
// has taken itself out of it, and the null stream may not be touched at all
bool g_captured_elsewhere = false;
thread_local hipStreamCaptureMode g_mode = hipStreamCaptureModeGlobal;
std::string g_disturbed;
hipError_t unsafe(const char* call, bool null_stream = false) {
  if (!g_captured_elsewhere || (g_mode == hipStreamCaptureModeRelaxed && !null_stream)) return hipSuccess;
  g_disturbed = call;
  return hipErrorStreamCaptureUnsupported;
}

// the two kernels of a question (lanes.hip): they meet if they were given to different queues
const void* g_handshake_kernel = nullptr;
unsigned* g_answer = nullptr;
hipStream_t g_asked_first = nullptr;
void handshake(void** args, hipStream_t s) {
  unsigned token;
  int polls;
  memcpy(&token, args[3], sizeof(token));
  memcpy(&polls, args[4], sizeof(polls));
  if (polls == 0) return;
  if (!g_asked_first) {
    g_asked_first = s;
    return;
  }
  const bool met = as_stream(s)->queue != as_stream(g_asked_first)->queue;
  g_asked_first = nullptr;
  if (g_answer) g_answer[0] = met ? token : 0, g_answer[1] = token;   // the one that comes second sees the other's flag either way
}


void reset(const int* load) {
  std::lock_guard<std::mutex> lock(g_mu);
  for (int q = 0; q < kQueues; ++q) {
    g_time[q] = 0.0;
    g_load[q] = load ? load[q] : 0;
  }
  g_spans.clear();
}
}  // namespace

extern "C" {
hipError_t hipStreamCreateWithFlags(hipStream_t* out, unsigned) {
  if (unsafe("hipStreamCreateWithFlags") != hipSuccess) return hipErrorStreamCaptureUnsupported;
  std::lock_guard<std::mutex> lock(g_mu);
  const int q = static_cast<int>(std::min_element(g_load, g_load + kQueues) - g_load);
  ++g_load[q];
  ++g_streams_alive;
  *out = reinterpret_cast<hipStream_t>(new Stream{q});
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  std::lock_guard<std::mutex> lock(g_mu);
  --g_load[as_stream(s)->queue];
  --g_streams_alive;
  delete as_stream(s);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* out, unsigned) {
  std::lock_guard<std::mutex> lock(g_mu);
  ++g_events_alive;
  *out = reinterpret_cast<hipEvent_t>(new Event);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* out) { return hipEventCreateWithFlags(out, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
  std::lock_guard<std::mutex> lock(g_mu);
  --g_events_alive;
  delete as_event(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  std::lock_guard<std::mutex> lock(g_mu);
  as_event(e)->done = g_time[as_stream(s)->queue];
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  std::lock_guard<std::mutex> lock(g_mu);
  double& t = g_time[as_stream(s)->queue];
  t = std::max(t, as_event(e)->done);
  return hipSuccess;
}
hipError_t hipExtLaunchKernel(const void*, dim3, dim3, void** args, size_t, hipStream_t s, hipEvent_t, hipEvent_t stop, int) {
  std::lock_guard<std::mutex> lock(g_mu);
  Launch what;
  memcpy(&what, args[0], sizeof(what));
  double& t = g_time[as_stream(s)->queue];
  if (g_spans.size() <= static_cast<size_t>(what.id)) g_spans.resize(static_cast<size_t>(what.id) + 1);
  g_spans[static_cast<size_t>(what.id)] = Span{t, t + what.duration};
  t += what.duration;
  if (stop) as_event(stop)->done = t;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* fn, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t s) {
  if (fn == g_handshake_kernel) {
    handshake(args, s);
    return hipSuccess;
  }
  return hipExtLaunchKernel(fn, grid, block, args, lds, s, nullptr, nullptr, 0);
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float*, hipEvent_t, hipEvent_t) { return hipErrorNotSupported; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st) {
  *st = hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "modelled"; }
hipError_t hipDeviceGetAttribute(int*, hipDeviceAttribute_t, int) { return hipErrorNotSupported; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* mode) {
  std::swap(*mode, g_mode);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (unsafe("hipHostMalloc") != hipSuccess) return hipErrorStreamCaptureUnsupported;
  *p = g_answer = static_cast<unsigned*>(calloc(1, n));
  return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** out, void* p, unsigned) {
  *out = p;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static unsigned flags[4];
  *p = flags;
  return hipSuccess;
}
hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return unsafe("hipMemcpy", true); }
// what the compiler emits for a file with kernels
void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  if (strstr(name, "handshake_kernel")) g_handshake_kernel = host;
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
namespace {
struct {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
} g_call;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
  g_call = {grid, block, lds, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) {
  *grid = g_call.grid;
  *block = g_call.block;
  *lds = g_call.lds;
  *s = g_call.stream;
  return hipSuccess;
}
hipError_t hipExtStreamCreateWithCUMask(hipStream_t* out, uint32_t, const uint32_t*) { return hipStreamCreateWithFlags(out, 0); }
}  // extern "C"

// ------------------------------------------------------------------------------------------------------- the checks
namespace {
using namespace tch;
int g_failures = 0;

void expect(bool ok, const std::string& what) {
  if (!ok && ++g_failures <= 20) fprintf(stderr, "FAILED: %s\n", what.c_str());
}

int on_other_queues(hipStream_t a, hipStream_t b) { return as_stream(a)->queue != as_stream(b)->queue; }

void launch(Context* ctx, int id, double duration) {
  Launch what{id, duration};
  submit(ctx, reinterpret_cast<const void*>(&g_failures), dim3(1), dim3(64), &what, sizeof(what), "kernel", 0.0, 1, 0.0);
}

// Ten sections of a main-lane kernel, a second-lane kernel that waits for it, and another main-lane kernel, with a join one
// point behind after each: a section starts when the main lane and the second lane's work of the section before the
// last one have ended -- not before, and not later, whatever streams the process has besides.
void lanes_one_point_behind(const int* load, bool through_queue) {
  reset(load);
  constexpr int kSections = 10;
  const double side_us[kSections] = {40, 5, 12, 60, 3, 25, 25, 8, 90, 10};
  hipStream_t main = nullptr;
  (void)hipStreamCreateWithFlags(&main, 0);
  {
    Context ctx(main);
    ctx.streams_meet = on_other_queues;
    Program prog;
    ctx.recording = &prog;
    for (int k = 0; k < kSections; ++k) {
      launch(&ctx, 3 * k, 10.0);
      ctx.lane = 1;
      ctx.wait_main = true;
      launch(&ctx, 3 * k + 1, side_us[k]);
      ctx.lane = 0;
      ctx.wait_main = false;
      launch(&ctx, 3 * k + 2, 5.0);
      ctx.record_join(true);
    }
    ctx.record_join();
    launch(&ctx, 3 * kSections, 1.0);
    ctx.recording = nullptr;
    ctx.prepare_lanes(prog);
    if (through_queue) ctx.queue = std::make_shared<LaunchQueue>(main, 16, 4);
    char where[96];
    snprintf(where, sizeof(where), "load %d %d %d %d, %s", load[0], load[1], load[2], load[3], through_queue ? "queue" : "direct");
    for (int replay = 0; replay < 2; ++replay) {
      for (size_t i = 0; i < prog.launches.size(); ++i)
        expect(ctx.dispatch(prog.launches[i], i + 1 < prog.launches.size() ? &prog.launches[i + 1] : nullptr) == 0, where);
      if (ctx.queue) expect(ctx.queue->synchronize() == 0, where);
      const std::vector<Span> at = g_spans;
      expect(at.size() == 3 * kSections + 1, where);
      for (int k = 0; k < kSections; ++k) {
        const std::string which = std::string(where) + ", section " + std::to_string(k);
        expect(at[3 * k + 1].start == std::max(at[3 * k].end, k ? at[3 * k - 2].end : 0.0), which + ": second lane");
        if (k >= 1)
          expect(at[3 * k].start == std::max(at[3 * k - 1].end, k >= 2 ? at[3 * (k - 2) + 1].end : 0.0), which + ": main lane");
      }
      expect(at[3 * kSections].start == std::max(at[3 * kSections - 1].end, at[3 * kSections - 2].end), std::string(where) + ": join");
    }
    ctx.queue.reset();
  }
  (void)hipStreamDestroy(main);
  expect(g_streams_alive == 0 && g_events_alive == 0, "streams or events left behind");
}

// ---- which stream becomes the second lane, with the answers of the streams given
std::vector<int> g_answers;   // one per ask; the last one for all that follow
size_t g_asked = 0;
int scripted(hipStream_t, hipStream_t) { return g_answers[std::min(g_asked++, g_answers.size() - 1)]; }

void record_two_lanes(Context* ctx, Program* prog) {
  ctx->recording = prog;
  launch(ctx, 0, 10.0);
  ctx->lane = 1;
  ctx->wait_main = true;
  launch(ctx, 1, 40.0);
  ctx->lane = 0;
  ctx->wait_main = false;
  launch(ctx, 2, 5.0);
  ctx->recording = nullptr;
  ctx->prepare_lanes(*prog);
}

void choice(const char* name, std::vector<int> answers, bool shown, size_t asks, size_t asks_later, bool shown_later) {
  reset(nullptr);
  g_answers = answers;
  g_asked = 0;
  hipStream_t main = nullptr;
  (void)hipStreamCreateWithFlags(&main, 0);
  {
    Context ctx(main);
    ctx.streams_meet = scripted;
    Program first, later;
    record_two_lanes(&ctx, &first);
    expect(ctx.side && ctx.side_shown == shown, std::string(name) + ": shown");
    expect(g_asked == asks, std::string(name) + ": asks " + std::to_string(g_asked));
    expect(g_streams_alive == 2, std::string(name) + ": refused streams are given back");
    for (auto& l : first.launches) expect(ctx.dispatch(l) == 0, name);
    const Span before = g_spans[1];
    g_asked = asks;
    for (int i = 0; i < 10; ++i) record_two_lanes(&ctx, &later);   // new plans
    expect(ctx.side_shown == shown_later, std::string(name) + ": shown later");
    expect(g_asked == asks_later, std::string(name) + ": asks later " + std::to_string(g_asked));
    expect(g_streams_alive <= 3, std::string(name) + ": streams");
    for (auto& l : first.launches) expect(ctx.dispatch(l) == 0, name);
    expect(g_spans[1].start >= before.end, std::string(name) + ": a new second lane starts where the old one stands");
  }
  (void)hipStreamDestroy(main);
  expect(g_streams_alive == 0 && g_events_alive == 0, std::string(name) + ": left behind");
}

// A recording that ends while another thread captures a graph: the second lane is chosen as ever, and no call disturbs the capture.
void beside_a_capture(const int* load) {
  reset(load);
  hipStream_t main = nullptr;
  (void)hipStreamCreateWithFlags(&main, 0);
  {
    Context ctx(main);
    ctx.streams_meet = run_at_the_same_time;
    Program prog;
    g_captured_elsewhere = true;
    g_disturbed.clear();
    record_two_lanes(&ctx, &prog);
    g_captured_elsewhere = false;
    expect(g_disturbed.empty(), "a capture in another thread is disturbed by " + g_disturbed);
    expect(g_mode == hipStreamCaptureModeGlobal, "the thread's capture mode is put back");
    expect(ctx.side && ctx.side_shown && on_other_queues(main, ctx.side), "second lane beside a capture");
  }
  (void)hipStreamDestroy(main);
}
}  // namespace

int main() {
  int cases = 0;
  constexpr int kAsks = Context::kAsks, kAll = Context::kAsks * Context::kCandidates;
  choice("meets at once", {1}, true, 1, 1, true);
  choice("missed, but meets when asked again", {0, 0, 1}, true, 3, 3, true);
  choice("shares the queue, the next one does not", {0, 0, 0, 1}, true, kAsks + 1, kAsks + 1, true);
  std::vector<int> last(kAll, 0);
  last[kAll - 1] = 1;
  choice("only the last one meets", last, true, kAll, kAll, true);
  choice("none ever meets", {0}, false, kAll, kAll * Context::kLooks, false);
  std::vector<int> later(kAll, 0);
  later.push_back(1);
  choice("chip held by another tenant at first", later, false, kAll, kAll + 1, true);
  choice("cannot be asked", {-1}, false, 1, Context::kLooks, false);
  cases += 7;
  for (int l = 0; l < 81; ++l) {
    const int load[kQueues] = {l % 3, l / 3 % 3, l / 9 % 3, l / 27};
    for (bool through_queue : {false, true}) {
      lanes_one_point_behind(load, through_queue);
      ++cases;
    }
    beside_a_capture(load);
    ++cases;
  }
  printf("%d cases, %d failures\n", cases, g_failures);
  return g_failures ? 1 : 0;
}
