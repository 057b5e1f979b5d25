// session.hip -- resident decoder sessions: the exported calls that do not depend on
// the model, and the part of a session every model shares.
//
// Takes the place of the generated ModelSession
// (tools/buddy-codegen/gen_session.py:1381-1452) and of the greedy part of the
// decode loop (runtime/llm/TextGeneration.cpp:215-266, Sampler.h:101-104).  Token
// id, position and step counter live in device memory, so a whole decode step is
// captured once into a hipGraph and replayed; greedy decoding feeds the argmax
// straight into the next step's embedding gather without a host round trip.
#include "session_base.h"

#include <algorithm>
#include <chrono>
#include <cstring>
#include <thread>
#include <vector>

namespace bh {
namespace {

constexpr size_t kGivenWord = 4, kHostWords = 8; // what is given, the logits in the pinned buffer

// State and n logits into the pinned buffer: one launch in place of a copy of the state and
// one of the logits through the runtime's staging, which blocks.  With the state of the
// step written by a kernel that the host does not wait for, 24 steps of a model of four
// layers behind a prompt of 45, each with its logits, took 7277 us instead of 7975.
__global__ void __launch_bounds__(256)
hand_out_kernel(const int *__restrict__ state, const float *__restrict__ logits, int n,
                int *__restrict__ out, int *__restrict__ done) {
  const int i = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (i == 0)
    for (int w = 0; w < 3; ++w)
      out[w] = state[w];
  float *dst = reinterpret_cast<float *>(out + kHostWords);
  if (i + 3 < n)
    *reinterpret_cast<float4 *>(dst + i) = *reinterpret_cast<const float4 *>(logits + i);
  else
    for (int e = i; e < n; ++e)
      dst[e] = logits[e];
  if (!done)
    return;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // a fence of all: 22 us for 608 KB, not 16
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(done + blockIdx.x, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
size_t done_word(int vocab) { return kHostWords + (size_t)round_up(vocab, 4); }
int hand_blocks(int n) { return (int)std::max<int64_t>(1, ceil_div(n, 1024)); }

// Memory that the runtime does not know: a copy to it goes through a buffer of its own,
// piece by piece, and blocks.
bool pageable(const void *p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

} // namespace

Session::~Session() {
  if (stream)
    (void)hipStreamSynchronize(stream);
  for (StepGraphs &kept : graphs)
    drop_graphs(kept);
  for (void *p : owned)
    (void)hipFree(p);
  if (host_state)
    (void)hipHostFree(host_state);
  if (own_stream)
    (void)hipStreamDestroy(stream);
}

int Session::init(int vocab_size, int capacity, hipStream_t on_stream) {
  vocab = vocab_size;
  max_len = capacity;
  stream = on_stream;
  if (!stream) {
    BH_CHECK_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    own_stream = true;
  }
  const size_t groups = (size_t)ceil_div(vocab, kTileN);
  token_log_cap = 65536;
  int rc = alloc(&logits, groups * kTileN);
  rc |= alloc(&state, 4);
  rc |= alloc(&token_log, (size_t)token_log_cap);
  rc |= alloc((char **)&amax_ws, argmax_workspace_bytes());
  rc |= alloc(&group_max_v, groups);
  rc |= alloc(&group_max_i, groups);
  if (rc)
    return rc;
  BH_CHECK_HIP(hipHostMalloc((void **)&host_state, 4 * (done_word(vocab) + (size_t)hand_blocks(vocab)),
                             hipHostMallocCoherent));
  BH_CHECK_HIP(hipMemsetAsync(state, 0, 4 * sizeof(int), stream));
  BH_CHECK_HIP(hipStreamSynchronize(stream));
  return BUDDY_HIP_OK;
}

void Session::drop_graphs(StepGraphs &kept) {
  for (auto &kv : kept) {
    if (kv.second.exec)
      (void)hipGraphExecDestroy(kv.second.exec);
    if (kv.second.graph)
      (void)hipGraphDestroy(kv.second.graph);
  }
  kept.clear();
}

// The position and step the device holds must stay inside the cache and the
// token log for every one of `steps` further steps.
int Session::check_steps(int steps, const char *who) const {
  BH_REQUIRE(next_pos >= 0, "%s: no token / position set (set_state first)", who);
  BH_REQUIRE(steps > 0 && (int64_t)next_pos + steps <= max_len,
             "%s: %d step(s) from position %d leave the cache (max_len %d)", who, steps,
             next_pos, max_len);
  BH_REQUIRE((int64_t)next_step + steps <= token_log_cap,
             "%s: %d step(s) from step %d overflow the token log (%d entries)", who,
             steps, next_step, token_log_cap);
  return BUDDY_HIP_OK;
}

int Session::enqueue_whole_step(bool hands) {
  int rc = BUDDY_HIP_OK;
  if (hands)
    rc = prepare_step({-1, 0, 0, host_state + kGivenWord});
  if (!rc)
    rc = enqueue_step(next_pos);
  return rc || !hands ? rc : enqueue_hand_out(vocab, true);
}

int Session::run_step(bool hands) {
  int rc = check_steps(1, "decode step");
  if (rc)
    return rc;
  if (!use_graph) {
    rc = enqueue_whole_step(hands);
  } else {
    const std::pair<int, int> key = step_key(next_pos);
    StepGraphs &kept = graphs[hands];
    auto it = kept.find(key);
    if (it == kept.end()) {
      if (kept.size() >= kMaxStepGraphs) {
        BH_CHECK_HIP(hipStreamSynchronize(stream)); // a replay may still be running
        drop_graphs(kept);
      }
      it = kept.emplace(key, StepGraph{}).first;
    }
    StepGraph &g = it->second;
    if (!g.exec) {
      BH_CHECK_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
      rc = enqueue_whole_step(hands);
      hipError_t e = hipStreamEndCapture(stream, &g.graph);
      if (!rc && e != hipSuccess)
        rc = fail(BUDDY_HIP_ERR_HIP, "hipStreamEndCapture: %s", hipGetErrorString(e));
      if (!rc && (e = hipGraphInstantiate(&g.exec, g.graph, nullptr, nullptr, 0)) != hipSuccess)
        rc = fail(BUDDY_HIP_ERR_HIP, "hipGraphInstantiate: %s", hipGetErrorString(e));
      if (rc) {
        drop_graphs(kept); // a half-built graph is not kept
        return rc;
      }
    }
    BH_CHECK_HIP(hipGraphLaunch(g.exec, stream));
  }
  if (!rc) {
    ++next_pos;
    ++next_step;
    stepped();
  }
  return rc;
}

// The captured step has kernel arguments baked in (weight, cache and embedding
// pointers): whoever may change one of them drops the graph first, and the
// next step captures a new one.
int Session::invalidate_graph() {
  for (StepGraphs &kept : graphs)
    if (!kept.empty()) {
      BH_CHECK_HIP(hipStreamSynchronize(stream));
      drop_graphs(kept);
    }
  return BUDDY_HIP_OK;
}

int Session::set_state(int token, int pos, int step) {
  int rc = seek(pos);
  if (rc)
    return rc;
  next_pos = pos;
  next_step = step;
  return prepare_step({token, pos, step});
}

int *Session::hand_done() const { return host_state + done_word(vocab); }

int Session::enqueue_hand_out(int n, bool says) {
  hipLaunchKernelGGL(hand_out_kernel, dim3((unsigned)hand_blocks(n)), dim3(256), 0, stream, state,
                     logits, n, host_state, says ? hand_done() : nullptr);
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}

// Its last kernel says in the pinned buffer that it is there.  The words are looked at for up to
// look_us; a step that takes longer, or has failed, is waited for (and reported) by the runtime, whose
// wait sleeps and takes up to 20 us to come back, and so are the steps behind it but every sixteenth,
// which looks whether steps have become shorter.
int Session::wait_hand_out(int n) {
  constexpr int kYieldUs = 100, kLooksSkipped = 15;
  const int blocks = hand_blocks(n);
  if (!look_us || looks_skipped > 0) {
    looks_skipped -= looks_skipped > 0;
    BH_CHECK_HIP(hipStreamSynchronize(stream));
    return BUDDY_HIP_OK;
  }
  const auto t0 = std::chrono::steady_clock::now();
  for (int b = 0; b < blocks;) {
    if (__atomic_load_n(hand_done() + b, __ATOMIC_ACQUIRE)) {
      ++b;
      continue;
    }
    const auto us = std::chrono::duration_cast<std::chrono::microseconds>(std::chrono::steady_clock::now() - t0);
    if (us.count() > look_us) {
      looks_skipped = kLooksSkipped;
      BH_CHECK_HIP(hipStreamSynchronize(stream));
      return BUDDY_HIP_OK;
    }
    if (us.count() > kYieldUs)
      std::this_thread::yield();
  }
  return BUDDY_HIP_OK;
}

int Session::hand_out(float *logits_out, int *next_token) {
  const bool staged = logits_out && pageable(logits_out);
  if (logits_out && !staged)
    BH_CHECK_HIP(hipMemcpyAsync(logits_out, logits, sizeof(float) * vocab, hipMemcpyDefault,
                                stream));
  const int n = staged ? vocab : 0;
  if (int rc = enqueue_hand_out(n, false))
    return rc;
  // (A prompt is waited for by the runtime: looking gained nothing there, and whoever waits for the
  // device behind it has the runtime's wait all the same, up to 50 us of a prompt of 2 tokens.)
  BH_CHECK_HIP(hipStreamSynchronize(stream));
  if (staged)
    std::memcpy(logits_out, host_state + kHostWords, sizeof(float) * vocab);
  if (next_token)
    *next_token = host_state[0];
  return BUDDY_HIP_OK;
}

int Session::step_and_hand_out(int token, int pos, float *logits_out, int *next_token) {
  // a step that other calls have captured serves the first of these too: capturing costs some 400 us
  bool apart = !logits_out || !pageable(logits_out);
  if (!apart && use_graph) {
    const auto it = graphs[0].find(step_key(pos));
    if (it != graphs[0].end() && !it->second.handed)
      apart = it->second.handed = true;
  }
  int rc;
  if (apart) {
    if ((rc = set_state(token, pos, 0)) || (rc = run_step()))
      return rc;
    return hand_out(logits_out, next_token);
  }
  if ((rc = seek(pos)))
    return rc;
  next_pos = pos;
  next_step = 0;
  int *given = host_state + kGivenWord;
  given[0] = token;
  given[1] = pos;
  given[2] = 0;
  std::fill_n(hand_done(), hand_blocks(vocab), 0);
  if ((rc = run_step(true)) || (rc = wait_hand_out(vocab)))
    return rc;
  std::memcpy(logits_out, host_state + kHostWords, sizeof(float) * vocab);
  if (next_token)
    *next_token = host_state[0];
  return BUDDY_HIP_OK;
}

} // namespace bh

using bh::Session;

extern "C" {

void buddy_hip_session_destroy(buddy_hip_session *hs) try {
  delete bh::as_session(hs);
} BH_CATCH_VOID("buddy_hip_session_destroy")

int buddy_hip_session_use_graph(buddy_hip_session *hs, int enable) try {
  Session *s = bh::as_session(hs);
  BH_REQUIRE(s, "session_use_graph: null session");
  s->use_graph = enable != 0;
  return BUDDY_HIP_OK;
} BH_CATCH_INT("buddy_hip_session_use_graph")

int buddy_hip_session_set_look_us(buddy_hip_session *hs, int us) try {
  Session *s = bh::as_session(hs);
  BH_REQUIRE(s, "session_set_look_us: null session");
  BH_REQUIRE(us >= 0, "session_set_look_us: %d us", us);
  s->look_us = us;
  s->looks_skipped = 0;
  return BUDDY_HIP_OK;
} BH_CATCH_INT("buddy_hip_session_set_look_us")

int buddy_hip_session_decode_mirror(buddy_hip_session *hs, int token, int pos,
                                    float *logits_out, float *kv_rows_out,
                                    int *next_token) try {
  Session *s = bh::as_session(hs);
  BH_REQUIRE(s, "session_decode: null session");
  int rc = s->ready();
  if (rc)
    return rc;
  BH_REQUIRE(token >= 0 && token < s->vocab, "session_decode: token %d", token);
  BH_REQUIRE(pos >= 0 && pos < s->max_len,
             "session_decode: position %d outside the cache (max_len %d)", pos,
             s->max_len);
  if (!kv_rows_out)
    return s->step_and_hand_out(token, pos, logits_out, next_token);
  // and the cache rows this step wrote, all layers
  if ((rc = s->set_state(token, pos, 0)) || (rc = s->run_step()) || (rc = s->copy_kv_rows(pos, 1, kv_rows_out)))
    return rc;
  return s->hand_out(logits_out, next_token);
} BH_CATCH_INT("buddy_hip_session_decode_mirror")

int buddy_hip_session_decode(buddy_hip_session *hs, int token, int pos,
                             float *logits_out, int *next_token) {
  return buddy_hip_session_decode_mirror(hs, token, pos, logits_out, nullptr, next_token);
}

int buddy_hip_session_decode_greedy(buddy_hip_session *hs, int first_token,
                                    int start_pos, int steps, int *tokens_out) try {
  Session *s = bh::as_session(hs);
  BH_REQUIRE(s && tokens_out, "session_decode_greedy: null argument");
  int rc = s->ready();
  if (rc)
    return rc;
  BH_REQUIRE(first_token >= 0 && first_token < s->vocab,
             "session_decode_greedy: token %d", first_token);
  BH_REQUIRE(steps > 0 && steps <= s->token_log_cap,
             "session_decode_greedy: steps %d", steps);
  BH_REQUIRE(start_pos >= 0 && start_pos + steps <= s->max_len,
             "session_decode_greedy: positions %d..%d outside the cache (max_len %d)",
             start_pos, start_pos + steps - 1, s->max_len);
  if ((rc = s->set_state(first_token, start_pos, 0)))
    return rc;
  for (int i = 0; i < steps; ++i)
    if ((rc = s->run_step()))
      return rc;
  BH_CHECK_HIP(hipMemcpyAsync(tokens_out, s->token_log, sizeof(int) * steps,
                              hipMemcpyDefault, s->stream));
  BH_CHECK_HIP(hipStreamSynchronize(s->stream));
  return BUDDY_HIP_OK;
} BH_CATCH_INT("buddy_hip_session_decode_greedy")

int buddy_hip_session_prefill(buddy_hip_session *hs, const int *tokens,
                              int n_tokens, int start_pos, float *logits_out,
                              int *next_token) try {
  Session *s = bh::as_session(hs);
  BH_REQUIRE(s && tokens, "session_prefill: null argument");
  int rc = s->ready();
  if (rc)
    return rc;
  BH_REQUIRE(n_tokens > 0 && start_pos >= 0 && start_pos + n_tokens <= s->max_len,
             "session_prefill: tokens %d..%d outside the cache (max_len %d)",
             start_pos, start_pos + n_tokens - 1, s->max_len);
  const int last = n_tokens - 1;
  if ((rc = s->prefill_rows(tokens, n_tokens, start_pos, &last, 1, s->logits)))
    return rc;
  if ((rc = bh::launch_argmax(s->logits, s->vocab, s->amax_ws, s->state, nullptr,
                              nullptr, s->stream)))
    return rc;
  return s->hand_out(logits_out, next_token);
} BH_CATCH_INT("buddy_hip_session_prefill")

int buddy_hip_session_prefill_rows(buddy_hip_session *hs, const int *tokens, int n_tokens,
                                   int start_pos, const int *rows, int n_rows,
                                   float *logits_out) try {
  Session *s = bh::as_session(hs);
  BH_REQUIRE(s && tokens && n_rows >= 0 && (n_rows == 0 || (rows && logits_out)),
             "session_prefill_rows: null argument");
  int rc = s->ready();
  if (rc)
    return rc;
  BH_REQUIRE(n_tokens > 0 && start_pos >= 0 && (int64_t)start_pos + n_tokens <= s->max_len,
             "session_prefill_rows: tokens %d..%d outside the cache (max_len %d)", start_pos,
             start_pos + n_tokens - 1, s->max_len);
  for (int i = 0; i < n_rows; ++i)
    BH_REQUIRE(rows[i] >= 0 && rows[i] < n_tokens && (i == 0 || rows[i] > rows[i - 1]),
               "session_prefill_rows: rows must ascend within the tokens");
  float *dev = nullptr;
  const size_t bytes = sizeof(float) * (size_t)n_rows * s->vocab;
  if (n_rows)
    BH_CHECK_HIP(hipMalloc((void **)&dev, bytes));
  rc = s->prefill_rows(tokens, n_tokens, start_pos, rows, n_rows, dev);
  if (!rc && n_rows &&
      hipMemcpyAsync(logits_out, dev, bytes, hipMemcpyDefault, s->stream) != hipSuccess)
    rc = bh::fail(BUDDY_HIP_ERR_HIP, "session_prefill_rows: copy failed");
  const hipError_t e = hipStreamSynchronize(s->stream);
  if (!rc && e != hipSuccess)
    rc = bh::fail(BUDDY_HIP_ERR_HIP, "session_prefill_rows: %s", hipGetErrorString(e));
  if (dev)
    (void)hipFree(dev);
  return rc;
} BH_CATCH_INT("buddy_hip_session_prefill_rows")

int buddy_hip_session_prefill_all_logits(buddy_hip_session *hs, const int *tokens,
                                         int n_tokens, int start_pos,
                                         float *logits_out) try {
  BH_REQUIRE(hs && tokens && logits_out && n_tokens > 0,
             "session_prefill_all_logits: bad argument");
  std::vector<int> rows((size_t)n_tokens);
  for (int i = 0; i < n_tokens; ++i)
    rows[(size_t)i] = i;
  return buddy_hip_session_prefill_rows(hs, tokens, n_tokens, start_pos, rows.data(), n_tokens,
                                        logits_out);
} BH_CATCH_INT("buddy_hip_session_prefill_all_logits")

void buddy_hip_session_adopt(buddy_hip_session *hs, void *device_ptr) try {
  Session *s = bh::as_session(hs);
  if (s && device_ptr)
    s->owned.push_back(device_ptr);
} BH_CATCH_VOID("buddy_hip_session_adopt")

int buddy_hip_session_enqueue_steps(buddy_hip_session *hs, int steps) try {
  Session *s = bh::as_session(hs);
  BH_REQUIRE(s && steps > 0, "session_enqueue_steps: bad argument");
  int rc = s->ready();
  if (rc)
    return rc;
  // refused as a whole: no step is enqueued when the last one would not fit
  if ((rc = s->check_steps(steps, "session_enqueue_steps")))
    return rc;
  for (int i = 0; i < steps; ++i)
    if ((rc = s->run_step()))
      return rc;
  return BUDDY_HIP_OK;
} BH_CATCH_INT("buddy_hip_session_enqueue_steps")

int buddy_hip_session_set_state(buddy_hip_session *hs, int token, int pos) try {
  Session *s = bh::as_session(hs);
  BH_REQUIRE(s, "session_set_state: null session");
  BH_REQUIRE(token >= 0 && token < s->vocab && pos >= 0 &&
                 pos < s->max_len,
             "session_set_state: token %d / position %d out of range", token, pos);
  int rc = s->ready();
  if (rc)
    return rc;
  if ((rc = s->set_state(token, pos, 0)))
    return rc;
  BH_CHECK_HIP(hipStreamSynchronize(s->stream));
  return BUDDY_HIP_OK;
} BH_CATCH_INT("buddy_hip_session_set_state")

const float *buddy_hip_session_logits(buddy_hip_session *hs) {
  Session *s = bh::as_session(hs);
  return s ? s->logits : nullptr;
}

int buddy_hip_session_reset(buddy_hip_session *hs) try {
  Session *s = bh::as_session(hs);
  BH_REQUIRE(s, "session_reset: null session");
  s->next_pos = -1; // the next step needs a token and a position first
  return s->reset();
} BH_CATCH_INT("buddy_hip_session_reset")

const char *buddy_hip_session_architecture(buddy_hip_session *hs) {
  return hs ? bh::as_session(hs)->architecture() : nullptr;
}

int buddy_hip_session_vocab(buddy_hip_session *hs) try {
  Session *s = bh::as_session(hs);
  return s ? s->vocab : 0;
} BH_CATCH_INT("buddy_hip_session_vocab")

buddy_hip_stream buddy_hip_session_stream(buddy_hip_session *hs) {
  Session *s = bh::as_session(hs);
  return s ? reinterpret_cast<buddy_hip_stream>(s->stream) : nullptr;
}
}
