// Host runtime of the GPT-2 token loop on MI355X, exported through the C ABI
// in include/rtgpu.h. It owns HBM-resident weights and KV caches and drives
// the gfx950 kernels of kernels.hip; it never computes model math on the CPU
// (sampling of non-greedy generation aside, which the reference also does on
// the host, gpt2.rs:871-1017).
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "../../include/rtgpu.h"
#include "decode_persistent.h"
#include "attn_pair.h"
#include "bgemv.h"
#include "copy_team.h"
#include "device_memory.h"
#include "gemm_pair.h"
#include "kernels.h"
#include "rows.h"
#include "safetensors_reader.h"
#include "scratch.h"

using namespace rtg;

namespace {

rtg_result ok() { return rtg_result{true, nullptr}; }

rtg_result err(const std::string& m) {
  char* s = (char*)malloc(m.size() + 1);
  memcpy(s, m.c_str(), m.size() + 1);
  return rtg_result{false, s};
}

std::string fmt(const char* f, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, f);
  vsnprintf(buf, sizeof buf, f, ap);
  va_end(ap);
  return buf;
}

// A C++ exception other than HipError (e.g. std::bad_alloc for a malformed
// tensor shape) as an error result: no exception crosses the C boundary.
rtg_result err_internal(const std::exception& ex) { return err(std::string("internal error: ") + ex.what()); }

struct HipError {
  std::string msg;
};

void hip_check(hipError_t e, const char* what) {
  if (e != hipSuccess) throw HipError{std::string("HIP error in ") + what + ": " + hipGetErrorString(e)};
}
#define HIPX(call) hip_check((call), #call)

std::string check_device() {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n == 0)
    return "no HIP device available: rtgpu requires an MI355X (gfx950) GPU";
  int dev = 0;
  hipGetDevice(&dev);
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return "hipGetDeviceProperties failed";
  if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return std::string("rtgpu is built for gfx950 (MI355X); found ") + prop.gcnArchName;
  return "";
}

size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// ---- results to the host ----
//
// A call's results reach the caller's pageable memory through page-locked
// staging buffers of the library's own: a small one (a token's logits) by one
// kernel that also carries the launch's error word, a large one in chunks, the
// next chunk's transfer running while helper threads copy this one out
// (copy_team.h); they first touch the destination's pages while the GPU computes
// (first writes to fresh memory were most of that time). Through the runtime's own staging, one
// batch-1 token of GPT-2 small took 259 us with its logits (a 205 us step) and
// a 333-token forward 4.9 ms with its 67 MB; now 235 us and 2.7 ms (3.0 without
// the early touch).

// Two chunks and a few words behind them, with an event per chunk.
struct HostStage {
  static constexpr size_t kChunk = (size_t)4 << 20;
  char* mem = nullptr;
  hipEvent_t ev[2] = {nullptr, nullptr};
  ~HostStage() {
    if (mem) (void)hipHostFree(mem);
    for (auto e : ev)
      if (e) (void)hipEventDestroy(e);
  }
};

// Stages not in use, at most kKeep of them (the rest are freed when returned);
// rtg_cleanup gives them all back. Each is in use by one call at a time.
struct HostStages {
  static constexpr size_t kKeep = 4;
  std::mutex mu;
  std::vector<std::pair<int, std::unique_ptr<HostStage>>> idle;  // by device
  // Null where there is no page-locked memory to be had (test hook
  // RTG_TEST_PINNED_FAIL=1).
  std::unique_ptr<HostStage> take(int device) {
    {
      std::lock_guard<std::mutex> g(mu);
      for (auto it = idle.begin(); it != idle.end(); ++it)
        if (it->first == device) {
          std::unique_ptr<HostStage> s = std::move(it->second);
          idle.erase(it);
          return s;
        }
    }
    std::unique_ptr<HostStage> s(new HostStage());
    const char* t = getenv("RTG_TEST_PINNED_FAIL");
    if ((t && t[0] == '1') || hipHostMalloc(reinterpret_cast<void**>(&s->mem), 2 * HostStage::kChunk + 256,
                                            hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      s->mem = nullptr;
      return nullptr;
    }
    for (auto& e : s->ev) HIPX(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    return s;
  }
  void give(int device, std::unique_ptr<HostStage> s) {
    std::lock_guard<std::mutex> g(mu);
    if (idle.size() < kKeep) idle.emplace_back(device, std::move(s));
  }
};
HostStages& host_stages() {
  static HostStages* s = new HostStages();  // (kept to the process's end: no HIP calls from static destructors)
  return *s;
}

// After the work enqueued on s: bytes (a multiple of 4) from device memory src
// to dst, and the value of the device word err (null: 0 is returned). The
// stream has drained when it returns.
unsigned copy_out(hipStream_t s, int device, void* dst, const void* src, size_t bytes, const unsigned* err) {
  if (bytes == 0 && !err) {
    HIPX(hipStreamSynchronize(s));
    return 0;
  }
  std::unique_ptr<HostStage> st = host_stages().take(device);
  unsigned e = 0;
  if (!st) {  // through the runtime's own staging
    if (bytes) HIPX(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s));
    HIPX(hipStreamSynchronize(s));
    if (err) HIPX(hipMemcpy(&e, err, 4, hipMemcpyDeviceToHost));
    return e;
  }
  uint32_t* word = reinterpret_cast<uint32_t*>(st->mem + 2 * HostStage::kChunk);
  if (bytes <= HostStage::kChunk) {
    launch_copy_out(s, static_cast<const uint32_t*>(src), bytes / 4, err, reinterpret_cast<uint32_t*>(st->mem));
    HIPX(hipGetLastError());
    HIPX(hipStreamSynchronize(s));
    if (bytes) memcpy(dst, st->mem, bytes);
    if (err) e = *reinterpret_cast<const volatile uint32_t*>(st->mem + bytes);
  } else {
    const char* from = static_cast<const char*>(src);
    CopyTeam team(static_cast<char*>(dst), bytes, HostStage::kChunk, st->mem, st->mem + HostStage::kChunk);
    auto fetch = [&](size_t i) {
      HIPX(hipMemcpyAsync(st->mem + (i & 1) * HostStage::kChunk, from + i * team.chunk, team.size(i),
                          hipMemcpyDeviceToHost, s));
      HIPX(hipEventRecord(st->ev[i & 1], s));
    };
    try {
      if (err) launch_copy_out(s, nullptr, 0, err, word);
      fetch(0);
      if (team.count() > 1) fetch(1);
      team.touch();
      for (size_t i = 0; i < team.count(); ++i) {
        HIPX(hipEventSynchronize(st->ev[i & 1]));
        team.copy(i);
        if (i + 2 < team.count()) fetch(i + 2);
      }
      HIPX(hipStreamSynchronize(s));
    } catch (...) {
      (void)hipStreamSynchronize(s);  // no transfer into the stage is in flight when it is given back
      throw;
    }
    if (err) e = *reinterpret_cast<const volatile uint32_t*>(word);
  }
  host_stages().give(device, std::move(st));
  return e;
}

}  // namespace

// ---------------------------------------------------------------------------
// Model
// ---------------------------------------------------------------------------

struct LayerW {
  void *wqkv, *waproj, *wfc, *wmproj;  // W^T [N][K] in storage type
  float *bqkv, *baproj, *bfc, *bmproj;
  float *ln1w, *ln1b, *ln2w, *ln2b;
};

// Tile-ordered copies of the decode GEMV weights and the folded LayerNorm
// constants for the batched decode step (bgemv.h), built on first use.
struct BatchedWeights {
  void* arena = nullptr;
  struct Layer {
    const void *qkv, *proj, *fc, *mproj;  // tiled W^T
    const float *sq, *cq, *sf, *cf;       // LN1 into c_attn, LN2 into c_fc
  };
  std::vector<Layer> layers;
  const void* lm = nullptr;  // tiled wte (the tied LM head)
  const float *sl = nullptr, *cl = nullptr;  // ln_f into the LM head
  BgemvPlan pq{}, pp{}, pf{}, pm{};          // c_attn, attn c_proj, c_fc, mlp c_proj
  BgemvPlan pl[2]{};                         // LM head: up to 16 sequences, and more
  ~BatchedWeights() {
    if (arena) hipFree(arena);
  }
};

// The weights as the prefill's pair GEMM reads them (gemm_pair.h), with the
// scales of the inputs they multiply; built with the model.
struct PrefillWeights {
  void* arena = nullptr;
  size_t bytes = 0;
  struct Layer {
    PairWeights qkv, proj, fc, mproj;
    const float *s1, *s2, *sh;  // input scales: LN1, LN2, gelu output
    AttnScales att;             // v: the attention output's scale too
  };
  std::vector<Layer> layers;
  PairWeights lm;              // wte
  const float* sf = nullptr;   // scale of LN_f
  ~PrefillWeights() {
    if (arena) hipFree(arena);
  }
};

// A model's PrefillWeights, as long as their memory is not needed for something
// that cannot be done without: every allocation that fails takes them back
// (device_memory.h) and the model's prefill runs the f32-MFMA GEMMs from then
// on. A pass holds them while it is being enqueued; freeing them waits for the
// device, and so for the passes enqueued.
class PrefillHolder final : public SpareMemory {
 public:
  PrefillHolder() { register_spare(this); }
  ~PrefillHolder() { unregister_spare(this); }
  PrefillHolder(const PrefillHolder&) = delete;
  PrefillHolder& operator=(const PrefillHolder&) = delete;
  std::shared_ptr<const PrefillWeights> get() const {
    std::lock_guard<std::mutex> g(mu_);
    return pw_;
  }
  void set(std::unique_ptr<PrefillWeights> pw, int device) {
    std::lock_guard<std::mutex> g(mu_);
    pw_ = std::move(pw);
    device_ = device;
  }
  bool give_back(int device) override {
    std::weak_ptr<const PrefillWeights> left;
    {
      std::shared_ptr<const PrefillWeights> pw;
      std::lock_guard<std::mutex> g(mu_);
      if (!pw_ || device != device_) return false;
      pw.swap(pw_);
      left = pw;
    }
    // passes that are being enqueued on other threads (milliseconds) let go
    for (int i = 0; i < 2000 && !left.expired(); ++i) std::this_thread::sleep_for(std::chrono::milliseconds(1));
    return true;
  }

 private:
  mutable std::mutex mu_;
  std::shared_ptr<const PrefillWeights> pw_;
  int device_ = -1;
};

struct rtg_model {
  rtg_config cfg;
  int hd = 0;
  int wtype = W_F32;
  int device = 0;
  void* arena = nullptr;
  size_t arena_bytes = 0;
  void* wte = nullptr;
  float* wpe = nullptr;
  float *lnfw = nullptr, *lnfb = nullptr;
  std::vector<LayerW> layers;
  size_t nparams = 0;
  PersistentPlan* pplan = nullptr;
  RowsPlan* rplan = nullptr;  // multi-row forward (short prompts), null where unsupported
  PrefillHolder pw;           // empty where the f32-MFMA GEMMs run the prefill
  std::mutex bw_mu;
  std::unique_ptr<BatchedWeights> bw;
  // Pool of caches reused by the generate entry points (keyed by batch).
  std::mutex pool_mu;
  std::multimap<size_t, rtg_cache*> pool;
  ~rtg_model();
};

// ---------------------------------------------------------------------------
// Cache (+ per-cache stream, work buffers and the captured decode graph)
// ---------------------------------------------------------------------------

struct rtg_cache {
  const rtg_model* m = nullptr;
  size_t batch = 1;
  size_t len = 0;
  hipStream_t stream = nullptr;
  float* k = nullptr;  // [L][B][H][P][hd]
  float* v = nullptr;
  size_t layer_stride = 0;  // floats per layer per K (or V)
  // decode state in device memory
  int* pos_dev = nullptr;
  int* step_dev = nullptr;
  unsigned long long* keys = nullptr;
  uint32_t* token_dev = nullptr;
  uint32_t* ids_dev = nullptr;   // [B][P] generated ids
  uint32_t* ids_in = nullptr;    // [B*P] prompt ids
  // work buffers, capacity in rows
  size_t rows_cap = 0;
  float *x = nullptr, *ln = nullptr, *qkv = nullptr, *att = nullptr, *h = nullptr;
  float* ws = nullptr;  // split-k partial tiles of the prefill GEMMs
  size_t ws_floats = 0;
  size_t logit_rows_cap = 0;
  float* logits = nullptr;
  // decode graph over the current buffers
  hipGraph_t graph = nullptr;
  hipGraphExec_t graph_exec = nullptr;
  int host_steps = 0;  // batched steps fed by forward_cached before the graph was captured
  hipEvent_t ev[3] = {nullptr, nullptr, nullptr};
  PersistentState* pstate = nullptr;
  RowsState* rstate = nullptr;  // the multi-row forward's flags and work rows
  // batched decode step (bgemv): split-k partials and counters, per-group
  // LayerNorm statistics partials of the residual stream
  float* bg_part = nullptr;
  unsigned* bg_cnt = nullptr;
  float* bg_spart = nullptr;
  void* sample_work = nullptr;  // of launch_sample, made for the first sampled token
  float* bg_cen = nullptr;  // [2][kBgemvRows]: per-row centres of the folded LayerNorms' inputs
};

static void free_work(rtg_cache* c) {
  for (float** p : {&c->x, &c->ln, &c->qkv, &c->att, &c->h, &c->ws}) {
    if (*p) hipFree(*p);
    *p = nullptr;
  }
  c->rows_cap = 0;
  c->ws_floats = 0;
}

static void destroy_graph(rtg_cache* c) {
  if (c->graph_exec) hipGraphExecDestroy(c->graph_exec);
  if (c->graph) hipGraphDestroy(c->graph);
  c->graph_exec = nullptr;
  c->graph = nullptr;
}

// Floats the layer GEMMs of a prefill over M rows use to split over k, on the
// pair GEMMs or on the f32-MFMA ones.
static size_t prefill_ws_floats(const rtg_model* m, size_t M, bool pair) {
  const int d = (int)m->cfg.n_embd, planes = m->wtype == W_F32 ? 2 : 1;
  size_t ws = 0;
  for (const auto& nk : {std::make_pair(3 * d, d), std::make_pair(d, d), std::make_pair(4 * d, d),
                         std::make_pair(d, 4 * d)})
    ws = std::max(ws, pair ? pair_gemm_ws_floats((int)M, nk.first, nk.second, planes)
                           : gemm_splitk_ws_floats((int)M, nk.first, nk.second));
  return ws;
}

// The split-k workspace for the largest need of the four layer GEMMs at any row
// count up to cap (the split depends on the row blocks).
static void ensure_ws(rtg_cache* c, size_t cap, bool pair) {
  size_t ws = 0;
  for (size_t r = 32; r < cap + 128; r += (pair || r < 128 ? 32 : 128))
    ws = std::max(ws, prefill_ws_floats(c->m, std::min(r, cap), pair));
  if (ws <= c->ws_floats) return;
  if (c->ws) hipFree(c->ws);
  c->ws = nullptr;
  c->ws_floats = 0;
  HIPX(device_malloc(&c->ws, ws * 4));
  c->ws_floats = ws;
}

static void ensure_rows(rtg_cache* c, size_t rows) {
  if (rows <= c->rows_cap) return;
  destroy_graph(c);
  free_work(c);
  const size_t d = c->m->cfg.n_embd;
  size_t cap = std::max<size_t>(rows, 16);
  HIPX(device_malloc(&c->x, cap * d * 4));
  HIPX(device_malloc(&c->ln, cap * d * 4));
  HIPX(device_malloc(&c->qkv, cap * 3 * d * 4));
  HIPX(device_malloc(&c->att, cap * d * 4));
  HIPX(device_malloc(&c->h, cap * 4 * d * 4));
  ensure_ws(c, cap, c->m->pw.get() != nullptr);
  c->rows_cap = cap;
}

static void ensure_logits(rtg_cache* c, size_t rows) {
  if (rows <= c->logit_rows_cap) return;
  destroy_graph(c);
  if (c->pstate) persistent_state_destroy(c->pstate);  // it holds the logits pointer
  c->pstate = nullptr;
  if (c->logits) hipFree(c->logits);
  c->logits = nullptr;
  size_t cap = std::max<size_t>(rows, 16);
  HIPX(device_malloc(&c->logits, cap * c->m->cfg.vocab_size * 4));
  c->logit_rows_cap = cap;
}

static void ensure_sample_work(rtg_cache* c) {
  if (!c->sample_work) HIPX(device_malloc(&c->sample_work, sample_work_bytes((int)c->m->cfg.vocab_size)));
}

static rtg_cache* cache_create(const rtg_model* m, size_t batch) {
  std::unique_ptr<rtg_cache> c(new rtg_cache());
  c->m = m;
  c->batch = batch;
  const size_t L = m->cfg.n_layer, H = m->cfg.n_head, P = m->cfg.n_positions, hd = m->hd;
  c->layer_stride = batch * H * P * hd;
  try {
    HIPX(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
    HIPX(device_malloc(&c->k, std::max<size_t>(L * c->layer_stride, 1) * 4));
    HIPX(device_malloc(&c->v, std::max<size_t>(L * c->layer_stride, 1) * 4));
    HIPX(device_malloc(&c->pos_dev, 256));
    HIPX(device_malloc(&c->step_dev, 256));
    HIPX(device_malloc(&c->keys, std::max<size_t>(batch, 1) * 8));
    HIPX(device_malloc(&c->token_dev, std::max<size_t>(batch, 1) * 4));
    HIPX(device_malloc(&c->ids_dev, std::max<size_t>(batch * P, 1) * 4));
    HIPX(device_malloc(&c->ids_in, std::max<size_t>(batch * P, 1) * 4));
    for (auto& e : c->ev) HIPX(hipEventCreate(&e));
    HIPX(hipMemsetAsync(c->pos_dev, 0, 256, c->stream));
    HIPX(hipMemsetAsync(c->step_dev, 0, 256, c->stream));
    launch_reset_keys(c->stream, (int)batch, c->keys);
    HIPX(hipStreamSynchronize(c->stream));
  } catch (...) {
    rtg_cache_destroy(c.release());
    throw;
  }
  return c.release();
}

rtg_model::~rtg_model() {
  for (auto& kv : pool) rtg_cache_destroy(kv.second);
  pool.clear();
  if (pplan) persistent_plan_destroy(pplan);
  if (rplan) rows_plan_destroy(rplan);
  if (arena) hipFree(arena);
}

// ---------------------------------------------------------------------------
// Pipelines
// ---------------------------------------------------------------------------

static KvDst kv_layer(const rtg_cache* c, size_t l) {
  KvDst kv;
  kv.k = c->k + l * c->layer_stride;
  kv.v = c->v + l * c->layer_stride;
  kv.n_head = (int)c->m->cfg.n_head;
  kv.n_pos = (int)c->m->cfg.n_positions;
  kv.d = (int)c->m->cfg.n_embd;
  return kv;
}

// Activation buffers of one forward pass: x, ln [M][d], qkv [M][3d],
// att [M][d], h [M][4d], the logits rows and the GEMMs' split-k workspace
// (ws_floats floats; null: the GEMMs run unsplit).
struct Work {
  float *x, *ln, *qkv, *att, *h, *logits;
  float* ws;
  size_t ws_floats;
};

static Work cache_work(const rtg_cache* c) {
  return Work{c->x, c->ln, c->qkv, c->att, c->h, c->logits, c->ws, c->ws_floats};
}

// The rows whose logits a prefill computes: all S*T, the last row of each
// sequence (written as S rows: all that generation reads, gpt2.rs:420-423), or
// none (a prompt read into the cache without logits_out).
enum LogitRows { LOGITS_ALL, LOGITS_LAST, LOGITS_NONE };

// forward_cached body for S sequences x T new tokens (gpt2.rs:376-396) on the
// pair GEMMs (gemm_pair.h): w.ln, w.att and w.h hold f16 pairs, 4 bytes per
// element like the f32 rows they replace.
static void enqueue_prefill_pair(rtg_cache* c, const PrefillWeights& pw, const Work& w, const uint32_t* ids_dev,
                                 size_t S, size_t T, size_t past, LogitRows logit_rows) {
  const rtg_model* m = c->m;
  const int d = (int)m->cfg.n_embd, V = (int)m->cfg.vocab_size, M = (int)(S * T);
  const float eps = m->cfg.layer_norm_epsilon;
  hipStream_t s = c->stream;
  uint16_t *ln = reinterpret_cast<uint16_t*>(w.ln), *att = reinterpret_cast<uint16_t*>(w.att),
           *h = reinterpret_cast<uint16_t*>(w.h);
  auto args = [&](const uint16_t* A, int K, const float* bias, float* C, long ldc, int epi) {
    PairGemmArgs a;
    a.A = A;
    a.lda = 2 * K;
    a.M = M;
    a.bias = bias;
    a.C = C;
    a.ldc = ldc;
    a.epi = epi;
    a.ws = w.ws;
    a.ws_floats = w.ws_floats;
    return a;
  };
  launch_embed(s, m->wte, m->wtype, m->wpe, ids_dev, M, (int)T, (int)past, nullptr, d, w.x);
  for (size_t l = 0; l < m->layers.size(); ++l) {
    const LayerW& L = m->layers[l];
    const PrefillWeights::Layer& P = pw.layers[l];
    KvDst kv = kv_layer(c, l);
    launch_layernorm_pair(s, w.x, d, L.ln1w, L.ln1b, eps, M, d, P.s1, ln);
    PairGemmArgs a = args(ln, d, L.bqkv, w.qkv, 3 * d, EPI_BIAS);
    a.kv = kv;
    a.kv_T = (int)T;
    a.kv_past = (int)past;
    launch_pair_gemm(s, P.qkv, a);
    if (m->hd == 64)
      launch_attn_pair(s, w.qkv, (int)S, (int)T, (int)past, kv.k, kv.v, kv.n_head, kv.n_pos, d, P.att, att);
    else
      launch_attn_prefill(s, w.qkv, (int)S, (int)T, (int)past, kv.k, kv.v, kv.n_head, kv.n_pos, d, nullptr, att,
                          P.att.v);
    launch_pair_gemm(s, P.proj, args(att, d, L.baproj, w.x, d, EPI_BIAS_RESID));
    launch_layernorm_pair(s, w.x, d, L.ln2w, L.ln2b, eps, M, d, P.s2, ln);
    a = args(ln, d, L.bfc, nullptr, 0, EPI_BIAS_GELU);
    a.P = h;
    a.p_scale = P.sh;
    launch_pair_gemm(s, P.fc, a);
    launch_pair_gemm(s, P.mproj, args(h, 4 * d, L.bmproj, w.x, d, EPI_BIAS_RESID));
  }
  if (logit_rows != LOGITS_NONE) {
    const bool all = logit_rows == LOGITS_ALL;
    const int rows = all ? M : (int)S;
    launch_layernorm_pair(s, w.x + (all ? 0 : (T - 1) * d), all ? d : (long)T * d, m->lnfw, m->lnfb, eps, rows, d,
                          pw.sf, ln);
    PairGemmArgs a = args(ln, d, nullptr, w.logits, V, EPI_NONE);
    a.M = rows;
    a.ws = nullptr;
    launch_pair_gemm(s, pw.lm, a);
  }
  HIPX(hipGetLastError());
}

// forward_cached body for S sequences x T new tokens (gpt2.rs:376-396) on the
// MFMA prefill path, on the activation buffers w. ids_dev holds S*T ids. for_draws:
// the logits go to the seeded sampler, which keeps the f32-MFMA GEMMs and the
// attention that go with them for every model. The pair GEMMs' logits are as
// close to 64 bits or closer, but differ by up to 1e-6; over a flat distribution
// (45000 kept tokens of 2e-5) that moves one draw in a few hundred to the next
// token, and the text behind a seed changes from there on.
static void enqueue_prefill(rtg_cache* c, const Work& w, const uint32_t* ids_dev, size_t S, size_t T, size_t past,
                            LogitRows logit_rows, bool for_draws = false) {
  const rtg_model* m = c->m;
  if (!for_draws)
    if (const auto pw = m->pw.get()) return enqueue_prefill_pair(c, *pw, w, ids_dev, S, T, past, logit_rows);
  const int d = (int)m->cfg.n_embd, V = (int)m->cfg.vocab_size, M = (int)(S * T);
  const float eps = m->cfg.layer_norm_epsilon;
  hipStream_t s = c->stream;
  launch_embed(s, m->wte, m->wtype, m->wpe, ids_dev, M, (int)T, (int)past, nullptr, d, w.x);
  for (size_t l = 0; l < m->layers.size(); ++l) {
    const LayerW& L = m->layers[l];
    KvDst kv = kv_layer(c, l);
    launch_layernorm(s, w.x, L.ln1w, L.ln1b, eps, M, d, w.ln);
    launch_gemm_qkv(s, w.ln, d, L.wqkv, m->wtype, L.bqkv, w.qkv, 3 * d, M, d, (int)S, (int)T, (int)past, kv, w.ws,
                    w.ws_floats);
    launch_attn_prefill(s, w.qkv, (int)S, (int)T, (int)past, kv.k, kv.v, kv.n_head, kv.n_pos, d, w.att);
    launch_gemm(s, w.att, d, L.waproj, m->wtype, L.baproj, w.x, d, M, d, d, EPI_BIAS_RESID, w.ws, w.ws_floats);
    launch_layernorm(s, w.x, L.ln2w, L.ln2b, eps, M, d, w.ln);
    launch_gemm(s, w.ln, d, L.wfc, m->wtype, L.bfc, w.h, 4 * d, M, 4 * d, d, EPI_BIAS_GELU, w.ws, w.ws_floats);
    launch_gemm(s, w.h, 4 * d, L.wmproj, m->wtype, L.bmproj, w.x, d, M, d, 4 * d, EPI_BIAS_RESID, w.ws,
                w.ws_floats);
  }
  if (logit_rows == LOGITS_NONE) return;
  launch_layernorm(s, w.x, m->lnfw, m->lnfb, eps, M, d, w.ln);
  if (logit_rows == LOGITS_ALL) {
    launch_gemm(s, w.ln, d, m->wte, m->wtype, nullptr, w.logits, V, M, V, d, EPI_NONE);
  } else {
    // Last row of each sequence: rows (s*T + T-1), stride T*d.
    launch_gemm(s, w.ln + (T - 1) * d, (int)(T * d), m->wte, m->wtype, nullptr, w.logits, V, (int)S, V, d,
                EPI_NONE);
  }
}

// ---- batched decode step on the tile-ordered GEMV (bgemv.h) ----

// The batched step needs every GEMV's K to be a whole number of k-tiles and at
// most kBgemvRows sequences; other shapes keep the per-op kernels below.
static bool batched_ok(const rtg_model* m, size_t B) {
  const size_t tk = m->wtype == W_F32 ? 16 : 32;
  // (the LayerNorm statistics of a row come in at most 128 panel groups)
  return B >= 1 && B <= (size_t)kBgemvRows && m->cfg.n_embd % tk == 0 && m->cfg.n_embd <= 2048;
}

// Builds the model's tile-ordered weight copies and folded LayerNorm constants
// (once; callers may race, the mutex serialises them).
static const BatchedWeights* ensure_batched(const rtg_model* mc) {
  rtg_model* m = const_cast<rtg_model*>(mc);
  std::lock_guard<std::mutex> g(m->bw_mu);
  if (m->bw) return m->bw.get();
  const int d = (int)m->cfg.n_embd, V = (int)m->cfg.vocab_size, L = (int)m->layers.size(), wt = m->wtype;
  std::unique_ptr<BatchedWeights> bw(new BatchedWeights());
  const size_t tq = tiled_weight_bytes(3 * d, d, wt), tp = tiled_weight_bytes(d, d, wt);
  const size_t tf = tiled_weight_bytes(4 * d, d, wt), tm = tiled_weight_bytes(d, 4 * d, wt);
  const size_t tl = tiled_weight_bytes(V, d, wt);
  const size_t per_layer = align_up(tq, 256) + align_up(tp, 256) + align_up(tf, 256) + align_up(tm, 256);
  const size_t fold_layer = (size_t)(2 * 3 * d + 2 * 4 * d) * 4;
  const size_t total = per_layer * L + align_up(tl, 256) + align_up(fold_layer, 256) * L + align_up((size_t)2 * V * 4, 256);
  HIPX(hipDeviceSynchronize());
  HIPX(device_malloc(&bw->arena, total));
  char* p = static_cast<char*>(bw->arena);
  auto take = [&](size_t n) {
    char* r = p;
    p += align_up(n, 256);
    return r;
  };
  auto tile = [&](const void* src, int N, int K, size_t bytes) {
    void* dst = take(bytes);
    if (!launch_tile_weights(nullptr, src, wt, N, K, dst)) throw HipError{"tile_weights launch failed"};
    return (const void*)dst;
  };
  for (int l = 0; l < L; ++l) {
    const LayerW& W = m->layers[l];
    BatchedWeights::Layer bl{};
    bl.qkv = tile(W.wqkv, 3 * d, d, tq);
    bl.proj = tile(W.waproj, d, d, tp);
    bl.fc = tile(W.wfc, 4 * d, d, tf);
    bl.mproj = tile(W.wmproj, d, 4 * d, tm);
    float* f = reinterpret_cast<float*>(take(fold_layer));
    float *sq = f, *cq = f + 3 * d, *sf = f + 6 * d, *cf = f + 10 * d;
    if (!ln_fold(W.wqkv, wt, 3 * d, d, W.ln1w, W.ln1b, W.bqkv, sq, cq) ||
        !ln_fold(W.wfc, wt, 4 * d, d, W.ln2w, W.ln2b, W.bfc, sf, cf))
      throw HipError{"ln_fold launch failed"};
    bl.sq = sq; bl.cq = cq; bl.sf = sf; bl.cf = cf;
    bw->layers.push_back(bl);
  }
  bw->lm = tile(m->wte, V, d, tl);
  float* fl = reinterpret_cast<float*>(take((size_t)2 * V * 4));
  if (!ln_fold(m->wte, wt, V, d, m->lnfw, m->lnfb, nullptr, fl, fl + V)) throw HipError{"ln_fold launch failed"};
  bw->sl = fl;
  bw->cl = fl + V;
  HIPX(hipDeviceSynchronize());
  bw->pq = bgemv_plan(3 * d, d, wt);
  bw->pp = bgemv_plan(d, d, wt);
  bw->pf = bgemv_plan(4 * d, d, wt);
  bw->pm = bgemv_plan(d, 4 * d, wt);
  bw->pl[0] = bgemv_plan(V, d, wt);
  // more than 16 rows: two panels per wave share each load of x (GPT-2 small
  // f32, 24 sequences: 532 us per step against 550 with one and 539 with four;
  // XL bf16: 508 against 516 with four)
  bw->pl[1] = bgemv_plan(V, d, wt, 2);
  m->bw = std::move(bw);
  return m->bw.get();
}

// The cache's workspace for the batched step (allocated once per cache).
static void ensure_bg_work(rtg_cache* c, const BatchedWeights* bw) {
  if (c->bg_part) return;
  size_t part = 1, groups = 1;
  for (const BgemvPlan* pl : {&bw->pq, &bw->pp, &bw->pf, &bw->pm, &bw->pl[c->batch > 16]}) {
    part = std::max(part, bgemv_work_floats(*pl, (int)c->batch));
    groups = std::max(groups, (size_t)pl->groups);
  }
  HIPX(device_malloc(&c->bg_part, part * 4));
  HIPX(device_malloc(&c->bg_cnt, groups * 4));
  HIPX(device_malloc(&c->bg_spart, groups * kBgemvRows * 2 * 4));
  HIPX(device_malloc(&c->bg_cen, 2 * kBgemvRows * 4));
  HIPX(hipMemsetAsync(c->bg_cnt, 0, groups * 4, c->stream));
  HIPX(hipStreamSynchronize(c->stream));
}

// Prepares the decode step of a cache without a batch-1 persistent state
// (before any capture): the batched weights and the step's workspace.
static void prepare_decode(rtg_cache* c) {
  if (c->pstate || !batched_ok(c->m, c->batch)) return;
  ensure_bg_work(c, ensure_batched(c->m));
}

// One decode step for B sequences: per layer four tile-ordered GEMVs with
// LayerNorm folded into c_attn / c_fc / the LM head (row statistics written by
// the residual epilogues) and the cached attention; forward_cached with one
// token per sequence (gpt2.rs:376-396, 477-538).
static void enqueue_decode_step_batched(rtg_cache* c) {
  const rtg_model* m = c->m;
  const BatchedWeights* bw = m->bw.get();
  const int d = (int)m->cfg.n_embd, V = (int)m->cfg.vocab_size, B = (int)c->batch;
  const float eps = m->cfg.layer_norm_epsilon;
  hipStream_t s = c->stream;
  auto base = [&]() {
    BgemvArgs a{};
    a.M = B;
    a.wtype = m->wtype;
    a.part = c->bg_part;
    a.cnt = c->bg_cnt;
    a.eps = eps;
    return a;
  };
  auto run = [&](const BgemvPlan& pl, const BgemvArgs& a) {
    if (!launch_bgemv(s, pl, a)) throw HipError{"bgemv launch failed"};
  };
  // c->ln holds x scaled by the gain of the LayerNorm folded into the next
  // GEMV (written by the embedding and by each residual epilogue); c->ln,
  // c->att and c->h are in the GEMV input layout (xt_index, tile width tk)
  const int tk = m->wtype == W_F32 ? 16 : 32;
  const size_t NL = m->layers.size();
  // Centres of the folded LayerNorms (two alternating per-row buffers): the
  // GEMV input c->ln holds (x - cen_cur) * g; each LayerNorm-folded GEMV
  // writes its rows' exact mean into the other buffer, and the residual
  // epilogue after it centres the next input on that mean, so the fold only
  // ever subtracts the drift of the mean between two LayerNorms.
  float* cen_cur = c->bg_cen;
  float* cen_next = c->bg_cen + kBgemvRows;
  if (!launch_embed_stats(s, m->wte, m->wtype, m->wpe, c->token_dev, c->pos_dev, B, d, c->x, c->bg_spart,
                          NL ? m->layers[0].ln1w : m->lnfw, c->ln, cen_cur))
    throw HipError{"embed_stats launch failed"};
  // shape of the statistics partials the last residual writer left
  int st_groups = 1, st_cols = d;
  auto ln_in = [&](BgemvArgs& a, const float* g, const float* sv, bool record) {
    a.ln_g = g; a.ln_s = sv; a.ln_part = c->bg_spart; a.ln_groups = st_groups; a.ln_cols = st_cols;
    a.cen_in = cen_cur;
    if (record) {
      cen_next = cen_cur == c->bg_cen ? c->bg_cen + kBgemvRows : c->bg_cen;
      a.cen_out = cen_next;
    }
  };
  auto resid_out = [&](BgemvArgs& a, const BgemvPlan& pl, const float* g_next) {
    a.stats_part = c->bg_spart;
    a.xg = c->ln;
    a.g_next = g_next;
    a.xg_cen = cen_next;
    cen_cur = cen_next;
    st_groups = pl.groups;
    st_cols = 16 * pl.npw;
  };
  for (size_t l = 0; l < m->layers.size(); ++l) {
    const LayerW& L = m->layers[l];
    const BatchedWeights::Layer& T = bw->layers[l];
    KvDst kv = kv_layer(c, l);
    {  // LN1 + c_attn; k/v of the new token into the cache
      BgemvArgs a = base();
      a.X = c->ln; a.Wt = T.qkv; a.N = 3 * d; a.K = d; a.bias = T.cq;
      ln_in(a, L.ln1w, T.sq, true);
      a.epi = EPI_BIAS;
      a.qkv = BgemvQkv{c->qkv, d, d, kv, c->pos_dev};
      run(bw->pq, a);
    }
    launch_attn_decode(s, B, c->qkv, d, kv.k, kv.v, kv.n_head, kv.n_pos, c->pos_dev, c->att, d, tk);
    {  // attention c_proj + residual; statistics partials for LN2
      BgemvArgs a = base();
      a.X = c->att; a.Wt = T.proj; a.N = d; a.K = d; a.bias = L.baproj;
      a.C = c->x; a.ldc = d; a.epi = EPI_BIAS_RESID;
      resid_out(a, bw->pp, L.ln2w);
      run(bw->pp, a);
    }
    {  // LN2 + c_fc + gelu_new
      BgemvArgs a = base();
      a.X = c->ln; a.Wt = T.fc; a.N = 4 * d; a.K = d; a.bias = T.cf;
      ln_in(a, L.ln2w, T.sf, true);
      a.C = c->h; a.c_tiled = true; a.epi = EPI_BIAS_GELU;
      run(bw->pf, a);
    }
    {  // mlp c_proj + residual; statistics partials for the next LayerNorm
      BgemvArgs a = base();
      a.X = c->h; a.Wt = T.mproj; a.N = d; a.K = 4 * d; a.bias = L.bmproj;
      a.C = c->x; a.ldc = d; a.epi = EPI_BIAS_RESID;
      resid_out(a, bw->pm, l + 1 < NL ? m->layers[l + 1].ln1w : m->lnfw);
      run(bw->pm, a);
    }
  }
  {  // ln_f + tied LM head (gpt2.rs:392-396)
    BgemvArgs a = base();
    a.X = c->ln; a.Wt = bw->lm; a.N = V; a.K = d; a.bias = bw->cl;
    ln_in(a, m->lnfw, bw->sl, false);
    a.C = c->logits; a.ldc = V; a.epi = EPI_BIAS;
    run(bw->pl[B > 16], a);
  }
  // (the argmax in the LM head's epilogue, a per-row atomic max per
  // workgroup, was measured slower than this separate kernel)
  launch_argmax(s, c->logits, V, B, V, c->keys);
}

// One decode step for all B sequences of the cache, reading the token from
// token_dev and the position from pos_dev (both device-resident), writing the
// argmax token back to token_dev and ids_dev[b][step]. Capturable.
static void enqueue_decode_step(rtg_cache* c, int pos = -1) {
  const rtg_model* m = c->m;
  const int d = (int)m->cfg.n_embd, V = (int)m->cfg.vocab_size, B = (int)c->batch;
  const float eps = m->cfg.layer_norm_epsilon;
  hipStream_t s = c->stream;
  const int P = (int)m->cfg.n_positions;
  if (c->pstate) {
    HIPX(persistent_decode_step(c->pstate, s, /*cooperative=*/false, pos));
  } else if (c->bg_part) {
    enqueue_decode_step_batched(c);
  } else {
    launch_embed(s, m->wte, m->wtype, m->wpe, c->token_dev, B, 1, 0, c->pos_dev, d, c->x);
    for (size_t l = 0; l < m->layers.size(); ++l) {
      const LayerW& L = m->layers[l];
      KvDst kv = kv_layer(c, l);
      launch_layernorm(s, c->x, L.ln1w, L.ln1b, eps, B, d, c->ln);
      launch_gemv_qkv(s, B, L.wqkv, m->wtype, L.bqkv, c->ln, d, c->qkv, d, d, kv, c->pos_dev);
      launch_attn_decode(s, B, c->qkv, d, kv.k, kv.v, kv.n_head, kv.n_pos, c->pos_dev, c->att, d);
      launch_gemv(s, B, L.waproj, m->wtype, L.baproj, c->att, d, c->x, d, d, d, EPI_BIAS_RESID);
      launch_layernorm(s, c->x, L.ln2w, L.ln2b, eps, B, d, c->ln);
      launch_gemv(s, B, L.wfc, m->wtype, L.bfc, c->ln, d, c->h, 4 * d, 4 * d, d, EPI_BIAS_GELU);
      launch_gemv(s, B, L.wmproj, m->wtype, L.bmproj, c->h, 4 * d, c->x, d, d, 4 * d, EPI_BIAS_RESID);
    }
    launch_layernorm(s, c->x, m->lnfw, m->lnfb, eps, B, d, c->ln);
    launch_gemv(s, B, m->wte, m->wtype, nullptr, c->ln, d, c->logits, V, V, d, EPI_NONE);
    launch_argmax(s, c->logits, V, B, V, c->keys);
  }
  if (!c->pstate)  // the persistent step finishes itself
    launch_finalize(s, B, c->keys, c->token_dev, c->ids_dev, P, c->pos_dev, c->step_dev, nullptr);
}

// The position and step counters (and, for a decode step from the host, its B
// tokens) as kernel arguments: one launch, no staging copy; never captured.
static void set_counters(rtg_cache* c, int pos, int step) {
  launch_set_step(c->stream, nullptr, c->pos_dev, pos, c->step_dev, step);
}
static void set_step(rtg_cache* c, const uint32_t* ids, size_t B) {
  if (B <= (size_t)kStepIds) {
    StepIds s{};
    memcpy(s.id, ids, B * 4);
    launch_set_step(c->stream, c->token_dev, c->pos_dev, (int)c->len, c->step_dev, 0, (int)B, s);
  } else {
    HIPX(hipMemcpyAsync(c->token_dev, ids, B * 4, hipMemcpyHostToDevice, c->stream));
    set_counters(c, (int)c->len, 0);
  }
}

// The multi-row forward runs S sequences x T tokens of a cache of batch S in
// one launch (RTG_NO_ROWS=1: the per-op prefill kernels instead).
static bool rows_path(const rtg_cache* c, size_t S, size_t T) {
  const char* off = getenv("RTG_NO_ROWS");
  if (off && off[0] == '1') return false;
  return c->m->rplan && S == c->batch && rows_supported(c->m->rplan, (int)S, (int)T);
}

// Enqueues the multi-row forward on the cache's stream (the caller holds
// persistent_launch_lock until the stream drains): ids_dev [S*T] at position
// past, logits [S*T][V] (null: no LM head); state st (default: the cache's own, made on first use).
static void enqueue_rows(rtg_cache* c, const uint32_t* ids_dev, size_t S, size_t T, size_t past, float* logits,
                         RowsState* st = nullptr, const RowsFinish* fin = nullptr) {
  const rtg_model* m = c->m;
  if (!st) {
    if (!c->rstate) {
      c->rstate = rows_state_create(m->rplan);
      if (!c->rstate) throw HipError{"multi-row forward: state allocation failed"};
    }
    st = c->rstate;
  }
  HIPX(rows_forward(m->rplan, st, c->stream, c->k, c->v, (long)c->layer_stride, ids_dev, (int)S, (int)T, (int)past,
                    nullptr, logits, fin));
}

// After the stream has drained: a bounded wait of the multi-row forward that
// timed out becomes an error (its word is cleared for the next launch).
static void check_rows(RowsState* st, unsigned e) {
  rows_dump_trace();
  if (e) {
    HIPX(hipMemset(rows_err(st), 0, 4));
    throw HipError{fmt("multi-row forward timed out waiting for a peer (phase %u)", e)};
  }
}

static void check_rows(RowsState* st) {
  unsigned e = 0;
  HIPX(hipMemcpy(&e, rows_err(st), 4, hipMemcpyDeviceToHost));
  check_rows(st, e);
}

static void ensure_graph(rtg_cache* c) {
  if (c->graph_exec) return;
  HIPX(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
  enqueue_decode_step(c);
  hipGraph_t g = nullptr;
  hipError_t e = hipStreamEndCapture(c->stream, &g);
  HIPX(e);
  c->graph = g;
  HIPX(hipGraphInstantiate(&c->graph_exec, c->graph, nullptr, nullptr, 0));
}

// ---------------------------------------------------------------------------
// Validation shared by the entry points (gpt2.rs:364-377, 616-618)
// ---------------------------------------------------------------------------

static std::string check_ids(const rtg_model* m, const uint32_t* ids, size_t n) {
  for (size_t i = 0; i < n; ++i)
    if (ids[i] >= m->cfg.vocab_size)
      return fmt("Token ID %zu out of range (vocab_size=%zu)", (size_t)ids[i], m->cfg.vocab_size);
  return "";
}

static std::string check_cached(const rtg_model* m, size_t past, const uint32_t* ids, size_t n) {
  if (n == 0) return "Empty input";
  const size_t total = past + n;
  if (total > m->cfg.n_positions)
    return fmt("Total sequence length %zu exceeds max position %zu", total, m->cfg.n_positions);
  return check_ids(m, ids, n);
}

// forward_cached for all sequences of a cache: ids [B][n].
static void forward_cached_impl(rtg_cache* c, const uint32_t* ids, size_t n, float* logits_out) {
  const rtg_model* m = c->m;
  const size_t B = c->batch, V = m->cfg.vocab_size;
  ensure_rows(c, B * n);
  ensure_logits(c, logits_out ? B * n : B);
  if (n == 1 && B == 1 && persistent_supported(m->pplan, 1)) {
    // one new token at batch 1: the persistent decode step, the kernel
    // generate_cached runs per token; its token is read from token_dev at
    // position *pos_dev = past, its logits land in c->logits
    if (!c->pstate) {
      c->pstate = persistent_state_create(m->pplan, c->k, c->v, 1, c->token_dev, c->pos_dev, c->logits, c->keys,
                                          c->ids_dev, c->step_dev);
      destroy_graph(c);
    }
  }
  if (n == 1 && B == 1 && c->pstate) {
    std::lock_guard<std::mutex> plock(persistent_launch_lock(m->device));
    set_step(c, ids, 1);
    HIPX(persistent_decode_step(c->pstate, c->stream, /*cooperative=*/false, (int)c->len));
    const unsigned e =
        copy_out(c->stream, m->device, logits_out, c->logits, logits_out ? V * 4 : 0, persistent_err(c->pstate));
    if (e) {
      HIPX(hipMemset(persistent_err(c->pstate), 0, 4));
      throw HipError{fmt("persistent decode step timed out waiting for a peer (code %u)", e)};
    }
    c->len += 1;
    return;
  }
  if (n == 1 && B >= 2 && !c->pstate && batched_ok(m, B)) {
    // one new token per sequence: the batched decode step (the same kernels
    // generate_cached_batched replays), its token read from token_dev at
    // position *pos_dev = past
    prepare_decode(c);
    set_step(c, ids, B);
    // a loop of such calls replays the step as a graph from its third step on
    // (capturing it costs more than two steps save)
    const char* ng = getenv("RTG_NO_GRAPH");
    if (!(ng && ng[0] == '1') && (c->graph_exec || ++c->host_steps > 2)) {
      ensure_graph(c);
      HIPX(hipGraphLaunch(c->graph_exec, c->stream));
    } else {
      enqueue_decode_step(c);
    }
  } else if (rows_path(c, B, n)) {
    std::lock_guard<std::mutex> plock(persistent_launch_lock(m->device));
    HIPX(hipMemcpyAsync(c->ids_in, ids, B * n * 4, hipMemcpyHostToDevice, c->stream));
    enqueue_rows(c, c->ids_in, B, n, c->len, logits_out ? c->logits : nullptr);
    check_rows(c->rstate, copy_out(c->stream, m->device, logits_out, c->logits, logits_out ? B * n * V * 4 : 0,
                                   rows_err(c->rstate)));
    c->len += n;
    return;
  } else {
    HIPX(hipMemcpyAsync(c->ids_in, ids, B * n * 4, hipMemcpyHostToDevice, c->stream));
    enqueue_prefill(c, cache_work(c), c->ids_in, B, n, c->len, logits_out ? LOGITS_ALL : LOGITS_NONE);
  }
  copy_out(c->stream, m->device, logits_out, c->logits, logits_out ? B * n * V * 4 : 0, nullptr);
  c->len += n;
}

static rtg_cache* pool_take(const rtg_model* mc, size_t batch) {
  rtg_model* m = const_cast<rtg_model*>(mc);
  {
    std::lock_guard<std::mutex> g(m->pool_mu);
    auto it = m->pool.find(batch);
    if (it != m->pool.end()) {
      rtg_cache* c = it->second;
      m->pool.erase(it);
      c->len = 0;
      return c;
    }
  }
  return cache_create(mc, batch);
}

static void pool_give(const rtg_model* mc, rtg_cache* c) {
  rtg_model* m = const_cast<rtg_model*>(mc);
  std::lock_guard<std::mutex> g(m->pool_mu);
  m->pool.emplace(c->batch, c);
}

struct PoolLease {
  const rtg_model* m;
  rtg_cache* c;
  PoolLease(const rtg_model* mm, size_t b) : m(mm), c(pool_take(mm, b)) {}
  ~PoolLease() {
    if (c) pool_give(m, c);
  }
};

// generate_cached over B equal-length prompts (gpt2.rs:405-441), greedy or,
// with sp (B = 1), choosing every token with the device sampler
// (sample_logits, gpt2.rs:871-906): the whole loop stays on the device.
static void generate_greedy(const rtg_model* m, const uint32_t* prompts, size_t B, size_t n, size_t max_new,
                            uint32_t* out, rtg_timing* timing, const SampleParams* sp = nullptr) {
  PoolLease lease(m, B);
  rtg_cache* c = lease.c;
  const size_t V = m->cfg.vocab_size, P = m->cfg.n_positions;
  const size_t steps = max_new > 0 ? max_new : 1;  // first token comes from prefill
  const bool rows = rows_path(c, B, n);
  // Draws read the last row of an LM head over all rows (as the f32-MFMA GEMM
  // sums it for that many; see enqueue_prefill).
  const bool draws = sp && sp->temperature > 0.0f, all = rows || draws;
  ensure_rows(c, B * n);
  if (draws && !rows) ensure_ws(c, B * n, false);
  ensure_logits(c, all ? B * n : B);
  if (sp) ensure_sample_work(c);
  hipStream_t s = c->stream;
  // overwrite the argmax token of the step just enqueued with the sampler's choice
  auto sample = [&](const float* row) {
    if (sp && !launch_sample(s, row, (int)V, c->ids_in, (int)n, c->ids_dev, c->step_dev, *sp, c->token_dev,
                             c->sample_work))
      throw HipError{"vocabulary too large for the device sampler"};
  };
  if (!c->pstate && persistent_supported(m->pplan, (int)B)) {
    c->pstate = persistent_state_create(m->pplan, c->k, c->v, (int)B, c->token_dev, c->pos_dev, c->logits, c->keys,
                                        c->ids_dev, c->step_dev);
    destroy_graph(c);  // the step graph changes shape
  }
  prepare_decode(c);
  // The persistent step's workgroups wait on each other: no second persistent
  // step of this process may be in flight on the device (another thread's
  // cache) until this stream has drained.
  if (rows && !c->rstate) {  // (allocated before the timed prefill)
    c->rstate = rows_state_create(m->rplan);
    if (!c->rstate) throw HipError{"multi-row forward: state allocation failed"};
  }
  std::unique_lock<std::mutex> plock;
  if (c->pstate || rows) plock = std::unique_lock<std::mutex>(persistent_launch_lock(m->device));
  HIPX(hipMemcpyAsync(c->ids_in, prompts, B * n * 4, hipMemcpyHostToDevice, s));
  HIPX(hipEventRecord(c->ev[0], s));
  // finalize advances pos by one: after it, pos = n, the position of the
  // prefill token that the first decode step consumes.
  set_counters(c, (int)n - 1, 0);
  if (rows) {
    // the prefill with the argmax of each sequence's last row and the
    // finalize in the same launch
    const RowsFinish fin{c->keys, c->token_dev, c->ids_dev, (int)P, c->pos_dev, c->step_dev};
    enqueue_rows(c, c->ids_in, B, n, 0, c->logits, nullptr, &fin);
  } else {
    // argmax of the last row of each sequence (extract_row(logits, n-1))
    enqueue_prefill(c, cache_work(c), c->ids_in, B, n, 0, all ? LOGITS_ALL : LOGITS_LAST, draws);
    launch_argmax(s, c->logits + (all ? (n - 1) * V : 0), (long)(all ? n * V : V), (int)B, (int)V, c->keys);
    launch_finalize(s, (int)B, c->keys, c->token_dev, c->ids_dev, (int)P, c->pos_dev, c->step_dev);
  }
  sample(all ? c->logits + (n - 1) * V : c->logits);
  HIPX(hipEventRecord(c->ev[1], s));
  // The persistent step (one kernel) is launched directly: replaying it as a
  // one-node graph was measured to leave ~8 us between launches instead of ~1.
  // RTG_NO_GRAPH=1 does the same for the batched step's kernels (for
  // per-kernel profiling; same results).
  const char* ng = getenv("RTG_NO_GRAPH");
  if (c->pstate || (ng && ng[0] == '1')) {
    for (size_t i = 1; i < steps; ++i) {
      enqueue_decode_step(c, (int)(n + i - 1));  // step i consumes the token at position n + i - 1
      sample(c->logits);
    }
  } else {
    ensure_graph(c);
    for (size_t i = 1; i < steps; ++i) {
      HIPX(hipGraphLaunch(c->graph_exec, s));
      sample(c->logits);
    }
  }
  HIPX(hipEventRecord(c->ev[2], s));
  // Optional profiling pass: rewind to the first decode step and replay the
  // steps launch by launch with events around the persistent kernel. Inputs
  // (tokens, positions, cache rows) are the same, so are the results.
  double kern_ms = 0.0;
  size_t kern_n = 0;
  if (timing && timing->profile_kernels && c->pstate && steps > 1 && !sp) {
    std::vector<hipEvent_t> evs(2 * (steps - 1));
    for (auto& e : evs) HIPX(hipEventCreate(&e));
    set_counters(c, (int)n, 1);
    HIPX(hipMemcpyAsync(c->token_dev, c->ids_dev, 4, hipMemcpyDeviceToDevice, s));
    for (size_t i = 1; i < steps; ++i) {
      HIPX(hipEventRecord(evs[2 * (i - 1)], s));
      HIPX(persistent_decode_step(c->pstate, s, /*cooperative=*/true, (int)(n + i - 1)));
      HIPX(hipEventRecord(evs[2 * (i - 1) + 1], s));
    }
    HIPX(hipStreamSynchronize(s));
    for (size_t i = 0; i + 1 < evs.size(); i += 2) {
      float ms = 0.f;
      HIPX(hipEventElapsedTime(&ms, evs[i], evs[i + 1]));
      kern_ms += ms;
      ++kern_n;
    }
    for (auto& e : evs) hipEventDestroy(e);
  }
  std::vector<uint32_t> gen(B * P);
  HIPX(hipMemcpyAsync(gen.data(), c->ids_dev, B * P * 4, hipMemcpyDeviceToHost, s));
  HIPX(hipStreamSynchronize(s));
  if (rows) check_rows(c->rstate);
  if (c->pstate) {
    persistent_dump_trace(c->pstate);
    unsigned e = 0;
    HIPX(hipMemcpy(&e, persistent_err(c->pstate), 4, hipMemcpyDeviceToHost));
    if (e) {
      HIPX(hipMemset(persistent_err(c->pstate), 0, 4));
      throw HipError{fmt("persistent decode step timed out waiting for a peer (code %u)", e)};
    }
  }
  c->len = n + steps - 1;  // the last generated token is never fed back
  const size_t outlen = n + steps;
  for (size_t b = 0; b < B; ++b) {
    memcpy(out + b * outlen, prompts + b * n, n * 4);
    memcpy(out + b * outlen + n, gen.data() + b * P, steps * 4);
  }
  if (timing) {
    float a = 0.f, b2 = 0.f;
    HIPX(hipEventElapsedTime(&a, c->ev[0], c->ev[1]));
    HIPX(hipEventElapsedTime(&b2, c->ev[1], c->ev[2]));
    timing->prefill_ms = a;
    timing->decode_ms = b2;
    timing->decode_steps = steps - 1;
    timing->decode_kernel_ms = kern_ms;
    timing->decode_kernel_launches = kern_n;
  }
}

// ---------------------------------------------------------------------------
// Model construction (gpt2.rs:214-263)
// ---------------------------------------------------------------------------

// Memory for the model's PrefillWeights (cfg, wtype and the layer count set).
// Null where the pair GEMM does not apply (n_embd not a multiple of 64, a
// negative epsilon) or where the copy does not fit the device: the f32-MFMA
// GEMMs then run the prefill.
static std::unique_ptr<PrefillWeights> alloc_prefill_weights(const rtg_model* m) {
  const int d = (int)m->cfg.n_embd, V = (int)m->cfg.vocab_size, L = (int)m->cfg.n_layer, wt = m->wtype;
  if (d % 64 != 0 || !(m->cfg.layer_norm_epsilon >= 0.f)) return nullptr;
  std::unique_ptr<PrefillWeights> pw(new PrefillWeights());
  struct Shape {
    int N, K;
  };
  const Shape sh[4] = {{3 * d, d}, {d, d}, {4 * d, d}, {d, 4 * d}};
  size_t total = 256;  // the flag
  for (const Shape& x : sh) total += L * (align_up(pair_weight_bytes(x.N, x.K, wt), 256) + align_up(x.N * 4, 256));
  const int H = (int)m->cfg.n_head;
  total += L * (3 * align_up(d * 4, 256) + align_up(3 * d * 4, 256) + align_up(4 * d * 4, 256) + align_up(H * 4, 256));
  total += align_up(pair_weight_bytes(V, d, wt), 256) + align_up((size_t)V * 4, 256) + align_up(d * 4, 256);
  if (hipMalloc(&pw->arena, total) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  pw->bytes = total;
  return pw;
}

// Fills and keeps them, unless a weight or a bound of an activation is not
// finite.
static void build_prefill_weights(rtg_model* m, std::unique_ptr<PrefillWeights> pw) {
  if (!pw) return;
  const int d = (int)m->cfg.n_embd, V = (int)m->cfg.vocab_size, H = (int)m->cfg.n_head, wt = m->wtype;
  char* p = static_cast<char*>(pw->arena);
  auto take = [&](size_t n) {
    char* r = p;
    p += align_up(n, 256);
    return r;
  };
  auto floats = [&](int n) { return reinterpret_cast<float*>(take((size_t)n * 4)); };
  hipStream_t s = nullptr;
  int* bad = reinterpret_cast<int*>(take(256));
  HIPX(hipMemset(bad, 0, 4));
  auto weights = [&](const void* W, int N, int K, const float* in_scale) {
    PairWeights w;
    w.planes = wt == W_F32 ? 2 : 1;
    w.N = N;
    w.K = K;
    w.w = reinterpret_cast<uint16_t*>(take(pair_weight_bytes(N, K, wt)));
    w.out_scale = floats(N);
    launch_pair_weights(s, W, wt, in_scale, w, bad);
    return w;
  };
  for (const LayerW& W : m->layers) {
    PrefillWeights::Layer l;
    float *s1 = floats(d), *sqkv = floats(3 * d), *s2 = floats(d), *sh4 = floats(4 * d), *sk = floats(d),
          *qk = floats(H);
    launch_pair_ln_scale(s, W.ln1w, W.ln1b, d, s1, bad);
    launch_pair_ln_scale(s, W.ln2w, W.ln2b, d, s2, bad);
    // attention averages value rows, so its output has the bound of c_attn's v
    launch_pair_row_scale(s, W.wqkv, wt, 3 * d, d, W.ln1w, W.ln1b, W.bqkv, sqkv, bad);
    if (m->hd == 64) launch_head_scale(s, sqkv, H, sk, qk, bad);
    l.att = AttnScales{sqkv, sk, qk, sqkv + 2 * d};
    launch_pair_row_scale(s, W.wfc, wt, 4 * d, d, W.ln2w, W.ln2b, W.bfc, sh4, bad);
    l.s1 = s1;
    l.s2 = s2;
    l.sh = sh4;
    l.qkv = weights(W.wqkv, 3 * d, d, s1);
    l.proj = weights(W.waproj, d, d, l.att.v);
    l.fc = weights(W.wfc, 4 * d, d, s2);
    l.mproj = weights(W.wmproj, d, 4 * d, sh4);
    pw->layers.push_back(l);
  }
  float* sf = floats(d);
  launch_pair_ln_scale(s, m->lnfw, m->lnfb, d, sf, bad);
  pw->sf = sf;
  pw->lm = weights(m->wte, V, d, sf);
  int flag = 0;
  HIPX(hipGetLastError());
  HIPX(hipMemcpy(&flag, bad, 4, hipMemcpyDeviceToHost));
  if (flag == 0) m->pw.set(std::move(pw), m->device);
}

namespace {
// A weight as the caller or the file holds it: f32, bf16 or f16 elements
// (uploaded as they are and converted on the device), or an f32 decode on the
// host of any other element type.
struct HostTensor {
  std::vector<size_t> shape;
  const void* data = nullptr;
  int stype = SRC_F32;
  std::vector<float> owned;
  size_t numel() const {
    size_t n = 1;
    for (size_t x : shape) n *= x;
    return n;
  }
  size_t bytes() const { return numel() * (stype == SRC_F32 ? 4 : 2); }
};

using Lookup = std::map<std::string, HostTensor>;

std::string shape_str(const std::vector<size_t>& s) {
  std::string r = "[";
  for (size_t i = 0; i < s.size(); ++i) r += (i ? ", " : "") + std::to_string(s[i]);
  return r + "]";
}

rtg_result build_model(const rtg_config* cfg, Lookup& lk, rtg_storage storage, rtg_model** out) {
  const size_t d = cfg->n_embd, L = cfg->n_layer, V = cfg->vocab_size, P = cfg->n_positions, H = cfg->n_head;
  // gpt2.rs:224-263: look up every name first, in the reference's order.
  std::vector<std::string> names = {"wte.weight", "wpe.weight", "ln_f.weight", "ln_f.bias"};
  const char* per[] = {"ln_1.weight", "ln_1.bias", "attn.c_attn.weight", "attn.c_attn.bias",
                       "attn.c_proj.weight", "attn.c_proj.bias", "ln_2.weight", "ln_2.bias",
                       "mlp.c_fc.weight", "mlp.c_fc.bias", "mlp.c_proj.weight", "mlp.c_proj.bias"};
  for (size_t i = 0; i < L; ++i)
    for (const char* p : per) names.push_back("h." + std::to_string(i) + "." + p);
  for (const auto& nm : names)
    if (!lk.count(nm)) return err("Missing weight: " + nm);
  if (H == 0 || d == 0 || d % H != 0) return err(fmt("n_embd %zu is not divisible by n_head %zu", d, H));
  const size_t hd = d / H;
  if (hd > 64) return err(fmt("head_dim %zu > 64 is not supported", hd));
  if (d % 8 != 0) return err(fmt("n_embd %zu must be a multiple of 8", d));
  // Shapes (the reference does not check them; a mismatch there is a panic or garbage).
  auto want = [&](const std::string& nm, std::vector<size_t> s) -> std::string {
    const auto& t = lk[nm];
    if (t.shape != s) return "Shape mismatch for " + nm + ": expected " + shape_str(s) + ", got " + shape_str(t.shape);
    return "";
  };
  std::string e;
  if (!(e = want("wte.weight", {V, d})).empty() || !(e = want("wpe.weight", {P, d})).empty() ||
      !(e = want("ln_f.weight", {d})).empty() || !(e = want("ln_f.bias", {d})).empty())
    return err(e);
  for (size_t i = 0; i < L; ++i) {
    std::string p = "h." + std::to_string(i) + ".";
    std::vector<std::pair<const char*, std::vector<size_t>>> sh = {
        {"ln_1.weight", {d}}, {"ln_1.bias", {d}}, {"attn.c_attn.weight", {d, 3 * d}}, {"attn.c_attn.bias", {3 * d}},
        {"attn.c_proj.weight", {d, d}}, {"attn.c_proj.bias", {d}}, {"ln_2.weight", {d}}, {"ln_2.bias", {d}},
        {"mlp.c_fc.weight", {d, 4 * d}}, {"mlp.c_fc.bias", {4 * d}}, {"mlp.c_proj.weight", {4 * d, d}},
        {"mlp.c_proj.bias", {d}}};
    for (auto& kv : sh)
      if (!(e = want(p + kv.first, kv.second)).empty()) return err(e);
  }
  std::string derr = check_device();
  if (!derr.empty()) return err(derr);

  std::unique_ptr<rtg_model> m(new rtg_model());
  m->cfg = *cfg;
  m->hd = (int)hd;
  m->wtype = storage == RTG_STORE_BF16 ? W_BF16 : W_F32;
  hipGetDevice(&m->device);
  const size_t wb = m->wtype == W_BF16 ? 2 : 4;
  // Arena layout: per layer [wqkv wproj wfc wmproj | biases | LN], then wte, wpe, ln_f.
  std::vector<size_t> offs;
  size_t cur = 0;
  auto take = [&](size_t bytes) {
    size_t o = cur;
    cur = align_up(cur + bytes, 256);
    return o;
  };
  struct LOff {
    size_t wqkv, waproj, wfc, wmproj, bqkv, baproj, bfc, bmproj, ln1w, ln1b, ln2w, ln2b;
  };
  std::vector<LOff> lo(L);
  for (size_t i = 0; i < L; ++i) {
    lo[i].wqkv = take(3 * d * d * wb);
    lo[i].waproj = take(d * d * wb);
    lo[i].wfc = take(4 * d * d * wb);
    lo[i].wmproj = take(4 * d * d * wb);
    lo[i].bqkv = take(3 * d * 4);
    lo[i].baproj = take(d * 4);
    lo[i].bfc = take(4 * d * 4);
    lo[i].bmproj = take(d * 4);
    lo[i].ln1w = take(d * 4);
    lo[i].ln1b = take(d * 4);
    lo[i].ln2w = take(d * 4);
    lo[i].ln2b = take(d * 4);
  }
  const size_t o_wte = take(V * d * wb), o_wpe = take(P * d * 4), o_lnfw = take(d * 4), o_lnfb = take(d * 4);
  float* staging = nullptr;
  bool own_staging = false;
  std::unique_ptr<PrefillWeights> pw;
  try {
    HIPX(device_malloc(&m->arena, cur));
    m->arena_bytes = cur;
    char* A = reinterpret_cast<char*>(m->arena);
    // (uploads pass through the memory of the prefill weights, which are made
    // last, where it is large enough: allocating 0.26 GB takes ~10 ms)
    const size_t stage_max = std::max({V * d, P * d, 4 * d * d}) * 4;
    pw = alloc_prefill_weights(m.get());
    own_staging = !pw || pw->bytes < stage_max;
    if (own_staging) {
      if (hipMalloc(&staging, stage_max) != hipSuccess) {
        (void)hipGetLastError();
        pw.reset();  // the load needs the staging, the prefill can do without its copy
        HIPX(device_malloc(&staging, stage_max));
      }
    } else staging = static_cast<float*>(pw->arena);
    hipStream_t s = nullptr;
    // Tensors go to the device in their own element type; widening,
    // narrowing to the storage type and the transpose run there.
    auto upload_f32 = [&](const std::string& nm, size_t off) {
      const auto& t = lk[nm];
      if (t.stype == SRC_F32) {
        HIPX(hipMemcpy(A + off, t.data, t.bytes(), hipMemcpyHostToDevice));
        return;
      }
      HIPX(hipMemcpy(staging, t.data, t.bytes(), hipMemcpyHostToDevice));
      launch_convert_to(s, staging, t.stype, (long)t.numel(), A + off, W_F32);
      HIPX(hipGetLastError());
      HIPX(hipDeviceSynchronize());
    };
    auto upload_wt = [&](const std::string& nm, size_t off) {  // [K][N] -> W^T [N][K] in storage type
      const auto& t = lk[nm];
      const size_t K = t.shape[0], N = t.shape[1];
      HIPX(hipMemcpy(staging, t.data, t.bytes(), hipMemcpyHostToDevice));
      launch_transpose_to(s, staging, t.stype, (int)K, (int)N, A + off, m->wtype);
      HIPX(hipGetLastError());
      HIPX(hipDeviceSynchronize());
    };
    m->layers.resize(L);
    for (size_t i = 0; i < L; ++i) {
      std::string p = "h." + std::to_string(i) + ".";
      upload_wt(p + "attn.c_attn.weight", lo[i].wqkv);
      upload_wt(p + "attn.c_proj.weight", lo[i].waproj);
      upload_wt(p + "mlp.c_fc.weight", lo[i].wfc);
      upload_wt(p + "mlp.c_proj.weight", lo[i].wmproj);
      upload_f32(p + "attn.c_attn.bias", lo[i].bqkv);
      upload_f32(p + "attn.c_proj.bias", lo[i].baproj);
      upload_f32(p + "mlp.c_fc.bias", lo[i].bfc);
      upload_f32(p + "mlp.c_proj.bias", lo[i].bmproj);
      upload_f32(p + "ln_1.weight", lo[i].ln1w);
      upload_f32(p + "ln_1.bias", lo[i].ln1b);
      upload_f32(p + "ln_2.weight", lo[i].ln2w);
      upload_f32(p + "ln_2.bias", lo[i].ln2b);
      LayerW& w = m->layers[i];
      w.wqkv = A + lo[i].wqkv;
      w.waproj = A + lo[i].waproj;
      w.wfc = A + lo[i].wfc;
      w.wmproj = A + lo[i].wmproj;
      w.bqkv = reinterpret_cast<float*>(A + lo[i].bqkv);
      w.baproj = reinterpret_cast<float*>(A + lo[i].baproj);
      w.bfc = reinterpret_cast<float*>(A + lo[i].bfc);
      w.bmproj = reinterpret_cast<float*>(A + lo[i].bmproj);
      w.ln1w = reinterpret_cast<float*>(A + lo[i].ln1w);
      w.ln1b = reinterpret_cast<float*>(A + lo[i].ln1b);
      w.ln2w = reinterpret_cast<float*>(A + lo[i].ln2w);
      w.ln2b = reinterpret_cast<float*>(A + lo[i].ln2b);
    }
    {
      const auto& t = lk["wte.weight"];
      HIPX(hipMemcpy(staging, t.data, t.bytes(), hipMemcpyHostToDevice));
      launch_convert_to(s, staging, t.stype, (long)(V * d), A + o_wte, m->wtype);
      HIPX(hipGetLastError());
      HIPX(hipDeviceSynchronize());
    }
    upload_f32("wpe.weight", o_wpe);
    upload_f32("ln_f.weight", o_lnfw);
    upload_f32("ln_f.bias", o_lnfb);
    m->wte = A + o_wte;
    m->wpe = reinterpret_cast<float*>(A + o_wpe);
    m->lnfw = reinterpret_cast<float*>(A + o_lnfw);
    m->lnfb = reinterpret_cast<float*>(A + o_lnfb);
    if (own_staging) HIPX(hipFree(staging));
    own_staging = false;
    build_prefill_weights(m.get(), std::move(pw));
  } catch (const HipError& he) {
    if (own_staging && staging) hipFree(staging);
    return err(he.msg);
  } catch (const std::exception& ex) {
    if (own_staging && staging) hipFree(staging);
    return err_internal(ex);
  }
  size_t np = V * d + P * d + 2 * d;
  np += L * (2 * d + d * 3 * d + 3 * d + d * d + d + 2 * d + d * 4 * d + 4 * d + 4 * d * d + d);
  m->nparams = np;
  {
    PersistentWeights pw;
    pw.cfg = m->cfg;
    pw.wtype = m->wtype;
    pw.wte = m->wte;
    pw.wpe = m->wpe;
    pw.lnfw = m->lnfw;
    pw.lnfb = m->lnfb;
    for (auto& l : m->layers)
      pw.layers.push_back({l.wqkv, l.waproj, l.wfc, l.wmproj, l.bqkv, l.baproj, l.bfc, l.bmproj, l.ln1w, l.ln1b,
                           l.ln2w, l.ln2b});
    m->pplan = persistent_plan_create(pw);
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess)
      m->rplan = rows_plan_create(pw, cus);
  }
  *out = m.release();
  return ok();
}

bool decode_f64(const void* data, size_t n, std::vector<float>* out) {
  out->resize(n);
  const uint8_t* raw = reinterpret_cast<const uint8_t*>(data);
  for (size_t i = 0; i < n; ++i) {
    double v;
    memcpy(&v, raw + 8 * i, 8);
    (*out)[i] = (float)v;
  }
  return true;
}
}  // namespace

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------

extern "C" {

void rtg_init(void) { hipInit(0); }
void rtg_cleanup(void) {
  std::lock_guard<std::mutex> g(host_stages().mu);
  host_stages().idle.clear();
}
const char* rtg_version(void) { return "rtgpu 0.1.0 (gfx950)"; }

void rtg_free_error_message(char* msg) { free(msg); }

rtg_result rtg_model_from_host(const rtg_config* cfg, const rtg_named_tensor* tensors, size_t n, rtg_storage storage,
                               rtg_model** out) {
  try {
    if (!cfg || !out) return err("null argument");
    Lookup lk;
    for (size_t i = 0; i < n; ++i) {
      const rtg_named_tensor& t = tensors[i];
      HostTensor& h = lk[t.name];
      h.shape.assign(t.shape, t.shape + t.ndim);
      switch (t.dtype) {
        case RTG_F32: h.stype = SRC_F32; h.data = t.data; break;
        case RTG_BF16: h.stype = SRC_BF16; h.data = t.data; break;
        case RTG_F16: h.stype = SRC_F16; h.data = t.data; break;
        case RTG_F64:
          decode_f64(t.data, h.numel(), &h.owned);
          h.stype = SRC_F32;
          h.data = h.owned.data();
          break;
        default: return err("Unsupported dtype for " + std::string(t.name));
      }
    }
    return build_model(cfg, lk, storage, out);
  } catch (const std::exception& ex) {
    return err_internal(ex);
  }
}

rtg_result rtg_model_from_safetensors(const char* path, const rtg_config* cfg, rtg_storage storage,
                                      rtg_model** out) {
  try {
    if (!cfg || !out || !path) return err("null argument");
    StFile f;
    std::string e = st_read_file(path, &f);
    if (!e.empty()) return err("Failed to load safetensors: " + e);
    // F32, BF16 and F16 tensors are used in place in the mapping (no host copy);
    // other element types are decoded to f32 (safetensors.rs:232-348).
    Lookup lk;
    for (auto& kv : f.entries) {
      const StEntry& en = kv.second;
      HostTensor& h = lk[kv.first];
      h.shape = en.shape;
      if (en.dtype == "F32" || en.dtype == "BF16" || en.dtype == "F16") {
        e = st_check_size(en, en.dtype == "F32" ? 4 : 2, en.dtype.c_str());
        h.stype = en.dtype == "F32" ? SRC_F32 : en.dtype == "BF16" ? SRC_BF16 : SRC_F16;
        h.data = st_data(f, en);
      } else {
        e = st_decode_f32(f, en, &h.owned);
        h.stype = SRC_F32;
        h.data = h.owned.data();
      }
      if (!e.empty()) return err("Failed to load safetensors: " + e);
    }
    return build_model(cfg, lk, storage, out);
  } catch (const std::exception& ex) {
    return err_internal(ex);
  }
}

void rtg_model_destroy(rtg_model* model) { delete model; }

size_t rtg_num_parameters(const rtg_model* model) { return model ? model->nparams : 0; }

rtg_result rtg_cache_new(const rtg_model* model, size_t batch, rtg_cache** out) {
  if (!model || !out) return err("null argument");
  if (batch == 0) return err("batch must be >= 1");
  try {
    *out = cache_create(model, batch);
  } catch (const HipError& e) {
    return err(e.msg);  } catch (const std::exception& ex) {
    return err_internal(ex);
  }
  return ok();
}

size_t rtg_cache_len(const rtg_cache* cache) { return cache ? cache->len : 0; }
bool rtg_cache_is_empty(const rtg_cache* cache) { return rtg_cache_len(cache) == 0; }
void rtg_cache_clear(rtg_cache* cache) {
  if (cache) cache->len = 0;
}

void rtg_cache_destroy(rtg_cache* c) {
  if (!c) return;
  if (c->stream) hipStreamSynchronize(c->stream);
  destroy_graph(c);
  if (c->pstate) persistent_state_destroy(c->pstate);
  if (c->rstate) rows_state_destroy(c->rstate);
  free_work(c);
  for (void* p : {(void*)c->k, (void*)c->v, (void*)c->pos_dev, (void*)c->step_dev, (void*)c->keys,
                  (void*)c->token_dev, (void*)c->ids_dev, (void*)c->ids_in, (void*)c->logits,
                  (void*)c->bg_part, (void*)c->bg_cnt, (void*)c->bg_spart, (void*)c->bg_cen,
                  c->sample_work})
    if (p) hipFree(p);
  for (auto e : c->ev)
    if (e) hipEventDestroy(e);
  if (c->stream) hipStreamDestroy(c->stream);
  delete c;
}

rtg_result rtg_cache_read(const rtg_cache* c, size_t layer, size_t head, size_t seq, int values, float* out) {
  if (!c || !out) return err("null argument");
  const rtg_model* m = c->m;
  if (layer >= m->cfg.n_layer || head >= m->cfg.n_head || seq >= c->batch) return err("index out of range");
  const size_t P = m->cfg.n_positions, hd = m->hd;
  const float* base = (values ? c->v : c->k) + layer * c->layer_stride + ((seq * m->cfg.n_head + head) * P) * hd;
  try {
    if (c->len) HIPX(hipMemcpy(out, base, c->len * hd * 4, hipMemcpyDeviceToHost));
  } catch (const HipError& e) {
    return err(e.msg);  } catch (const std::exception& ex) {
    return err_internal(ex);
  }
  return ok();
}

rtg_result rtg_forward_cached_batched(const rtg_model* model, rtg_cache* cache, const uint32_t* ids, size_t n,
                                      float* logits_out) {
  if (!model || !cache) return err("null argument");
  if (cache->m != model) return err("the cache belongs to another model");
  std::string e = check_cached(model, cache->len, ids, n);
  if (e.empty() && cache->batch > 1) e = check_ids(model, ids, n * cache->batch);
  if (!e.empty()) return err(e);
  try {
    forward_cached_impl(cache, ids, n, logits_out);
  } catch (const HipError& he) {
    return err(he.msg);  } catch (const std::exception& ex) {
    return err_internal(ex);
  }
  return ok();
}

rtg_result rtg_forward_cached(const rtg_model* model, rtg_cache* cache, const uint32_t* ids, size_t n,
                              float* logits_out) {
  if (cache && cache->batch != 1) return err("rtg_forward_cached needs a batch-1 cache");
  return rtg_forward_cached_batched(model, cache, ids, n, logits_out);
}

// rtg_forward_cached_noalloc for a prompt the multi-row forward takes: its
// state in the scratch array (the 64 KiB head, then its work rows), the
// logits after it; the same kernel and inputs as rtg_forward_cached's.
static rtg_result noalloc_rows(const rtg_model* model, rtg_cache* cache, const uint32_t* ids, size_t n,
                               float* logits_out) {
  const size_t V = model->cfg.vocab_size;
  const size_t state = align_up(rows_state_bytes(model->rplan, false), 256) / 4;
  if (state + n * V > kScratchHeadFloats + kScratchFloats)
    return err(fmt("rtg_forward_cached_noalloc: %zu new tokens need %zu bytes of scratch; it holds %zu", n,
                   (state + n * V - kScratchHeadFloats) * 4, kScratchFloats * 4));
  try {
    hipError_t he = hipSuccess;
    float* sp = scratch_device_ptr(model->device, &he);
    HIPX(he);
    static_assert(rows_state_head_bytes() == kScratchHeadFloats * sizeof(float), "scratch head");
    std::lock_guard<std::mutex> slock(scratch_lock(model->device));
    std::lock_guard<std::mutex> plock(persistent_launch_lock(model->device));
    RowsState st;  // over the scratch array (one region per buffer): nothing is allocated
    st.mem = sp;
    st.fresh = false;
    float* logits = sp + state;
    HIPX(hipMemcpyAsync(cache->ids_in, ids, n * 4, hipMemcpyHostToDevice, cache->stream));
    enqueue_rows(cache, cache->ids_in, 1, n, cache->len, logits_out ? logits : nullptr, &st);
    if (logits_out) HIPX(hipMemcpyAsync(logits_out, logits, n * V * 4, hipMemcpyDeviceToHost, cache->stream));
    HIPX(hipStreamSynchronize(cache->stream));
    check_rows(&st);
    cache->len += n;
  } catch (const HipError& he) {
    return err(he.msg);
  } catch (const std::exception& ex) {
    return err_internal(ex);
  }
  return ok();
}

rtg_result rtg_forward_cached_noalloc(const rtg_model* model, rtg_cache* cache, const uint32_t* ids, size_t n,
                                      float* logits_out) {
  if (!model || !cache || (n && !ids)) return err("null argument");
  // the pass runs cache->m's kernels on buffers sized from model's shape
  if (cache->m != model) return err("rtg_forward_cached_noalloc: the cache belongs to another model");
  if (cache->batch != 1) return err("rtg_forward_cached_noalloc needs a batch-1 cache");
  std::string e = check_cached(model, cache->len, ids, n);
  if (!e.empty()) return err(e);
  // x, ln, att [n][d], qkv [n][3d], h [n][4d], logits [n][V] in the device's
  // scratch array, each part on a 256-byte boundary like a hipMalloc'd buffer
  // (the same alignment, so the same kernels as rtg_forward_cached run)
  const size_t d = model->cfg.n_embd, V = model->cfg.vocab_size;
  const size_t pd = align_up(n * d, 64), p3 = align_up(3 * n * d, 64), p4 = align_up(4 * n * d, 64);
  const size_t pv = align_up(n * V, 64);
  // the split-k partial tiles the pass's GEMMs use at n rows (as much as the
  // cache's own workspace would hold for them, so the same kernels run)
  size_t pw = prefill_ws_floats(model, n, model->pw.get() != nullptr);
  pw = align_up(pw, 64);
  const size_t need = 3 * pd + p3 + p4 + pv;
  if (need > kScratchFloats)
    return err(fmt("rtg_forward_cached_noalloc: %zu new tokens need %zu bytes of scratch; it holds %zu", n,
                   need * 4, kScratchFloats * 4));
  // where the GEMMs' split-k partials do not fit beside the activations the
  // GEMMs run unsplit (the same sums in another order), so the limit is
  // exactly the activations' size and grows monotonically with n
  if (need + pw > kScratchFloats) pw = 0;
  if (rows_path(cache, 1, n)) return noalloc_rows(model, cache, ids, n, logits_out);
  try {
    hipError_t he = hipSuccess;
    float* sp = scratch_device_ptr(model->device, &he);
    HIPX(he);
    sp += kScratchHeadFloats;
    // every call on this device shares the array: one pass at a time (the
    // call has drained its stream when it returns)
    std::lock_guard<std::mutex> slock(scratch_lock(model->device));
    // Nothing here has to start at zero: every kernel of the pass writes its
    // output rows in full before they are read (the residual epilogues add
    // into x after the embedding has written it).
    Work w;
    w.x = sp;
    w.ln = w.x + pd;
    w.att = w.ln + pd;
    w.qkv = w.att + pd;
    w.h = w.qkv + p3;
    w.logits = w.h + p4;
    w.ws = pw ? w.logits + pv : nullptr;
    w.ws_floats = pw;
    HIPX(hipMemcpyAsync(cache->ids_in, ids, n * 4, hipMemcpyHostToDevice, cache->stream));
    enqueue_prefill(cache, w, cache->ids_in, 1, n, cache->len, logits_out ? LOGITS_ALL : LOGITS_NONE);
    HIPX(hipGetLastError());
    if (logits_out)
      HIPX(hipMemcpyAsync(logits_out, w.logits, n * V * 4, hipMemcpyDeviceToHost, cache->stream));
    HIPX(hipStreamSynchronize(cache->stream));
    cache->len += n;
  } catch (const HipError& he) {
    return err(he.msg);
  } catch (const std::exception& ex) {
    return err_internal(ex);
  }
  return ok();
}

rtg_result rtg_forward(const rtg_model* model, const uint32_t* ids, size_t n, float* logits_out) {
  if (!model) return err("null argument");
  // gpt2.rs:269-279
  if (n == 0) return err("Empty input");
  if (n > model->cfg.n_positions)
    return err(fmt("Sequence length %zu exceeds max position %zu", n, model->cfg.n_positions));
  std::string e = check_ids(model, ids, n);
  if (!e.empty()) return err(e);
  try {
    PoolLease lease(model, 1);
    forward_cached_impl(lease.c, ids, n, logits_out);
  } catch (const HipError& he) {
    return err(he.msg);  } catch (const std::exception& ex) {
    return err_internal(ex);
  }
  return ok();
}

rtg_result rtg_generate_cached_batched(const rtg_model* model, const uint32_t* prompts, size_t batch, size_t n,
                                       size_t max_new, uint32_t* out, rtg_timing* timing) {
  if (!model || !out) return err("null argument");
  if (batch == 0) return err("batch must be >= 1");
  const size_t P = model->cfg.n_positions;
  std::string e = check_cached(model, 0, prompts, n);
  if (e.empty() && batch > 1) e = check_ids(model, prompts, n * batch);
  if (!e.empty()) return err(e);
  // The reference fails at the first decode step whose total exceeds
  // n_positions and discards the partial result (gpt2.rs:369-374, 427-433).
  const size_t steps = max_new > 0 ? max_new : 1;
  if (n + steps - 1 > P) return err(fmt("Total sequence length %zu exceeds max position %zu", P + 1, P));
  try {
    generate_greedy(model, prompts, batch, n, max_new, out, timing);
  } catch (const HipError& he) {
    return err(he.msg);  } catch (const std::exception& ex) {
    return err_internal(ex);
  }
  return ok();
}

rtg_result rtg_generate_cached(const rtg_model* model, const uint32_t* prompt, size_t n, size_t max_new,
                               float temperature, uint64_t seed, uint32_t* out) {
  if (temperature <= 0.0f) return rtg_generate_cached_batched(model, prompt, 1, n, max_new, out, nullptr);
  if (!model || !out) return err("null argument");
  // Sampling path (gpt2.rs:405-441 with sample_with_temperature, :996-1017),
  // tokens chosen on the device.
  std::string e = check_cached(model, 0, prompt, n);
  if (!e.empty()) return err(e);
  const size_t P = model->cfg.n_positions;
  const size_t steps = max_new > 0 ? max_new : 1;
  if (n + steps - 1 > P) return err(fmt("Total sequence length %zu exceeds max position %zu", P + 1, P));
  const SampleParams sp{temperature, 0, 1.0f, 1.0f, seed, 0};
  try {
    generate_greedy(model, prompt, 1, n, max_new, out, nullptr, &sp);
  } catch (const HipError& he) {
    return err(he.msg);  } catch (const std::exception& ex) {
    return err_internal(ex);
  }
  return ok();
}

rtg_result rtg_generate_with_config(const rtg_model* model, const uint32_t* prompt, size_t n,
                                    const rtg_gen_config* cfg, uint32_t* out) {
  if (!model || !out || !cfg) return err("null argument");
  if (cfg->temperature <= 0.0f && cfg->repetition_penalty == 1.0f)
    return rtg_generate_cached_batched(model, prompt, 1, n, cfg->max_new_tokens, out, nullptr);
  std::string e = check_cached(model, 0, prompt, n);
  if (!e.empty()) return err(e);
  const size_t P = model->cfg.n_positions;
  const size_t steps = cfg->max_new_tokens > 0 ? cfg->max_new_tokens : 1;
  if (n + steps - 1 > P) return err(fmt("Total sequence length %zu exceeds max position %zu", P + 1, P));
  // sample_logits (gpt2.rs:871-906) on the device after every step
  const int k = cfg->top_k > (size_t)INT32_MAX ? INT32_MAX : (int)cfg->top_k;
  const SampleParams sp{cfg->temperature, k, cfg->top_p, cfg->repetition_penalty, cfg->seed, 0};
  try {
    generate_greedy(model, prompt, 1, n, cfg->max_new_tokens, out, nullptr, &sp);
  } catch (const HipError& he) {
    return err(he.msg);  } catch (const std::exception& ex) {
    return err_internal(ex);
  }
  return ok();
}

rtg_result rtg_generate(const rtg_model* model, const uint32_t* prompt, size_t n, size_t max_new, float temperature,
                        uint64_t seed, uint32_t* out) {
  if (!model || !out) return err("null argument");
  // gpt2.rs:311-346: each step runs forward() over the last n_positions
  // tokens and picks the next token from the last row's logits. The tokens
  // live in one device buffer: the step reads its window from there and the
  // device sampler appends its choice, so the loop never waits for the host.
  const size_t V = model->cfg.vocab_size, P = model->cfg.n_positions;
  if (max_new == 0) {
    memcpy(out, prompt, n * 4);
    return ok();
  }
  if (n == 0) return err("Empty input");
  // forward() checks the ids of each window; later windows add only sampled ids
  const size_t start0 = n > P ? n - P : 0;
  std::string e = check_ids(model, prompt + start0, n - start0);
  if (!e.empty()) return err(e);
  const size_t total = n + max_new;
  uint32_t* toks = nullptr;
  int* steps = nullptr;
  try {
    PoolLease lease(model, 1);
    rtg_cache* c = lease.c;
    hipStream_t s = c->stream;
    HIPX(device_malloc(&toks, total * 4));
    HIPX(device_malloc(&steps, max_new * 4));
    std::vector<int> step_no(max_new);
    for (size_t i = 0; i < max_new; ++i) step_no[i] = (int)(i + 1);  // the sampler's generation index + 1
    HIPX(hipMemcpyAsync(toks, prompt, n * 4, hipMemcpyHostToDevice, s));
    HIPX(hipMemcpyAsync(steps, step_no.data(), max_new * 4, hipMemcpyHostToDevice, s));
    c->len = 0;
    ensure_rows(c, std::min(total - 1, P));
    if (temperature > 0.0f) ensure_ws(c, std::min(total - 1, P), false);
    ensure_logits(c, 1);
    ensure_sample_work(c);
    // sample_with_temperature (gpt2.rs:996-1017); argmax for temperature <= 0.
    // Draw k of the seeded sequence goes to generation index k - 1.
    const SampleParams sp{temperature, 0, 1.0f, 1.0f, seed, 0};
    for (size_t i = 0; i < max_new; ++i) {
      const size_t len = n + i;
      const size_t start = len > P ? len - P : 0;
      enqueue_prefill(c, cache_work(c), toks + start, 1, len - start, 0, LOGITS_LAST, temperature > 0.0f);
      if (!launch_sample(s, c->logits, (int)V, toks, (int)n, toks + n, steps + i, sp, c->token_dev,
                         c->sample_work))
        throw HipError{"vocabulary too large for the device sampler"};
    }
    HIPX(hipMemcpyAsync(out, toks, total * 4, hipMemcpyDeviceToHost, s));
    HIPX(hipStreamSynchronize(s));
    c->len = 0;
  } catch (const HipError& he) {
    if (toks) hipFree(toks);
    if (steps) hipFree(steps);
    return err(he.msg);  } catch (const std::exception& ex) {
    if (toks) hipFree(toks);
    if (steps) hipFree(steps);
    return err_internal(ex);
  }
  hipFree(toks);
  hipFree(steps);
  return ok();
}

}  // extern "C"
