// The dense path around the MoE block: the rest of a GPT-OSS decoder step as
// CpuModel::prepare_step runs it (crates/gpt-oss-model-runner/src/
// cpu_runner.rs:2103-2333, forward_layer_batch :2335-2586), on the GPU: a step
// is one copy in (the embedding rows), launches on the context's stream, one
// copy out (the logits) and one synchronization. Each layer's MoE half
// (post-attention RMSNorm, moe_batch, residual add) goes through
// gossmx_moe_forward_residual. The steps used to run norms, RoPE and attention
// on host threads with two round trips a layer: a 63-token prefill and 8
// decodes of two GPT-OSS-20B layers went from 9.76 to 4.67 ms.
//
// - bf16 projections: Kernels::bf16_matvec (gpt-oss-cpu-kernels lib.rs:314-341)
//   with its 16 fixed reduction lanes, multiply then add, lanes folded 0..15
//   (scalar_bf16_dot lib.rs:1007-1029), then += bias (project_bf16[_batch]
//   cpu_runner.rs:2689-2792): dense_proj_kernel and dense_gemv_kernel, over
//   copies of the Q/K/V/O weights and lm_head made in HBM when the model is
//   created.
// - RMSNorm boundaries: norm_boundary (:2680-2687) over Kernels::rms_norm
//   (lib.rs:699-730, the same 16-lane sum of squares): dense_norm_kernel.
// - YaRN RoPE (YarnRope :3927-4013) with its bf16 boundaries, by the host's
//   cosines and sines: qkv_finish_kernel.
// - Attention with learned sinks over the visible KV window
//   (attention_one_staged :3840-3924): attention_kernel. The KV cache of
//   CpuKvCache (:653-740): a sliding layer keeps sliding_window tokens, a full
//   layer context_cap. A step's rows count as cached only when the whole step
//   succeeded (PreparedCpuStep::commit, :1081-1113).
// - Residual adds (add_residual :3732-3738), the final norm, lm_head and its
//   bf16 round trip with the finiteness check (:2255-2312).
// powf, cosf, sinf and log are the host C library's, as is expf in
// gossmx_attention: the functions Rust's f32/f64 methods call on x86_64 Linux
// (attention_kernel's expf_glibc has the same results).

#include "../../include/gossmx.h"
#include "gossmx_internal.h"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <new>
#include <type_traits>
#include <utility>
#include <vector>

namespace {

int err(int status, const char* message) { return gossmx::set_error(status, message); }

inline uint32_t f2u(float f) { uint32_t u; std::memcpy(&u, &f, 4); return u; }
inline float u2f(uint32_t u) { float f; std::memcpy(&f, &u, 4); return f; }
// bf16::from_f32 of half 2.7.1: round to nearest even, NaN quieted.
inline uint16_t bf16_bits(float f) {
  const uint32_t u = f2u(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
  const uint32_t round_bit = 0x8000u;
  const uint32_t up = ((u & round_bit) != 0 && (u & (3 * round_bit - 1)) != 0) ? 1u : 0u;
  return (uint16_t)((u >> 16) + up);
}
inline float bf16_f32(uint16_t b) { return u2f((uint32_t)b << 16); }
inline float bf16_round(float f) { return bf16_f32(bf16_bits(f)); }

// ---------------------------------------------------------------------------
// YaRN RoPE (YarnRope::new / apply, cpu_runner.rs:3933-4013).

struct Rope {
  std::vector<float> inv_freq;
  float attention_scale = 1.0f;
  size_t head_dim = 0;
};

Rope make_rope(const gossmx_model_config& c) {
  Rope r;
  const size_t dim = c.head_dim;
  r.head_dim = dim;
  const float theta = (float)c.rope_theta;
  if (!c.rope_yarn) {
    for (size_t i = 0; i < dim; i += 2) r.inv_freq.push_back(1.0f / powf(theta, (float)i / (float)dim));
    return r;
  }
  const double two_pi = 6.283185307179586;
  auto correction = [&](double rotations) {
    return ((double)dim * std::log((double)c.rope_original_max_positions / (rotations * two_pi))) /
           (2.0 * std::log(c.rope_theta));
  };
  double low = correction(c.rope_beta_fast), high = correction(c.rope_beta_slow);
  if (c.rope_truncate) {
    low = std::floor(low);
    high = std::ceil(high);
  }
  low = std::max(low, 0.0);
  high = std::min(high, (double)(dim - 1));
  const double range = std::max(std::fabs(high - low), 0.001);
  for (size_t i = 0; i < dim / 2; ++i) {
    const float frequency = powf(theta, (float)(i * 2) / (float)dim);
    const float extrapolation = 1.0f / frequency;
    const float interpolation = 1.0f / ((float)c.rope_factor * frequency);
    float ramp = ((float)i - (float)low) / (float)range;
    ramp = std::min(std::max(ramp, 0.0f), 1.0f);
    r.inv_freq.push_back(interpolation * ramp + extrapolation * (1.0f - ramp));
  }
  r.attention_scale = (float)(0.1 * std::log(c.rope_factor) + 1.0);
  return r;
}

// The bf16 cosines, then sines, of a position: they depend on (position, i)
// only and every head shares them.
void rope_row(const Rope& r, size_t position, float* table) {
  const size_t half = r.head_dim / 2;
  for (size_t i = 0; i < half; ++i) {
    const float angle = (float)position * r.inv_freq[i];
    table[i] = bf16_round(cosf(angle) * r.attention_scale);
    table[half + i] = bf16_round(sinf(angle) * r.attention_scale);
  }
}

void rope_apply(const Rope& r, float* v, size_t heads, size_t position) {
  const size_t half = r.head_dim / 2;
  std::vector<float> table(2 * half);
  rope_row(r, position, table.data());
  for (size_t h = 0; h < heads; ++h) {
    float* p = v + h * r.head_dim;
    for (size_t i = 0; i < half; ++i) {
      const float cosine = table[i], sine = table[half + i];
      const float left = bf16_round(p[i]), right = bf16_round(p[half + i]);
      const float left_cosine = bf16_round(left * cosine), right_sine = bf16_round(right * sine);
      const float right_cosine = bf16_round(right * cosine), left_sine = bf16_round(left * sine);
      p[i] = bf16_round(left_cosine - right_sine);
      p[half + i] = bf16_round(right_cosine + left_sine);
    }
  }
}

// ---------------------------------------------------------------------------
// Attention for one query over `tokens` visible key/value rows, oldest first
// (attention_one_staged): bf16 QK dot, bf16 scale, softmax with the sink in
// the denominator, bf16 probabilities, f32 accumulation, bf16 output.
// keys and values are rows of kv_heads * head_dim. gossmx_attention's; a
// model's steps run attention_kernel, with the same float chains.

float attention_scale(size_t head_dim) { return 1.0f / std::sqrt((float)head_dim); }

void attention(const float* q_all, size_t tokens, const uint16_t* keys, const uint16_t* values, const float* sinks,
               size_t heads, size_t kv_heads, size_t head_dim, float* out) {
  const size_t groups = heads / kv_heads, width = kv_heads * head_dim;
  const float scale = attention_scale(head_dim);
  std::vector<float> scores(tokens);
  for (size_t h = 0; h < heads; ++h) {
    const float* q = q_all + h * head_dim;
    const size_t kvh = h / groups;
    for (size_t t = 0; t < tokens; ++t) {
      const uint16_t* k = keys + t * width + kvh * head_dim;
      float dot = 0.0f;
      for (size_t d = 0; d < head_dim; ++d) dot += q[d] * bf16_f32(k[d]);
      dot = bf16_round(dot);
      scores[t] = bf16_round(dot * scale);
    }
    float maximum = sinks[h];
    for (size_t t = 0; t < tokens; ++t) maximum = std::fmax(maximum, scores[t]);
    float sum = 0.0f;
    for (size_t t = 0; t < tokens; ++t) sum += expf(scores[t] - maximum);
    const float denominator = expf(sinks[h] - maximum) + sum;
    float* o = out + h * head_dim;
    for (size_t d = 0; d < head_dim; ++d) o[d] = 0.0f;
    for (size_t t = 0; t < tokens; ++t) {
      const float p = bf16_round(expf(scores[t] - maximum) / denominator);
      const uint16_t* v = values + t * width + kvh * head_dim;
      for (size_t d = 0; d < head_dim; ++d) o[d] += p * bf16_f32(v[d]);
    }
    for (size_t d = 0; d < head_dim; ++d) o[d] = bf16_round(o[d]);
  }
}

// The KV cache of one layer (CpuKvCache): the last min(positions, capacity)
// tokens are committed. On the device it is a ring of `slots` rows, position p
// in slot p % slots, with room for the m rows of a step beside every committed
// row that a later step can still see (the last capacity - 1): a step writes
// its rows there, and committing them is the host's `len` and `start` alone.
struct KvCache {
  size_t capacity = 0, len = 0, start = 0;
  size_t slots = 0;
  uint16_t *k = nullptr, *v = nullptr;
  void append(size_t p) {
    if (len == capacity) ++start;
    else ++len;
    if (len == 1) start = p;
  }
};

double seconds_since(std::chrono::steady_clock::time_point t0) {
  return std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
}

int check_config(const gossmx_model_config* c) {
  if (!c) return err(GOSSMX_ERR_INVALID_ARGUMENT, "null model config");
  if (!c->vocab || !c->hidden || !c->layers || !c->heads || !c->kv_heads || !c->head_dim || c->head_dim % 2 ||
      c->heads % c->kv_heads || !c->sliding_window || !c->context_cap)
    return err(GOSSMX_ERR_INVALID_DIMENSIONS,
               "model config needs non-zero sizes, an even head_dim and heads divisible by kv_heads");
  if (c->rope_yarn && (c->rope_factor <= 0.0 || !c->rope_original_max_positions))
    return err(GOSSMX_ERR_INVALID_DIMENSIONS, "YaRN scaling needs a positive factor and original positions");
  return GOSSMX_OK;
}

}  // namespace

// The model's device side: its dense tensors but the embedding copied to HBM,
// the RoPE table, and grow-only buffers for a step's rows.
struct DenseDevice {
  struct Layer {
    const uint16_t *q, *k, *v, *o;
    const float *qb, *kb, *vb, *ob;
    const float *input_norm, *post_norm, *sinks;
  };
  int device = 0;
  std::vector<void*> weights;  // device allocations of the copies
  std::vector<Layer> layers;
  const uint16_t* lm_head = nullptr;
  const float* final_norm = nullptr;
  float* rope = nullptr;  // cosines and sines (rope_row) of the positions below rope_rows
  size_t rope_rows = 0;
  char *work = nullptr, *host_in = nullptr, *host_out = nullptr;  // a step's device rows; pinned input and results
  size_t work_cap = 0, in_cap = 0, out_cap = 0;                  // bytes
  double clock_hz = 1e8;  // of wall_clock64
  ~DenseDevice() {
    (void)hipSetDevice(device);
    for (void* p : weights) (void)hipFree(p);
    (void)hipFree(rope);
    (void)hipFree(work);
    (void)hipHostFree(host_in);
    (void)hipHostFree(host_out);
  }
};

struct gossmx_model {
  gossmx_ctx* ctx = nullptr;
  gossmx_model_config cfg{};
  const uint16_t* embedding = nullptr;
  std::vector<gossmx_dense_layer> layers;
  Rope rope;
  std::vector<KvCache> caches;
  size_t position = 0;
  DenseDevice dev;
  double dense_seconds = 0.0, moe_seconds = 0.0;
  ~gossmx_model() {
    (void)hipSetDevice(dev.device);
    for (KvCache& kv : caches) {
      (void)hipFree(kv.k);
      (void)hipFree(kv.v);
    }
  }
};

namespace {

int hip_err(hipError_t e, const char* what) {
  char msg[256];
  std::snprintf(msg, sizeof msg, "%s: %s", what, hipGetErrorString(e));
  return err(e == hipErrorOutOfMemory ? GOSSMX_ERR_OUT_OF_MEMORY : GOSSMX_ERR_DEVICE, msg);
}

#define DENSE_HIP(expr, what)                        \
  do {                                               \
    const hipError_t e_ = (expr);                    \
    if (e_ != hipSuccess) return hip_err(e_, what);  \
  } while (0)

// A copy of n elements of T in device memory, owned by the model.
template <class T>
int upload(DenseDevice& D, const T* src, size_t n, const T** dst) {
  void* p = nullptr;
  DENSE_HIP(hipMalloc(&p, n * sizeof(T)), "model weights allocation");
  D.weights.push_back(p);
  gossmx::count_transfer(gossmx::kTransferUpload, n * sizeof(T));
  DENSE_HIP(hipMemcpy(p, src, n * sizeof(T), hipMemcpyHostToDevice), "model weights upload");
  *dst = static_cast<const T*>(p);
  return GOSSMX_OK;
}

// Grows a device (or, pinned, a host) buffer to n bytes; its contents go.
int grow(char** p, size_t* cap, size_t n, bool pinned) {
  if (n <= *cap) return GOSSMX_OK;
  if (pinned) (void)hipHostFree(*p);
  else (void)hipFree(*p);
  *p = nullptr;
  *cap = 0;
  if (pinned) DENSE_HIP(hipHostMalloc((void**)p, n), "step staging");
  else DENSE_HIP(hipMalloc((void**)p, n), "step buffer");
  *cap = n;
  return GOSSMX_OK;
}

// The RoPE table covers positions below `rows`. It doubles, so a sequence
// computes each position's cosines and sines (host cosf and sinf) about twice
// at most.
int grow_rope(gossmx_model* M, size_t rows, hipStream_t stream) {
  DenseDevice& D = M->dev;
  if (rows <= D.rope_rows) return GOSSMX_OK;
  const size_t dim = M->cfg.head_dim;
  const size_t n = std::max(rows, std::min(std::max<size_t>(2 * D.rope_rows, 64), M->cfg.context_cap));
  std::vector<float> table(n * dim);
  for (size_t p = 0; p < n; ++p) rope_row(M->rope, p, &table[p * dim]);
  float* d = nullptr;
  DENSE_HIP(hipMalloc((void**)&d, n * dim * sizeof(float)), "rotation table");
  gossmx::count_transfer(gossmx::kTransferUpload, n * dim * sizeof(float));
  hipError_t e = hipMemcpyAsync(d, table.data(), n * dim * sizeof(float), hipMemcpyHostToDevice, stream);
  if (e == hipSuccess) e = hipStreamSynchronize(stream);
  if (e != hipSuccess) {
    (void)hipFree(d);
    return hip_err(e, "rotation table copy");
  }
  (void)hipFree(D.rope);
  D.rope = d;
  D.rope_rows = n;
  return GOSSMX_OK;
}

// Room for m rows at position `base` in a layer's ring (KvCache). A larger
// ring takes the committed rows that can still be seen to their new slots.
int grow_ring(gossmx_model* M, KvCache& kv, size_t base, size_t m, hipStream_t stream) {
  const size_t needed = std::min(base, kv.capacity - 1) + m;
  if (needed <= kv.slots) return GOSSMX_OK;
  const size_t width = M->cfg.kv_heads * M->cfg.head_dim;
  const size_t n = std::max(needed, std::min(std::max<size_t>(2 * kv.slots, 256), M->cfg.context_cap));
  uint16_t* ring[2] = {nullptr, nullptr};
  hipError_t e = hipMalloc((void**)&ring[0], n * width * 2);
  if (e == hipSuccess) e = hipMalloc((void**)&ring[1], n * width * 2);
  const size_t keep = std::min(kv.len, kv.capacity - 1);
  for (size_t p = base - keep; p < base && e == hipSuccess;) {
    const size_t from = p % kv.slots, to = p % n, run = std::min(base - p, std::min(kv.slots - from, n - to));
    for (int i = 0; i < 2 && e == hipSuccess; ++i)
      e = hipMemcpyAsync(ring[i] + to * width, (i ? kv.v : kv.k) + from * width, run * width * 2,
                         hipMemcpyDeviceToDevice, stream);
    p += run;
  }
  if (e == hipSuccess) e = hipStreamSynchronize(stream);
  if (e != hipSuccess) {
    (void)hipStreamSynchronize(stream);
    (void)hipFree(ring[0]);
    (void)hipFree(ring[1]);
    return hip_err(e, "KV cache growth");
  }
  (void)hipFree(kv.k);
  (void)hipFree(kv.v);
  kv.k = ring[0];
  kv.v = ring[1];
  kv.slots = n;
  return GOSSMX_OK;
}

// Up to three projections of one input (project_bf16[_batch]) in one launch.
// One token through small matrices (Q/K/V, O): work-groups stage their whole K
// range at once; batches: the K-chunked kernel.
hipError_t project(const gossmx::DenseSet& set, int count, const float* in, size_t cols, size_t m, hipStream_t stream) {
  size_t rows = 0;
  for (int i = 0; i < count; ++i) rows += set.rows[i];
  return m == 1 && cols % 8 == 0 && cols <= 4096 && rows <= 65536
             ? gossmx::launch_dense_gemv(set, count, in, (int)cols, stream)
             : gossmx::launch_dense_proj(set, count, in, (int)cols, (int)m, stream);
}

// A step's buffers in DenseDevice::work: m rows each.
struct StepRows {
  uint16_t *hidden, *after, *next;      // [hidden] bf16
  float *x, *q, *k, *v, *proj;          // the next projections' input; Q, K, V and O outputs
  char* out;                            // the results that go to the host: marks, logits
};

size_t out_bytes(const gossmx_model_config& c) { return c.layers * sizeof(gossmx::ModelMark) + c.vocab * 2; }

// Enqueues one layer-major step over the m rows whose embeddings are in
// host_in, and the copy of its marks and the last row's logits to host_out.
// *enqueued counts the layers whose MoE call was enqueued.
int enqueue_step(gossmx_model* M, size_t m, const StepRows& R, hipStream_t stream, size_t* enqueued) {
  const gossmx_model_config& c = M->cfg;
  DenseDevice& D = M->dev;
  const size_t H = c.hidden, QW = c.heads * c.head_dim, KW = c.kv_heads * c.head_dim, n = m * H;
  const size_t base = M->position;
  gossmx::ModelMark* marks = reinterpret_cast<gossmx::ModelMark*>(R.out);
  uint16_t* logits = reinterpret_cast<uint16_t*>(R.out + c.layers * sizeof(gossmx::ModelMark));
  const int* flags = gossmx::context_error_flags(M->ctx);
  gossmx::count_transfer(gossmx::kTransferActivation, n * 2);
  DENSE_HIP(hipMemcpyAsync(R.hidden, D.host_in, n * 2, hipMemcpyHostToDevice, stream), "embedding rows copy");
  uint16_t *hidden = R.hidden, *next = R.next;
  for (size_t li = 0; li < c.layers; ++li) {
    const DenseDevice::Layer& L = D.layers[li];
    KvCache& kv = M->caches[li];
    DENSE_HIP(gossmx::launch_dense_norm(hidden, L.input_norm, (int)m, (int)H, c.rms_norm_eps, R.x,
                                        li ? marks + li - 1 : nullptr, flags, stream),
              "input norm launch");
    gossmx::DenseSet qkv{};
    const uint16_t* w[3] = {L.q, L.k, L.v};
    const float* bias[3] = {L.qb, L.kb, L.vb};
    float* out[3] = {R.q, R.k, R.v};
    for (int i = 0; i < 3; ++i) {
      qkv.w[i] = w[i];
      qkv.bias[i] = bias[i];
      qkv.out[i] = out[i];
      qkv.rows[i] = (int)(i ? KW : QW);
    }
    DENSE_HIP(project(qkv, 3, R.x, H, m, stream), "projection launch");
    gossmx::AttnArgs a{};
    a.q = R.q;
    a.k_new = R.k;
    a.v_new = R.v;
    a.rope = D.rope;
    a.k = kv.k;
    a.v = kv.v;
    a.sinks = L.sinks;
    a.out = R.x;
    a.base = base;
    a.len = kv.len;
    a.capacity = kv.capacity;
    a.slots = kv.slots;
    a.m = (int)m;
    a.heads = (int)c.heads;
    a.kv_heads = (int)c.kv_heads;
    a.head_dim = (int)c.head_dim;
    a.scale = attention_scale(c.head_dim);
    DENSE_HIP(gossmx::launch_attention(a, stream), "attention launch");
    gossmx::DenseSet o{};
    o.w[0] = L.o;
    o.bias[0] = L.ob;
    o.out[0] = R.proj;
    o.rows[0] = (int)H;
    DENSE_HIP(project(o, 1, R.x, QW, m, stream), "projection launch");
    DENSE_HIP(gossmx::launch_residual_add(hidden, R.proj, R.after, n, &marks[li].begin, stream), "residual add launch");
    // The MoE half (norm_boundary(after, post_attention_norm), moe_batch,
    // add_residual) -> the next layer's rows. The block's profile records carry
    // the layer and the phase.
    (void)gossmx_profile_tag(M->ctx, (int)li, base == 0 || m > 1 ? GOSSMX_PHASE_PREFILL : GOSSMX_PHASE_DECODE);
    gossmx_moe_io io{};
    io.x = R.after;
    io.m = m;
    io.memory = GOSSMX_MEM_DEVICE;
    const int st = gossmx_moe_forward_residual(M->ctx, M->layers[li].moe, &io, L.post_norm, c.rms_norm_eps, next);
    (void)gossmx_profile_tag(M->ctx, -1, GOSSMX_PHASE_UNKNOWN);
    if (st != GOSSMX_OK) return st;
    ++*enqueued;
    std::swap(hidden, next);
  }
  // Final norm and lm_head for the last row (the only row whose logits are required).
  DENSE_HIP(gossmx::launch_dense_norm(hidden + (m - 1) * H, D.final_norm, 1, (int)H, c.rms_norm_eps, R.x,
                                      marks + c.layers - 1, flags, stream),
            "final norm launch");
  DENSE_HIP(gossmx::launch_lm_head(D.lm_head, R.x, logits, (int)c.vocab, (int)H, stream), "projection launch");
  gossmx::count_transfer(gossmx::kTransferOutput, out_bytes(c));
  DENSE_HIP(hipMemcpyAsync(D.host_out, R.out, out_bytes(c), hipMemcpyDeviceToHost, stream), "logits copy");
  return GOSSMX_OK;
}

// The GPU side of a step: one copy in, its launches, one copy out, one
// synchronization. The MoE calls' error flags are reported as the first layer
// that raised any left them; *moe becomes the time between the marks.
int gpu_step(gossmx_model* M, const uint32_t* tokens, size_t m, double* moe) {
  const gossmx_model_config& c = M->cfg;
  DenseDevice& D = M->dev;
  // The context's stream is read on every step: gossmx_ctx_set_stream may have
  // replaced it since the last one.
  const hipStream_t stream = gossmx::context_stream(M->ctx);
  const size_t H = c.hidden, QW = c.heads * c.head_dim, KW = c.kv_heads * c.head_dim;
  DENSE_HIP(hipSetDevice(D.device), "hipSetDevice");
  StepRows R{};
  size_t bytes = 0;
  auto place = [&](auto** p, size_t n) {
    *p = reinterpret_cast<std::remove_reference_t<decltype(*p)>>(reinterpret_cast<uintptr_t>(D.work) + bytes);
    bytes += (n * sizeof(**p) + 255) / 256 * 256;
  };
  for (int pass = 0; pass < 2; ++pass) {  // sizes, then addresses
    bytes = 0;
    place(&R.hidden, m * H);
    place(&R.after, m * H);
    place(&R.next, m * H);
    place(&R.x, m * std::max(H, QW));
    place(&R.q, m * QW);
    place(&R.k, m * KW);
    place(&R.v, m * KW);
    place(&R.proj, m * H);
    place(&R.out, out_bytes(c));
    if (int st = grow(&D.work, &D.work_cap, bytes, false)) return st;
  }
  if (int st = grow(&D.host_in, &D.in_cap, m * H * 2, true)) return st;
  if (int st = grow(&D.host_out, &D.out_cap, out_bytes(c), true)) return st;
  if (int st = grow_rope(M, M->position + m, stream)) return st;
  for (KvCache& kv : M->caches)
    if (int st = grow_ring(M, kv, M->position, m, stream)) return st;
  for (size_t r = 0; r < m; ++r)
    std::memcpy(D.host_in + r * H * 2, M->embedding + (size_t)tokens[r] * H, H * 2);
  size_t enqueued = 0;
  const int st = enqueue_step(M, m, R, stream, &enqueued);
  if (st != GOSSMX_OK) {
    (void)hipStreamSynchronize(stream);  // the staging buffers' copies end before the next step reuses them
    // An earlier layer may have raised the error flags: its error comes first,
    // and the flags are not left for the next call.
    const int raised = enqueued ? gossmx::context_errors(M->ctx) : GOSSMX_OK;
    return raised != GOSSMX_OK ? raised : st;
  }
  DENSE_HIP(hipStreamSynchronize(stream), "model step");
  const gossmx::ModelMark* marks = reinterpret_cast<const gossmx::ModelMark*>(D.host_out);
  uint64_t ticks = 0;
  for (size_t li = 0; li < c.layers; ++li) {
    if (marks[li].flags) return gossmx::error_flags_result(M->ctx, marks[li].flags);
    ticks += marks[li].end - marks[li].begin;
  }
  *moe = (double)ticks / D.clock_hz;
  return GOSSMX_OK;
}

// One layer-major step over m rows at positions model->position + r
// (prepare_step with every row in one sequence). Writes the last row's logits.
// The caches change only when the step succeeds. A run-time failure on the GPU
// (HIP error, out of memory) opens the circuit breaker, as a failed projection
// call does.
int run_step(gossmx_model* M, const uint32_t* tokens, size_t m, float* logits) {
  const gossmx_model_config& c = M->cfg;
  for (size_t r = 0; r < m; ++r)
    if (tokens[r] >= c.vocab) return err(GOSSMX_ERR_INVALID_ARGUMENT, "token id is not below vocab");
  if (M->position + m > c.context_cap)
    return err(GOSSMX_ERR_INVALID_DIMENSIONS, "the step would pass the sequence's context cap");
  const auto t_step = std::chrono::steady_clock::now();
  double moe = 0.0;
  if (int st = gossmx::run_time_result(M->ctx, gpu_step(M, tokens, m, &moe))) return st;
  // The logits are bf16 values; an exponent of all ones is an infinity or a NaN.
  const uint16_t* bits =
      reinterpret_cast<const uint16_t*>(M->dev.host_out + c.layers * sizeof(gossmx::ModelMark));
  uint32_t not_finite = 0;
  for (size_t i = 0; i < c.vocab; ++i) {
    not_finite |= (bits[i] & 0x7f80u) == 0x7f80u;
    logits[i] = bf16_f32(bits[i]);
  }
  if (not_finite) return err(GOSSMX_ERR_NON_FINITE_LOGITS, "CPU model produced non-finite logits");
  // Commit the step's rows.
  for (KvCache& kv : M->caches)
    for (size_t r = 0; r < m; ++r) kv.append(M->position + r);
  M->position += m;
  M->moe_seconds += moe;
  M->dense_seconds += std::max(0.0, seconds_since(t_step) - moe);
  return GOSSMX_OK;
}

// Empty caches; the rings stay allocated.
void reset_caches(gossmx_model* M) {
  M->caches.resize(M->cfg.layers);
  for (size_t li = 0; li < M->cfg.layers; ++li) {
    KvCache& kv = M->caches[li];
    kv.capacity = M->layers[li].sliding ? M->cfg.sliding_window : M->cfg.context_cap;
    kv.len = kv.start = 0;
  }
  M->position = 0;
}

}  // namespace

extern "C" {

int gossmx_model_create(gossmx_ctx* ctx, const gossmx_model_config* config, const uint16_t* embedding,
                        const float* final_norm, const uint16_t* lm_head, const gossmx_dense_layer* layers,
                        gossmx_model** out) {
  if (!ctx || !embedding || !final_norm || !lm_head || !layers || !out)
    return err(GOSSMX_ERR_INVALID_ARGUMENT, "null argument");
  *out = nullptr;
  if (int st = check_config(config)) return st;
  for (size_t li = 0; li < config->layers; ++li) {
    const gossmx_dense_layer& L = layers[li];
    if (!L.input_norm || !L.q_weight || !L.q_bias || !L.k_weight || !L.k_bias || !L.v_weight || !L.v_bias ||
        !L.o_weight || !L.o_bias || !L.sinks || !L.post_attention_norm || !L.moe)
      return err(GOSSMX_ERR_INVALID_ARGUMENT, "null layer tensor");
    const gossmx_moe_config* mc = gossmx::layer_config(L.moe);
    if (mc->hidden != config->hidden)
      return err(GOSSMX_ERR_INVALID_DIMENSIONS, "MoE layer hidden size differs from the model's");
  }
  gossmx_model* M = new (std::nothrow) gossmx_model;
  if (!M) return err(GOSSMX_ERR_OUT_OF_MEMORY, "model allocation failed");
  M->ctx = ctx;
  M->cfg = *config;
  M->embedding = embedding;
  M->layers.assign(layers, layers + config->layers);
  M->rope = make_rope(*config);
  reset_caches(M);
  // The dense tensors but the embedding go to the context's GPU.
  const size_t H = config->hidden, QW = config->heads * config->head_dim, KW = config->kv_heads * config->head_dim;
  DenseDevice& D = M->dev;
  D.device = gossmx::context_device(ctx);
  int st = hipSetDevice(D.device) == hipSuccess ? GOSSMX_OK : err(GOSSMX_ERR_DEVICE, "hipSetDevice failed");
  int khz = 0;
  if (st == GOSSMX_OK && hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, D.device) == hipSuccess && khz > 0)
    D.clock_hz = 1e3 * khz;
  D.layers.resize(config->layers);
  for (size_t li = 0; li < config->layers && st == GOSSMX_OK; ++li) {
    const gossmx_dense_layer& L = layers[li];
    DenseDevice::Layer& DL = D.layers[li];
    if (!st) st = upload(D, L.q_weight, QW * H, &DL.q);
    if (!st) st = upload(D, L.k_weight, KW * H, &DL.k);
    if (!st) st = upload(D, L.v_weight, KW * H, &DL.v);
    if (!st) st = upload(D, L.o_weight, H * QW, &DL.o);
    if (!st) st = upload(D, L.q_bias, QW, &DL.qb);
    if (!st) st = upload(D, L.k_bias, KW, &DL.kb);
    if (!st) st = upload(D, L.v_bias, KW, &DL.vb);
    if (!st) st = upload(D, L.o_bias, H, &DL.ob);
    if (!st) st = upload(D, L.input_norm, H, &DL.input_norm);
    if (!st) st = upload(D, L.post_attention_norm, H, &DL.post_norm);
    if (!st) st = upload(D, L.sinks, config->heads, &DL.sinks);
  }
  if (!st) st = upload(D, final_norm, H, &D.final_norm);
  if (!st) st = upload(D, lm_head, config->vocab * H, &D.lm_head);
  if (st) {
    delete M;
    return st;
  }
  *out = M;
  return GOSSMX_OK;
}

void gossmx_model_destroy(gossmx_model* model) { delete model; }

int gossmx_model_reset(gossmx_model* model) {
  if (!model) return err(GOSSMX_ERR_INVALID_ARGUMENT, "null model");
  reset_caches(model);
  return GOSSMX_OK;
}

int gossmx_model_prefill(gossmx_model* model, const uint32_t* tokens, size_t n, float* logits) {
  if (!model || !tokens || !logits) return err(GOSSMX_ERR_INVALID_ARGUMENT, "null argument");
  if (!n) return err(GOSSMX_ERR_INVALID_DIMENSIONS, "CPU prefill is empty");
  reset_caches(model);
  return run_step(model, tokens, n, logits);
}

int gossmx_model_append(gossmx_model* model, const uint32_t* tokens, size_t n, float* logits) {
  if (!model || !tokens || !logits) return err(GOSSMX_ERR_INVALID_ARGUMENT, "null argument");
  if (!n) return err(GOSSMX_ERR_INVALID_DIMENSIONS, "CPU step is empty");
  return run_step(model, tokens, n, logits);
}

int gossmx_model_decode(gossmx_model* model, uint32_t token, float* logits) {
  if (!model || !logits) return err(GOSSMX_ERR_INVALID_ARGUMENT, "null argument");
  if (!model->position) return err(GOSSMX_ERR_INVALID_ARGUMENT, "CPU decode requires an existing prefill cache");
  return run_step(model, &token, 1, logits);
}

int gossmx_model_position(const gossmx_model* model, size_t* position) {
  if (!model || !position) return err(GOSSMX_ERR_INVALID_ARGUMENT, "null argument");
  *position = model->position;
  return GOSSMX_OK;
}

int gossmx_model_cache(const gossmx_model* model, size_t layer, size_t* len, size_t* start_position) {
  if (!model || !len || !start_position) return err(GOSSMX_ERR_INVALID_ARGUMENT, "null argument");
  if (layer >= model->cfg.layers) return err(GOSSMX_ERR_INVALID_ARGUMENT, "layer index out of range");
  *len = model->caches[layer].len;
  *start_position = model->caches[layer].start;
  return GOSSMX_OK;
}

int gossmx_model_times(const gossmx_model* model, double* dense_seconds, double* moe_seconds) {
  if (!model || !dense_seconds || !moe_seconds) return err(GOSSMX_ERR_INVALID_ARGUMENT, "null argument");
  *dense_seconds = model->dense_seconds;
  *moe_seconds = model->moe_seconds;
  return GOSSMX_OK;
}

int gossmx_greedy_token(const float* logits, size_t n, uint32_t* token) {
  if (!logits || !token) return err(GOSSMX_ERR_INVALID_ARGUMENT, "null argument");
  // A pass over integers that the compiler vectorizes: the bits of a finite
  // float as an int of the same order (-0.0 as +0.0), the lowest int for the
  // others. Then the first index that holds the largest.
  constexpr int32_t kNone = INT32_MIN;
  auto key = [](float f) -> int32_t {
    const int32_t b = (int32_t)f2u(f), magnitude = b & 0x7fffffff;
    const int32_t ordered = b < 0 ? -magnitude : magnitude;
    return magnitude < 0x7f800000 ? ordered : kNone;
  };
  int32_t largest = kNone;
  for (size_t i = 0; i < n; ++i) {
    const int32_t v = key(logits[i]);
    largest = v > largest ? v : largest;
  }
  if (largest == kNone) return err(GOSSMX_ERR_NON_FINITE_LOGITS, "model returned no finite logits");
  size_t best = 0;
  while (key(logits[best]) != largest) ++best;
  *token = (uint32_t)best;
  return GOSSMX_OK;
}

int gossmx_yarn_rope(const gossmx_model_config* config, float* values, size_t heads, size_t position) {
  if (!config || !values) return err(GOSSMX_ERR_INVALID_ARGUMENT, "null argument");
  if (!config->head_dim || config->head_dim % 2)
    return err(GOSSMX_ERR_INVALID_DIMENSIONS, "head_dim must be even and non-zero");
  if (config->rope_yarn && (config->rope_factor <= 0.0 || !config->rope_original_max_positions))
    return err(GOSSMX_ERR_INVALID_DIMENSIONS, "YaRN scaling needs a positive factor and original positions");
  rope_apply(make_rope(*config), values, heads, position);
  return GOSSMX_OK;
}

int gossmx_attention(const float* query, const uint16_t* keys, const uint16_t* values, size_t tokens, size_t window,
                     const float* sinks, size_t heads, size_t kv_heads, size_t head_dim, float* out) {
  if (!query || !sinks || !out || (tokens && (!keys || !values)))
    return err(GOSSMX_ERR_INVALID_ARGUMENT, "null argument");
  if (!heads || !kv_heads || heads % kv_heads || !head_dim || !window)
    return err(GOSSMX_ERR_INVALID_DIMENSIONS, "invalid CPU attention dimensions");
  const size_t visible = std::min(tokens, window), first = tokens - visible, KW = kv_heads * head_dim;
  attention(query, visible, keys + first * KW, values + first * KW, sinks, heads, kv_heads, head_dim, out);
  return GOSSMX_OK;
}

}  // extern "C"
