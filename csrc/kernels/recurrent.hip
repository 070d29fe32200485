// Gated linear recurrence with a short causal convolution in front (the recurrent block of Griffin-style designs), over
// the engine's per-sequence state slots.
//
//   conv_state   out[t, c] = b[c] + sum_k taps[c, k] * in[t - (K - 1) + k, c]; inputs before the step's first row come
//                from the slot's tail (the last K - 1 inputs of the sequence), an empty (zero) history at position 0.  The
//                tail is rewritten with the step's last K - 1 inputs (shifted in place when the step is shorter).  An
//                optional SiLU on the output, or the row's own input added to it (in + conv(in)).
//   lru_scan     r = sigmoid(gate_r), i = sigmoid(gate_i), log a = -c r softplus(lam), S = a S + sqrt(1 - a^2) i u,
//                out = S * y.  The state S is fp32 and lives in the sequence's slot; a sequence's first step starts from
//                S = 0 (position 0 is not special-cased beyond that: the recurrence's own formula applies to it).
//
// The convolution and the recurrence's coefficients (every sigmoid, softplus, exponential and root) are computed for
// all rows in parallel; only S = a S + b and the product with the gelu branch walk a sequence's rows in order, one
// thread per (sequence, channel) -- a decode step is one iteration.  The biases of the two input projections and the
// gelu of the branch are applied here, so those projections are plain GEMMs with fp32 output.  Everything here is fp32
// whatever the element type of the projections around it.
#include <algorithm>

#include "api_layers.h"

namespace dsse {
namespace {

DEV float sigmoidf(float x) { return 1.0f / (1.0f + expf(-x)); }
DEV float softplusf(float x) { return x > 20.0f ? x : log1pf(expf(x)); }
DEV float gelu_tanh_f(float z) { return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z))); }

constexpr int kConvRows = 8;   // rows per workgroup of the convolution (its rows are independent of each other)

template <typename T>
__global__ __launch_bounds__(256) void conv_state_kernel(ConvStateParams p) {
  const int seq = blockIdx.y;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int ql = p.q_len[seq];
  const int t0 = blockIdx.z * kConvRows;
  if (c >= p.C || t0 >= ql) return;
  // single: one launch block per sequence walks all of its rows (one, in a decode step) and then moves the tail itself
  const int t1 = p.single ? ql : (t0 + kConvRows < ql ? t0 + kConvRows : ql);
  const int K = p.K, Kt = K - 1;
  const int row0 = p.q_start[seq];
  const bool fresh = p.ctx_len[seq] - ql == 0;  // the sequence starts in this step: nothing before it
  float* tail = p.tail + (int64_t)p.state_slot[seq] * Kt * p.C + c;  // tail[j * C]: input at offset j - Kt
  const T* taps = reinterpret_cast<const T*>(p.taps) + (int64_t)c * K;
  const float bias = p.bias ? (float)reinterpret_cast<const T*>(p.bias)[c] : 0.0f;
  const float ib = p.in_bias ? (float)reinterpret_cast<const T*>(p.in_bias)[c] : 0.0f;  // the input projection's bias
  const float* in = p.in + (int64_t)row0 * p.ld_in + c;
  for (int t = t0; t < t1; ++t) {
    float v = bias;
    for (int k = 0; k < K; ++k) {
      const int i = t - Kt + k;
      const float x = i >= 0 ? in[(int64_t)i * p.ld_in] + ib : (fresh ? 0.0f : tail[(int64_t)(Kt + i) * p.C]);
      v += (float)taps[k] * x;
    }
    if (p.act == 1) v = v / (1.0f + expf(-v));
    else if (p.act == 2) v += in[(int64_t)t * p.ld_in] + ib;
    if (p.out) p.out[(int64_t)(row0 + t) * p.C + c] = v;
    if (p.out_b) reinterpret_cast<T*>(p.out_b)[(int64_t)(row0 + t) * p.C + c] = (T)v;
  }
  if (p.single)  // this thread alone reads and writes its (slot, channel): ascending, as in conv_tail_kernel
    for (int j = 0; j < Kt; ++j) {
      const int i = ql - Kt + j;
      tail[(int64_t)j * p.C] = i >= 0 ? in[(int64_t)i * p.ld_in] + ib : (fresh ? 0.0f : tail[(int64_t)(Kt + i) * p.C]);
    }
}

// The same with four taps, four channels per thread and the last three inputs in registers: an input is read once instead of
// four times (3000 rows of 4096: 74 -> 26 us).  Only a sequence's first rows read the old tail, so their thread writes the new
// one as well: no second launch (4.5 us in a decode step).
template <typename T>
__global__ __launch_bounds__(256) void conv_state4_kernel(ConvStateParams p) {
  constexpr int K = 4, Kt = K - 1;
  const int seq = blockIdx.y, c = 4 * (blockIdx.x * blockDim.x + threadIdx.x);
  const int ql = p.q_len[seq], t0 = blockIdx.z * kConvRows;
  if (c >= p.C || t0 >= ql) return;
  const int t1 = t0 + kConvRows < ql ? t0 + kConvRows : ql;
  const int row0 = p.q_start[seq];
  const bool fresh = p.ctx_len[seq] - ql == 0;
  float* tail = p.tail + (int64_t)p.state_slot[seq] * Kt * p.C + c;
  const f32x4 zero{0.f, 0.f, 0.f, 0.f};
  f32x4 taps[4];  // of channel c + e
#pragma unroll
  for (int e = 0; e < 4; ++e) taps[e] = ld4(reinterpret_cast<const T*>(p.taps) + (int64_t)(c + e) * K);
  const f32x4 bias = p.bias ? ld4(reinterpret_cast<const T*>(p.bias) + c) : zero;
  const f32x4 ib = p.in_bias ? ld4(reinterpret_cast<const T*>(p.in_bias) + c) : zero;
  const float* in = p.in + (int64_t)row0 * p.ld_in + c;
  f32x4 x[K], next[kConvRows];
#pragma unroll
  for (int j = 0; j < Kt; ++j) {
    const int i = t0 - Kt + j;
    x[j] = i >= 0 ? ld4(in + (int64_t)i * p.ld_in) + ib : (fresh ? zero : ld4(tail + (int64_t)(Kt + i) * p.C));
  }
#pragma unroll
  for (int t = 0; t < kConvRows; ++t) next[t] = t0 + t < t1 ? ld4(in + (int64_t)(t0 + t) * p.ld_in) : zero;
  if (t0 == 0) {
    f32x4 last[Kt];  // the input at offset ql - Kt + j, for a shorter step an entry of the old tail (ql + j)
#pragma unroll
    for (int j = 0; j < Kt; ++j) {
      const int i = ql - Kt + j;
      last[j] = i >= 0 ? ld4(in + (int64_t)i * p.ld_in) + ib : (ql + j == 1 ? x[1] : x[2]);
    }
#pragma unroll
    for (int j = 0; j < Kt; ++j) st4(tail + (int64_t)j * p.C, last[j]);
  }
#pragma unroll
  for (int t = 0; t < kConvRows; ++t) {
    if (t0 + t >= t1) break;
    x[3] = next[t] + ib;
    f32x4 v = bias;
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += taps[e][k] * x[k][e];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (p.act == 1) v[e] = v[e] / (1.0f + expf(-v[e]));
      else if (p.act == 2) v[e] += x[3][e];
    }
    const int64_t at = (int64_t)(row0 + t0 + t) * p.C + c;
    if (p.out) st4(p.out + at, v);
    if (p.out_b) st4(reinterpret_cast<T*>(p.out_b) + at, v);
    x[0] = x[1], x[1] = x[2], x[2] = x[3];
  }
}

// After every row of the step has read the old tail: the slot's new tail = the step's last K - 1 inputs.  Ascending:
// entry j takes the input at offset ql - Kt + j, which for a short step is the old entry j + ql (> j, not yet
// overwritten).
template <typename T>
__global__ __launch_bounds__(256) void conv_tail_kernel(ConvStateParams p) {
  const int seq = blockIdx.y;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int ql = p.q_len[seq];
  if (c >= p.C || ql <= 0) return;
  const int Kt = p.K - 1;
  const bool fresh = p.ctx_len[seq] - ql == 0;
  float* tail = p.tail + (int64_t)p.state_slot[seq] * Kt * p.C + c;
  const float ib = p.in_bias ? (float)reinterpret_cast<const T*>(p.in_bias)[c] : 0.0f;
  const float* in = p.in + (int64_t)p.q_start[seq] * p.ld_in + c;
  for (int j = 0; j < Kt; ++j) {
    const int i = ql - Kt + j;
    tail[(int64_t)j * p.C] = i >= 0 ? in[(int64_t)i * p.ld_in] + ib : (fresh ? 0.0f : tail[(int64_t)(Kt + i) * p.C]);
  }
}

// (a, b) of S = a S + b: a = exp(-c sigmoid(g_r) softplus(lam)), b = sqrt(1 - a^2) sigmoid(g_i) u
DEV void lru_coeff(float gr, float gi, float u, float c, float sp, float& a, float& b) {
  const float log_a = -c * sigmoidf(gr) * sp;
  a = expf(log_a);
  b = sqrtf(-expm1f(2.0f * log_a)) * sigmoidf(gi) * u;  // sqrt(1 - a^2) without cancellation near a = 1
}

// Everything of the recurrence that does not depend on the state, for every row at once: the gates' pre-activations
// [recurrence gate | input gate] of each block are overwritten with (a, b) of S = a S + b.
// R rows per thread: their loads are in flight together and the channel's softplus is made once (3000 rows of 4096: 80 ->
// 53 us, some 100 vector instructions per element)
template <typename T, int R>
__global__ __launch_bounds__(256) void lru_coeff_kernel(LruScanParams p, int rows) {
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  const int64_t row0 = (int64_t)blockIdx.x * R;
  if (c >= p.C) return;
  const float sp = softplusf((float)reinterpret_cast<const T*>(p.lam)[c]);
  const int b = c / p.bw, o = c % p.bw;
  float* g = const_cast<float*>(p.gates) + row0 * 2 * p.C + (int64_t)b * 2 * p.bw + o;
  const float* u = p.u + row0 * p.C + c;
  const int n = (int)(rows - row0 < R ? rows - row0 : R);
  float gr[R], gi[R], ui[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int64_t at = i < n ? i : 0;
    gr[i] = g[at * 2 * p.C];
    gi[i] = g[at * 2 * p.C + p.bw];
    ui[i] = u[at * p.C];
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (i >= n) break;
    float a, bb;
    lru_coeff(gr[i], gi[i], ui[i], p.c, sp, a, bb);
    g[(int64_t)i * 2 * p.C] = a;
    g[(int64_t)i * 2 * p.C + p.bw] = bb;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void lru_scan_kernel(LruScanParams p) {
  const int seq = blockIdx.y;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int ql = p.q_len[seq];
  if (c >= p.C || ql <= 0) return;
  const int row0 = p.q_start[seq];
  float* st = p.state + (int64_t)p.state_slot[seq] * p.C + c;
  float S = p.ctx_len[seq] - ql == 0 ? 0.0f : *st;
  const int b = c / p.bw, o = c % p.bw;
  const float yb = p.y_bias ? (float)reinterpret_cast<const T*>(p.y_bias)[c] : 0.0f;
  const float* ab = p.gates + (int64_t)row0 * 2 * p.C + (int64_t)b * 2 * p.bw + o;
  const float* y = p.y + (int64_t)row0 * p.C + c;
  T* out = reinterpret_cast<T*>(p.out) + (int64_t)row0 * p.C + c;
  int t = 0;
  for (; t + 4 <= ql; t += 4) {  // the loads of four steps are in flight before the four dependent updates
    float a[4], bb[4], yy[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a[i] = ab[(int64_t)(t + i) * 2 * p.C];
      bb[i] = ab[(int64_t)(t + i) * 2 * p.C + p.bw];
      yy[i] = y[(int64_t)(t + i) * p.C];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      S = a[i] * S + bb[i];
      out[(int64_t)(t + i) * p.C] = (T)(S * gelu_tanh_f(yy[i] + yb));
    }
  }
  for (; t < ql; ++t) {
    S = ab[(int64_t)t * 2 * p.C] * S + ab[(int64_t)t * 2 * p.C + p.bw];
    out[(int64_t)t * p.C] = (T)(S * gelu_tanh_f(y[(int64_t)t * p.C] + yb));
  }
  *st = S;
}

// A step that is all of u's rows and few of every sequence (decode): coefficients and walk in one launch, the gates stay as they are
// (one row each of 160 sequences x 2560 channels: 20.1 us in four launches, 6.4 in this one; 16 sequences 9.0 in two, 4.7).  Its
// chain is the longest sequence's, 0.46 us a row (lru_takes_step).
template <typename T>
__global__ __launch_bounds__(256) void lru_step_kernel(LruScanParams p) {
  const int seq = blockIdx.y;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int ql = p.q_len[seq];
  if (c >= p.C || ql <= 0) return;
  const int row0 = p.q_start[seq];
  float* st = p.state + (int64_t)p.state_slot[seq] * p.C + c;
  const int b = c / p.bw, o = c % p.bw;
  const float* g = p.gates + (int64_t)row0 * 2 * p.C + (int64_t)b * 2 * p.bw + o;
  const float* u = p.u + (int64_t)row0 * p.C + c;
  const float* y = p.y + (int64_t)row0 * p.C + c;
  T* out = reinterpret_cast<T*>(p.out) + (int64_t)row0 * p.C + c;
  float S = p.ctx_len[seq] - ql == 0 ? 0.0f : *st;
  const float yb = p.y_bias ? (float)reinterpret_cast<const T*>(p.y_bias)[c] : 0.0f;
  const float sp = softplusf((float)reinterpret_cast<const T*>(p.lam)[c]);
  for (int t = 0; t < ql; ++t) {
    float a, bb;
    lru_coeff(g[(int64_t)t * 2 * p.C], g[(int64_t)t * 2 * p.C + p.bw], u[(int64_t)t * p.C], p.c, sp, a, bb);
    S = a * S + bb;
    out[(int64_t)t * p.C] = (T)(S * gelu_tanh_f(y[(int64_t)t * p.C] + yb));
  }
  *st = S;
}

// Prompt portions: the walk in three phases so that no thread takes more than ~3 x 32 dependent steps.  A chunk is
// kScanRows rows of one sequence; its scratch slot is (first row) / kScanRows + (sequence index), which is unique because
// sequences are packed in row order.
//   1. per chunk, in parallel: A = prod a_t and B = the chunk's walk from S = 0          (S_end = A S_in + B); a call that holds
//      all rows makes the coefficients here, for one reading of the gates
//   2. per sequence: the chunks in order -- each chunk's incoming state replaces its B, the last one is the slot's state
//   3. per chunk, in parallel: the walk from the incoming state, times gelu(branch + bias)
// A few chunks (kFoldChunks) take no second phase: the first leaves (S_in, S_end) of a sequence's first chunk, and every thread of
// the third folds the chunks before its own.  Rows go in batches whose loads are in flight together.  Per layer (coefficients
// and walk), four launches before / now: 200 rows of 2560 35 / 24 us, 700 42 / 30, 3000 rows of 4096 127 / 105.
constexpr int kScanRows = 32;
constexpr int kChunkedFrom = 128;  // rows of a step from which the walk is chunked (below: one thread per sequence)

DEV int scan_slot(int row0, int t0, int seq) { return (row0 + t0) / kScanRows + seq; }

constexpr int kScanBatch = 8;    // rows whose loads are in flight together
constexpr int kFoldChunks = 32;  // chunks of a step up to which the third phase folds

template <typename T, bool COEFF>
__global__ __launch_bounds__(256) void lru_chunk_reduce_kernel(LruScanParams p, int fold) {
  const int seq = blockIdx.y, c = blockIdx.x * blockDim.x + threadIdx.x;
  const int ql = p.q_len[seq], t0 = blockIdx.z * kScanRows;
  if (c >= p.C || t0 >= ql) return;
  const int t1 = t0 + kScanRows < ql ? t0 + kScanRows : ql;
  const int row0 = p.q_start[seq];
  const int b = c / p.bw, o = c % p.bw;
  float* ab = const_cast<float*>(p.gates) + (int64_t)row0 * 2 * p.C + (int64_t)b * 2 * p.bw + o;
  const float* u = p.u + (int64_t)row0 * p.C + c;
  const float sp = COEFF ? softplusf((float)reinterpret_cast<const T*>(p.lam)[c]) : 0.0f;
  float A = 1.0f, B = 0.0f;
  for (int t = t0; t < t1; t += kScanBatch) {
    float ga[kScanBatch], gb[kScanBatch], ui[kScanBatch];
#pragma unroll
    for (int i = 0; i < kScanBatch; ++i) {
      const int64_t at = t + i < t1 ? t + i : t;
      ga[i] = ab[at * 2 * p.C];
      gb[i] = ab[at * 2 * p.C + p.bw];
      if (COEFF) ui[i] = u[at * p.C];
    }
#pragma unroll
    for (int i = 0; i < kScanBatch; ++i) {
      if (t + i >= t1) break;
      float a = ga[i], bb = gb[i];
      if (COEFF) {
        lru_coeff(ga[i], gb[i], ui[i], p.c, sp, a, bb);
        ab[(int64_t)(t + i) * 2 * p.C] = a;
        ab[(int64_t)(t + i) * 2 * p.C + p.bw] = bb;
      }
      B = a * B + bb;
      A *= a;
    }
  }
  const int64_t s = (int64_t)scan_slot(row0, t0, seq) * p.C + c;
  if (fold && t0 == 0) {
    const float S = p.ctx_len[seq] - ql == 0 ? 0.0f : p.state[(int64_t)p.state_slot[seq] * p.C + c];
    B = A * S + B;
    A = S;
  }
  p.chunk_a[s] = A;
  p.chunk_b[s] = B;
}

__global__ __launch_bounds__(256) void lru_chunk_carry_kernel(LruScanParams p) {
  const int seq = blockIdx.y, c = blockIdx.x * blockDim.x + threadIdx.x;
  const int ql = p.q_len[seq];
  if (c >= p.C || ql <= 0) return;
  const int row0 = p.q_start[seq], chunks = (ql + kScanRows - 1) / kScanRows;
  float* st = p.state + (int64_t)p.state_slot[seq] * p.C + c;
  float S = p.ctx_len[seq] - ql == 0 ? 0.0f : *st;
  const int64_t s0 = (int64_t)scan_slot(row0, 0, seq) * p.C + c;  // a sequence's slots follow each other
  for (int k = 0; k < chunks; k += kScanBatch) {
    float a[kScanBatch], bb[kScanBatch];
#pragma unroll
    for (int i = 0; i < kScanBatch; ++i) {
      const int64_t s = s0 + (int64_t)(k + i < chunks ? k + i : k) * p.C;
      a[i] = p.chunk_a[s];
      bb[i] = p.chunk_b[s];
    }
#pragma unroll
    for (int i = 0; i < kScanBatch; ++i) {
      if (k + i >= chunks) break;
      p.chunk_b[s0 + (int64_t)(k + i) * p.C] = S;  // the chunk's incoming state
      S = a[i] * S + bb[i];
    }
  }
  *st = S;
}

template <typename T>
__global__ __launch_bounds__(256) void lru_chunk_apply_kernel(LruScanParams p, int fold) {
  const int seq = blockIdx.y, c = blockIdx.x * blockDim.x + threadIdx.x;
  const int ql = p.q_len[seq], t0 = blockIdx.z * kScanRows;
  if (c >= p.C || t0 >= ql) return;
  const int t1 = t0 + kScanRows < ql ? t0 + kScanRows : ql;
  const int row0 = p.q_start[seq];
  const int b = c / p.bw, o = c % p.bw;
  const float yb = p.y_bias ? (float)reinterpret_cast<const T*>(p.y_bias)[c] : 0.0f;
  const float* ab = p.gates + (int64_t)row0 * 2 * p.C + (int64_t)b * 2 * p.bw + o;
  const float* y = p.y + (int64_t)row0 * p.C + c;
  T* out = reinterpret_cast<T*>(p.out) + (int64_t)row0 * p.C + c;
  const int64_t s0 = (int64_t)scan_slot(row0, 0, seq) * p.C + c;
  const int chunk = blockIdx.z;
  float S;
  if (!fold) {
    S = p.chunk_b[s0 + (int64_t)chunk * p.C];
  } else if (chunk == 0) {
    S = p.chunk_a[s0];
  } else {
    S = p.chunk_b[s0];
#pragma unroll 8
    for (int k = 1; k < chunk; ++k) S = p.chunk_a[s0 + (int64_t)k * p.C] * S + p.chunk_b[s0 + (int64_t)k * p.C];
  }
  for (int t = t0; t < t1; t += kScanBatch) {
    float a[kScanBatch], bb[kScanBatch], yy[kScanBatch];
#pragma unroll
    for (int i = 0; i < kScanBatch; ++i) {
      const int64_t at = t + i < t1 ? t + i : t;
      a[i] = ab[at * 2 * p.C];
      bb[i] = ab[at * 2 * p.C + p.bw];
      yy[i] = y[at * p.C];
    }
#pragma unroll
    for (int i = 0; i < kScanBatch; ++i) {
      if (t + i >= t1) break;
      S = a[i] * S + bb[i];
      out[(int64_t)(t + i) * p.C] = (T)(S * gelu_tanh_f(yy[i] + yb));
    }
  }
  if (fold && t1 == ql) p.state[(int64_t)p.state_slot[seq] * p.C + c] = S;
}

// One launch or the other forms, by the longest sequence: coefficients in parallel and a walk of 0.19 us a row below kChunkedFrom
// rows, chunks (a workgroup for every 32 rows of the step per sequence) from there on.  One launch / the others, 2560 channels:
// 8 rows 6.2 / 6.4, 12 8.0 / 7.1; 63 of 1 row and one of 8 6.9 / 7.5, of 12 8.7 / 8.3, of 32 18 / 12; chunks: 8 of 16 rows 10.0 / 12.6,
// of 24 13.7 / 16.4, 63 of 1 row and one of 190 89 / 33; 159 of 1 row and one of 24 16 / 23, of 48 27 / 27, 255 and one of 48 28 / 33.
bool lru_takes_step(const LruScanParams& p, bool chunked) {
  return p.longest <= (chunked ? std::max(24, std::min(48, p.nseq / 4)) : 8);
}

}  // namespace
}  // namespace dsse

extern "C" hipError_t dsse_conv_state(const dsse::ConvStateParams* p, hipStream_t st) {
  if (p->nseq <= 0 || p->rows <= 0) return hipSuccess;
  dim3 grid((p->C + 255) / 256, p->nseq, p->single ? 1 : (p->rows + dsse::kConvRows - 1) / dsse::kConvRows);
  dim3 tgrid((p->C + 255) / 256, p->nseq);
  const bool tails = p->K > 1 && !p->single;
  const bool four = p->K == 4 && !p->single && p->C % 4 == 0 && p->ld_in % 4 == 0 &&
                    dsse::fours({p->in, p->tail, p->taps, p->bias, p->in_bias, p->out, p->out_b});
  const dim3 fgrid((p->C / 4 + 255) / 256, grid.y, grid.z);
  if (four) {
    if (p->f32) hipLaunchKernelGGL(dsse::conv_state4_kernel<float>, fgrid, dim3(256), 0, st, *p);
    else hipLaunchKernelGGL(dsse::conv_state4_kernel<bf16>, fgrid, dim3(256), 0, st, *p);
  } else if (p->f32) {
    hipLaunchKernelGGL(dsse::conv_state_kernel<float>, grid, dim3(256), 0, st, *p);
    if (tails) hipLaunchKernelGGL(dsse::conv_tail_kernel<float>, tgrid, dim3(256), 0, st, *p);
  } else {
    hipLaunchKernelGGL(dsse::conv_state_kernel<bf16>, grid, dim3(256), 0, st, *p);
    if (tails) hipLaunchKernelGGL(dsse::conv_tail_kernel<bf16>, tgrid, dim3(256), 0, st, *p);
  }
  return hipGetLastError();
}

extern "C" hipError_t dsse_lru_scan(const dsse::LruScanParams* p, hipStream_t st) {
  using namespace dsse;
  if (p->nseq <= 0 || p->rows <= 0) return hipSuccess;
  dim3 grid((p->C + 255) / 256, p->nseq);
  const bool alone = p->coeff && p->alone;
  const bool chunked = p->chunk_a && p->chunk_b && p->rows >= kChunkedFrom;  // prompt portions
  if (alone && lru_takes_step(*p, chunked)) {
    if (p->f32) hipLaunchKernelGGL(lru_step_kernel<float>, grid, dim3(256), 0, st, *p);
    else hipLaunchKernelGGL(lru_step_kernel<bf16>, grid, dim3(256), 0, st, *p);
    return hipGetLastError();
  }
  if (p->coeff && !(alone && chunked)) {
    const int per = p->rows >= 256 ? 4 : 1;  // few rows: a thread per element fills more of the chip
    dim3 cgrid((p->rows + per - 1) / per, (p->C + 255) / 256);
    if (p->f32 && per == 4) hipLaunchKernelGGL((lru_coeff_kernel<float, 4>), cgrid, dim3(256), 0, st, *p, p->rows);
    else if (p->f32) hipLaunchKernelGGL((lru_coeff_kernel<float, 1>), cgrid, dim3(256), 0, st, *p, p->rows);
    else if (per == 4) hipLaunchKernelGGL((lru_coeff_kernel<bf16, 4>), cgrid, dim3(256), 0, st, *p, p->rows);
    else hipLaunchKernelGGL((lru_coeff_kernel<bf16, 1>), cgrid, dim3(256), 0, st, *p, p->rows);
  }
  if (chunked) {
    dim3 zgrid((p->C + 255) / 256, p->nseq, (p->rows + kScanRows - 1) / kScanRows);
    const int fold = (int)zgrid.z <= kFoldChunks;
    if (!alone) hipLaunchKernelGGL((lru_chunk_reduce_kernel<float, false>), zgrid, dim3(256), 0, st, *p, fold);
    else if (p->f32) hipLaunchKernelGGL((lru_chunk_reduce_kernel<float, true>), zgrid, dim3(256), 0, st, *p, fold);
    else hipLaunchKernelGGL((lru_chunk_reduce_kernel<bf16, true>), zgrid, dim3(256), 0, st, *p, fold);
    if (!fold) hipLaunchKernelGGL(lru_chunk_carry_kernel, grid, dim3(256), 0, st, *p);
    if (p->f32) hipLaunchKernelGGL(lru_chunk_apply_kernel<float>, zgrid, dim3(256), 0, st, *p, fold);
    else hipLaunchKernelGGL(lru_chunk_apply_kernel<bf16>, zgrid, dim3(256), 0, st, *p, fold);
    return hipGetLastError();
  }
  if (p->f32) hipLaunchKernelGGL(lru_scan_kernel<float>, grid, dim3(256), 0, st, *p);
  else hipLaunchKernelGGL(lru_scan_kernel<bf16>, grid, dim3(256), 0, st, *p);
  return hipGetLastError();
}
