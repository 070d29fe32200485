// Row-wise fp32 pieces of pre-norm designs with matrix-state mixers:
//
//   stream_step      resid += mult * y + embed[id] + vec, then xb = tanh(alpha * resid) * w + b (the element-wise norm
//                    that needs no row statistic, so the add and the norm are one pass over the row)
//   gated_act        h = act(gate) * up from the fused gate | up projection's fp32 output (SiLU or tanh-form gelu)
//   norm_rope_rows   a row of heads: RMS norm over the whole row with a gain, a unit vector per head, an RMS norm per
//                    head with one gain vector for all heads (or without a gain), or nothing;
//                    rotate-half rotation of each head's leading coordinates; a scale; written to a chosen output row
//                    (a cache row: keys and values go straight into their pages) in fp32 or bf16
//   gate_math        decays and gates in place: exp(-exp(A) softplus(x + dt)), sigmoid(x), sigmoid(x)^(1/tau), or the first of
//                    these on a row's left half and the second on its right half
//   gated_head_norm  out = o / rms(o) * w * silu(gate) per (row, head), or * sigmoid(gate)
//   rms_mix          out = c * (rms-norm(ya) * wa + rms-norm(yb) * wb)
//   logit_cap        logits * scale, then cap * tanh(. / cap)
//
// Everything is computed in fp32; only xb / h / out of the element type and bf16 cache rows are rounded.
#include <algorithm>

#include "api_mixers.h"

namespace dsse {
namespace {

DEV float sigmoid_f(float x) { return 1.0f / (1.0f + expf(-x)); }
DEV float silu_f(float x) { return x / (1.0f + expf(-x)); }
DEV float softplus_f(float x) { return x > 20.0f ? x : log1pf(expf(x)); }
DEV float gelu_tanh_f(float z) { return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z))); }

DEV float block_sum256(float v, float* red) {
  v = wave_sum(v);
  const int wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[wave] = v;
  __syncthreads();
  float s = 0.f;
  for (int i = 0; i < nw; ++i) s += red[i];
  return s;
}

// VEC elements per thread, a row over as many workgroups as it takes (16 rows of 4096: one workgroup per row
// waited 9.6 us on its chain of loads, now 2.5; 3000 rows 37 -> 28)
template <typename T, int VEC>
__global__ __launch_bounds__(256) void stream_step_kernel(StreamStepParams p) {
  const int row = blockIdx.x, d = (blockIdx.y * 256 + threadIdx.x) * VEC;
  if (d >= p.W) return;
  float* resid = p.resid + (int64_t)row * p.W + d;
  const float* y = p.y ? p.y + (int64_t)row * p.nsum * p.W + d : nullptr;
  const T* e = nullptr;
  if (p.embed) {
    int id = p.ids[row];
    id = (unsigned)id < (unsigned)p.vocab ? id : 0;  // padded / inactive rows carry any id
    e = reinterpret_cast<const T*>(p.embed) + (int64_t)id * p.W + d;
  }
  if constexpr (VEC == 4) {
    f32x4 v = ld4(resid);
    if (y) v += p.mult * add_parts<f32x4>(p.nsum, [&](int s) { return ld4(y + (int64_t)s * p.W); });
    if (e) v += ld4(e);
    if (p.vec) v += ld4(p.vec + d);
    if (y || e || p.vec) st4(resid, v);
    if (p.w) {
      const float alpha = p.alpha[0];
      const f32x4 w = ld4(p.w + d), b = ld4(p.b + d);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = tanhf(alpha * v[i]) * w[i] + b[i];
      st4(reinterpret_cast<T*>(p.xb) + (int64_t)row * p.W + d, v);
    }
  } else {
    float v = *resid;
    if (y) v += p.mult * add_parts<float>(p.nsum, [&](int s) { return y[(int64_t)s * p.W]; });
    if (e) v += (float)*e;
    if (p.vec) v += p.vec[d];
    if (y || e || p.vec) *resid = v;
    if (p.w) reinterpret_cast<T*>(p.xb)[(int64_t)row * p.W + d] = (T)(tanhf(p.alpha[0] * v) * p.w[d] + p.b[d]);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void gated_act_kernel(const float* gu, int ldg, T* h, int M, int F, int kind) {
  const int64_t n = (int64_t)M * F;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / F;
    const int c = (int)(i - r * F);
    const float g = gu[r * ldg + c], u = gu[r * ldg + F + c];
    h[i] = (T)((kind == 0 ? silu_f(g) : gelu_tanh_f(g)) * u);
  }
}

// One wave per head, four heads to a workgroup where their norms do not need the whole row; else a row's workgroup of 4 waves
// (a decode step's: up to 16) walks them.  16 rows of 32 heads of 128, one workgroup of four waves per row before: per-head
// norms 11.2 -> 3.0 us, row norms 10.4 -> 5.7 us.  A head's normed values pass through the wave's LDS strip so
// that a coordinate and its rotation partner are both at hand whatever lane loaded them, and so that the kernel works
// in place (out == x): a head is read completely before any of it is written.
constexpr int kMaxHeadDim = 512;

// WAVES: most waves of a workgroup
template <typename OutT, int WAVES>
DEV void norm_rope_row(const NormRopeParams& p, int gy, float* strips, float* red) {
  const int row = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = WAVES == 4 ? 4 : blockDim.x >> 6;
  const float* x = p.x + (int64_t)row * p.ldx;
  const int N = p.nh * p.D;
  float inv_row = 1.0f;
  if (p.kind == 1) {
    float ss = 0.f;
    for (int d = threadIdx.x; d < N; d += blockDim.x) ss += x[d] * x[d];
    ss = block_sum256(ss, red);
    inv_row = 1.0f / sqrtf(ss / (float)N + p.eps);
  }
  int orow = p.out_rows ? p.out_rows[row] : row;
  if (orow < 0 || orow >= p.num_out_rows) return;  // uniform for the workgroup; after the only block-wide barrier
  OutT* out = reinterpret_cast<OutT*>(p.out) + (int64_t)orow * p.ldo;
  int pos = p.rope ? p.positions[row] : 0;
  pos = pos < 0 ? 0 : (pos >= p.rope_len ? p.rope_len - 1 : pos);
  const float2* cs = p.rope ? p.rope + (int64_t)pos * p.half : nullptr;
  const int dims = p.rope ? 2 * p.half : 0;
  float* s = strips + wave * p.D;
  for (int h0 = nw * blockIdx.y; h0 < p.nh; h0 += nw * gy) {  // uniform trip count: the barriers below are reached by every wave
    const int h = h0 + wave;
    const bool on = h < p.nh;
    const float* xh = x + (on ? h : 0) * p.D;
    float inv = inv_row;
    if (p.kind >= 2) {
      float ss = 0.f;
      for (int i = lane; i < p.D; i += 64) ss += xh[i] * xh[i];
      ss = wave_sum(ss);
      inv = 1.0f / sqrtf((p.kind == 3 ? ss / (float)p.D : ss) + p.eps);
    }
    if (on)
      for (int i = lane; i < p.D; i += 64)
        s[i] = xh[i] * inv * (p.kind == 1 ? p.norm_w[h * p.D + i] : (p.kind == 3 && p.norm_w ? p.norm_w[i] : 1.0f));
    __syncthreads();  // the strip is written before it is read
    if (on)
      for (int i = lane; i < p.D; i += 64) {
        float v = s[i];
        if (i < dims) {
          const bool lo = i < p.half;
          const float2 c = cs[lo ? i : i - p.half];
          const float o = s[lo ? i + p.half : i - p.half];
          v = lo ? v * c.x - o * c.y : v * c.x + o * c.y;
        }
        out[h * p.D + i] = (OutT)(v * p.scale);
        if (p.out_t) {  // the same number once more where the MFMA attention's value operand wants it
          const int page = orow / kBS, off = orow % kBS;
          const int at = ((off & 15) >> 2) * 8 + ((off >> 4) & 1) * 4 + (off & 3);
          reinterpret_cast<OutT*>(p.out_t)[(((int64_t)page * p.nh + h) * p.D + i) * kBS + at] = (OutT)(v * p.scale);
        }
      }
    __syncthreads();  // the strip is read before the next head overwrites it
  }
}

// The same with four neighbouring numbers to a lane: a head of 4 n numbers is n lanes, a wave takes 64 / n heads, sums and rotation
// partners (half / 4 lanes away) come from shuffles; no strips, no barriers.  norm_rope_fours() says which sets it takes.  1500
// rows, by ones / by fours: unit q and k of 8 heads of 128 9.8 / 7.3 us, rotation of 16 and 16 heads in place 15.1 / 8.7, row-normed
// and rotated q and k with v (16, 8, 8 heads) 17.7 / 12.3; 300 rows 8.1 / 4.8.
template <typename OutT>
DEV void norm_rope_fours_row(const NormRopeParams& p, int gy, float* red) {
  const int row = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int n = p.D >> 2, e = 4 * (lane & (n - 1)), hpw = 64 / n, N = p.nh * p.D;
  const float* x = p.x + (int64_t)row * p.ldx;
  float inv_row = 1.0f;
  if (p.kind == 1) {
    f32x4 sq{0.f, 0.f, 0.f, 0.f};
    for (int d = 4 * threadIdx.x; d < N; d += 4 * blockDim.x) {
      const f32x4 v = ld4(x + d);
      sq += v * v;
    }
    inv_row = 1.0f / sqrtf(block_sum256((sq[0] + sq[1]) + (sq[2] + sq[3]), red) / (float)N + p.eps);
  }
  const int orow = p.out_rows ? p.out_rows[row] : row;
  if (orow < 0 || orow >= p.num_out_rows) return;  // uniform for the workgroup; after the only block-wide barrier
  OutT* out = reinterpret_cast<OutT*>(p.out) + (int64_t)orow * p.ldo;
  const int dims = p.rope ? 2 * p.half : 0;
  f32x4 cs0{1.f, 0.f, 1.f, 0.f}, cs1 = cs0;  // (cos, sin) of the lane's four numbers
  float side = 0.f;                          // how their partners enter: v cos + side * partner sin
  if (e < dims) {
    int pos = p.positions[row];
    pos = pos < 0 ? 0 : (pos >= p.rope_len ? p.rope_len - 1 : pos);
    const float* c = reinterpret_cast<const float*>(p.rope + (int64_t)pos * p.half + (e < p.half ? e : e - p.half));
    cs0 = ld4(c), cs1 = ld4(c + 4);
    side = e < p.half ? -1.f : 1.f;
  }
  f32x4 w{1.f, 1.f, 1.f, 1.f};
  if (p.kind == 3 && p.norm_w) w = ld4(p.norm_w + e);
  for (int h0 = nw * hpw * blockIdx.y; h0 < p.nh; h0 += nw * hpw * gy) {
    const int h = h0 + wave * hpw + lane / n;
    const bool on = h < p.nh;
    f32x4 v = ld4(x + (on ? h : 0) * p.D + e);
    if (p.bias) v += ld4(p.bias + (on ? h : 0) * p.D + e);
    float inv = inv_row;
    if (p.kind >= 2) {
      float ss = (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
      for (int o = n >> 1; o >= 1; o >>= 1) ss += __shfl_xor(ss, o);
      inv = 1.0f / sqrtf((p.kind == 3 ? ss / (float)p.D : ss) + p.eps);
    } else if (p.kind == 1) {
      w = ld4(p.norm_w + (on ? h : 0) * p.D + e);
    }
    v = v * inv * w;
    if (dims) {
      f32x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = side * __shfl_xor(v[i], p.half >> 2);
      // numbers past the rotated ones stay as they are, whatever they were paired with: 0 * inf is no zero
      if (e < dims)
        v = f32x4{v[0] * cs0[0] + o[0] * cs0[1], v[1] * cs0[2] + o[1] * cs0[3], v[2] * cs1[0] + o[2] * cs1[1], v[3] * cs1[2] + o[3] * cs1[3]};
    }
    v = v * p.scale;
    if (!on) continue;
    st4(out + h * p.D + e, v);
    if (p.out_t) {  // the same numbers once more where the MFMA attention's value operand wants them
      const int page = orow / kBS, off = orow % kBS;
      const int at = ((off & 15) >> 2) * 8 + ((off >> 4) & 1) * 4 + (off & 3);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        reinterpret_cast<OutT*>(p.out_t)[(((int64_t)page * p.nh + h) * p.D + e + i) * kBS + at] = (OutT)v[i];
    }
  }
}

// Values on their way into pages and transposed pages.  By token the transposed ones are 2-byte writes from 32 workgroups behind eight
// L2s; where the 32 packed rows around a row are one page in order, wherever in the launch they begin, the page's workgroups take
// columns instead: each a part of the page's columns for all of its 32 rows, so that a value's 32 tokens, 64 bytes, are written at
// once.  The others go by token.  Both kinds move a row's worth of numbers per workgroup, behind one load of the slots.  8 heads of
// 128, us, all by token / whole pages only at multiples of 32 packed rows, a workgroup to 32 rows of a head / this: one prompt of 1500 rows
// 13.2 / 6.0 / 5.0, three of together 1500 13.0 / 8.9 / 5.1, of 300 4.9 / 5.6 / 3.9, 344 rows behind 20 decode rows 5.4 / 6.2 / 4.1; beside
// queries and keys 23.7 / 14.0 / 13.6, 23.7 / 18.4 / 13.7, 9.5 / 6.5 / 5.4, 11.3 / 7.5 / 5.8, and 192 decode rows 8.6 / 8.1 / 6.9 (8 of 64, one
// prompt of 1500: 15.3 / 9.5 / 10.6).
constexpr int kPageCols = 64;  // columns that pass through LDS together
constexpr int kPageLds = kBS * (kPageCols + 4) * sizeof(bf16);

// Returns false, in every thread, where the row's page is not whole.  gy workgroups of the set per row.
DEV bool value_pages(const NormRopeParams& p, int gy, bf16* tile) {
  const int row = blockIdx.x, lane = threadIdx.x & 63;
  const int near = row + lane - (kBS - 1);  // lane kBS - 1: the row itself
  const int slot = near >= 0 && near < p.T ? p.out_rows[near] : -1;
  const int own = __shfl(slot, kBS - 1);
  if (own < 0 || own >= p.num_out_rows) return false;
  const int off = own % kBS, first = own - off, from = kBS - 1 - off;  // the lane of the page's first row
  const int i = lane - from;
  if (first + kBS > p.num_out_rows || !__all(i < 0 || i >= kBS || slot == first + i)) return false;
  const int t0 = row - off, N = p.nh * p.D;
  const int each = max((N / 4 + kBS * gy - 1) / (kBS * gy), 8);  // groups of four columns of a workgroup: whole lines of x
  const int g0 = (off * gy + (int)blockIdx.y) * each, g1 = min(g0 + each, N / 4);
  bf16* out = reinterpret_cast<bf16*>(p.out) + (int64_t)first * p.ldo;
  bf16* pages = reinterpret_cast<bf16*>(p.out_t) + (int64_t)first * N;
  constexpr int ldt = kPageCols + 4;
  for (int g = g0; g < g1; g += kPageCols / 4) {
    const int n = min(kPageCols / 4, g1 - g);
    for (int u = threadIdx.x; u < kBS * n; u += blockDim.x) {
      const int r = u / n, q = u - r * n, d = 4 * (g + q);
      f32x4 v = ld4(p.x + (int64_t)(t0 + r) * p.ldx + d);
      if (p.bias) v += ld4(p.bias + d);
      v = v * p.scale;
      const bf16x4 b{(bf16)v[0], (bf16)v[1], (bf16)v[2], (bf16)v[3]};
      *reinterpret_cast<bf16x4*>(tile + r * ldt + 4 * q) = b;
      *reinterpret_cast<bf16x4*>(out + (int64_t)r * p.ldo + d) = b;
    }
    __syncthreads();
    for (int u = threadIdx.x; u < 16 * n; u += blockDim.x) {  // (column, 8 places): tokens 4 q .. + 3 and 16 + 4 q .. + 3
      const int d = u >> 2, q = u & 3;
      bf16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = tile[(4 * q + (j & 3) + 16 * (j >> 2)) * ldt + d];
      *reinterpret_cast<bf16x8*>(pages + (int64_t)(4 * g + d) * kBS + 8 * q) = o;
    }
    __syncthreads();
  }
  return true;
}

// Heads of 32, 64, 128 or 256 numbers in 16-byte pieces, rotation partners a power of two of lanes apart
inline bool norm_rope_fours(const NormRopeParams& p) {
  auto power = [](int n) { return n > 0 && (n & (n - 1)) == 0; };
  return p.D % 32 == 0 && p.D <= 256 && power(p.D) && p.ldx % 4 == 0 && p.ldo % 4 == 0 && fours({p.x, p.out, p.norm_w, p.rope, p.bias}) &&
         (!p.rope || (p.half % 4 == 0 && power(p.half / 4) && 2 * p.half <= p.D));
}

// A layer's queries, keys and values (blockIdx.z) in one launch.  What bounds it in a decode step: the launch, 4 to 5 us whatever it
// moves.  Surodra-wide, 16 rows, ten launches fewer (two of them gates): 703 -> 678 us; 1500 prompt rows of surodra-mid 1813 -> 1792.
template <int WAVES>
__global__ __launch_bounds__(64 * WAVES) void norm_rope_rows_kernel(NormRopeList l) {
  extern __shared__ float strips[];  // [waves][D]
  __shared__ float red[16];
  const NormRopeParams& p = l.p[blockIdx.z];
  const int gy = l.gy[blockIdx.z];
  if ((int)blockIdx.y >= gy) return;  // uniform: another set's share of the grid
  if (l.pages[blockIdx.z] && value_pages(p, gy, reinterpret_cast<bf16*>(strips))) return;
  if (l.fours[blockIdx.z]) {
    if (p.out_f32) norm_rope_fours_row<float>(p, gy, red);
    else norm_rope_fours_row<bf16>(p, gy, red);
    return;
  }
  if (p.out_f32) norm_rope_row<float, WAVES>(p, gy, strips, red);
  else norm_rope_row<bf16, WAVES>(p, gy, strips, red);
}

__global__ __launch_bounds__(256) void gate_math_kernel(float* x, int ld, int M, int N, int kind, const float* p1,
                                                        int rep1, const float* p2, int rep2, float c) {
  const int64_t n = (int64_t)M * N;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / N;
    const int col = (int)(i - r * N);
    float* px = x + r * ld + col;
    const float v = *px;
    float o;
    if (kind == 0 || (kind == 3 && 2 * col < N)) {
      o = expf(-expf(p1[col / rep1]) * softplus_f(v + p2[col / rep2]));
    } else if (kind == 1 || kind == 3) {
      o = sigmoid_f(v);
    } else {
      const float ls = fminf(v, 0.0f) - log1pf(expf(-fabsf(v)));  // log sigmoid(v)
      o = expf(ls / c);
    }
    *px = o;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void gated_head_norm_kernel(const float* o, const float* w, const float* gate, int ldg,
                                                              T* out, int M, int H, int V, float eps, int gate_kind) {
  const int lane = threadIdx.x & 63;
  const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);  // (row, head)
  if (item >= (int64_t)M * H) return;
  const int64_t row = item / H;
  const int h = (int)(item - row * H);
  const float* oh = o + item * V;
  const float* g = gate + row * ldg + (int64_t)h * V;
  T* dst = out + item * V;
  float ss = 0.f;
  for (int i = lane; i < V; i += 64) ss += oh[i] * oh[i];
  const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)V + eps);
  for (int i = lane; i < V; i += 64) dst[i] = (T)(oh[i] * inv * (w ? w[i] : 1.0f) * (gate_kind == 1 ? sigmoid_f(g[i]) : silu_f(g[i])));
}

// The same for heads of 32, 64, 128 or 256 values, V / 4 lanes each: 16-byte pieces, 256 / V heads to a wave (1500 rows of 16 heads of
// 128: 10.4 -> 7.7 us)
template <typename T>
__global__ __launch_bounds__(256) void gated_head_norm_fours_kernel(const float* o, const float* w, const float* gate, int ldg, T* out,
                                                                    int64_t items, int H, int V, float eps, int gate_kind) {
  const int n = V >> 2, e = 4 * (threadIdx.x & (n - 1));
  const int64_t item = (int64_t)blockIdx.x * (256 / n) + threadIdx.x / n;  // (row, head)
  if (item >= items) return;  // whole heads: the lanes of a head leave together
  const int64_t row = item / H;
  const f32x4 v = ld4(o + item * V + e), g = ld4(gate + row * ldg + (item - row * H) * V + e);
  f32x4 k{1.f, 1.f, 1.f, 1.f};
  if (w) k = ld4(w + e);
  float ss = (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
  for (int x = n >> 1; x >= 1; x >>= 1) ss += __shfl_xor(ss, x);
  const float inv = 1.0f / sqrtf(ss / (float)V + eps);
  f32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = v[i] * inv * k[i] * (gate_kind == 1 ? sigmoid_f(g[i]) : silu_f(g[i]));
  st4(out + item * V + e, r);
}

__global__ __launch_bounds__(256) void rms_mix_kernel(const float* ya, int na, const float* wa, const float* yb, int nb, const float* wb,
                                                      float* out, int W, float eps, float coef) {
  __shared__ float red[4];
  const int64_t row = blockIdx.x;
  auto a = [&](int d) { return add_parts<float>(na, [&](int s) { return ya[(row * na + s) * W + d]; }); };
  auto b = [&](int d) { return add_parts<float>(nb, [&](int s) { return yb[(row * nb + s) * W + d]; }); };
  float sa = 0.f, sb = 0.f;
  for (int d = threadIdx.x; d < W; d += blockDim.x) {
    const float u = a(d), v = b(d);
    sa += u * u;
    sb += v * v;
  }
  sa = block_sum256(sa, red);
  sb = block_sum256(sb, red);
  const float ia = 1.0f / sqrtf(sa / (float)W + eps), ib = 1.0f / sqrtf(sb / (float)W + eps);
  for (int d = threadIdx.x; d < W; d += blockDim.x) out[row * W + d] = coef * (a(d) * ia * wa[d] + b(d) * ib * wb[d]);
}

// The same with a row's values in registers, NV groups of four per thread: one read of each row, a decode step's row on up to
// 1024 threads (16 rows of 4096: 6.9 -> 3.2 us, 3000 rows 39 -> 23)
template <int NV>
__global__ __launch_bounds__(1024) void rms_mix_vec_kernel(const float* ya, int na, const float* wa, const float* yb, int nb, const float* wb,
                                                           float* out, int W, float eps, float coef) {
  __shared__ float red[2][16];
  const int64_t row = blockIdx.x;
  f32x4 a[NV], b[NV];
  float sa = 0.f, sb = 0.f;
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int d = 4 * (threadIdx.x + n * blockDim.x);
    a[n] = b[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (d < W) {
      a[n] = add_parts<f32x4>(na, [&](int s) { return ld4(ya + (row * na + s) * W + d); });
      b[n] = add_parts<f32x4>(nb, [&](int s) { return ld4(yb + (row * nb + s) * W + d); });
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) sa += a[n][i] * a[n][i], sb += b[n][i] * b[n][i];
  }
  sa = wave_sum(sa), sb = wave_sum(sb);
  const int wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if ((threadIdx.x & 63) == 0) red[0][wave] = sa, red[1][wave] = sb;
  __syncthreads();
  sa = sb = 0.f;
  for (int i = 0; i < nw; ++i) sa += red[0][i], sb += red[1][i];
  const float ia = 1.0f / sqrtf(sa / (float)W + eps), ib = 1.0f / sqrtf(sb / (float)W + eps);
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int d = 4 * (threadIdx.x + n * blockDim.x);
    if (d >= W) continue;
    const f32x4 u = ld4(wa + d), v = ld4(wb + d);
    f32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = coef * (a[n][i] * ia * u[i] + b[n][i] * ib * v[i]);
    st4(out + row * W + d, o);
  }
}

__global__ __launch_bounds__(256) void logit_cap_kernel(float* x, int64_t n, float scale, float cap) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float v = x[i] * scale;
    x[i] = cap > 0.0f ? cap * tanhf(v / cap) : v;
  }
}

inline int flat_blocks(int64_t n) {
  const int64_t b = (n + 255) / 256;
  return (int)(b < 1 ? 1 : (b > 4096 ? 4096 : b));
}

}  // namespace
}  // namespace dsse

extern "C" hipError_t dsse_stream_step(const dsse::StreamStepParams* p, hipStream_t st) {
  if (p->M <= 0) return hipSuccess;
  if (p->y && p->nsum < 1) return hipErrorInvalidValue;
  const bool vec = p->W % 4 == 0 && dsse::fours({p->resid, p->y, p->embed, p->vec, p->w, p->b, p->xb});
  const dim3 grid(p->M, (p->W + (vec ? 1023 : 255)) / (vec ? 1024 : 256));
  if (p->f32 && vec) hipLaunchKernelGGL((dsse::stream_step_kernel<float, 4>), grid, dim3(256), 0, st, *p);
  else if (p->f32) hipLaunchKernelGGL((dsse::stream_step_kernel<float, 1>), grid, dim3(256), 0, st, *p);
  else if (vec) hipLaunchKernelGGL((dsse::stream_step_kernel<bf16, 4>), grid, dim3(256), 0, st, *p);
  else hipLaunchKernelGGL((dsse::stream_step_kernel<bf16, 1>), grid, dim3(256), 0, st, *p);
  return hipGetLastError();
}

extern "C" hipError_t dsse_gated_act(const float* gu, int ldg, void* h, int M, int F, int kind, int f32, hipStream_t st) {
  if (M <= 0 || F <= 0) return hipSuccess;
  const int blocks = dsse::flat_blocks((int64_t)M * F);
  if (f32)
    hipLaunchKernelGGL(dsse::gated_act_kernel<float>, dim3(blocks), dim3(256), 0, st, gu, ldg, reinterpret_cast<float*>(h),
                       M, F, kind);
  else
    hipLaunchKernelGGL(dsse::gated_act_kernel<bf16>, dim3(blocks), dim3(256), 0, st, gu, ldg, reinterpret_cast<bf16*>(h),
                       M, F, kind);
  return hipGetLastError();
}

// Every set in fours: the only form that adds biases
extern "C" bool dsse_norm_rope_all_fours(const dsse::NormRopeList& l) {
  for (int i = 0; i < l.n; ++i)
    if (!dsse::norm_rope_fours(l.p[i]) || (l.p[i].kind == 1 && l.p[i].bias)) return false;
  return true;
}

extern "C" hipError_t dsse_norm_rope_rows(dsse::NormRopeList l, hipStream_t st) {
  if (l.n < 1 || l.n > dsse::NormRopeList::kMost) return hipErrorInvalidValue;
  int waves = 4, width = 0, most = 0;
  for (int i = 0; i < l.n; ++i) {
    const dsse::NormRopeParams& p = l.p[i];
    if (p.T != l.p[0].T || p.D > dsse::kMaxHeadDim) return hipErrorInvalidValue;
    l.fours[i] = dsse::norm_rope_fours(p);
    // a row's workgroup of up to 16 waves; in fours 96 rows of 16 heads take 4.7 us with four waves and 5.5 with 16, 64 rows 4.6 / 4.5
    if (p.kind == 1 && p.T <= (l.fours[i] ? 64 : 512) && p.nh > 4) waves = std::max(waves, std::min(p.nh, 16));
    if (!l.fours[i]) width = std::max(width, p.D);
  }
  const int T = l.p[0].T;
  if (T <= 0) return hipSuccess;
  size_t lds = 0;
  // one walk of the heads per workgroup while the rows alone leave the chip idle, then more of them: a workgroup's start (lengths, places,
  // position) costs as much as a group of narrow heads.  One group / all groups per workgroup / this rule, rows x heads x width:
  // 512 x 32 x 64 normed in place 8.4 / 11.4 / 8.2 us, 1000 x 32 x 128 15.3 / 17.5 / 14.7; rotated into bf16, 4096 x 16 x 64
  // 16.8 / 11.2 / 11.4, 4096 x 64 x 64 54.1 / 33.7 / 35.5, 1500 x 32 x 128 16.7 / 15.6 / 16.1.
  const int each = T <= 512 ? 1 : (T < 1500 ? 2 : (T < 3000 ? 4 : 8));
  for (int i = 0; i < l.n; ++i) {
    const dsse::NormRopeParams& p = l.p[i];
    const int heads = waves * (l.fours[i] ? 256 / p.D : 1), groups = (p.nh + heads - 1) / heads;  // of one walk
    l.gy[i] = p.nh <= 0 ? 0 : (p.kind == 1 ? 1 : std::min((groups + each - 1) / each, 65535));
    // from 128 rows on: with fewer they are decode rows, each in a page of its own
    l.pages[i] = waves == 4 && l.fours[i] && p.out_t && dsse::fours({p.out_t}) && p.out_rows && !p.out_f32 && p.kind == 0 && !p.rope && p.nh > 0 && T >= 128;
    if (l.pages[i]) lds = std::max(lds, (size_t)dsse::kPageLds);
    most = std::max(most, l.gy[i]);
  }
  if (most <= 0) return hipSuccess;
  const dim3 grid(T, most, l.n);
  lds = std::max(lds, (size_t)waves * width * sizeof(float));
  if (waves == 4) hipLaunchKernelGGL(dsse::norm_rope_rows_kernel<4>, grid, dim3(256), lds, st, l);
  else hipLaunchKernelGGL(dsse::norm_rope_rows_kernel<16>, grid, dim3(64 * waves), lds, st, l);
  return hipGetLastError();
}

extern "C" hipError_t dsse_gate_math(float* x, int ld, int M, int N, int kind, const float* p1, int rep1, const float* p2,
                                     int rep2, float c, hipStream_t st) {
  if (M <= 0 || N <= 0) return hipSuccess;
  if (rep1 < 1 || rep2 < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(dsse::gate_math_kernel, dim3(dsse::flat_blocks((int64_t)M * N)), dim3(256), 0, st, x, ld, M, N, kind,
                     p1, rep1, p2, rep2, c);
  return hipGetLastError();
}

extern "C" hipError_t dsse_gated_head_norm(const float* o, const float* w, const float* gate, int ldg, void* out, int M,
                                           int H, int V, float eps, int gate_kind, int f32, hipStream_t st) {
  if (M <= 0 || H <= 0) return hipSuccess;
  if (V % 32 == 0 && V <= 256 && (V & (V - 1)) == 0 && ldg % 4 == 0 && dsse::fours({o, w, gate, out})) {
    const int64_t items = (int64_t)M * H, heads = 1024 / V;
    const dim3 grid((unsigned)((items + heads - 1) / heads));
    if (f32)
      hipLaunchKernelGGL(dsse::gated_head_norm_fours_kernel<float>, grid, dim3(256), 0, st, o, w, gate, ldg,
                         reinterpret_cast<float*>(out), items, H, V, eps, gate_kind);
    else
      hipLaunchKernelGGL(dsse::gated_head_norm_fours_kernel<bf16>, grid, dim3(256), 0, st, o, w, gate, ldg,
                         reinterpret_cast<bf16*>(out), items, H, V, eps, gate_kind);
    return hipGetLastError();
  }
  const int blocks = (int)(((int64_t)M * H + 3) / 4);
  if (f32)
    hipLaunchKernelGGL(dsse::gated_head_norm_kernel<float>, dim3(blocks), dim3(256), 0, st, o, w, gate, ldg,
                       reinterpret_cast<float*>(out), M, H, V, eps, gate_kind);
  else
    hipLaunchKernelGGL(dsse::gated_head_norm_kernel<bf16>, dim3(blocks), dim3(256), 0, st, o, w, gate, ldg,
                       reinterpret_cast<bf16*>(out), M, H, V, eps, gate_kind);
  return hipGetLastError();
}

extern "C" hipError_t dsse_rms_mix(const float* ya, int na, const float* wa, const float* yb, int nb, const float* wb, float* out, int M,
                                   int W, float eps, float coef, hipStream_t st) {
  if (M <= 0) return hipSuccess;
  if (na < 1 || nb < 1) return hipErrorInvalidValue;
  if (W % 4 == 0 && W <= 16384 && dsse::fours({ya, wa, yb, wb, out})) {
    const int threads = dsse::row_threads(M, W), nv = (W / 4 + threads - 1) / threads;
#define DSSE_MIX(n) hipLaunchKernelGGL(dsse::rms_mix_vec_kernel<n>, dim3(M), dim3(threads), 0, st, ya, na, wa, yb, nb, wb, out, W, eps, coef)
    if (nv <= 1) DSSE_MIX(1);
    else if (nv <= 2) DSSE_MIX(2);
    else DSSE_MIX(4);
#undef DSSE_MIX
    return hipGetLastError();
  }
  hipLaunchKernelGGL(dsse::rms_mix_kernel, dim3(M), dim3(256), 0, st, ya, na, wa, yb, nb, wb, out, W, eps, coef);
  return hipGetLastError();
}

extern "C" hipError_t dsse_logit_cap(float* logits, long long n, float scale, float cap, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(dsse::logit_cap_kernel, dim3(dsse::flat_blocks(n)), dim3(256), 0, st, logits, (int64_t)n, scale, cap);
  return hipGetLastError();
}
