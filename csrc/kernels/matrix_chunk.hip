// Matrix-state recurrences of prompt portions in chunks of 64 tokens on the fp32 matrix cores: decays that are one number per
// head (or per token and head, or none), with or without the delta rule.
//
// What bounds it: the chain from chunk to chunk.  The token walk (matrix_scan.hip) spends some 75 vector instructions per
// token and wave, 0.46 us per token of a sequence; a chunk of 64 tokens is five small products here, 6.4 us with the delta
// rule and 4.4 us without.  2048 tokens, 16 heads, 128 x 128: 946 -> 221 us and 919 -> 150 us; prompts of 582, 352 and 566
// tokens 281 -> 140 us and 268 -> 87 us (two-level walk of matrix_scan_chunked: some 220 us).  With A_t the
// product of the decays up to token t of the chunk, R[t][i] = A_t / A_i (formed as the product of the decays between them, so
// a decay of zero is no division), S the incoming state and u_i the written values,
//
//     S_t  = A_t S + sum_{i <= t} R[t][i] k_i u_i^T
//     u    = T (v - A (K S)),  T = (1 + L)^-1 diag(beta),  L[t][i] = beta_t R[t][i] k_t . k_i  for i < t   (delta rule)
//     u    = v                                                                                              (without)
//     o    = A (Q S) + M u,    M[t][i] = R[t][i] q_t . k_i  for i <= t
//     S'   = A_C S + K^T (E u),  E_i = R[C - 1][i]
//
// (the chunkwise form of the delta rule: Yang et al., "Parallelizing Linear Transformers with the Delta Rule over Sequence
// Length", 2024)
//
// Two launches: T, M, A and E depend on the inputs alone and are made for all chunks at once; the second walks the chunks of
// a (sequence, head, 16 value columns).  All products are v_mfma_f32_16x16x4_f32, 32-bit like the walk.  The accumulator
// layout (rows 4 g + i of column r) IS the B operand of a product whose k index runs 4 g + i over i, so the state, the
// written values and their scaled copy go from one product to the next without a change of layout; they meet between the four
// waves (16 tokens and D / 4 state rows each) in LDS.  The next chunk's operands are in registers a whole chunk ahead.
//
// A chunk's products run over its later tokens with weights of zero, so a token that is not finite would make the outputs of its
// whole chunk NaN.  Where an output is not finite, the sequence's columns are walked once more token by token (walk_tokens): such
// a token reaches the tokens after it and none before it.  The same walk serves sequences that the launch has no chunks for.
#include <algorithm>
#include <climits>

#include "api_mixers.h"

namespace dsse {
namespace {

constexpr int kC = 64;         // tokens per chunk
constexpr int kTwoLevelRows = 256;  // rows of a launch from which the two-level walk pays
constexpr int kScanCols = 16;  // value columns per workgroup: a tile of the state entry (matrix_scan.hip)

// floats of one (chunk, head): M | A | E | T
constexpr int kUnitA = kC * kC, kUnitE = kUnitA + kC, kUnitT = kUnitE + kC;
DEV int64_t unit_floats(bool delta) { return delta ? kUnitT + kC * kC : kUnitT; }

// chunks of the sequences before `seq` (wave-uniform; every lane calls it)
DEV int chunks_before(const int* q_len, int seq, int lane) {
  int sum = 0;
  for (int s0 = 0; s0 < seq; s0 += 64) {
    const int n = s0 + lane < seq ? q_len[s0 + lane] : 0;
    int c = n > 0 ? (n + kC - 1) / kC : 0;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) c += __shfl_xor(c, o);
    sum += c;
  }
  return __builtin_amdgcn_readfirstlane(sum);
}

// rows of four consecutive floats at p + row * ld, zero past the end
DEV f32x4 row4(const float* p, int64_t ld, int row, int rows) {
  const f32x4 v = ld_global<f32x4>(p + (int64_t)(row < rows ? row : 0) * ld);
  return row < rows ? v : f32x4{0.f, 0.f, 0.f, 0.f};
}

// Sums over the key width in kSums parts, added pairwise: a chain of 32 dependent products would round more than the token
// walk's tree over the lanes does.  Error of a layer's outputs against 64 bits, root mean square: 1.2e-7..1.4e-7 here and
// 1.0e-7..1.4e-7 in the walk; 2.3e-7 and 3.2e-7 where decays stay near one; of whole fp32 models 1.2e-6 and 1.3e-6.
constexpr int kSums = 8;
DEV f32x4 total(const f32x4 (&s)[4]) { return (s[0] + s[1]) + (s[2] + s[3]); }
DEV f32x4 total(const f32x4 (&s)[kSums]) { return ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7])); }

template <int NT, bool DELTA>
__global__ __launch_bounds__(256) void chunk_prepare_kernel(MatrixScanParams p, float* __restrict__ ws) {
  __shared__ float a_s[kC], b_s[kC], R[kC][kC + 1];
  __shared__ __align__(16) float Ls[DELTA ? kC : 1][kC + 4];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
  const int h = blockIdx.y;
  // the sequence and the place in it of chunk blockIdx.x
  int seq = -1, c = 0, before = 0;
  for (int s0 = 0; s0 < p.nseq && seq < 0; s0 += 64) {
    const int n = s0 + lane < p.nseq ? p.q_len[s0 + lane] : 0;
    const int own = n > 0 ? (n + kC - 1) / kC : 0;
    int upto = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(upto, o);
      if (lane >= o) upto += v;
    }
    const int at = (int)blockIdx.x - before;
    const uint64_t hit = __ballot(at >= upto - own && at < upto);
    if (hit) {
      const int l = __builtin_ctzll(hit);
      seq = s0 + l;
      c = at - __builtin_amdgcn_readlane(upto - own, l);
    }
    before += __builtin_amdgcn_readlane(upto, 63);
  }
  if (seq < 0) return;  // uniform for the workgroup: past the last chunk
  const int ql = p.q_len[seq], cnt = ql - c * kC < kC ? ql - c * kC : kC;
  const int64_t row0 = p.q_start[seq] + c * kC;
  const int grp = h / (p.H / p.G);
  float* unit = ws + ((int64_t)blockIdx.x * p.H + h) * unit_floats(DELTA);
  if (tid < kC) {
    float a = 1.0f, b = 0.0f;
    if (tid < cnt) {
      a = p.decay_kind == 1 ? p.decay[h] : (p.decay_kind == 2 ? p.decay[(row0 + tid) * p.ldd + h] : 1.0f);
      if (DELTA) b = p.beta[(row0 + tid) * p.ldb + h];
    }
    a_s[tid] = a;
    b_s[tid] = b;
  }
  __syncthreads();
  if (w == 3) {  // the wave with the most products makes them; this wave's column of R first (its products are independent)
    const float mine = a_s[lane];
    float v = 0.f;
#pragma unroll 8
    for (int t = 0; t < kC; ++t) {
      const float at = __shfl(mine, t);  // by every lane, also by the one that starts its column here
      v = t == lane ? 1.0f : v * at;
      R[t][lane] = v;
    }
  }
  // rows 16 w .. of K K^T and Q K^T, the tiles at and left of the diagonal
  const float* K = p.k + row0 * p.ldk + grp * p.D + 4 * g;
  const float* Q = p.q + row0 * p.ldq + grp * p.D + 4 * g;
  f32x4 kk[4][kSums], qk[4][kSums];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int s = 0; s < kSums; ++s) kk[j][s] = qk[j][s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const f32x4 qa = row4(Q + 16 * t, p.ldq, 16 * w + r, cnt);
    f32x4 kb[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j <= w) kb[j] = row4(K + 16 * t, p.ldk, 16 * j + r, cnt);  // uniform
    const f32x4 ka = row4(K + 16 * t, p.ldk, 16 * w + r, cnt);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j <= w)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (DELTA) kk[j][t % kSums] = mfma16x16x4(ka[i], kb[j][i], kk[j][t % kSums]);
          qk[j][t % kSums] = mfma16x16x4(qa[i], kb[j][i], qk[j][t % kSums]);
        }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const f32x4 qs = total(qk[j]), ks = total(kk[j]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 16 * w + 4 * g + i, col = 16 * j + r;
      const float rt = R[t][col];
      unit[t * kC + col] = col <= t ? rt * qs[i] * p.q_scale : 0.0f;
      if (DELTA) Ls[t][col] = col < t ? b_s[t] * rt * ks[i] : 0.0f;
    }
  }
  if (tid < kC) {
    unit[kUnitA + tid] = a_s[0] * R[tid][0];
    unit[kUnitE + tid] = R[kC - 1][tid];
  }
  if constexpr (DELTA) {
    __syncthreads();
    if (w != 0) return;
    // column `lane` of (1 + L)^-1 by forward substitution: a row of L is the same for all lanes
    float x[kC];
#pragma unroll
    for (int t = 0; t < kC; ++t) {
      float s[4] = {t == lane ? 1.0f : 0.0f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < t; i += 4) {
        const f32x4 l4 = *reinterpret_cast<const f32x4*>(&Ls[t][i]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (i + e < t) s[e] -= l4[e] * x[i + e];
      }
      x[t] = (s[0] + s[1]) + (s[2] + s[3]);
      unit[kUnitT + t * kC + lane] = x[t] * b_s[lane];
    }
  }
}

DEV f32x4 buf4(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
DEV float buf1(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}

// Operands of one chunk in a wave's registers (16 tokens 16 w .. of it)
template <int NT, bool DELTA>
struct Chunk {
  static constexpr int kOwn = NT >= 4 ? NT / 4 : 1;  // state row tiles of a wave
  f32x4 k[NT], q[NT], t[DELTA ? 4 : 1], m[4], v, a, e;
  float last;  // the product of the chunk's decays
};

// One wave's walk of a sequence, token by token: 16 value columns of a head, state rows 16 t + 4 g + i of column r in a lane
template <int NT, bool DELTA>
DEV void walk_tokens(const MatrixScanParams& p, int h, int64_t row0, int ql, bool fresh, int col, int r, int g, float* to) {
  const int grp = h / (p.H / p.G);
  f32x4 S[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) S[t][i] = fresh ? 0.0f : to[(16 * t + 4 * g + i) * kScanCols];
  for (int64_t row = row0; row < row0 + ql; ++row) {
    const float* k = p.k + row * p.ldk + grp * p.D + 4 * g;
    const float* q = p.q + row * p.ldq + grp * p.D + 4 * g;
    const float a = p.decay_kind == 1 ? p.decay[h] : (p.decay_kind == 2 ? p.decay[row * p.ldd + h] : 1.0f);
    float u = p.v[row * p.ldv + h * p.V + col], part = 0.0f, o = 0.0f;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      S[t] = S[t] * a;
      const f32x4 k4 = ld_global<f32x4>(k + 16 * t);
      if (DELTA)
#pragma unroll
        for (int i = 0; i < 4; ++i) part += S[t][i] * k4[i];
    }
    if (DELTA) u = p.beta[row * p.ldb + h] * (u - rows4_sum(part));
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const f32x4 k4 = ld_global<f32x4>(k + 16 * t), q4 = ld_global<f32x4>(q + 16 * t);
      S[t] += k4 * u;
#pragma unroll
      for (int i = 0; i < 4; ++i) o += S[t][i] * (q4[i] * p.q_scale);
    }
    o = rows4_sum(o);
    if (g == 0) p.out[(row * p.H + h) * p.V + col] = o;
  }
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) to[(16 * t + 4 * g + i) * kScanCols] = S[t][i];
}

template <int NT, bool DELTA>
__global__ __launch_bounds__(256, 1) void chunk_walk_kernel(MatrixScanParams p, const float* __restrict__ ws, int chunks) {
  using Ch = Chunk<NT, DELTA>;
  constexpr int kOwn = Ch::kOwn;
  constexpr int kKeyRow = 16 * NT + 4;  // floats of a key row in LDS: rows four apart start 16 banks apart
  __shared__ f32x4 bB[4][64], bU[4][64], bE[4][64], bS[NT][64];
  __shared__ int votes[4];
  __shared__ __align__(16) float keys[kC * kKeyRow];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  // heads fastest: the column blocks of a head read the same keys, queries and T, M, and land on one XCD's L2 when the heads
  // are a multiple of eight
  const int seq = blockIdx.z, h = blockIdx.x, cb = blockIdx.y, grp = h / (p.H / p.G);
  const int ql = p.q_len[seq];
  if (ql <= 0) return;  // uniform
  const int first = chunks_before(p.q_len, seq, lane), n = (ql + kC - 1) / kC;
  const int64_t row0 = p.q_start[seq];
  constexpr int units = DELTA ? kUnitT + kC * kC : kUnitT;
  const int col = cb * kScanCols + r;
  const bool owner = w * kOwn < NT;  // narrow states have fewer row tiles than waves
  // Buffer loads: the lane's offsets never change, a chunk's place is in the descriptor's base and its rows past the
  // sequence's end are past the descriptor's range, so they read as zeros
  const int own = 16 * w + r;
  const uint32_t q_vo = (uint32_t)(own * p.ldq + 4 * g) * 4, k_vo = (uint32_t)(own * p.ldk + 4 * g) * 4,
                 m_vo = (uint32_t)(own * kC + 4 * g) * 4,
                 v_vo = (uint32_t)((16 * w + 4 * g) * p.ldv + r) * 4, v_row = (uint32_t)p.ldv * 4;
  auto request = [&](int c, Ch& x) {  // chunks past the last one read it again
    c = c < n ? c : n - 1;
    const int left = ql - c * kC < kC ? ql - c * kC : kC;
    const int64_t at = row0 + (int64_t)c * kC;
    const __amdgpu_buffer_rsrc_t qr = make_rsrc(p.q + at * p.ldq + grp * p.D, (uint32_t)((left - 1) * p.ldq + p.D) * 4);
    const __amdgpu_buffer_rsrc_t kr = make_rsrc(p.k + at * p.ldk + grp * p.D, (uint32_t)((left - 1) * p.ldk + p.D) * 4);
    const __amdgpu_buffer_rsrc_t vr =
        make_rsrc(p.v + at * p.ldv + h * p.V + cb * kScanCols, (uint32_t)((left - 1) * p.ldv + kScanCols) * 4);
    const __amdgpu_buffer_rsrc_t ur = make_rsrc(ws + ((int64_t)(first + c) * p.H + h) * units, (uint32_t)units * 4);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      x.k[t] = buf4(kr, k_vo + 64 * t, 0);
      x.q[t] = buf4(qr, q_vo + 64 * t, 0);
    }
    x.a = buf4(ur, (kUnitA + 16 * w + 4 * g) * 4, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) x.v[i] = buf1(vr, v_vo + i * v_row, 0);  // the scalar offset is not range-checked
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if constexpr (DELTA) x.t[t] = buf4(ur, kUnitT * 4 + m_vo + 64 * t, 0);
    x.e = buf4(ur, (kUnitE + 16 * w + 4 * g) * 4, 0);
#pragma unroll
    for (int t = 0; t < 4; ++t) x.m[t] = buf4(ur, m_vo + 64 * t, 0);
    x.last = buf1(ur, (kUnitA + kC - 1) * 4, 0);
  };
  // the state entry is tile-major [H][V / 16][D][16] (V % 16 == 0)
  float* to = p.state + p.state_slot[seq] * ((int64_t)p.H * p.D * p.V) + (int64_t)h * p.D * p.V +
              (int64_t)cb * p.D * kScanCols + r;
  const bool fresh = p.ctx_len[seq] - ql == 0;
  if (first + n > chunks) {  // uniform: sequences longer than the caller said, or sharing rows; no units were made for this one
    if (w == 0) walk_tokens<NT, DELTA>(p, h, row0, ql, fresh, col, r, g, to);
    return;
  }
  f32x4 S[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) S[t][i] = fresh ? 0.0f : to[(16 * t + 4 * g + i) * kScanCols];

  float odd = 0.0f;  // NaN once an output is not finite
  auto walk = [&](int c, const Ch& x, Ch& next) {
    request(c + 1, next);  // in flight across this chunk
    // the chunk's key rows: the state's update reads them by columns
#pragma unroll
    for (int t = 0; t < NT; ++t) *reinterpret_cast<f32x4*>(&keys[own * kKeyRow + 16 * t + 4 * g]) = x.k[t];
    f32x4 P[kSums], u = x.v;
#pragma unroll
    for (int q = 0; q < kSums; ++q) P[q] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (DELTA) {
      f32x4 W[kSums];
#pragma unroll
      for (int q = 0; q < kSums; ++q) W[q] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          W[t % kSums] = mfma16x16x4(x.k[t][i], S[t][i], W[t % kSums]), P[t % kSums] = mfma16x16x4(x.q[t][i], S[t][i], P[t % kSums]);
      const f32x4 ws4 = total(W);
#pragma unroll
      for (int i = 0; i < 4; ++i) u[i] = x.v[i] - x.a[i] * ws4[i];
      bB[w][lane] = u;
      lds_barrier();
      f32x4 ut[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const f32x4 b = bB[t][lane];
        ut[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) ut[t] = mfma16x16x4(x.t[t][i], b[i], ut[t]);
      }
      u = total(ut);
    }
    bU[w][lane] = u;
    bE[w][lane] = x.e * u;
    if constexpr (!DELTA) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) P[t % kSums] = mfma16x16x4(x.q[t][i], S[t][i], P[t % kSums]);
    }
    lds_barrier();
    const f32x4 ps = total(P);
    f32x4 o[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t) o[t] = mfma16x16x4(x.m[t][i], bU[t][lane][i], o[t]);
    f32x4 res = total(o);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      res[i] += x.a[i] * (ps[i] * p.q_scale);
      odd += res[i] * 0.0f;
    }
    if (owner) {
      f32x4 s[kOwn];
#pragma unroll
      for (int o = 0; o < kOwn; ++o) s[o] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < NT; ++t)  // this wave's tiles, picked without indexing registers at run time
#pragma unroll
        for (int o = 0; o < kOwn; ++o)
          if (t == w * kOwn + o) s[o] = S[t] * x.last;  // uniform
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const f32x4 b = bE[t][lane];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int o = 0; o < kOwn; ++o) s[o] = mfma16x16x4(keys[(16 * t + 4 * g + i) * kKeyRow + 16 * (w * kOwn + o) + r], b[i], s[o]);
      }
#pragma unroll
      for (int o = 0; o < kOwn; ++o) bS[w * kOwn + o][lane] = s[o];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int tok = c * kC + 16 * w + 4 * g + i;
      if (tok < ql) p.out[((row0 + tok) * p.H + h) * p.V + col] = res[i];
    }
    lds_barrier();
#pragma unroll
    for (int t = 0; t < NT; ++t) S[t] = bS[t][lane];
  };
  Ch x, y;
  request(0, x);
  for (int c = 0; c < n; c += 2) {
    walk(c, x, y);
    if (c + 1 < n) walk(c + 1, y, x);  // uniform
  }
  const bool mine = __any(odd != 0.0f);
  if (lane == 0) votes[w] = mine;
  lds_barrier();
  if (votes[0] | votes[1] | votes[2] | votes[3]) {  // uniform for the workgroup
    __syncthreads();                                // every wave's outputs are written
    if (w == 0) walk_tokens<NT, DELTA>(p, h, row0, ql, fresh, col, r, g, to);
    return;
  }
#pragma unroll
  for (int t = 0; t < NT; ++t)
    if (t / kOwn == w)  // uniform
#pragma unroll
      for (int i = 0; i < 4; ++i) to[(16 * t + 4 * g + i) * kScanCols] = S[t][i];
}

template <int NT, bool DELTA>
hipError_t launch_chunks(const MatrixScanParams& p, float* ws, int chunks, hipStream_t st) {
  hipLaunchKernelGGL((chunk_prepare_kernel<NT, DELTA>), dim3(chunks, p.H), dim3(256), 0, st, p, ws);
  hipLaunchKernelGGL((chunk_walk_kernel<NT, DELTA>), dim3(p.H, p.V / kScanCols, p.nseq), dim3(256), 0, st, p, ws, chunks);
  return hipGetLastError();
}

}  // namespace

// Time in us of the walk by tokens and of the chunks: each is a start, then its longest chain or the work of all its column blocks,
// whichever is more.  Fitted per key width over 1..128 sequences of 16..4096 rows of 2..1024 column blocks (both within 11 % rms);
// of 864 timings the slower of the two is taken by more than 6 % in seven, by 9 % at most.  Walk against
// chunks, H x D x V: delta rule, 16 x 128 x 128, one sequence of 64 rows 31 / 38, 128 rows 56 / 44, 2048 rows 995 / 217, 128 of 32
// rows 388 / 531; 32 x 64 x 64, 64 of 64 rows 223 / 290 (one chunk each: the delta rule's start is not made up for); without it,
// 16 x 128 x 128, 64 rows 28 / 22, 2048 rows 913 / 146, 128 of 32 rows 360 / 491; 16 x 32 x 64, 64 of 64 rows 76 / 62.
struct ScanCost {
  double walk0, row, row_block, chunk0, chunk, chunk_block, seq_block;
};
static bool chunks_pay(const MatrixScanParams& p, int64_t rows, int64_t chunks, int64_t longest) {
  static const ScanCost kDelta[3] = {{5.3, 0.269, 0.044, 24.2, 2.53, 1.93, 0.42},   // widths 32, 64, 128
                                     {5.5, 0.301, 0.061, 25.8, 3.33, 2.22, 1.17},
                                     {5.5, 0.425, 0.118, 29.9, 5.24, 3.54, 1.17}};
  static const ScanCost kPlain[3] = {{5.4, 0.233, 0.039, 12.1, 1.84, 1.11, 0.46},
                                     {5.4, 0.270, 0.051, 13.7, 2.38, 1.34, 0.44},
                                     {5.2, 0.380, 0.107, 17.0, 4.03, 2.23, 1.18}};
  if (p.beta && longest <= kC) return false;
  const ScanCost& c = (p.beta ? kDelta : kPlain)[p.D == 32 ? 0 : (p.D == 64 ? 1 : 2)];
  const double blocks = (double)p.H * (p.V / kScanCols) / 128.0, n = (double)((longest + kC - 1) / kC);
  const double walk = c.walk0 + std::max(c.row * longest, c.row_block * rows * blocks);
  return walk > c.chunk0 + std::max(c.chunk * n, (c.chunk_block * chunks + c.seq_block * p.nseq) * blocks);
}

// chunks of `rows` rows at most: the launch's workgroups find theirs by the lengths
static int64_t chunk_bound(const MatrixScanParams& p, int64_t rows, int64_t longest) {
  return std::min(rows / kC + p.nseq, p.nseq * ((longest + kC - 1) / kC));
}

// Whether the chunks take the shape, and their workspace floats
static int64_t chunk_room(const MatrixScanParams& p, int rows, int64_t longest) {
  auto aligned = [](const float* x, int ld) { return reinterpret_cast<uintptr_t>(x) % 16 == 0 && ld % 4 == 0; };
  if (longest <= 0 || p.nseq <= 0 || p.src_idx || p.decay_kind > 2 || (p.D != 32 && p.D != 64 && p.D != 128) ||
      p.V % kScanCols || !aligned(p.q, p.ldq) || !aligned(p.k, p.ldk))
    return 0;
  // rows of a chunk lie within 31-bit offsets of its first one
  const int64_t ld = std::max(std::max((int64_t)p.ldq, (int64_t)p.ldk), (int64_t)p.ldv);
  const int64_t chunks = chunk_bound(p, rows, longest);
  if (chunks > 65535 || p.nseq > 65535 || p.H > 65535 || ld * kC * 4 > INT32_MAX) return 0;
  const int64_t floats = chunks * p.H * (p.beta ? kUnitT + kC * kC : kUnitT);
  return floats <= (int64_t{1} << 28) ? floats : 0;  // a gigabyte: 128k rows of 16 heads; the token walk needs no workspace
}

int64_t scan_chunk_floats(const MatrixScanParams& p, int rows, int64_t longest) {
  const int64_t floats = chunk_room(p, rows, longest);
  if (!floats) return 0;
  return chunks_pay(p, std::min<int64_t>(rows, p.nseq * longest), chunk_bound(p, rows, longest), longest) ? floats : 0;
}

// Without the delta rule.  Where the chunks are out of the question (decays per key channel, other widths, unaligned rows) two
// levels beat one long chain; where they are not, only for a long sequence of a few column blocks, whose chunks follow one
// another on a mostly empty chip.  Chunks against two levels: 2 heads of 128 x 128, 700 rows 59 / 66, 1000 rows 77 / 72; 2 heads of
// 64 x 64, 1000 rows 49 / 57, 2048 rows 84 / 74; 2 of 32 x 16, 2048 rows 66 / 68, 4096 rows 120 / 98; 16 x 64 x 64, 4096 rows 170 / 257.
bool scan_two_levels(const MatrixScanParams& p, int rows, int64_t longest) {
  if (p.beta || rows < kTwoLevelRows) return false;
  if (!chunk_room(p, rows, longest)) return true;
  const int64_t from = p.D == 128 ? 900 : (p.D == 64 ? 1500 : 2500);
  return longest >= from && (int64_t)p.nseq * p.H * (p.V / kScanCols) <= 16;
}

}  // namespace dsse

extern "C" hipError_t dsse_scan_chunks(const dsse::MatrixScanParams* p, float* ws, int rows, int64_t longest, hipStream_t st) {
  if (p->nseq <= 0 || p->H <= 0 || rows <= 0) return hipSuccess;
  if (p->H % p->G || !dsse::scan_chunk_floats(*p, rows, longest)) return hipErrorInvalidValue;
  const int chunks = (int)dsse::chunk_bound(*p, rows, longest);
#define DSSE_CHUNK_CASE(n)                                                            \
  case 16 * n:                                                                        \
    return p->beta ? dsse::launch_chunks<n, true>(*p, ws, chunks, st) : dsse::launch_chunks<n, false>(*p, ws, chunks, st);
  switch (p->D) {
    DSSE_CHUNK_CASE(2)
    DSSE_CHUNK_CASE(4)
    DSSE_CHUNK_CASE(8)
  }
#undef DSSE_CHUNK_CASE
  return hipErrorInvalidValue;
}
