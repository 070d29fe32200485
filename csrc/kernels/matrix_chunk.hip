// Matrix-state recurrences of prompt portions in chunks of 16 tokens on the fp32 matrix cores: with or without the delta rule, under
// decays that are one number per head, per token and head, or per token, head and key channel (or none).
//
// What bounds it: the chain from chunk to chunk.  The token walk (matrix_scan.hip) spends some 75 vector instructions per token and
// wave, 0.46 us per token of a sequence.  A chunk of 16 is 29 products of 16 x 16 x 4 per wave with the delta rule and 17 without,
// 0.42 and 0.25 us of matrix time, and takes 1.1 and 0.63 us (key width 128): the rest is LDS, the barrier and dependent products.
// With P[t][i] the product of the decays after token i up to token t (P[t][-1]: from the chunk's start), per key channel, S the
// incoming state and u_i the written values, all products with P elementwise along the key width,
//
//     W    = (K P[.][-1]) S,   u = T (v - W),   T = (1 + L)^-1 diag(beta),  L[t][i] = beta_t k_t . (P[t][i] k_i) for i < t   (delta rule)
//     u    = v                                                                                                         (without)
//     o    = (Q P[.][-1]) S + M u,   M[t][i] = q_t . (P[t][i] k_i)  for i <= t
//     S'   = P[15][-1] S + (K P[15][.])^T u
//
// (the chunkwise form of the delta rule: Yang et al., "Parallelizing Linear Transformers with the Delta Rule over Sequence Length",
// 2024).  Every P is formed as the product of the decays between the two tokens, so a decay of zero is no division; a chunk no longer
// than a tile of the matrix cores is what makes that affordable per key channel.
//
// Two launches: the scaled rows, T, M and the chunk's decay depend on the inputs alone and are made for all chunks at once, laid out
// as operands; the second walks the chunks of a (sequence, head, 16 or 32 value columns), each of its waves holding D / 4 state rows.
// All products are v_mfma_f32_16x16x4_f32, 32-bit like the walk.  The accumulator layout (rows 4 g + i of column r) IS the B operand
// of a product whose k index runs 4 g + i over i, so the state and the written values go from one product to the next without a
// change of layout; only the waves' shares of W and o meet in LDS, those of o behind the next chunk's products.
//
// Measured, us, key and value width 128 (before: chunks of 64 tokens for decays per head, two parallel token walks per key channel):
// delta rule, 16 heads: prompts of 582, 352 and 566 tokens 140 -> 81, one of 2048 217 -> 147, of 200 58 -> 25; retention 87 -> 54,
// 146 -> 89, 30 -> 16; decays per channel, 8 heads: 146 -> 39, 210 -> 88, one of 200 (token walk) 74 -> 19.  Error of the outputs
// against 64 bits, root mean square: 1.1e-7 with the delta rule (walk 1.0e-7, chunks of 64 1.2e-7 .. 1.4e-7), 2.7e-7 under decays near
// one (walk 3.2e-7, chunks of 64 2.3e-7 .. 3.2e-7), 1.3e-7 per channel (walk and two walks 1.3e-7).
//
// A chunk's products run over its later tokens with weights of zero, so a token that is not finite would make the outputs of its
// whole chunk NaN.  Where an output is not finite, the sequence's columns are walked once more token by token (walk_tokens): such
// a token reaches the tokens after it and none before it.  The same walk serves sequences that the launch has no chunks for.
//
// The workspace is 17 (25) KB per chunk and head at width 128; past kRoom the launch goes by segments of every sequence, which meet in
// the state entries.
#include <algorithm>
#include <climits>

#include "api_mixers.h"

namespace dsse {
namespace {

constexpr int kC = 16;         // tokens per chunk: a tile of the matrix cores
constexpr int kTwoLevelRows = 256;  // rows of a launch from which the two-level walk pays
constexpr int kScanCols = 16;  // value columns of a tile of the state entry (matrix_scan.hip)
constexpr int64_t kRoom = int64_t{1} << 26;   // workspace floats of a segment: 268 MB
constexpr int64_t kMostRows = int64_t{1} << 22;  // rows x heads

// floats of one (chunk, head): Q' | K^ | (K') | M | (T) | A; the first three as tiles of 16 key channels
__host__ __device__ constexpr int unit_floats(int D, bool delta) {
  return (delta ? 3 : 2) * kC * D + (delta ? 2 : 1) * kC * kC + D;
}

// The launch's part of each sequence: its chunks [c0, c0 + span)
struct Segment {
  int c0, span;
};
DEV int chunks_of(int ql, Segment sg) {
  const int n = ql > 0 ? (ql + kC - 1) / kC - sg.c0 : 0;
  return n < 0 ? 0 : (n < sg.span ? n : sg.span);
}
// chunks of the sequences before `seq` (wave-uniform; every lane calls it)
DEV int chunks_before(const int* q_len, int seq, int lane, Segment sg) {
  int sum = 0;
  for (int s0 = 0; s0 < seq; s0 += 64) {
    int c = s0 + lane < seq ? chunks_of(q_len[s0 + lane], sg) : 0;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) c += __shfl_xor(c, o);
    sum += c;
  }
  return __builtin_amdgcn_readfirstlane(sum);
}

template <int CTRL>
DEV float row_rotated(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
DEV float row16_sum(float v) {
  v += row_rotated<0x128>(v);
  v += row_rotated<0x124>(v);
  v += row_rotated<0x122>(v);
  v += row_rotated<0x121>(v);
  return v;
}

template <int N, typename T>
DEV T pairwise(const T* x) {
  if constexpr (N == 1) return x[0];
  else return pairwise<N / 2>(x) + pairwise<N / 2>(x + N / 2);
}

// One (chunk, head): everything that does not depend on the state.  CHAN: the decays differ between key channels.
template <int NT, bool DELTA, bool CHAN>
__global__ __launch_bounds__(256) void chunk_prepare_kernel(MatrixScanParams p, float* __restrict__ ws, Segment sg) {
  constexpr int D = 16 * NT, kPer = NT, kVec = kPer < 4 ? kPer : 4;  // channels per lane of a row of 16 lanes, in vectors
  using vec = float __attribute__((ext_vector_type(kVec)));
  constexpr int kRow = D + 4;  // rows start four banks apart
  __shared__ __align__(16) float qs[kC][kRow], ks[kC][kRow], as[kC][CHAN ? kRow : 1];
  __shared__ __align__(16) float Ls[DELTA ? kC : 1][kC];
  __shared__ float bs[kC];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = blockIdx.y;
  // the sequence and the place in it of chunk blockIdx.x
  int seq = -1, c = 0, before = 0;
  for (int s0 = 0; s0 < p.nseq && seq < 0; s0 += 64) {
    const int own = s0 + lane < p.nseq ? chunks_of(p.q_len[s0 + lane], sg) : 0;
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
  const int first = (sg.c0 + c) * kC, left = p.q_len[seq] - first, cnt = left < kC ? left : kC;
  const int64_t row0 = p.q_start[seq] + first;
  const int grp = h / (p.H / p.G);
  float* unit = ws + ((int64_t)blockIdx.x * p.H + h) * unit_floats(D, DELTA);
  float* uk = unit + kC * D;
  float* ub = uk + kC * D;
  float* um = ub + (DELTA ? kC * D : 0);
  float* ut = um + kC * kC;
  float* ua = um + (DELTA ? 2 : 1) * kC * kC;
  // tokens past the sequence's end: no key, no query, no decay
  for (int i = tid; i < kC * D / 4; i += 256) {
    const int t = i / (D / 4), d = 4 * (i % (D / 4));
    const bool on = t < cnt;
    const int64_t row = row0 + (on ? t : 0);
    f32x4 q = ld_global<f32x4>(p.q + row * p.ldq + grp * D + d), k = ld_global<f32x4>(p.k + row * p.ldk + grp * D + d);
#pragma unroll
    for (int e = 0; e < 4; ++e) q[e] = on ? q[e] * p.q_scale : 0.0f, k[e] = on ? k[e] : 0.0f;
    *reinterpret_cast<f32x4*>(&qs[t][d]) = q;
    *reinterpret_cast<f32x4*>(&ks[t][d]) = k;
    if constexpr (CHAN) {
      f32x4 a = ld_global<f32x4>(p.decay + row * p.ldd + h * D + d);
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] = on ? a[e] : 1.0f;
      *reinterpret_cast<f32x4*>(&as[t][d]) = a;
    }
  }
  if (!CHAN && tid < kC)
    as[tid][0] = tid >= cnt || p.decay_kind == 0 ? 1.0f : (p.decay_kind == 1 ? p.decay[h] : p.decay[(row0 + tid) * p.ldd + h]);
  if (DELTA && tid < kC) bs[tid] = tid < cnt ? p.beta[(row0 + tid) * p.ldb + h] : 0.0f;
  __syncthreads();
  auto decay = [&](int t, int d) {
    if constexpr (CHAN) return *reinterpret_cast<const f32x4*>(&as[t][d]);
    else return f32x4{as[t][0], as[t][0], as[t][0], as[t][0]};
  };
  // the state's view of the tokens: rows times the decays up to them, keys times the decays after them
  if (w >= 2 && lane < D / 4) {  // the waves with the fewest pairs, or none
    const int d = 4 * lane, at = d / 16 * (16 * kC) + d % 16;
    f32x4 a{1.f, 1.f, 1.f, 1.f};
    if (w == 2) {
#pragma unroll
      for (int t = 0; t < kC; ++t) {
        a *= decay(t, d);
        *reinterpret_cast<f32x4*>(unit + at + 16 * t) = *reinterpret_cast<const f32x4*>(&qs[t][d]) * a;
        if (DELTA) *reinterpret_cast<f32x4*>(ub + at + 16 * t) = *reinterpret_cast<const f32x4*>(&ks[t][d]) * a;
      }
      *reinterpret_cast<f32x4*>(ua + d) = a;
    } else {
      f32x4 x[kC];
#pragma unroll
      for (int t = kC - 1; t >= 0; --t) {
        x[t] = *reinterpret_cast<const f32x4*>(&ks[t][d]) * a;
        a *= decay(t, d);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t = 0; t < kC; t += 4)
          *reinterpret_cast<f32x4*>(uk + (d + e) * kC + t) = f32x4{x[t][e], x[t + 1][e], x[t + 2][e], x[t + 3][e]};
    }
  }
  if constexpr (!CHAN) {
    // pairs of tokens: the rows' products on the matrix cores, times the decays between the two
    if (w < (DELTA ? 2 : 1)) {  // uniform: queries against keys, keys against keys
      const int r = lane & 15, g = lane >> 4;
      const float(&rows)[kC][kRow] = w ? ks : qs;
      f32x4 s[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(&rows[r][16 * t + 4 * g]), b = *reinterpret_cast<const f32x4*>(&ks[r][16 * t + 4 * g]);
#pragma unroll
        for (int i = 0; i < 4; ++i) s[t] = mfma16x16x4(a[i], b[i], s[t]);
      }
      f32x4 R{0.f, 0.f, 0.f, 0.f};
      float v = 0.f;
#pragma unroll
      for (int t = 0; t < kC; ++t) {
        v = t == r ? 1.0f : v * as[t][0];
        if (g == t / 4) R[t % 4] = v;
      }
      const f32x4 x = R * pairwise<NT>(s);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 4 * g + i;
        if (w == 0) um[t * kC + r] = r <= t ? x[i] : 0.0f;
        else if (DELTA) Ls[t][r] = r < t ? bs[t] * x[i] : 0.0f;
      }
    }
  } else {
  // pairs of tokens: key i, decayed from token to token, against the queries (and keys) of the tokens from it on
  {
    const int dg = lane & 15, i = 4 * (lane >> 4) + w;
    vec kr[kPer / kVec];
#pragma unroll
    for (int e = 0; e < kPer / kVec; ++e) kr[e] = *reinterpret_cast<const vec*>(&ks[i][kVec * (dg + 16 * e)]);
    float m = 0.f, l = 0.f;
#pragma unroll
    for (int t = 0; t < kC; ++t) {
      if (t < w) continue;  // uniform: none of the wave's keys is at or before t
      float sq[kVec], sk[kVec];
#pragma unroll
      for (int j = 0; j < kVec; ++j) sq[j] = sk[j] = 0.f;
#pragma unroll
      for (int e = 0; e < kPer / kVec; ++e) {
        const int d = kVec * (dg + 16 * e);
        const vec a = *reinterpret_cast<const vec*>(&as[t][d]), q = *reinterpret_cast<const vec*>(&qs[t][d]);
        if (t > i) kr[e] *= a;
#pragma unroll
        for (int j = 0; j < kVec; ++j) sq[j] += q[j] * kr[e][j];
        if (DELTA) {
          const vec k = *reinterpret_cast<const vec*>(&ks[t][d]);
#pragma unroll
          for (int j = 0; j < kVec; ++j) sk[j] += k[j] * kr[e][j];
        }
      }
      auto sum = [](const float (&s)[kVec]) {
        if constexpr (kVec == 4) return (s[0] + s[1]) + (s[2] + s[3]);
        else return s[0] + s[1];
      };
      const float mt = row16_sum(sum(sq));
      if (dg == t) m = mt;
      if (DELTA) {
        const float lt = row16_sum(sum(sk));
        if (dg == t) l = lt;
      }
    }
    um[dg * kC + i] = i <= dg ? m : 0.0f;
    if (DELTA) Ls[dg][i] = i < dg ? bs[dg] * l : 0.0f;
  }
  }
  if constexpr (DELTA) {
    __syncthreads();
    if (tid >= kC) return;
    // column `tid` of (1 + L)^-1 by forward substitution: a row of L is the same for all lanes
    float x[kC];
#pragma unroll
    for (int t = 0; t < kC; ++t) {
      float s[4] = {t == tid ? 1.0f : 0.0f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < t; i += 4) {
        const f32x4 l4 = *reinterpret_cast<const f32x4*>(&Ls[t][i]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (i + e < t) s[e] -= l4[e] * x[i + e];
      }
      x[t] = (s[0] + s[1]) + (s[2] + s[3]);
      ut[t * kC + tid] = x[t] * bs[tid];
    }
  }
}

DEV f32x4 buf4(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
DEV float buf1(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}

// One wave's walk of a sequence, token by token: 16 value columns of a head, state rows 16 t + 4 g + i of column r in a lane
template <int NT, bool DELTA>
DEV void walk_tokens(const MatrixScanParams& p, int h, int64_t row0, int ql, bool fresh, int col, int g, float* to) {
  const int grp = h / (p.H / p.G);
  f32x4 S[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) S[t][i] = fresh ? 0.0f : to[(16 * t + 4 * g + i) * kScanCols];
  for (int64_t row = row0; row < row0 + ql; ++row) {
    const float* k = p.k + row * p.ldk + grp * p.D + 4 * g;
    const float* q = p.q + row * p.ldq + grp * p.D + 4 * g;
    const bool chan = p.decay_kind == 3;
    const float* ac = p.decay + row * p.ldd + h * p.D + 4 * g;
    const float a = p.decay_kind == 1 ? p.decay[h] : (p.decay_kind == 2 ? p.decay[row * p.ldd + h] : 1.0f);
    float u = p.v[row * p.ldv + h * p.V + col], part = 0.0f, o = 0.0f;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if (chan) S[t] *= ld_global<f32x4>(ac + 16 * t);  // uniform
      else S[t] = S[t] * a;
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

// CT tiles of 16 value columns per workgroup
template <int NT, bool DELTA, int CT>
__global__ __launch_bounds__(64 * (NT < 4 ? NT : 4), 2) void chunk_walk_kernel(MatrixScanParams p, const float* __restrict__ ws,
                                                                              int chunks, Segment sg) {
  constexpr int NW = NT < 4 ? NT : 4, OWN = NT / NW, MI = 4 / NW;  // waves, state row tiles and products with M of each
  constexpr int D = 16 * NT, kUnit = unit_floats(D, DELTA);
  constexpr int kAhead = DELTA ? 2 : (CT == 1 ? 4 : 3);  // chunks whose operands are in registers or on their way
  constexpr int kB = 2 * kC * D, kM = kB + (DELTA ? kC * D : 0), kT = kM + kC * kC, kA = kM + (DELTA ? 2 : 1) * kC * kC;
  __shared__ f32x4 bO[2][NW][CT][64], bW[DELTA ? 2 : 1][NW][CT][64];
  __shared__ int votes[NW];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  // heads fastest: the column blocks of a head read the same units and land on one XCD's L2 when the heads are a multiple of eight
  const int seq = blockIdx.z, h = blockIdx.x, cb = blockIdx.y;
  const int n = chunks_of(p.q_len[seq], sg);
  if (n <= 0) return;  // uniform
  const int first = chunks_before(p.q_len, seq, lane, sg);
  const int64_t row0 = (int64_t)p.q_start[seq] + (int64_t)sg.c0 * kC;
  const int all = p.q_len[seq] - sg.c0 * kC, ql = all < sg.span * kC ? all : sg.span * kC;
  const bool fresh = sg.c0 == 0 && p.ctx_len[seq] - p.q_len[seq] == 0;
  // the state entry is tile-major [H][V / 16][D][16] (V % 16 == 0)
  float* to = p.state + p.state_slot[seq] * ((int64_t)p.H * D * p.V) + (int64_t)h * D * p.V + (int64_t)cb * CT * D * kScanCols + r;
  const int col = cb * CT * kScanCols + r;
  auto by_tokens = [&]() {
#pragma unroll
    for (int x = 0; x < CT; ++x)
      walk_tokens<NT, DELTA>(p, h, row0, ql, fresh, col + 16 * x, g, to + x * D * kScanCols);
  };
  if (first + n > chunks) {  // uniform: sequences longer than the caller said, or sharing rows; no units were made for this one
    if (w == 0) by_tokens();
    return;
  }
  struct Operands {
    f32x4 q[OWN], k[OWN], b[DELTA ? OWN : 1], a[OWN], t, v[CT];
    float m[MI];
  };
  // Chunks are requested one after another: what is left of the sequence, and where its next unit and value rows lie.  The
  // value rows past its end, and every operand of a chunk past the last one, are past their descriptor's range: zeros, no traffic.
  const float* next_unit = ws + ((int64_t)first * p.H + h) * kUnit;
  const float* next_v = p.v + row0 * p.ldv + h * p.V + cb * CT * kScanCols;
  int ahead = ql;
  const int64_t unit_step = (int64_t)p.H * kUnit, v_step = (int64_t)kC * p.ldv;
  const uint32_t u_vo = (uint32_t)(16 * r + 4 * g) * 4, v_vo = (uint32_t)(4 * g * p.ldv + r) * 4, v_row = (uint32_t)p.ldv * 4;
  auto range = [&](int rows, uint32_t row) {  // bytes of CT tiles of the last of up to 16 rows, and of the rows before it
    rows = rows < kC ? rows : kC;
    return rows > 0 ? (uint32_t)(rows - 1) * row + CT * kScanCols * 4 : 0u;
  };
  auto request = [&](Operands& x) {
    const __amdgpu_buffer_rsrc_t ur = make_rsrc(next_unit, ahead > 0 ? kUnit * 4 : 0);
    const __amdgpu_buffer_rsrc_t vr = make_rsrc(next_v, range(ahead, v_row));
    next_unit += unit_step, next_v += v_step, ahead -= kC;
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      const int t = w * OWN + o;
      if constexpr (DELTA) x.b[o] = buf4(ur, u_vo, (kB + 256 * t) * 4);
      x.q[o] = buf4(ur, u_vo, 256 * t * 4);
      x.k[o] = buf4(ur, u_vo, (kC * D + 256 * t) * 4);
      x.a[o] = buf4(ur, 16 * g, (kA + 16 * t) * 4);
    }
    if constexpr (DELTA) x.t = buf4(ur, u_vo, kT * 4);
#pragma unroll
    for (int i = 0; i < MI; ++i) x.m[i] = buf1(ur, u_vo, (kM + w + NW * i) * 4);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) x.v[ct][i] = buf1(vr, v_vo + i * v_row + 64 * ct, 0);  // the scalar offset is not range-checked
  };
  f32x4 S[OWN][CT];
#pragma unroll
  for (int o = 0; o < OWN; ++o)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        S[o][ct][i] = fresh ? 0.0f : to[(ct * D + 16 * (w * OWN + o) + 4 * g + i) * kScanCols];
  float odd = 0.0f;  // NaN once an output is not finite
  const uint32_t o_row = (uint32_t)(p.H * p.V) * 4;
  float part[CT][MI][NW];
  auto collect = [&](int c) {  // every wave's share of chunk c's rows 4 g + w (+ NW)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int o = 0; o < NW; ++o) part[ct][i][o] = reinterpret_cast<const float*>(&bO[c & 1][o][ct][lane])[w + NW * i];
  };
  float* next_out = p.out + (row0 * p.H + h) * p.V + cb * CT * kScanCols;
  int behind = ql;
  auto write = [&]() {  // chunk after chunk; rows past the sequence's end are out of the descriptor's range
    const __amdgpu_buffer_rsrc_t to_out = make_rsrc(next_out, range(behind, o_row));
    next_out += (int64_t)kC * p.H * p.V, behind -= kC;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        float s = part[ct][i][0] + part[ct][i][1];
        if constexpr (NW == 4) s += part[ct][i][2] + part[ct][i][3];
        odd += s * 0.0f;
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(s), to_out, (4 * g + w + NW * i) * o_row + r * 4 + 64 * ct, 0, 0);
      }
  };
  const f32x4 zero{0.f, 0.f, 0.f, 0.f};
  // One chunk: the outputs of the chunk before leave LDS meanwhile, behind the barrier that the delta rule needs anyway
  auto step = [&](int c, Operands& x) {
    f32x4 u[CT], O[OWN][CT];
    auto read_out = [&](int i0, int i1) {
#pragma unroll
      for (int i = i0; i < i1; ++i)
#pragma unroll
        for (int o = 0; o < OWN; ++o)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) O[o][ct] = mfma16x16x4(x.q[o][i], S[o][ct][i], i ? O[o][ct] : zero);
    };
    if constexpr (DELTA) {
      f32x4 W[OWN][CT];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int o = 0; o < OWN; ++o)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) W[o][ct] = mfma16x16x4(x.b[o][i], S[o][ct][i], i ? W[o][ct] : zero);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        f32x4 s = W[0][ct];
#pragma unroll
        for (int o = 1; o < OWN; ++o) s += W[o][ct];
        bW[c & 1][w][ct][lane] = s;
      }
      read_out(0, 2);
      lds_barrier();
      f32x4 ws4[CT][NW];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int o = 0; o < NW; ++o) ws4[ct][o] = bW[c & 1][o][ct][lane];
      collect(c > 0 ? c - 1 : 0);
      __builtin_amdgcn_sched_barrier(0);
      read_out(2, 4);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        f32x4 s = ws4[ct][0] + ws4[ct][1];
        if constexpr (NW == 4) s += ws4[ct][2] + ws4[ct][3];
        const f32x4 d = x.v[ct] - s;
        f32x4 t0 = mfma16x16x4(x.t[0], d[0], zero), t1 = mfma16x16x4(x.t[1], d[1], zero);
        t0 = mfma16x16x4(x.t[2], d[2], t0);
        t1 = mfma16x16x4(x.t[3], d[3], t1);
        u[ct] = t0 + t1;
      }
    } else {
      read_out(0, 4);
      lds_barrier();
      collect(c > 0 ? c - 1 : 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) u[ct] = x.v[ct];
    }
#pragma unroll
    for (int o = 0; o < OWN; ++o)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) S[o][ct] *= x.a[o];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int o = 0; o < OWN; ++o)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) S[o][ct] = mfma16x16x4(x.k[o][i], u[ct][i], S[o][ct]);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      f32x4 s = O[0][ct];
#pragma unroll
      for (int o = 1; o < OWN; ++o) s += O[o][ct];
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        float uw = u[ct][NW * i];
#pragma unroll
        for (int k = 1; k < NW; ++k) uw = w == k ? u[ct][NW * i + k] : uw;
        s = mfma16x16x4(x.m[i], uw, s);
      }
      bO[c & 1][w][ct][lane] = s;
    }
    if (c > 0) write();  // uniform
    __builtin_amdgcn_sched_barrier(0);  // requests stay in the order of their use
    request(x);
    __builtin_amdgcn_sched_barrier(0);
  };
  Operands x[kAhead];
#pragma unroll
  for (int i = 0; i < kAhead; ++i) {
    request(x[i]);
    __builtin_amdgcn_sched_barrier(0);
  }
  int c = 0;
  for (; c + kAhead <= n; c += kAhead)  // no branch between the steps: each waits for its own operands alone
#pragma unroll
    for (int i = 0; i < kAhead; ++i) step(c + i, x[i]);
#pragma unroll
  for (int i = 0; i + 1 < kAhead; ++i)
    if (c + i < n) step(c + i, x[i]);  // uniform
  lds_barrier();
  collect(n - 1);
  write();
  const bool mine = __any(odd != 0.0f);
  if (lane == 0) votes[w] = mine;
  lds_barrier();
  int any = 0;
#pragma unroll
  for (int i = 0; i < NW; ++i) any |= votes[i];
  if (any) {          // uniform for the workgroup
    __syncthreads();  // every wave's outputs are written
    if (w == 0) by_tokens();
    return;
  }
#pragma unroll
  for (int o = 0; o < OWN; ++o)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) to[(ct * D + 16 * (w * OWN + o) + 4 * g + i) * kScanCols] = S[o][ct][i];
}

// two column tiles per workgroup once single ones are more than the CUs
bool scan_pairs(const MatrixScanParams& p) {
  return p.V % (2 * kScanCols) == 0 && (int64_t)p.H * (p.V / kScanCols) * p.nseq > 256;
}

// chunks of `rows` rows at most, `longest` in the longest sequence, in segments of `span` chunks of each
int64_t chunk_bound(const MatrixScanParams& p, int64_t rows, int64_t longest, int64_t span) {
  return std::min(rows / kC + p.nseq, p.nseq * std::min(span, (longest + kC - 1) / kC));
}
// the segment's chunks per sequence: all of them where the workspace has the room
int64_t segment_span(const MatrixScanParams& p, int64_t rows, int64_t longest) {
  const int64_t n = (longest + kC - 1) / kC, unit = (int64_t)p.H * unit_floats(p.D, p.beta);
  if (chunk_bound(p, rows, longest, n) * unit <= kRoom) return n;
  return std::max<int64_t>(1, kRoom / unit / p.nseq);
}

template <int NT, bool DELTA>
hipError_t launch_chunks(const MatrixScanParams& p, float* ws, int64_t rows, int64_t longest, hipStream_t st) {
  const int64_t n = (longest + kC - 1) / kC, span = segment_span(p, rows, longest);
  const int chunks = (int)chunk_bound(p, rows, longest, span);
  const bool pairs = scan_pairs(p);
  // a sequence may be longer than the caller said: the last segment takes what is left of it
  for (int64_t c0 = 0; c0 < n; c0 += span) {
    const Segment sg{(int)c0, c0 + span < n ? (int)span : INT_MAX / kC - (int)c0};
    if (p.decay_kind == 3)
      hipLaunchKernelGGL((chunk_prepare_kernel<NT, DELTA, true>), dim3(chunks, p.H), dim3(256), 0, st, p, ws, sg);
    else
      hipLaunchKernelGGL((chunk_prepare_kernel<NT, DELTA, false>), dim3(chunks, p.H), dim3(256), 0, st, p, ws, sg);
    const dim3 block(64 * (NT < 4 ? NT : 4));
    if (pairs)
      hipLaunchKernelGGL((chunk_walk_kernel<NT, DELTA, 2>), dim3(p.H, p.V / (2 * kScanCols), p.nseq), block, 0, st, p, ws, chunks, sg);
    else
      hipLaunchKernelGGL((chunk_walk_kernel<NT, DELTA, 1>), dim3(p.H, p.V / kScanCols, p.nseq), block, 0, st, p, ws, chunks, sg);
  }
  return hipGetLastError();
}

}  // namespace

// Time in us of the walk by tokens and of the chunks.  The walk: a start, then its longest chain or the work of all its column blocks, whichever
// is more (decode-sized launches, up to two rows a sequence on average, walk another kernel's chain).  The chunks: a start, the
// preparation of every (chunk, head), which costs the same however few its column blocks, and the longest chain or all column blocks.
// Fitted per key width over 1..180 sequences of 3..8192 rows of 1..1024 column blocks (each within 12 % rms); of 2784 timings the slower of
// the two is taken by more than 6 % in 58, by 10 % in 32; on average 0.4 % is lost.  Walk against chunks, H x D x V: delta rule, 16 x
// 128 x 128, one sequence of 17 rows 12.6 / 11.9, 64 rows 30 / 14, 2048 rows 962 / 147, 16 of 8 rows 27 / 24, 64 of 64 rows 372 / 165; without
// it, 17 rows 11.6 / 9.9, 64 rows 27 / 11, 64 of 64 rows 328 / 105; 2 x 128 x 128, 16 rows, decays per channel 10 / 12; few column blocks,
// 16 x 64 x 16, 64 of 32 rows 21 / 29, 128 of 24 rows, decays per channel 32 / 53; 2 x 128 x 32, 64 of 17 13 / 17; 8 x 128 x 16, 64 of 16 13 / 20.
struct ScanCost {
  double walk0, row, row_block, walk_seq, chunk0, channels, unit, chunk, chunk_block, seq_block;
};
static bool chunks_pay(const MatrixScanParams& p, int64_t rows, int64_t chunks, int64_t longest) {
  static const ScanCost kDelta[3] = {{4.7, 0.264, 0.041, 0.205, 8.7, 2.2, 0.083, 0.580, 0.120, 0.087},   // widths 32, 64, 128
                                     {4.4, 0.326, 0.058, 0.311, 9.2, 2.5, 0.109, 0.575, 0.286, 0.222},
                                     {4.9, 0.441, 0.106, 0.500, 9.6, 3.5, 0.207, 1.130, 0.300, 0.417}};
  static const ScanCost kPlain[3] = {{4.6, 0.224, 0.038, 0.229, 7.9, 1.4, 0.056, 0.260, 0.113, 0.091},
                                     {4.2, 0.288, 0.047, 0.338, 8.0, 1.9, 0.077, 0.343, 0.161, 0.205},
                                     {4.8, 0.390, 0.093, 0.513, 8.8, 2.7, 0.155, 0.707, 0.163, 0.466}};
  const ScanCost& c = (p.beta ? kDelta : kPlain)[p.D == 32 ? 0 : (p.D == 64 ? 1 : 2)];
  const double blocks = (double)p.H * (p.V / kScanCols) / 128.0, n = (double)((longest + kC - 1) / kC);
  const double walk = c.walk0 + std::max(c.row * (p.portions ? 1.0 : 1.8) * longest, (c.row_block * rows + c.walk_seq * p.nseq) * blocks);
  const bool chan = p.decay_kind == 3;
  const double prepare = c.chunk0 + (chan ? c.channels : 0.0) + c.unit * (chan ? 1.25 : 1.0) * chunks * p.H / 16;
  return walk > prepare + std::max(c.chunk * n, (c.chunk_block * chunks + c.seq_block * p.nseq) * blocks);
}

// Whether the chunks take the shape
static bool chunk_room(const MatrixScanParams& p, int64_t rows, int64_t longest) {
  auto aligned = [](const float* x, int ld) { return reinterpret_cast<uintptr_t>(x) % 16 == 0 && ld % 4 == 0; };
  if (longest <= 0 || p.nseq <= 0 || p.src_idx || p.decay_kind > 3 || (p.D != 32 && p.D != 64 && p.D != 128) ||
      p.V % kScanCols || !aligned(p.q, p.ldq) || !aligned(p.k, p.ldk) || (p.decay_kind == 3 && !aligned(p.decay, p.ldd)))
    return false;
  // value rows of a chunk lie within 31-bit offsets of its first one
  if (p.nseq > 65535 || p.H > 65535 || std::max<int64_t>(p.ldv, (int64_t)p.H * p.V) * kC * 4 > INT32_MAX || rows * p.H > kMostRows) return false;
  return (int64_t)p.nseq * p.H * unit_floats(p.D, p.beta) <= (int64_t{1} << 29);  // a chunk of each sequence: 2 GB
}

int64_t scan_chunk_floats(const MatrixScanParams& p, int rows, int64_t longest) {
  if (!chunk_room(p, rows, longest)) return 0;
  const int64_t all = (longest + kC - 1) / kC;
  if (!chunks_pay(p, std::min<int64_t>(rows, p.nseq * longest), chunk_bound(p, rows, longest, all), longest)) return 0;
  return chunk_bound(p, rows, longest, segment_span(p, rows, longest)) * p.H * unit_floats(p.D, p.beta);
}

// Without the delta rule.  Where the chunks are out of the question (other widths, unaligned rows) two levels beat one long chain;
// where they are not, only for a very long sequence of a few column blocks, whose chunks follow one another on a mostly empty chip.
// Chunks against two levels, decays per channel: 2 heads of 128 x 128, 2048 rows 84 / 84, 8192 rows 290 / 237; 4 of 64 x 64, 2048 rows
// 57 / 60, 4096 104 / 82; 4 of 32 x 32, 4096 rows 85 / 61.  One line for all decays: those per head take 81 / 101, 287 / 315; 55 / 75,
// 102 / 120; 83 / 100 (chunks of 64 took 138 and 509, 86 and 167, 121).
bool scan_two_levels(const MatrixScanParams& p, int rows, int64_t longest) {
  if (p.beta || rows < kTwoLevelRows) return false;
  if (!chunk_room(p, rows, longest)) return true;
  const int64_t from = p.D == 32 ? 4096 : 2048;
  return longest >= from && (int64_t)p.nseq * p.H * (p.V / kScanCols) <= 16;
}

}  // namespace dsse

extern "C" hipError_t dsse_scan_chunks(const dsse::MatrixScanParams* p, float* ws, int rows, int64_t longest, hipStream_t st) {
  if (p->nseq <= 0 || p->H <= 0 || rows <= 0) return hipSuccess;
  if (p->H % p->G || !dsse::scan_chunk_floats(*p, rows, longest)) return hipErrorInvalidValue;
#define DSSE_CHUNK_CASE(n)                                                            \
  case 16 * n:                                                                        \
    return p->beta ? dsse::launch_chunks<n, true>(*p, ws, rows, longest, st) : dsse::launch_chunks<n, false>(*p, ws, rows, longest, st);
  switch (p->D) {
    DSSE_CHUNK_CASE(2)
    DSSE_CHUNK_CASE(4)
    DSSE_CHUNK_CASE(8)
  }
#undef DSSE_CHUNK_CASE
  return hipErrorInvalidValue;
}
