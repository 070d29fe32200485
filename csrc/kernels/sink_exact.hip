// Sink attention of prompt portions in the exact mode (fp32 keys, values and outputs; head widths up to 128, multiples of 16) on
// the fp32 matrix cores: four column tiles (hb heads of one key/value group x rt tiles of 16 query rows) per workgroup, one per
// wave, over pages staged in LDS once for all of them.
//
//   S^T[key, row] = K[key, :] . Q[row, :]     A = key rows from LDS, B = the rows' queries in registers; the k index of step
//                                             (t, i) is dim 16 t + 4 g + i on both sides, so a lane reads four steps at once
//   O^T[dim, row] += V^T[dim, key] P^T[key, row]  the score accumulators (key 4 g + i of row r) ARE the B operand of step i,
//                                             A = V[key 4 g + i][dim] from LDS
//
// All arithmetic is 32-bit as in the row kernel (sink_attention.hip); scores are summed in four chains and outputs in pieces,
// so an output's error against 64 bits is no larger: 400 rows of 16 heads of 128 2.0e-7 (row kernel 3.3e-7), 64 rows
// behind 2000 keys 3.1e-7 (5.7e-7).
//
// A page's values meet all 16 rows of a tile, with weights of zero for keys that a row does not see: later tokens, keys behind
// the window, places of the page that hold nothing yet (or what an earlier sequence left).  Where such a value is not finite the
// row would be NaN, so a wave whose outputs are not all finite makes its rows once more one by one, from the keys they see.
//
// What bounds it: a page costs a wave 2 x 64 v_mfma_f32_16x16x4_f32 at widths of 128, 4096 cycles.  The row kernel (four waves
// walk one row's keys, a load per key and value) took 371 us for 400 rows of 16 heads of 128; here 56; 1000 rows 1460
// us and 130; 8 rows of each of 16 sequences behind 50 keys 97 and 14.
#include "sink_rows.h"

namespace dsse {
namespace {

constexpr int kExactTiles = 4;  // column tiles (waves) of a workgroup

// One row by one wave
DEV void exact_row(const SinkAttnParams& p, int seq, int h, int64_t row, int pos) {
  const int lane = threadIdx.x & 63;
  float m = -INFINITY, l = 0.f, acc[2] = {0.f, 0.f};  // V <= 128
  walk_row<float>(p, seq, h, pos, p.q + (row * p.H + h) * p.D, 0, 1, m, l, acc);
  float f = 1.0f;
  if (p.sink) {
    const float sk = p.sink[h], mm = fmaxf(m, sk);
    f = expf(m - mm);
    l = l * f + expf(sk - mm);
  }
  float gate = 1.0f;
  if (p.gate && !p.gate_wide) gate = 1.0f / (1.0f + expf(-p.gate[row * p.ldg + h]));
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int d = 64 * a + lane;
    if (d >= p.V) continue;
    float o = acc[a] * f / l * gate;
    if (p.gate_wide) o *= 1.0f / (1.0f + expf(-p.gate[row * p.ldg + h * p.V + d]));
    reinterpret_cast<float*>(p.out)[row * p.ldo + h * p.V + d] = o * p.out_scale;
  }
}

// NT = V / 16; KT = D / 16 when it equals NT, else 0: read from the parameters
template <int NT, int KT>
__global__ __launch_bounds__(64 * kExactTiles) void sink_exact_kernel(SinkAttnParams p, int hb, int rt) {
  extern __shared__ __align__(16) float smem[];
  constexpr int V = 16 * NT, KMAX = KT ? KT : 8, TH = 64 * kExactTiles;
  constexpr int KC = (KMAX * 16 * kBS / 4 + TH - 1) / TH, VC = (V * kBS / 4 + TH - 1) / TH;
  const int D = KT ? 16 * KT : p.D, kt = D / 16, ldk = D + 4, ldv = V + 4;
  float* keys = smem;
  float* vals = smem + kBS * ldk;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, g = lane >> 4;
  const int seq = p.work_seq[blockIdx.y], tile = p.work_tile[blockIdx.y];
  const int ql = p.q_len[seq], row_first = tile * 16 * rt;
  if (row_first >= ql) return;  // uniform for the workgroup
  const int h_first = blockIdx.x * hb, kvh = h_first / (p.H / p.G), head = h_first + wave / rt;
  const int q0 = p.q_start[seq], pos0 = p.ctx_len[seq] - ql;
  const int row_last = row_first + 16 * rt < ql ? row_first + 16 * rt - 1 : ql - 1;
  const int hi = pos0 + row_last;
  int lo = pos0 + row_first - p.window + 1;
  lo = lo > 0 ? lo : 0;
  const int pg_lo = lo / kBS;
  int kept_pages = 0;  // whole pages of kept keys before the window's first page
  if (p.keep_first > 0) {
    kept_pages = (p.keep_first + kBS - 1) / kBS;
    kept_pages = kept_pages < pg_lo ? kept_pages : pg_lo;
  }
  const int walk = kept_pages + hi / kBS - pg_lo + 1;
  const int* bt = p.block_tables + (int64_t)seq * p.max_blocks;
  auto page_at = [&](int it) { return it < kept_pages ? it : pg_lo + it - kept_pages; };
  const int tile_first = row_first + 16 * (wave % rt), off = tile_first + r;
  const bool on = off < ql;
  const int64_t row = q0 + (on ? off : 0);
  const int pos = on ? pos0 + off : -1;
  const int tile_hi = pos0 + (tile_first + 15 < ql ? tile_first + 15 : ql - 1);
  f32x4 qf[KMAX];
#pragma unroll
  for (int t = 0; t < KMAX; ++t) {
    qf[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    if ((KT || t < kt) && on) qf[t] = ld_global<f32x4>(p.q + (row * p.H + head) * D + 16 * t + 4 * g);
  }
  // staging: 16-byte pieces of the page's key and value rows; the next page is in registers while this one is used
  const float* kc = reinterpret_cast<const float*>(p.k);
  const float* vc = reinterpret_cast<const float*>(p.v);
  f32x4 nk[KC], nv[VC];
  auto request = [&](int it) {  // pages past the walk read its last one again
    int blk = bt[page_at(it < walk ? it : walk - 1)];
    blk = (unsigned)blk < (unsigned)p.num_blocks ? blk : 0;
    const float* kp = kc + ((int64_t)blk * kBS * p.G + kvh) * D;
    const float* vp = vc + ((int64_t)blk * kBS * p.G + kvh) * V;
#pragma unroll
    for (int i = 0; i < KC; ++i) {
      const int idx = tid + TH * i, kr = idx / (D / 4), c = idx - kr * (D / 4);
      nk[i] = ld_global<f32x4>(kp + (kr < kBS ? (int64_t)kr * p.G * D + 4 * c : 0));
    }
#pragma unroll
    for (int i = 0; i < VC; ++i) {
      const int idx = tid + TH * i, vr = idx / (V / 4), c = idx - vr * (V / 4);
      nv[i] = ld_global<f32x4>(vp + (vr < kBS ? (int64_t)vr * p.G * V + 4 * c : 0));
    }
  };
  auto stash = [&]() {
#pragma unroll
    for (int i = 0; i < KC; ++i) {
      const int idx = tid + TH * i, kr = idx / (D / 4), c = idx - kr * (D / 4);
      if (kr < kBS) *reinterpret_cast<f32x4*>(&keys[kr * ldk + 4 * c]) = nk[i];
    }
#pragma unroll
    for (int i = 0; i < VC; ++i) {
      const int idx = tid + TH * i, vr = idx / (V / 4), c = idx - vr * (V / 4);
      if (vr < kBS) *reinterpret_cast<f32x4*>(&vals[vr * ldv + 4 * c]) = nv[i];
    }
  };
  // outputs: sums over kSumPages pages, joined in `all`: one chain over a long walk would round more than the row kernel's
  // four waves with a part of the keys each.  The groups are pages of the sequence, not of the walk, and a page that a row does
  // not see adds exactly nothing to it: a row's result is the same however its prompt was cut into portions.
  constexpr int kSumPages = 4;
  int group = -1;
  f32x4 O[NT], all[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) O[n] = all[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  const float* rel = p.rel ? p.rel + (int64_t)head * p.rel_len : nullptr;
  request(0);
  for (int it = 0; it < walk; ++it) {
    const int pg = page_at(it);
    if (it) lds_barrier();  // every wave is done with the page before
    stash();
    lds_barrier();
    request(it + 1);
    if (pg * kBS > tile_hi) continue;  // uniform for the wave: none of its rows sees this page
    float w[8];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4 s[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) s[q] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < KMAX; ++t)
        if (KT || t < kt) {
          const f32x4 k4 = *reinterpret_cast<const f32x4*>(&keys[(16 * h + r) * ldk + 16 * t + 4 * g]);
#pragma unroll
          for (int i = 0; i < 4; ++i) s[i] = mfma16x16x4(k4[i], qf[t][i], s[i]);
        }
      const f32x4 sum = (s[0] + s[1]) + (s[2] + s[3]);
#pragma unroll
      for (int i = 0; i < 4; ++i) w[4 * h + i] = sum[i] * p.scale;
    }
    if (p.softcap > 0.f)
#pragma unroll
      for (int i = 0; i < 8; ++i) w[i] = p.softcap * tanhf(w[i] / p.softcap);
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int key = pg * kBS + 16 * (i >> 2) + 4 * g + (i & 3), dist = pos - key;
      const bool seen = dist >= 0 && (dist < p.window || key < p.keep_first);
      if (rel && seen) w[i] += rel[dist < p.rel_len ? dist : p.rel_len - 1];
      w[i] = seen ? w[i] : -INFINITY;
      mx = fmaxf(mx, w[i]);
    }
    const float mn = fmaxf(m, rows4_max(mx));
    const float at = mn == -INFINITY ? 0.0f : mn;  // nothing seen yet: exp(-inf - 0) is 0
    const float corr = expf(m - at);
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      w[i] = expf(w[i] - at);
      ps += w[i];
    }
    l = l * corr + rows4_sum(ps);
    m = mn;
    if (!__all(corr == 1.0f)) {
#pragma unroll
      for (int n = 0; n < NT; ++n) O[n] = O[n] * corr, all[n] = all[n] * corr;
    }
    if (pg / kSumPages != group) {  // uniform
      group = pg / kSumPages;
#pragma unroll
      for (int n = 0; n < NT; ++n) all[n] += O[n], O[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int n = 0; n < NT; ++n)
          O[n] = mfma16x16x4(vals[(16 * h + 4 * g + i) * ldv + 16 * n + r], w[4 * h + i], O[n]);
  }
  float odd = 0.0f;  // NaN once an output is not finite
  if (on) {
    float den = l, f = 1.0f;
    if (p.sink) {
      const float sk = p.sink[head], mm = fmaxf(m, sk);
      f = expf(m - mm);
      den = l * f + expf(sk - mm);
    }
    float gate = 1.0f;
    if (p.gate && !p.gate_wide) gate = 1.0f / (1.0f + expf(-p.gate[row * p.ldg + head]));
    const float* gw = p.gate_wide ? p.gate + row * p.ldg + head * V + 4 * g : nullptr;
    float* out = reinterpret_cast<float*>(p.out) + row * p.ldo + head * V + 4 * g;
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float o = (all[n][i] + O[n][i]) * f / den * gate;
        if (gw) o *= 1.0f / (1.0f + expf(-gw[16 * n + i]));
        out[16 * n + i] = o * p.out_scale;
        odd += o * 0.0f;
      }
  }
  if (!__any(odd != 0.0f)) return;
  for (int i = 0; i < 16 && tile_first + i < ql; ++i) exact_row(p, seq, head, q0 + tile_first + i, pos0 + tile_first + i);
}

template <int NT>
void launch_exact(dim3 grid, size_t lds, const SinkAttnParams& p, int hb, int rt, hipStream_t st) {
  if (p.D == p.V) hipLaunchKernelGGL((sink_exact_kernel<NT, NT>), grid, dim3(64 * kExactTiles), lds, st, p, hb, rt);
  else hipLaunchKernelGGL((sink_exact_kernel<NT, 0>), grid, dim3(64 * kExactTiles), lds, st, p, hb, rt);
}

}  // namespace

bool sink_exact_ok(const SinkAttnParams& p, int64_t num_work) {
  auto aligned = [](const void* x) { return reinterpret_cast<uintptr_t>(x) % 16 == 0; };
  const int rt = p.qt / 16;
  return p.f32 && p.qt % 16 == 0 && (rt == 1 || rt == 2 || rt == 4) && p.D % 16 == 0 && p.V % 16 == 0 && p.D <= 128 &&
         p.V <= 128 && !p.out_rope && p.H % p.G == 0 && (p.H / p.G) % (kExactTiles / rt) == 0 && num_work <= 65535 &&
         aligned(p.q) && aligned(p.k) && aligned(p.v);
}

}  // namespace dsse

extern "C" hipError_t dsse_sink_exact(int num_work, const dsse::SinkAttnParams* p, hipStream_t st) {
  if (num_work <= 0 || p->H <= 0) return hipSuccess;
  if (!dsse::sink_exact_ok(*p, num_work)) return hipErrorInvalidValue;
  const int rt = p->qt / 16, hb = dsse::kExactTiles / rt;
  const dim3 grid(p->H / hb, num_work);
  const size_t lds = dsse::kBS * (size_t)(p->D + 4 + p->V + 4) * sizeof(float);
  switch (p->V / 16) {
#define DSSE_EXACT_CASE(n) case n: dsse::launch_exact<n>(grid, lds, *p, hb, rt, st); break;
    DSSE_EXACT_CASE(1) DSSE_EXACT_CASE(2) DSSE_EXACT_CASE(3) DSSE_EXACT_CASE(4) DSSE_EXACT_CASE(5) DSSE_EXACT_CASE(6)
    DSSE_EXACT_CASE(7) DSSE_EXACT_CASE(8)
#undef DSSE_EXACT_CASE
  }
  return hipGetLastError();
}
