// One wave's walk of a query row's keys, shared by the row kernel (sink_attention.hip) and by the rows that the exact mode's
// shared-page form hands back (sink_exact.hip): 64 keys at a time, one per lane for the scores, then one output coordinate per
// lane and 64 broadcast weights for the values.  Keys that the row does not see are not read.
#pragma once
#include "api_mixers.h"

namespace dsse {
namespace {

// query (fp32, LDS or global) . key row (global): 16-byte loads when the row width allows
DEV float dot_row(const float* q, const bf16* k, int D) {
  float s = 0.f;
  int d = 0;
  if (D % 8 == 0) {
    for (; d < D; d += 8) {
      const bf16x8 kv = *reinterpret_cast<const bf16x8*>(k + d);
#pragma unroll
      for (int e = 0; e < 8; ++e) s += q[d + e] * (float)kv[e];
    }
  }
  for (; d < D; ++d) s += q[d] * (float)k[d];
  return s;
}
DEV float dot_row(const float* q, const float* k, int D) {
  float s = 0.f;
  int d = 0;
  if (D % 4 == 0) {
    for (; d < D; d += 4) {
      const f32x4 kv = *reinterpret_cast<const f32x4*>(k + d);
#pragma unroll
      for (int e = 0; e < 4; ++e) s += q[d + e] * kv[e];
    }
  }
  for (; d < D; ++d) s += q[d] * k[d];
  return s;
}

// The keys 64 c .. of c = first, first + step, ..: running maximum m and sum l, sums acc of output coordinates 64 a + lane
template <typename T, int ACCS>
DEV void walk_row(const SinkAttnParams& p, int seq, int h, int pos, const float* q, int first, int step, float& m, float& l,
                  float (&acc)[ACCS]) {
  const int lane = threadIdx.x & 63, D = p.D, V = p.V, g = h / (p.H / p.G);
  const int lo = pos - p.window + 1 > 0 ? pos - p.window + 1 : 0;
  const int kept = p.keep_first < lo ? p.keep_first : lo;  // keys 0 .. kept - 1 are walked ahead of the window's
  const int nkeys = kept + pos - lo + 1;
  const int last_rel = p.rel_len - 1;
  const float* rel = p.rel ? p.rel + (int64_t)h * p.rel_len : nullptr;
  const int* bt = p.block_tables + (int64_t)seq * p.max_blocks;
  const T* kc = reinterpret_cast<const T*>(p.k);
  const T* vc = reinterpret_cast<const T*>(p.v);
  for (int c = first; c * 64 < nkeys; c += step) {
    const int jj = c * 64 + lane;
    const bool on = jj < nkeys;
    const int j0 = on ? jj : 0;
    const int j = j0 < kept ? j0 : lo + j0 - kept;
    int page = bt[j / kBS];
    page = (unsigned)page < (unsigned)p.num_blocks ? page : 0;
    const int krow = (page * kBS + j % kBS) * p.G + g;
    const float s_dot = dot_row(q, kc + (int64_t)krow * D, D);
    float s = s_dot * p.scale;
    if (p.softcap > 0.f) s = p.softcap * tanhf(s / p.softcap);
    if (rel) s += rel[pos - j < last_rel ? pos - j : last_rel];
    s = on ? s : -INFINITY;
    const float m_new = fmaxf(m, wave_max(s));  // finite: the piece holds at least one key
    const float w = on ? expf(s - m_new) : 0.f;
    const float f = expf(m - m_new);            // 0 when m was -inf
    l = l * f + wave_sum(w);
    m = m_new;
#pragma unroll
    for (int a = 0; a < ACCS; ++a) acc[a] *= f;
    const int cnt = nkeys - c * 64 < 64 ? nkeys - c * 64 : 64;
    for (int t = 0; t < cnt; ++t) {
      const float wt = __shfl(w, t);
      const int vrow = __shfl(krow, t);
      const T* vp = vc + (int64_t)vrow * V;
#pragma unroll
      for (int a = 0; a < ACCS; ++a)
        if (a * 64 + lane < V) acc[a] += wt * (float)vp[a * 64 + lane];
    }
  }
}

}  // namespace
}  // namespace dsse
