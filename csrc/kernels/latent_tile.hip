// Latent attention of prompt portions in the folded form (latent_attention.hip), 128 query columns per workgroup (bf16).
//
// What bounds it: LDS traffic beside the matrix cores.  A column is a (row, head) pair; the one-wave form walks a page of
// keys and values for 16 of them (69 KB read per 1.1 MFLOP at rank 512); here eight waves share every page, staged in LDS
// once for eight column tiles:
//
//   scores   wave w owns column tile w: its 16 query vectors stay in registers as MFMA operands, the page's keys come from
//            LDS; online softmax in fp32, the weights go to LDS as bf16 operands of the second product, the factor of the
//            sums so far beside them;
//   sums     wave w owns the value dimensions [w rk / 8, (w + 1) rk / 8) of ALL 128 columns: every value fragment is read
//            from LDS by one wave only, and eight products share it.
//
// One barrier per page: step i makes the scores of page i and the sums of page i - 1, while the keys of page i + 1 and the
// values of page i are on their way into the other halves of their double buffers by LDS-DMA (a whole step in flight before
// the wait that ends the step).  Key rows (2 D bytes, D a multiple of 64) are stored with the 16-byte pieces of every
// 128-byte group swizzled by (row >> 1) & 5, transposed value rows (four pieces) by -(row >> 2) & 3, both on the source
// address: fragment reads are free of bank conflicts.
//
// Measured (one MI355X, against the one-wave form): 32 heads, rank 512, prompts of 1932 + 1068 tokens 1303 -> 316 us (537
// TFLOP/s), 4096 tokens 4178 -> 756 us (773 TFLOP/s); 16 heads, 1024 tokens 267 -> 101 us; rank 128, 2000 tokens 243 -> 94 us.
// Filling the page's 69 KB takes a CU longer than its products (about 1.5 us against 1), which is what is left.
#include "api_layers.h"
#include "lds_dma.h"

namespace dsse {
namespace {
namespace lt {

DEV int value_swizzle(int row) { return -(row >> 2) & 3; }

constexpr int kWaves = 8;
constexpr int kRot = 64;
constexpr float kLog2e = 1.4426950408889634f;

constexpr size_t lds_bytes(int rk) {
  return 2 * (size_t)kBS * (rk + kRot) * 2 + 2 * (size_t)rk * kBS * 2 + 2 * kWaves * 1024 + 2 * kWaves * 16 * 4;
}

}  // namespace lt

// NT: rk / 16 value tiles; the rotated part is 64 wide
template <int NT>
__global__ void __launch_bounds__(512, 2)
latent_tile_kernel(LatentAttnParams p, const bf16* __restrict__ vt, int rt, int hp) {
  using namespace lt;
  constexpr int rk = 16 * NT, D = rk + kRot, KS = D / 32, NW = NT / kWaves;  // k-steps of 32 per key, value tiles per wave
  constexpr int kKey = kBS * D * 2;                                // bytes of a page's keys
  constexpr int kVal = rk * kBS * 2;                               // bytes of a page's values
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  char* const keys = smem;                                     // two pages
  char* const vals = smem + 2 * kKey;                          // two pages
  char* const wts = vals + 2 * kVal;                           // [2][column tile][1 KB]
  float* const fac = reinterpret_cast<float*>(wts + 2 * kWaves * 1024);  // [2][column tile][16]
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const int seq = p.work_seq[blockIdx.x], tile = p.work_tile[blockIdx.x];
  const int ql = p.q_len[seq];
  if (tile * rt >= ql) return;  // uniform for the workgroup
  const int q0 = p.q_start[seq], pos0 = p.ctx_len[seq] - ql;
  // this lane's column, in column tile w
  const int c_off = tile * rt + r / hp, c_head = (blockIdx.y * kWaves + w) * hp + r % hp;
  const bool c_ok = c_off < ql && c_head < p.H;
  const int c_pos = c_ok ? pos0 + c_off : -1;
  const int64_t c_row = q0 + (c_ok ? c_off : 0);
  // the page walk of the workgroup's rows
  const int row_first = pos0 + tile * rt, row_last = pos0 + (tile * rt + rt < ql ? tile * rt + rt : ql) - 1;
  int lo = row_first - p.window + 1;
  lo = lo > 0 ? lo : 0;
  const int pg0 = lo / kBS, n = row_last / kBS - pg0 + 1;
  const int* bt = p.block_tables + (int64_t)seq * p.max_blocks;
  auto ids_from = [&](int i0) {
    const int b = i0 + lane < n ? bt[pg0 + i0 + lane] : 0;
    return (unsigned)b < (unsigned)p.num_blocks ? b : 0;  // a stale table entry never leaves the cache
  };
  int kid = ids_from(0), vid = kid;  // 64 page ids each, of the keys' and of the values' chunk of the walk

  // DMA pieces: keys 32 rows x D / 8 pieces, values rk rows x 4 pieces, 64 pieces per instruction
  constexpr int KI = (kKey / 1024 + kWaves - 1) / kWaves, VI = rk * 4 / 64 / kWaves;
  uint32_t k_vo[KI], v_vo[VI];
#pragma unroll
  for (int i = 0; i < KI; ++i) {
    const int piece = (i * kWaves + w) * 64 + lane, row = piece / (D / 8), slot = piece - row * (D / 8);
    k_vo[i] = (uint32_t)(row * D * 2 + (((slot & ~7) | ((slot & 7) ^ piece_swizzle(row))) << 4));
  }
#pragma unroll
  for (int i = 0; i < VI; ++i) {
    const int piece = (i * kWaves + w) * 64 + lane, row = piece >> 2;
    v_vo[i] = (uint32_t)(row * kBS * 2 + (((piece & 3) ^ value_swizzle(row & 15)) << 4));
  }
  auto issue_keys = [&](int i) {
    if ((i & 63) == 0 && i > 0) kid = ids_from(i);
    const int blk = __builtin_amdgcn_readlane(kid, i & 63);
    const __amdgpu_buffer_rsrc_t src = make_rsrc(reinterpret_cast<const char*>(p.cache) + (int64_t)blk * kKey, (uint32_t)kKey);
    char* dst = keys + (i & 1) * kKey;
#pragma unroll
    for (int j = 0; j < KI; ++j)
      if ((j + 1) * kWaves * 1024 <= kKey || (j * kWaves + w) * 1024 < kKey)  // uniform
        lds_dma(src, dst + (j * kWaves + w) * 1024, k_vo[j]);
  };
  auto issue_vals = [&](int i) {
    if ((i & 63) == 0 && i > 0) vid = ids_from(i);
    const int blk = __builtin_amdgcn_readlane(vid, i & 63);
    const __amdgpu_buffer_rsrc_t src = make_rsrc(vt + (int64_t)blk * rk * kBS, (uint32_t)kVal);
    char* dst = vals + (i & 1) * kVal;
#pragma unroll
    for (int j = 0; j < VI; ++j) lds_dma(src, dst + (j * kWaves + w) * 1024, v_vo[j]);
  };
  issue_keys(0);

  // the column's query vector [q_abs | rot(q)] as operands: k-step u = 2 q + s holds elements 64 q + 16 g + 8 s ..
  bf16x8 qf[KS];
  {
    // a column that does not exist reads its first row's: it is masked below and never stored
    const int64_t at = c_row * p.H + (c_ok ? c_head : 0);
    const float* qa = p.q_abs + at * rk;
#pragma unroll
    for (int u = 0; u < NT / 2; ++u) {
      const int d = 64 * (u >> 1) + 16 * g + 8 * (u & 1);
      const f32x4 a = ld_global<f32x4>(qa + d), b = ld_global<f32x4>(qa + d + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) qf[u][j] = (bf16)a[j], qf[u][4 + j] = (bf16)b[j];
    }
    const bf16* qr = reinterpret_cast<const bf16*>(p.q) + at * (p.dn + kRot) + p.dn;
    const int pp = c_pos < 0 ? 0 : (c_pos >= p.rope_len ? p.rope_len - 1 : c_pos);
    const float2* cs = p.rope + (int64_t)pp * (kRot / 2);
#pragma unroll
    for (int u = NT / 2; u < KS; ++u) {
      const int d = 16 * g + 8 * (u & 1);
#pragma unroll
      for (int j = 0; j < 8; j += 2) {
        const float a = (float)qr[d + j], b = (float)qr[d + j + 1];
        const float2 t = cs[(d + j) / 2];
        qf[u][j] = (bf16)(a * t.x - b * t.y);
        qf[u][j + 1] = (bf16)(b * t.x + a * t.y);
      }
    }
  }
  int k_rd[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) k_rd[s] = r * D * 2 + (((2 * g + s) ^ piece_swizzle(r)) << 4);
  const int v_rd = (w * NW * 16 + r) * kBS * 2 + ((g ^ value_swizzle(r)) << 4);

  f32x4 O[NW][kWaves];  // [value tile][column tile]
#pragma unroll
  for (int t = 0; t < NW; ++t)
#pragma unroll
    for (int c = 0; c < kWaves; ++c) O[t][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  const float scale2 = p.scale * kLog2e;

  auto scores = [&](int i) {
    const char* kb = keys + (i & 1) * kKey;
    f32x4 s0 = f32x4{0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      const bf16x8 k0 = *reinterpret_cast<const bf16x8*>(kb + k_rd[u & 1] + 128 * (u >> 1));
      const bf16x8 k1 = *reinterpret_cast<const bf16x8*>(kb + k_rd[u & 1] + 128 * (u >> 1) + 16 * D * 2);
      s0 = mfma16x16x32(k0, qf[u], s0);
      s1 = mfma16x16x32(k1, qf[u], s1);
    }
    // lane (r, g): column r, keys 4 g + j (s0) and 16 + 4 g + j (s1) of the page
    const int key0 = (pg0 + i) * kBS;
    float sv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) sv[j] = (j < 4 ? s0[j] : s1[j - 4]) * scale2;
    if (!(key0 + kBS - 1 <= row_first && row_last - key0 < p.window && __all(c_ok))) {  // some key is hidden from some column
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int key = key0 + (j < 4 ? 4 * g + j : 16 + 4 * g + (j - 4));
        sv[j] = c_ok && key <= c_pos && c_pos - key < p.window ? sv[j] : -INFINITY;
      }
    }
    float mx = sv[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) mx = fmaxf(mx, sv[j]);
    const float mn = fmaxf(m, rows4_max(mx));
    const float at = mn == -INFINITY ? 0.0f : mn;  // nothing seen yet: exp2(-inf - 0) is 0
    const float corr = __builtin_amdgcn_exp2f(m - at);
    bf16x8 pf;
    float ps = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float e = __builtin_amdgcn_exp2f(sv[j] - at);
      ps += e;
      pf[j] = (bf16)e;
    }
    l = l * corr + rows4_sum(ps);
    m = mn;
    *reinterpret_cast<bf16x8*>(wts + ((i & 1) * kWaves + w) * 1024 + lane * 16) = pf;
    if (g == 0) fac[((i & 1) * kWaves + w) * 16 + r] = corr;
  };
  auto sums = [&](int i) {
    const char* vb = vals + (i & 1) * kVal;
    bf16x8 vf[NW];
#pragma unroll
    for (int t = 0; t < NW; ++t) vf[t] = *reinterpret_cast<const bf16x8*>(vb + v_rd + t * 16 * kBS * 2);
#pragma unroll
    for (int c = 0; c < kWaves; ++c) {
      const bf16x8 pf = *reinterpret_cast<const bf16x8*>(wts + ((i & 1) * kWaves + c) * 1024 + lane * 16);
      const float corr = fac[((i & 1) * kWaves + c) * 16 + r];
      if (!__all(corr == 1.0f)) {  // a maximum moved
#pragma unroll
        for (int t = 0; t < NW; ++t)
#pragma unroll
          for (int j = 0; j < 4; ++j) O[t][c][j] *= corr;
      }
#pragma unroll
      for (int t = 0; t < NW; ++t) O[t][c] = mfma16x16x32(vf[t], pf, O[t][c]);
    }
  };
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  for (int i = 0; i <= n; ++i) {
    if (i + 1 < n) issue_keys(i + 1);
    if (i < n) {
      issue_vals(i);
      scores(i);
    }
    if (i > 0) sums(i - 1);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
  // one over every column's sum, through LDS to the waves that hold its value dimensions
  if (g == 0) fac[w * 16 + r] = l > 0.f ? 1.0f / l : 0.0f;
  lds_barrier();
#pragma unroll
  for (int c = 0; c < kWaves; ++c) {
    const int off = tile * rt + r / hp, head = (blockIdx.y * kWaves + c) * hp + r % hp;
    if (off >= ql || head >= p.H) continue;
    const float inv = fac[c * 16 + r];
    bf16* out = reinterpret_cast<bf16*>(p.out) + ((int64_t)(q0 + off) * p.H + head) * rk + w * NW * 16 + 4 * g;
#pragma unroll
    for (int t = 0; t < NW; ++t) {
      bf16x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = (bf16)(O[t][c][j] * inv);
      *reinterpret_cast<bf16x4*>(out + 16 * t) = v;
    }
  }
}

template <int NT>
hipError_t launch_latent_tile(int num_work, const LatentAttnParams& p, const bf16* vt, int rt, int hp, hipStream_t st) {
  constexpr size_t lds = lt::lds_bytes(16 * NT);
  static bool attr_set = false;
  if (!attr_set) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&latent_tile_kernel<NT>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    attr_set = true;
  }
  const int gy = (p.H + hp - 1) / hp;
  hipLaunchKernelGGL(latent_tile_kernel<NT>, dim3(num_work, (gy + lt::kWaves - 1) / lt::kWaves), dim3(512), lds, st, p, vt, rt,
                     hp);
  return hipGetLastError();
}

}  // namespace
}  // namespace dsse

// rt rows x hp heads = 16 columns per tile, tiles of eight: the heads' tiles of the same rows
extern "C" hipError_t dsse_latent_tile(int num_work, const dsse::LatentAttnParams* p, const void* vt, int rt, int hp,
                                       hipStream_t st) {
  if (num_work <= 0) return hipSuccess;
  if (p->f32 || rt * hp != 16 || p->dr != dsse::lt::kRot || p->nparts > 1) return hipErrorInvalidValue;
  const bf16* v = reinterpret_cast<const bf16*>(vt);
  switch (p->rk) {
    case 128: return dsse::launch_latent_tile<8>(num_work, *p, v, rt, hp, st);
    case 256: return dsse::launch_latent_tile<16>(num_work, *p, v, rt, hp, st);
    case 512: return dsse::launch_latent_tile<32>(num_work, *p, v, rt, hp, st);
  }
  return hipErrorInvalidValue;
}
