// Paged GQA attention on MFMA for gfx950 (K5 decode and K12 prefill of SURVEY.md §2.4).
//
// KV cache layout (engine-owned, page = 32 tokens):
//   K: [blocks, Hkv, 32, 128]   one key row = 256 contiguous bytes
//   V: [blocks, Hkv, 128, 32]   transposed, tokens permuted inside the page by vperm() so the
//                               PV operand of lane group g is one 16-byte run
//
// One MFMA tile column is a (query token, q-head of the GQA group) pair: with G = Hq/Hkv heads
// per kv head, a 16-column tile holds QT = 16/G query tokens of one sequence.  Decode uses
// QT = 1 token (G columns live), prefill uses all 16 columns.  Scores are computed swapped,
// Sᵀ[key, col] = K · Qᵀ, so the softmax statistics of a column live in one lane column and
// the exponentiated scores are already the B operand of Oᵀ = Vᵀ · Pᵀ — no LDS round trip and
// no transposes inside the key loop.
//
// Work decomposition: a workgroup = QW × KWV waves.  The QW waves take consecutive query tiles
// (prefill: they share K/V lines through L1), the KWV waves split the key range and are merged
// in LDS; grid.z splits the key range into partitions of `part` keys (flash-decoding), merged
// by attn_combine_kernel.  Online softmax in base 2 with a finite initial max, so fully masked
// columns stay finite and produce zeros.
#include <cstdlib>

#include "attention_decode.h"

namespace dsse {

// One-wave decode workgroups (256+ streams) are held to 4 waves per SIMD: the folded QKV epilogue (FQ) otherwise
// raises the register peak from 127 to 159 and costs a wave per SIMD; 104 VGPRs, no spills.
// PD: KV pages in flight per wave (a register ring of PD pages, each wave's next PD-1 pages issued before the
// current one is computed).  One-wave workgroups with PD > 1 are held to 2 waves per SIMD (256 VGPRs): the
// 2048-workgroup grid they serve (256 streams x 8 kv heads) puts 2 waves on each SIMD anyway.
template <int QW, int KWV, int PD = 1, int FQG = 0>
__global__ void __launch_bounds__(64 * QW * KWV, QW * KWV == 1 ? (PD > 1 ? 2 : 4) : 1)
paged_attention_kernel(AttnParams p) {
  __shared__ __attribute__((aligned(16))) DecodeLds<QW, KWV, FQG> lds;
  decode_attention<QW, KWV, PD, FQG, false>(p, blockIdx.x, blockIdx.y, blockIdx.z, threadIdx.x >> 6, lds);
}

// Merge flash-decoding partitions: grid (num_work, hkv, QW), block 256 = (16 columns × 16 lanes),
// each thread owns 8 head dims of one column.
template <int QW>
__global__ void __launch_bounds__(256) attn_combine_kernel(AttnParams p) {
  const int item = blockIdx.x, h = blockIdx.y, qw = blockIdx.z;
  const int col = threadIdx.x >> 4, sub = threadIdx.x & 15;
  const int b = p.work_seq[item];
  const int qlen = p.q_len[b], ctx = p.ctx_len[b];
  const int G = p.group, QT = 16 / G;
  const int qi = (p.work_tile[item] * QW + qw) * QT + col / G;
  if (qi >= qlen) return;
  const int last_q = min(qlen, (p.work_tile[item] + 1) * QW * QT) - 1;
  const int kmax = ctx - qlen + last_q + 1;
  const int part = part_keys(p, kmax);
  const int np = min(p.nparts, (kmax + part - 1) / part);
  float mm = -1e30f;
  for (int z = 0; z < np; ++z) {
    const size_t base = (((size_t)item * p.hkv + h) * p.nparts + z) * QW + qw;
    mm = fmaxf(mm, p.part_ml[base * 16 + col].x);
  }
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  float ll = 0.f;
  for (int z = 0; z < np; ++z) {
    const size_t base = (((size_t)item * p.hkv + h) * p.nparts + z) * QW + qw;
    const float2 ml = p.part_ml[base * 16 + col];
    const float sc = exp2f(ml.x - mm);
    ll += ml.y * sc;
    const float4* po = reinterpret_cast<const float4*>(p.part_o + (base * 16 + col) * kD + 8 * sub);
    const float4 a = po[0], c = po[1];
    acc[0] += a.x * sc; acc[1] += a.y * sc; acc[2] += a.z * sc; acc[3] += a.w * sc;
    acc[4] += c.x * sc; acc[5] += c.y * sc; acc[6] += c.z * sc; acc[7] += c.w * sc;
  }
  const float inv = ll > 0.f ? 1.f / ll : 0.f;
  bf16x8 ov;
#pragma unroll
  for (int j = 0; j < 8; ++j) ov[j] = f2bf(acc[j] * inv);
  bf16* op = p.out + ((size_t)(p.q_start[b] + qi) * p.hq + h * G + (col % G)) * kD + 8 * sub;
  *reinterpret_cast<bf16x8*>(op) = ov;
}

template <int G>
hipError_t launch_folded(int kwv, int pd, dim3 grid, const AttnParams& p, hipStream_t st) {
  if (kwv == 8) hipLaunchKernelGGL((paged_attention_kernel<1, 8, 1, G>), grid, dim3(512), 0, st, p);
  else if (kwv == 1 && pd == 2) hipLaunchKernelGGL((paged_attention_kernel<1, 1, 2, G>), grid, dim3(64), 0, st, p);
  else if (kwv == 1) hipLaunchKernelGGL((paged_attention_kernel<1, 1, 1, G>), grid, dim3(64), 0, st, p);
  else if (kwv == 2 && pd == 2) hipLaunchKernelGGL((paged_attention_kernel<1, 2, 2, G>), grid, dim3(128), 0, st, p);
  else if (kwv == 2) hipLaunchKernelGGL((paged_attention_kernel<1, 2, 1, G>), grid, dim3(128), 0, st, p);
  else hipLaunchKernelGGL((paged_attention_kernel<1, 4, 1, G>), grid, dim3(256), 0, st, p);
  return hipGetLastError();
}

}  // namespace dsse

// the combine launch of decode partitions (nparts > 1)
extern "C" hipError_t dsse_attn_combine(int num_work, const dsse::AttnParams* p, hipStream_t st) {
  hipLaunchKernelGGL((dsse::attn_combine_kernel<1>), dim3(num_work, p->hkv, 1), dim3(256), 0, st, *p);
  return hipGetLastError();
}

// mode 0 = decode (QW = 1, KWV = 4), mode 1 = prefill (QW = 4, KWV = 1), mode 3 = decode reading q from the
// QKV GEMM's split-K slabs and writing the step's K / V (AttnParams::qkv_part).
extern "C" hipError_t dsse_paged_attention(int mode, int num_work, const dsse::AttnParams* p,
                                           hipStream_t st) {
  using namespace dsse;
  if (num_work <= 0) return hipSuccess;
  if (mode == 3) {
    // decode with the QKV epilogue folded in; GQA group 1, 2 or 4.  Every key-split wave sums its q slabs, so
    // fewer waves per workgroup than mode 0 pay off: 2 from 512 workgroups (64 streams: 4.58 vs 4.60 ms/step,
    // 8 waves 4.67-4.71; profiles/experiments_r2.md); from 2048 one wave without look-ahead beat two (9.95 vs
    // 10.20), two with a 2-page ring beat both (below)
    const dim3 grid(num_work, p->hkv, p->nparts);
    const int nwg = grid.x * grid.y * grid.z;
    // 2048+ workgroups (256 streams): one wave per (sequence, kv head), one page in flight -- with the
    // non-temporal K/V loads 9.70 / 9.71 ms/step vs 10.11 / 10.16 for 2 waves x 2 pages (the round-2 choice
    // under default-policy loads) and 10.31 for 2 waves x 1 page (profiles/r3/r3n_ab256.log); 512-2047: 2 waves
    // (128 streams 6.00-6.03 vs 6.23 with 4; 64 streams: look-ahead measured slower)
    const int kwv = p->kwv ? p->kwv : (nwg >= 2048 ? 1 : (nwg >= 512 ? 2 : 4));
    const int pd = p->pd ? p->pd : 1;
    hipError_t e;
    if (p->group == 1) e = launch_folded<1>(kwv, pd, grid, *p, st);
    else if (p->group == 2) e = launch_folded<2>(kwv, pd, grid, *p, st);
    else if (p->group == 4) e = launch_folded<4>(kwv, pd, grid, *p, st);
    else return hipErrorInvalidValue;
    if (e != hipSuccess) return e;
    if (p->nparts > 1 && !p->comb_cnt)
      hipLaunchKernelGGL((attn_combine_kernel<1>), dim3(num_work, p->hkv, 1), dim3(256), 0, st, *p);
  } else if (mode == 0) {
    // decode: p->kwv (attn_kwv in DSSE_KERNEL_CFG, read by the bindings) = waves per workgroup splitting the keys (1/2/4/8).
    // 1 / 2 / 4 waves, us, 512 keys on average (0.7 to 1.3 of it), 8 kv heads, non-temporal loads: 64 streams 122 / 28.6 / 29.6,
    // 128 streams 138 / 54.2 / 55.9, 256 streams 173 / 108 / 100; 256 streams of 128 keys 36.9 / 25.8 / 25.9.  (A next-page
    // register prefetch variant cost 2-10 % and was removed.)
    const dim3 grid(num_work, p->hkv, p->nparts);
    const unsigned nwg = grid.x * grid.y * grid.z;
    const int kwv = p->kwv ? p->kwv : (nwg >= 512 && nwg < 1536 ? 2 : 4);
    const int pd = p->pd == 2 && kwv <= 2 ? 2 : 1;  // attn_pd=2 (DSSE_KERNEL_CFG): 2-page register ring (1 / 2 waves)
    if (kwv == 8) hipLaunchKernelGGL((paged_attention_kernel<1, 8, 1>), grid, dim3(512), 0, st, *p);
    else if (kwv == 1 && pd == 2) hipLaunchKernelGGL((paged_attention_kernel<1, 1, 2>), grid, dim3(64), 0, st, *p);
    else if (kwv == 2 && pd == 2) hipLaunchKernelGGL((paged_attention_kernel<1, 2, 2>), grid, dim3(128), 0, st, *p);
    else if (kwv == 1) hipLaunchKernelGGL((paged_attention_kernel<1, 1, 1>), grid, dim3(64), 0, st, *p);
    else if (kwv == 2) hipLaunchKernelGGL((paged_attention_kernel<1, 2, 1>), grid, dim3(128), 0, st, *p);
    else hipLaunchKernelGGL((paged_attention_kernel<1, 4, 1>), grid, dim3(256), 0, st, *p);
    if (p->nparts > 1 && !p->comb_cnt)
      hipLaunchKernelGGL((attn_combine_kernel<1>), dim3(num_work, p->hkv, 1), dim3(256), 0, st, *p);
  } else {
    hipLaunchKernelGGL((paged_attention_kernel<4, 1>), dim3(num_work, p->hkv, p->nparts), dim3(256),
                       0, st, *p);
    if (p->nparts > 1)
      hipLaunchKernelGGL((attn_combine_kernel<4>), dim3(num_work, p->hkv, 4), dim3(256), 0, st, *p);
  }
  return hipGetLastError();
}

DSSE_CHECK_READER(dsse_check_attention)
