// Flash prefill attention on MFMA for gfx950 (K12 of SURVEY.md §2.4): causal, GQA, paged KV,
// chunked prefill (queries = the last q_len positions of a ctx_len context).
//
// Measured need (profiles/ttft_r1.md): the decode-derived kernel in attention.hip (no LDS, K/V read
// straight from the paged cache by every wave) ran an 8k-token causal prefill at ~157 TFLOP/s,
// 56 % of the TTFT.  This kernel is the classic LDS-staged flash structure, laid out for CDNA4:
//
//   workgroup  = one KV head x 64 query tokens; 2G waves (G = Hq/Hkv q heads x 2 halves of 32
//                queries), so every K/V byte staged in LDS feeds 2G waves (GQA reuse in LDS);
//   key loop   = 64 keys (two 32-token pages) per block, a 4-block LDS ring (4 x 32 KiB) filled by LDS-DMA
//                two blocks ahead;
//   scores     = Sᵀ = K·Qᵀ (keys on MFMA rows, queries on lanes): a query's softmax statistics live
//                in one lane column, and the exponentiated scores are already the B operand of
//                Oᵀ = Vᵀ·Pᵀ — the V cache stores each page transposed with the token permutation
//                vperm(), so lane group g's 8 keys {4g..4g+3, 16+4g..16+4g+3} are one 16-byte run;
//   LDS images = K [64 keys][256 B] with the XOR-swizzled 16-byte chunks of gemm_xlds, a page's Vᵀ [128 d][64 B] with
//                chunk ^= (-(d >> 2)) & 3: both read with conflict-free ds_read_b128, both filled by instructions that read
//                one contiguous KiB of a page;
//   softmax    = online, base 2, masked scores contribute exactly 0 (fully masked columns stay 0).
//
// Schedule: two phases per key block with a barrier before each, the products PV(j - 1) and QKᵀ(j) | softmax(j), and the two
// query halves staggered by one barrier.  Waves w and w + 4 share a SIMD (G = 4: the same head, the two query halves), so one
// runs its 64 MFMAs (1075 clocks) while the other runs its softmax (32 exponentials per lane and what goes with them: some 1100
// clocks beside MFMAs).  Vᵀ fragments are read in the softmax phase, K fragments under the PV products; the running max is off the
// critical chain (the softmax's comment).  One MI355X, 32 heads over 8, us: 8192 tokens 594 (925 TFLOP/s) with QKᵀ | softmax + PV as the
// phases, a block's maximum before its exponentials and Vᵀ read right before its products, 467 (1175) now; 6000 377 / 293, 4096 184 / 145, 2048
// 82 / 62, 1024 44 / 34, 512 27 / 21, 300 18.6 / 15.1, four of 2048 193 / 156; 16 heads over 8, 8192 tokens 681 / 365.  Left out in a copy, the
// LDS reads are 85 us of the 465, the DMA 6, the softmax 46; reads of a block further ahead, DMA in other places and other wave
// priorities 0 to 4 % slower.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "attention_flash.h"

namespace dsse {
using namespace flash;

template <int G, int HG, bool STAMP>
__global__ void __launch_bounds__(128 * HG) flash_prefill_kernel(AttnParams p, unsigned* stamps) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  flash_prefill<G, HG, STAMP>(p, stamps, blockIdx.x, smem);
}

// Merge the key ranges of split tiles (flash prefill key split): grid (ncomb, Hkv, G), 256 threads = 64 query rows x 4
// quarters of the head dimension; each thread reads its 32 dims of every slot once (the slots' O is relative to their
// own running max m, in log2 units: weight 2^(m - M)).
__global__ void __launch_bounds__(256) flash_combine_kernel(AttnParams p) {
  const int c = blockIdx.x, h = blockIdx.y, hl = blockIdx.z, G = p.group;
  const int qrow = threadIdx.x >> 2, dq = threadIdx.x & 3;
  const int b = p.comb[4 * c], tile = p.comb[4 * c + 1], s0 = p.comb[4 * c + 2], ns = p.comb[4 * c + 3];
  const int qi = tile * kBQ + qrow;
  if (qi >= p.q_len[b]) return;
  float mm = -1e30f;
  for (int k = 0; k < ns; ++k) mm = fmaxf(mm, p.part_ml[((size_t)((s0 + k) * p.hkv + h) * G + hl) * kBQ + qrow].x);
  f32x4 acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float ll = 0.f;
  for (int k = 0; k < ns; ++k) {
    const size_t row = ((size_t)((s0 + k) * p.hkv + h) * G + hl) * kBQ + qrow;
    const float2 ml = p.part_ml[row];
    const float wgt = __builtin_amdgcn_exp2f(ml.x - mm);
    ll += ml.y * wgt;
    const f32x4* po = reinterpret_cast<const f32x4*>(p.part_o + row * kD + 32 * dq);
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] += po[j] * wgt;
  }
  const float inv = ll > 0.f ? 1.f / ll : 0.f;
  bf16* op = p.out + ((size_t)(p.q_start[b] + qi) * p.hq + h * G + hl) * kD + 32 * dq;
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    bf16x8 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = f2bf(acc[j][i] * inv);
      v[4 + i] = f2bf(acc[j + 1][i] * inv);
    }
    *reinterpret_cast<bf16x8*>(op + 4 * j) = v;
  }
}

}  // namespace dsse

namespace {
template <int G, int HG, bool STAMP>
hipError_t launch_flash(int num_work, const dsse::AttnParams* p, hipStream_t st, unsigned* stamps) {
  using namespace dsse;
  constexpr int lds = kRing * kStage + (STAMP ? 2 * HG * kStampsPerBlock * kStampBlocks * 4 : 0);
  static bool attr_set = false;
  if (!attr_set) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&flash_prefill_kernel<G, HG, STAMP>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    attr_set = true;
  }
  hipLaunchKernelGGL((flash_prefill_kernel<G, HG, STAMP>), dim3(num_work * p->hkv * (G / HG)), dim3(128 * HG), lds, st,
                     *p, stamps);
  return hipGetLastError();
}

// DSSE_FLASH_STAMPS=<file>: the diagnostic build of the kernel; after each call the stamps of the first kStampWgs
// workgroups ([wg][wave][block][6] u32 shader-clock values) overwrite <file> (synchronises the device: never set it in
// serving)
hipError_t launch_stamped(int num_work, const dsse::AttnParams* p, hipStream_t st, const char* path) {
  using namespace dsse;
  if (p->group != 4) return hipErrorInvalidValue;
  const size_t n = (size_t)kStampWgs * 8 * kStampsPerBlock * kStampBlocks;
  static unsigned* buf = nullptr;
  if (buf == nullptr && hipMalloc(&buf, n * sizeof(unsigned)) != hipSuccess) return hipErrorOutOfMemory;
  (void)hipMemsetAsync(buf, 0, n * sizeof(unsigned), st);
  hipError_t e = launch_flash<4, 4, true>(num_work, p, st, buf);
  if (e != hipSuccess) return e;
  std::vector<unsigned> host(n);
  if ((e = hipStreamSynchronize(st)) != hipSuccess) return e;
  if ((e = hipMemcpy(host.data(), buf, n * sizeof(unsigned), hipMemcpyDeviceToHost)) != hipSuccess) return e;
  if (FILE* f = fopen(path, "wb")) {
    fwrite(host.data(), sizeof(unsigned), n, f);
    fclose(f);
  }
  return hipSuccess;
}
}  // namespace

// Work items: (sequence, 64-query tile) pairs; grid = num_work x Hkv workgroups, kv head fastest.  Requires
// G = Hq/Hkv in {1, 2, 4}.  (Splitting a kv head's q heads over G workgroups for short prompts -- 256 workgroups of
// 2 waves instead of 64 of 8 at 512 tokens -- measured 38.9 vs 28.8 us and was dropped; profiles/r4.)
// p->kwv (mode 2): q heads per workgroup (flash_hg in DSSE_KERNEL_CFG), 0 = the whole group.  Round 6 re-measured the
// split for a long prompt on ONE kv head (a TP = 8 rank: 4 q heads, 128 workgroups of 8 waves at 8k tokens, half the
// CUs idle): 2 q heads per workgroup 323 us, 1 q head 383 us, the whole group 264 us at T = 8192 (85 / 94 / 72 us
// at 2048; profiles/r6/flash_tp8_r6.log) -- every split stages the same K / V once more per workgroup, and the LDS
// fill, not the idle CUs, sets the time.
extern "C" hipError_t dsse_flash_prefill(int num_work, const dsse::AttnParams* p, hipStream_t st) {
  if (num_work <= 0) return hipSuccess;
  static const char* stamps = getenv("DSSE_FLASH_STAMPS");
  if (stamps != nullptr && stamps[0] != '\0') return launch_stamped(num_work, p, st, stamps);
  int hg = p->kwv;
  if (hg == 0 || p->work_kb) hg = p->group;  // the key split writes partial slots per whole group
  hipError_t e;
  switch (p->group) {
    case 1: e = launch_flash<1, 1, false>(num_work, p, st, nullptr); break;
    case 2: e = hg == 1 ? launch_flash<2, 1, false>(num_work, p, st, nullptr)
                        : launch_flash<2, 2, false>(num_work, p, st, nullptr); break;
    case 4: e = hg == 1 ? launch_flash<4, 1, false>(num_work, p, st, nullptr)
                        : hg == 2 ? launch_flash<4, 2, false>(num_work, p, st, nullptr)
                                  : launch_flash<4, 4, false>(num_work, p, st, nullptr); break;
    default: return hipErrorInvalidValue;
  }
  if (e != hipSuccess || !p->work_kb || p->ncomb <= 0) return e;
  hipLaunchKernelGGL(dsse::flash_combine_kernel, dim3(p->ncomb, p->hkv, p->group), dim3(256), 0, st, *p);
  return hipGetLastError();
}

DSSE_CHECK_READER(dsse_check_attention_prefill)
