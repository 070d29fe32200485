// The row-major GEMM of the exact mode in strips: chosen, and compared with the 64 x 64 tiles, in gemm_rowmajor.hip (gemm_rm_form_rows).
#include "api_layers.h"
#include "frag.h"
#include "lds_dma.h"

namespace dsse {
namespace {

constexpr int kStages = 4;

// gemm_rm_lds_kernel (gemm_rowmajor.hip) in fp32 with tiles of 16 TM rows x 64 columns, a wave taking all rows of 16 columns: rows in steps of 16 where 64 x 64 tiles
// leave part of their rows empty, and products of one k on all TM accumulators in a row, none of which waits for another.
// Measured (one MI355X), 64 x 64 tiles / this, us: 16384 x 2048, 130 rows 143 / 115, 400 rows 251 / 229; 6272 x 2048, 400 rows 129 / 93;
// 6144 x 4096, 400 rows 218 / 178; 4096 x 2048, 300 rows 71 / 57; 8192 x 2048, 130 rows 70 / 56.  With 64 rows it is the 64 x 64 form
// that is 2 % faster: two of its fragments feed four products.
template <int TM>
__global__ __launch_bounds__(256) void gemm_rm_strip_kernel(GemmRmParams p) {
  constexpr int kRows = 16 * TM, kPieces = 2 * TM + 8, kPer = (kPieces + 3) / 4;  // DMA instructions (8 rows) of a chunk, per wave
  constexpr int kSlot = 4 * kPer * 1024;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int nbm = (p.M + kRows - 1) / kRows, nbn = (p.N + 63) / 64, n = gridDim.x;
  const int xcd = blockIdx.x & 7, q8 = n >> 3, rem = n & 7;
  const int lid = (xcd < rem ? xcd * (q8 + 1) : rem * (q8 + 1) + (xcd - rem) * q8) + (blockIdx.x >> 3);
  const int grp = lid / (8 * nbn), gsz = min(8, nbm - 8 * grp), in = lid - grp * 8 * nbn;
  const int m0 = (8 * grp + in % gsz) * kRows, n0 = in / gsz * 64;
  const int z = blockIdx.z;
  const float* X = reinterpret_cast<const float*>(p.x) + (int64_t)z * p.xbs;
  const float* W = reinterpret_cast<const float*>(p.w) + (int64_t)z * p.wbs;
  const int nk = p.K / 32;
  __amdgpu_buffer_rsrc_t src[kPer];
  uint32_t vo[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int q = w * kPer + i;  // every instruction is of one operand; those past the last piece bring zeros without traffic
    const bool is_x = q < 2 * TM;
    const int rows = is_x ? p.M : p.N, ld = is_x ? p.ldx : p.ldw, row = 8 * (is_x ? q : q - 2 * TM) + (lane >> 3);
    const int global = (is_x ? m0 : n0) + row;
    src[i] = make_rsrc(is_x ? X : W, (uint32_t)(((size_t)(rows - 1) * ld + p.K) * sizeof(float)));
    vo[i] = q < kPieces && global < rows ? (uint32_t)((size_t)global * ld * sizeof(float)) + 16 * ((lane & 7) ^ piece_swizzle(row)) : kOOB;
  }
  auto issue = [&](int t) {
    char* base = smem + t % kStages * kSlot + w * kPer * 1024;
#pragma unroll
    for (int i = 0; i < kPer; ++i) lds_dma(src[i], base + i * 1024, t < nk ? vo[i] : kOOB, (uint32_t)t * 128);
  };
  int a_rd[2], b_rd[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int piece = ((2 * g + s) ^ piece_swizzle(r)) << 4;
    a_rd[s] = r * 128 + piece;
    b_rd[s] = (kRows + 16 * w + r) * 128 + piece;
  }
  f32x4 acc[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < kStages - 1; ++t) issue(t);
  for (int t = 0; t < nk; ++t) {
    // this wave's part of chunk t has landed and its fragments of chunk t - 1 are in registers, then everybody's
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((kStages - 2) * kPer) : "memory");
    issue(t + kStages - 1);
    const char* buf = smem + t % kStages * kSlot;
    f32x4 a[2][TM], b[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      b[s] = *reinterpret_cast<const f32x4*>(buf + b_rd[s]);
#pragma unroll
      for (int i = 0; i < TM; ++i) a[s][i] = *reinterpret_cast<const f32x4*>(buf + a_rd[s] + i * 2048);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < TM; ++i) acc[i] = mfma16x16x4(a[s][i][e], b[s][e], acc[i]);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the look-ahead past K: nothing lands in LDS any more
  const int col = n0 + 16 * w + r;
  if (col >= p.N) return;
  const float bv = p.bias ? reinterpret_cast<const float*>(p.bias)[(int64_t)z * p.bbs + col] : 0.0f;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = m0 + 16 * i + 4 * g + e;
      if (row >= p.M) continue;
      float v = acc[i][e] + bv;
      if (p.act == 1) v = gelu_tanh(v);
      reinterpret_cast<float*>(p.out)[(int64_t)z * p.obs + (int64_t)row * p.ldo + col] = v;
    }
}

template <int TM>
hipError_t launch_strip(const GemmRmParams& p, hipStream_t st) {
  constexpr int kLds = kStages * ((2 * TM + 8 + 3) / 4) * 4096;
  static bool attr_set = false;
  if (!attr_set) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_rm_strip_kernel<TM>), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    attr_set = true;
  }
  const int64_t tiles = (int64_t)((p.M + 16 * TM - 1) / (16 * TM)) * ((p.N + 63) / 64);
  hipLaunchKernelGGL((gemm_rm_strip_kernel<TM>), dim3((unsigned)tiles, 1, p.batch), dim3(256), kLds, st, p);
  return hipGetLastError();
}

}  // namespace

hipError_t gemm_rm_strip(int rows, const GemmRmParams& p, hipStream_t st) {
  return rows == 48 ? launch_strip<3>(p, st) : (rows == 80 ? launch_strip<5>(p, st) : hipErrorInvalidValue);
}

}  // namespace dsse
