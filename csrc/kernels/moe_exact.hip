// The grouped expert GEMMs of the exact mode (fp32): both operands staged through LDS by DMA.
//
//   MODE 0   h = act(x . up^T, x . gate^T)     32 hidden units of an expert (64 without a gate) x one 64-row tile of its list
//   MODE 1   o = weight * (h . down^T)         64 output columns x one tile
//
// What bounds it: the 32-bit matrix rate.  A wave takes 16 weight rows -- 8 units' gate rows and the same units' up rows, so that
// the two sums of a unit sit eight lanes apart -- times the tile's live 16-row sub-tiles; a chunk is 128 bytes of every row, four of
// them in flight, one counted wait and one barrier per chunk, as in gemm_rowmajor.hip.  Every fourth chunk goes to the same
// accumulator: four partial sums per output, as many as the register-direct kernels (moe.hip) have waves.
// Measured (one MI355X), both products, register-direct kernels / this, us: 2048 wide, 16 experts of 1408, top 2 and a shared one of
// 2816: 1 row 62 / 54, 8 rows 127 / 117, 16 rows 161 / 135, 32 rows 236 / 166, 64 rows 322 / 216, 150 rows 341 / 254, 300 rows 488 /
// 330, 600 rows 766 / 534; error against 64 bits 7.3e-7 both.
#include "api_layers.h"
#include "lds_dma.h"
#include "moe_rows.h"

namespace dsse {
namespace {

constexpr int kExactStages = 4;
constexpr int kExactSlot = (kMoeRows + 64) * 128;  // a chunk: the rows of x or h, then 64 weight rows

template <int MODE, bool GATED>
__global__ __launch_bounds__(256) void moe_exact_kernel(MoeGroupedParams p) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  __shared__ int ids[kMoeRows];
  const int t = blockIdx.y;
  if (t >= *p.num_tiles) return;
  const int e = p.tile_expert[t];
  const bool sh = e >= p.E;
  const int Fe = sh ? p.Fs : p.F, K = MODE == 1 ? Fe : p.W, N = MODE == 1 ? p.W : Fe;
  constexpr int kCols = MODE == 0 && GATED ? 32 : 64;  // columns or units of a workgroup
  const int n0 = blockIdx.x * kCols;
  if (n0 >= N) return;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  if (threadIdx.x < kMoeRows) ids[threadIdx.x] = p.sorted[t * kMoeRows + threadIdx.x];
  __syncthreads();
  // an expert's ids fill its tiles from the front
  int subs = 1;
#pragma unroll
  for (int i = 1; i < 4; ++i) subs += __builtin_amdgcn_readfirstlane(ids[16 * i]) >= 0;
  const float* X = reinterpret_cast<const float*>(MODE == 1 ? p.h : p.x);
  const int ldx = MODE == 1 ? p.ldh : p.W, xrows = MODE == 1 ? p.M * p.S : p.M;
  auto matrix = [&](const void* routed, const void* shared) {
    return sh ? reinterpret_cast<const float*>(shared) : reinterpret_cast<const float*>(routed) + (int64_t)e * p.F * p.W;
  };
  const float* W1 = MODE == 1 ? matrix(p.down, p.sdown) : matrix(p.up, p.sup);
  const float* W0 = MODE == 0 && GATED ? matrix(p.gate, p.sgate) : W1;
  // waves 0 and 1 stage the rows, 2 and 3 the weights, in kPer DMA instructions of eight rows each
  const bool is_x = w < 2;
  const uint32_t wbytes = (uint32_t)((size_t)N * K * 4);
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(X, (uint32_t)(((size_t)(xrows - 1) * ldx + K) * 4)), r0 = make_rsrc(W0, wbytes),
                               r1 = make_rsrc(W1, wbytes);
  constexpr int kPer = 4;
  static_assert(4 * kPer * 1024 == kExactSlot, "a chunk in the waves' instructions");
  uint32_t vo[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int row = (w & 1) * 32 + 8 * i + (lane >> 3);  // of the 64 rows or weight rows
    uint32_t at = kOOB;
    if (is_x) {
      const int id = ids[row];
      if (id >= 0) at = (uint32_t)((size_t)(MODE == 1 ? id : id / p.S) * ldx * 4);
    } else {
      // weight rows 16 v .. + 15 are wave v's columns; an instruction's eight are of one matrix
      const int n = n0 + (MODE == 0 && GATED ? 8 * (row >> 4) + (row & 7) : row);
      if (n < N) at = (uint32_t)((size_t)n * K * 4);
    }
    vo[i] = at == kOOB ? kOOB : at + 16 * ((lane & 7) ^ piece_swizzle(row));
  }
  const int nk = K / 32;
  auto issue = [&](int c, int slot) {
    char* base = smem + slot * kExactSlot + w * kPer * 1024;
#pragma unroll
    for (int i = 0; i < kPer; ++i) lds_dma(is_x ? rx : (i & 1 ? r1 : r0), base + i * 1024, c < nk ? vo[i] : kOOB, (uint32_t)c * 128);
  };
  int a_rd[2], b_rd[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int piece = ((2 * g + s) ^ piece_swizzle(r)) << 4;
    a_rd[s] = r * 128 + piece;
    b_rd[s] = (kMoeRows + 16 * w + r) * 128 + piece;
  }
  f32x4 acc[4][4];  // [chunk mod 4][sub-tile]
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[q][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < kExactStages - 1; ++c) issue(c, c);
  auto walk = [&](auto live) {
    constexpr int TM = decltype(live)::value;
    for (int c0 = 0; c0 < nk; c0 += 4) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {  // chunks past K hold zeros
        // this wave's part of chunk c0 + q has landed and its fragments of the chunk before are in registers, then everybody's
        asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        issue(c0 + q + 3, (q + 3) & 3);
        const char* buf = smem + q * kExactSlot;
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
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int i = 0; i < TM; ++i) acc[q][i] = mfma16x16x4(a[s][i][u], b[s][u], acc[q][i]);
      }
    }
  };
  static_assert(kExactStages == 4 && kPer == 4, "slots and sums by chunk mod 4, the wait above");
  if (subs == 1) walk(std::integral_constant<int, 1>{});
  else if (subs == 2) walk(std::integral_constant<int, 2>{});
  else if (subs == 3) walk(std::integral_constant<int, 3>{});
  else walk(std::integral_constant<int, 4>{});
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the look-ahead past K: nothing lands in LDS any more
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float v = (acc[0][i][u] + acc[1][i][u]) + (acc[2][i][u] + acc[3][i][u]);  // row 16 i + 4 g + u, the wave's column r
      const int id = ids[16 * i + 4 * g + u];
      if constexpr (MODE == 1) {
        const int d = n0 + 16 * w + r;
        if (id >= 0 && d < N) p.o[(int64_t)id * p.W + d] = out_weight(p, id / p.S, id % p.S) * v;
      } else if constexpr (GATED) {
        const float up = __shfl_xor(v, 8);  // lanes r < 8 hold a unit's gate sum
        const int f = n0 + 8 * w + r;
        if (r < 8 && id >= 0 && f < N) {
          const float wi = in_weight(p, id), gv = v * wi;
          reinterpret_cast<float*>(p.h)[(int64_t)id * p.ldh + f] = gv / (1.0f + expf(-gv)) * (up * wi);
        }
      } else {
        const int f = n0 + 16 * w + r;
        if (id >= 0 && f < N) {
          const float uv = v * in_weight(p, id);
          reinterpret_cast<float*>(p.h)[(int64_t)id * p.ldh + f] = uv > 0.0f ? uv * uv : 0.0f;
        }
      }
    }
}

template <int MODE, bool GATED>
hipError_t launch_exact(const MoeGroupedParams& p, int cols, int n, hipStream_t st) {
  constexpr int lds = kExactStages * kExactSlot;
  static bool attr_set = false;
  if (!attr_set) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&moe_exact_kernel<MODE, GATED>), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    attr_set = true;
  }
  hipLaunchKernelGGL((moe_exact_kernel<MODE, GATED>), dim3((n + cols - 1) / cols, p.max_tiles), dim3(256), lds, st, p);
  return hipGetLastError();
}

}  // namespace

// Whole chunks of 32 numbers, four of them at least, 16-byte-aligned operands inside a 2 GiB buffer range each
bool moe_exact_ok(const MoeGroupedParams& p) {
  const int64_t range = (int64_t)1 << 31;
  return p.f32 && p.parts == p.S && p.W >= 128 && p.F >= 128 && p.W % 32 == 0 && p.F % 32 == 0 && p.Fs % 32 == 0 && p.ldh % 4 == 0 && p.max_tiles <= 65535 &&
         fours({p.x, p.gate, p.up, p.down, p.sgate, p.sup, p.sdown, p.h}) && (int64_t)p.M * p.W * 4 < range &&
         (int64_t)p.M * p.S * p.ldh * 4 < range && (int64_t)p.F * p.W * 4 < range && (int64_t)p.Fs * p.W * 4 < range;
}

}  // namespace dsse

extern "C" hipError_t dsse_moe_exact(const dsse::MoeGroupedParams* p, hipStream_t st) {
  if (!dsse::moe_exact_ok(*p)) return hipErrorInvalidValue;
  const int fmax = p->F > p->Fs ? p->F : p->Fs;
  const hipError_t err = p->gate ? dsse::launch_exact<0, true>(*p, 32, fmax, st) : dsse::launch_exact<0, false>(*p, 64, fmax, st);
  return err != hipSuccess ? err : dsse::launch_exact<1, true>(*p, 64, p->W, st);
}
