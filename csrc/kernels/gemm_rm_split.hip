// The row-major GEMM of the exact mode with every wave on all of a tile's outputs: chosen, and compared with the other forms, in gemm_rowmajor.hip.
#include "api_layers.h"
#include "frag.h"
#include "lds_dma.h"

#include <type_traits>

namespace dsse {
namespace {

// Tiles of 16 TM rows x 16 TN columns; KW waves, each with 32 / KW k of every chunk of 32 for all TM TN accumulators, meet in LDS at the end.
//
// What bounds it: the fp32 matrix rate, and behind it the DMA instructions: one that misses L1 keeps its wave from issuing for some 40 clocks, whatever is
// in flight (with loads that all hit L1, or none, a tile of 7 x 2 takes 104 to 110 us at K = 8192, with these 130; more stages, other cache policies,
// waves that only load, loads by one wave at a time, fragments straight from memory and starts of K apart gave nothing or cost 5 to 30 %).  No fragment is read from LDS twice, so tiles can be
// as flat as the grid wants them: 64 x 64 tiles of 2 x 2 waves leave 448 rows and 224 workgroups for 400 rows of 2048 columns, 7 x 2 fills 256.
// Measured (one MI355X), the other forms / this, us: 400 rows, 2048 x 2048 43 / 37, 2048 x 8192 145 / 130, 8192 x 2048 141 / 130, 6272 x 2048 96 / 87; 300
// rows, 2048 x 2048 40 / 29; 64 rows, 8192 x 2048 34 / 25; 67 rows, 32768 x 2048 104 / 91; 130 rows, 16384 x 2048 95 / 84.
template <int TM, int TN, int KW, int STAGES>
__global__ __launch_bounds__(64 * KW) void gemm_rm_split_kernel(GemmRmParams p) {
  constexpr int kRows = 16 * TM, kCols = 16 * TN, kPieces = 2 * (TM + TN), kPer = (kPieces + KW - 1) / KW;  // DMA instructions (8 rows), per wave
  constexpr int kSlot = KW * kPer * 1024, E = 8 / KW, T = TM * TN;
  static_assert(KW == 4, "a wave's part of a fragment is two k");
  typedef __attribute__((ext_vector_type(2))) float V;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int nbm = (p.M + kRows - 1) / kRows, nbn = (p.N + kCols - 1) / kCols, n = gridDim.x;
  const int xcd = blockIdx.x & 7, q8 = n >> 3, rem = n & 7;
  const int lid = (xcd < rem ? xcd * (q8 + 1) : rem * (q8 + 1) + (xcd - rem) * q8) + (blockIdx.x >> 3);
  const int grp = lid / (8 * nbn), gsz = min(8, nbm - 8 * grp), in = lid - grp * 8 * nbn;
  const int m0 = (8 * grp + in % gsz) * kRows, n0 = in / gsz * kCols;
  const int z = blockIdx.z;
  const float* X = reinterpret_cast<const float*>(p.x) + (int64_t)z * p.xbs;
  const float* W = reinterpret_cast<const float*>(p.w) + (int64_t)z * p.wbs;
  const int nk = p.K / 32;
  auto swizzle = [](int row) { return (row >> 1) & 7; };  // a wave's part of 16 rows: 16 pieces in 16 slots
  __amdgpu_buffer_rsrc_t src[kPer];
  uint32_t vo[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int q = w * kPer + i;  // every instruction is of one operand; those past the last piece bring zeros without traffic
    const bool is_x = q < 2 * TM;
    const int rows = is_x ? p.M : p.N, ld = is_x ? p.ldx : p.ldw, row = 8 * (is_x ? q : q - 2 * TM) + (lane >> 3);
    const int global = (is_x ? m0 : n0) + row;
    src[i] = make_rsrc(is_x ? X : W, (uint32_t)(((size_t)(rows - 1) * ld + p.K) * sizeof(float)));
    vo[i] = q < kPieces && global < rows ? (uint32_t)((size_t)global * ld * sizeof(float)) + 16 * ((lane & 7) ^ swizzle(row)) : kOOB;
  }
  auto issue = [&](int t) {
    char* base = smem + t % STAGES * kSlot + w * kPer * 1024;
#pragma unroll
    for (int i = 0; i < kPer; ++i) lds_dma(src[i], base + i * 1024, t < nk ? vo[i] : kOOB, (uint32_t)t * 128);
  };
  const int at = (128 / KW) * w + 4 * E * g;  // of a row's 128 bytes
  const int rd = r * 128 + (((at >> 4) ^ swizzle(r)) << 4) + (at & 15);
  V a[2][TM], b[2][TN];
  f32x4 acc[T];
#pragma unroll
  for (int i = 0; i < T; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Fragments k, k + 1 of the chunk at `buf`: the TN of W, then the TM of X
  auto read = [&](auto set, const char* buf, int k) {
    constexpr int s = decltype(set)::value;
#pragma unroll
    for (int f = k; f < k + 2 && f < TM + TN; ++f) {
      const V v = *reinterpret_cast<const V*>(buf + rd + (f < TN ? kRows * 128 + f * 2048 : (f - TN) * 2048));
      if (f < TN) b[s][f] = v;
      else a[s][f - TN] = v;
    }
  };
  // Chunk t, in the slot at `now`; the fragments of chunk t + 1 are read and chunk t + STAGES is requested under its products.  The first product
  // takes the fragment that was read last, so the compiler's own wait for the fragments stands before the next reads and costs nothing.
  constexpr int kReads = (TM + TN + 1) / 2, kSide = kReads + kPer, kProducts = T * E;
  auto step = [&](auto set, int t, char* now, const char* next) {
    constexpr int cur = decltype(set)::value;
    // this wave's part of chunk t + 1 has landed and its fragments of chunk t are in registers, then everybody's: t's slot is free
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((STAGES - 2) * kPer) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    const bool more = t + STAGES < nk;
    auto products = [&](auto self, auto m) {
      constexpr int q = decltype(m)::value;
      if constexpr (q < kProducts) {
        constexpr int e = q / T, i = T - 1 - q % T;
        acc[i] = mfma16x16x4(a[cur][i / TN][e], b[cur][i % TN][e], acc[i]);
        __builtin_amdgcn_sched_barrier(0);
        constexpr int s0 = q * kSide / kProducts, s1 = (q + 1) * kSide / kProducts;
#pragma unroll
        for (int s = s0; s < s1; ++s) {
          if (s < kReads) {
            read(std::integral_constant<int, 1 - cur>{}, next, 2 * s);
          } else {
            lds_dma(src[s - kReads], now + w * kPer * 1024 + (s - kReads) * 1024, more ? vo[s - kReads] : kOOB, (uint32_t)(t + STAGES) * 128);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        self(self, std::integral_constant<int, q + 1>{});
      }
    };
    products(products, std::integral_constant<int, 0>{});
  };
#pragma unroll
  for (int t = 0; t < STAGES; ++t) issue(t);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((STAGES - 1) * kPer) : "memory");
#pragma unroll
  for (int k = 0; k < TM + TN; k += 2) read(std::integral_constant<int, 0>{}, smem, k);
  char* now = smem;
  auto after = [&](char* s) { return s + kSlot == smem + STAGES * kSlot ? smem : s + kSlot; };
  for (int t = 0; t < nk; t += 2) {  // an odd last chunk is followed by one of zeros
    char* second = after(now);
    char* third = after(second);
    step(std::integral_constant<int, 0>{}, t, now, second);
    step(std::integral_constant<int, 1>{}, t + 1, second, third);
    now = third;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the look-ahead past K: nothing lands in LDS any more
  __syncthreads();
  f32x4* red = reinterpret_cast<f32x4*>(smem) + lane;  // [output tile][wave]; tile i is finished by wave i % KW
#pragma unroll
  for (int i = 0; i < T; ++i)
    if (i % KW != w) red[(i * (KW - 1) + w - (w > i % KW)) * 64] = acc[i];
  __syncthreads();
  const float* bias = p.bias ? reinterpret_cast<const float*>(p.bias) + (int64_t)z * p.bbs : nullptr;
#pragma unroll
  for (int i = 0; i < T; ++i) {
    if (i % KW != w) continue;  // uniform
    f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < KW; ++v) s += v == i % KW ? acc[i] : red[(i * (KW - 1) + v - (v > i % KW)) * 64];
    const int col = n0 + 16 * (i % TN) + r;
    if (col >= p.N) continue;
    const float bv = bias ? bias[col] : 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = m0 + 16 * (i / TN) + 4 * g + e;
      if (row >= p.M) continue;
      float v = s[e] + bv;
      if (p.act == 1) v = gelu_tanh(v);
      reinterpret_cast<float*>(p.out)[(int64_t)z * p.obs + (int64_t)row * p.ldo + col] = v;
    }
  }
}

template <int TM, int TN, int KW, int STAGES>
hipError_t launch_split(const GemmRmParams& p, hipStream_t st) {
  constexpr int kPer = (2 * (TM + TN) + KW - 1) / KW, kRing = STAGES * kPer * KW * 1024, kRed = TM * TN * (KW - 1) * 1024, kLds = kRing > kRed ? kRing : kRed;
  static_assert(kLds <= 160 * 1024 && STAGES >= 2, "LDS");
  static bool attr_set = false;
  if (!attr_set) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_rm_split_kernel<TM, TN, KW, STAGES>), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    attr_set = true;
  }
  const int64_t tiles = (int64_t)((p.M + 16 * TM - 1) / (16 * TM)) * ((p.N + 16 * TN - 1) / (16 * TN));
  hipLaunchKernelGGL((gemm_rm_split_kernel<TM, TN, KW, STAGES>), dim3((unsigned)tiles, 1, p.batch), dim3(64 * KW), kLds, st, p);
  return hipGetLastError();
}

// us at K = 2048, measured: a round of 512 workgroups (two per CU), up to 256 that have the chip to themselves, up to 256 behind full rounds (5 x 4: 41 to 80
// from process to process, 400 rows of 16384 213 to 252 in all)
struct Form {
  int tm, tn, round, only, rest;
  hipError_t (*launch)(const GemmRmParams&, hipStream_t);
};
constexpr Form kForms[] = {{5, 4, 86, 48, 70, launch_split<5, 4, 4, 4>}, {9, 2, 79, 45, 72, launch_split<9, 2, 4, 3>},
                           {7, 2, 63, 37, 59, launch_split<7, 2, 4, 4>}, {5, 2, 48, 28, 40, launch_split<5, 2, 4, 4>},
                           {4, 2, 39, 23, 20, launch_split<4, 2, 4, 4>}, {3, 2, 31, 20, 13, launch_split<3, 2, 4, 4>}};

const Form& pick(int M, int N, int batch, int64_t& us) {
  const Form* best = nullptr;
  for (const Form& f : kForms) {
    const int64_t tiles = (int64_t)((M + 16 * f.tm - 1) / (16 * f.tm)) * ((N + 16 * f.tn - 1) / (16 * f.tn)) * batch, full = tiles / 512, left = tiles % 512;
    const int64_t t = full * f.round + (left > 256 ? f.round : left == 0 ? 0 : full == 0 ? f.only : f.rest);
    if (!best || t < us) best = &f, us = t;
  }
  return *best;
}

}  // namespace

int64_t gemm_rm_split_us(int M, int N, int batch) {
  int64_t us = 0;
  pick(M, N, batch, us);
  return us;
}

int gemm_rm_split_form(int M, int N, int batch) {
  int64_t us = 0;
  const Form& f = pick(M, N, batch, us);
  return 10 * f.tm + f.tn;
}

hipError_t gemm_rm_split(const GemmRmParams& p, hipStream_t st) {
  int64_t us = 0;
  return pick(p.M, p.N, p.batch, us).launch(p, st);
}

}  // namespace dsse
