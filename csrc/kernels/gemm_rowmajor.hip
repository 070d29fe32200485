// General row-major GEMM on MFMA: out[M, N] = act(X[M, K] . W[N, K]^T + bias), any M, N, K, batched over blockIdx.z.
//
// The engine's tiled-layout GEMMs (gemm_skinny / gemm_stream / gemm_wide / gemm_tiled / gemm_pipe) want N % 16 == 0 and
// K % 128 == 0 and a pre-tiled weight.  Layer designs whose inner sizes come from a checkpoint's configuration (expert
// widths, latent ranks, per-head slices, block-diagonal gates) need a kernel with no shape contract: this one reads both
// operands straight from global memory as MFMA fragments (K is the contiguous axis of X and of W, so a lane's fragment is
// one 16-byte load), zero-fills past M, N and K, and strides over a batch axis (per-head or per-block weights).
//
// Two element types: bf16 (v_mfma_f32_16x16x32_bf16) and fp32 (v_mfma_f32_16x16x4_f32, true 32-bit products) -- the
// latter is the engine's exact mode.  A lane (r = lane & 15, g = lane >> 4) holds PER consecutive k of row r; which k a
// (lane group, element) pair stands for only has to agree between the A and the B fragment, so both use k0 + PER g + j.
#include "api_layers.h"
#include "frag.h"
#include "lds_dma.h"

namespace dsse {
namespace {

// TM x TN 16x16 tiles per wave, WGM x WGN waves per workgroup (4 waves).
template <typename T, int TM, int TN, int WGM, int WGN>
__global__ __launch_bounds__(256) void gemm_rm_kernel(GemmRmParams p) {
  using F = Frag<T>;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int wm = wave / WGN, wn = wave % WGN;
  const int row0 = blockIdx.y * (WGM * TM * 16) + wm * TM * 16;
  const int col0 = blockIdx.x * (WGN * TN * 16) + wn * TN * 16;
  const int z = blockIdx.z;
  const T* X = reinterpret_cast<const T*>(p.x) + (int64_t)z * p.xbs;
  const T* W = reinterpret_cast<const T*>(p.w) + (int64_t)z * p.wbs;
  const T* bias = p.bias ? reinterpret_cast<const T*>(p.bias) + (int64_t)z * p.bbs : nullptr;
  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const T* xr[TM];
  const T* wr[TN];
  bool xv[TM], wv[TN];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int row = row0 + 16 * i + r;
    xv[i] = row < p.M;
    xr[i] = X + (int64_t)(xv[i] ? row : 0) * p.ldx;
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int col = col0 + 16 * j + r;
    wv[j] = col < p.N;
    wr[j] = W + (int64_t)(wv[j] ? col : 0) * p.ldw;
  }
  const bool vx = p.vecx != 0, vw = p.vecw != 0;
  for (int k0 = 0; k0 < p.K; k0 += F::KS) {
    const int k = k0 + F::PER * g;
    typename F::V a[TM], b[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) a[i] = load_frag<T>(xr[i], k, p.K, xv[i], vx);
#pragma unroll
    for (int j = 0; j < TN; ++j) b[j] = load_frag<T>(wr[j], k, p.K, wv[j], vw);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = mma(a[i], b[j], acc[i][j]);
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = col0 + 16 * j + r;
      if (col >= p.N) continue;
      const float bv = bias ? (float)bias[col] : 0.0f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = row0 + 16 * i + 4 * g + e;
        if (row >= p.M) continue;
        float v = acc[i][j][e] + bv;
        if (p.act == 1) v = gelu_tanh(v);
        const int64_t o = (int64_t)z * p.obs + (int64_t)row * p.ldo + col;
        if (p.out_f32) reinterpret_cast<float*>(p.out)[o] = v;
        else reinterpret_cast<T*>(p.out)[o] = (T)v;
      }
    }
}

// Aligned shapes with work for the matrix cores: both operands staged through LDS by DMA, kStages chunks deep.
//
// What bounds it: the matrix rate in fp32 (v_mfma_f32_16x16x4_f32, 157 TFLOP/s), LDS traffic in bf16.  The kernel above has
// no load in flight while it multiplies; here a chunk is 128 bytes of every row (32 fp32 or 64 bf16 k), 16-byte pieces
// swizzled by (row >> 1) & 5 on the source address so that fragment reads are free of bank conflicts; the chunk read next
// was requested kStages - 1 chunks ago, one counted wait and one barrier per chunk.  The slot refilled after that barrier
// held the chunk that every wave has finished reading.  Rows past M and N and chunks past K load as zeros without traffic.
// Measured (one MI355X): 400 rows in fp32, 2048 x 2048 205 -> 42 us, 16384 x 2048 330 -> 250 us (108 TFLOP/s), 2048 x 8192
// 788 -> 148 us; 1000 rows in bf16, 576 x 4096 119 -> 17 us; 3000 rows of 32 slices of 128 x 512 91 -> 39 us.
constexpr int kStages = 4;

// WS x WS waves of 32 x 32 outputs make the tile; KG such groups work on alternate chunks of K and meet in LDS.
template <typename T, int WS, int KG>
__global__ __launch_bounds__(64 * WS * WS * KG) void gemm_rm_lds_kernel(GemmRmParams p) {
  constexpr int kTile = 32 * WS, kWaves = WS * WS, kPer = 8 / WS;  // DMA instructions (8 rows) per wave and chunk
  constexpr int kSlot = 2 * kTile * 128;                           // a chunk: the X rows, then the W rows
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wave / kWaves, w = wave % kWaves;
  const int r = lane & 15, g = lane >> 4, wm = w / WS, wn = w % WS;
  // each XCD takes a contiguous run of tiles, row tiles fastest in groups of 8: neighbours share their operands in its L2
  const int nbm = (p.M + kTile - 1) / kTile, nbn = (p.N + kTile - 1) / kTile, n = gridDim.x;
  const int xcd = blockIdx.x & 7, q8 = n >> 3, rem = n & 7;
  const int lid = (xcd < rem ? xcd * (q8 + 1) : rem * (q8 + 1) + (xcd - rem) * q8) + (blockIdx.x >> 3);
  const int grp = lid / (8 * nbn), gsz = min(8, nbm - 8 * grp), in = lid - grp * 8 * nbn;
  const int m0 = (8 * grp + in % gsz) * kTile, n0 = in / gsz * kTile;
  const int z = blockIdx.z;
  const T* X = reinterpret_cast<const T*>(p.x) + (int64_t)z * p.xbs;
  const T* W = reinterpret_cast<const T*>(p.w) + (int64_t)z * p.wbs;
  const int nk = p.K * (int)sizeof(T) / 128, steps = (nk + KG - 1) / KG;
  // a group's waves stage its chunks in equal parts; every instruction is of one operand
  __amdgpu_buffer_rsrc_t src[WS == 1 ? 2 : 1];
  uint32_t vo[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int at = (w * kPer + i) * 8;
    const bool is_x = at < kTile;
    const int rows = is_x ? p.M : p.N, ld = is_x ? p.ldx : p.ldw, row = at % kTile + (lane >> 3);
    const int global = (is_x ? m0 : n0) + row;
    if (i % (WS == 1 ? 4 : kPer) == 0)
      src[WS == 1 ? i / 4 : 0] = make_rsrc(is_x ? X : W, (uint32_t)(((size_t)(rows - 1) * ld + p.K) * sizeof(T)));
    vo[i] = global < rows ? (uint32_t)((size_t)global * ld * sizeof(T)) + 16 * ((lane & 7) ^ piece_swizzle(row)) : kOOB;
  }
  auto issue = [&](int t) {
    const int c = t * KG + kg;
    char* base = smem + ((t % kStages) * KG + kg) * kSlot + w * kPer * 1024;
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      lds_dma(src[WS == 1 ? i / 4 : 0], base + i * 1024, c < nk ? vo[i] : kOOB, (uint32_t)c * 128);
  };
  int a_rd[2], b_rd[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int piece = ((2 * g + s) ^ piece_swizzle(r)) << 4;
    a_rd[s] = (wm * 32 + r) * 128 + piece;
    b_rd[s] = (kTile + wn * 32 + r) * 128 + piece;
  }
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i) acc[i][0] = acc[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < kStages - 1; ++t) issue(t);
  for (int t = 0; t < steps; ++t) {
    // this wave's part of step t has landed (those of the two younger steps may be in flight) and its fragments of step t - 1
    // are in registers, then everybody's
    static_assert(kStages == 4 && (kPer == 4 || kPer == 8), "the waits below");
    if constexpr (kPer == 4) asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    issue(t + kStages - 1);
    const char* buf = smem + ((t % kStages) * KG + kg) * kSlot;
    typename Frag<T>::V a[2][2], b[2][2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        a[i][s] = *reinterpret_cast<const typename Frag<T>::V*>(buf + a_rd[s] + i * 2048);
        b[i][s] = *reinterpret_cast<const typename Frag<T>::V*>(buf + b_rd[s] + i * 2048);
      }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mma(a[i][s], b[j][s], acc[i][j]);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the look-ahead past K: nothing lands in LDS any more
  if constexpr (KG > 1) {
    __syncthreads();
    f32x4* red = reinterpret_cast<f32x4*>(smem);
    if (kg > 0) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) red[(((kg - 1) * kWaves + w) * 4 + 2 * i + j) * 64 + lane] = acc[i][j];
    }
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int k = 1; k < KG; ++k)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] += red[(((k - 1) * kWaves + w) * 4 + 2 * i + j) * 64 + lane];
  }
  const T* bias = p.bias ? reinterpret_cast<const T*>(p.bias) + (int64_t)z * p.bbs : nullptr;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int col = n0 + (wn * 2 + j) * 16 + r;
    if (col >= p.N) continue;
    const float bv = bias ? (float)bias[col] : 0.0f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = m0 + (wm * 2 + i) * 16 + 4 * g + e;
        if (row >= p.M) continue;
        float v = acc[i][j][e] + bv;
        if (p.act == 1) v = gelu_tanh(v);
        const int64_t o = (int64_t)z * p.obs + (int64_t)row * p.ldo + col;
        if (p.out_f32) reinterpret_cast<float*>(p.out)[o] = v;
        else reinterpret_cast<T*>(p.out)[o] = (T)v;
      }
  }
}

// Up to 16 rows (decode buckets, per-head and per-block slices), or many rows of a NARROW output (a router's logits, a
// few-column gate: up to 64 columns): a workgroup owns one 16 x 16 output tile and its four waves split the K axis
// (k-steps w, w + 4, ...), meeting in LDS.  Four times the workgroups of a 16 x 64 tile and a quarter of the dependent
// k-steps per wave: these launches are latency-bound, not bandwidth-bound -- a narrow output leaves the 64 x 64 tiles
// of the general kernel a handful of workgroups that each walk the whole K axis.
// NW waves per workgroup: four, or sixteen when the launch has few tiles and a long K axis (a router's logits for a
// decode step are ONE tile: sixteen waves walk a sixteenth of K each instead of four a quarter).
template <typename T, int NW>
__global__ __launch_bounds__(NW * 64) void gemm_rm_skinny_kernel(GemmRmParams p) {
  using F = Frag<T>;
  __shared__ float red[NW * 4 * 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int col0 = blockIdx.x * 16, row0 = blockIdx.y * 16;
  const int z = blockIdx.z;
  const T* X = reinterpret_cast<const T*>(p.x) + (int64_t)z * p.xbs;
  const T* W = reinterpret_cast<const T*>(p.w) + (int64_t)z * p.wbs;
  const T* bias = p.bias ? reinterpret_cast<const T*>(p.bias) + (int64_t)z * p.bbs : nullptr;
  const bool xv = row0 + r < p.M, wv = col0 + r < p.N;
  const T* xr = X + (int64_t)(xv ? row0 + r : 0) * p.ldx;
  const T* wr = W + (int64_t)(wv ? col0 + r : 0) * p.ldw;
  const bool vx = p.vecx != 0, vw = p.vecw != 0;
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  int k0 = wave * F::KS;
  // Whole fragments, four steps' loads at a time, in the order of the loop below (the same sums); a row or column past the end reads the
  // first one and is not stored.  Where four waves walk the K axis a step's latency was most of the time: 3000 rows of 17 x 2048 in fp32
  // 24.9 -> 17.1 us, of 17 x 4096 44 -> 31, in bf16 21 -> 17; 16 rows of 2048 x 512 5.2 -> 4.4, of 4096 x 1024 in bf16 4.6 -> 4.2.  Sixteen waves stay
  // at 9.5 us for 16 rows of 16 x 2048 in fp32: 16 half lines per load and wave, whatever the order of K or the loads in flight.
  constexpr int U = 4;
  if (vx && vw)
    for (; k0 + ((U - 1) * NW + 1) * F::KS <= p.K; k0 += U * NW * F::KS) {
      typename F::V a[U], b[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        a[u] = ld_global<typename F::V>(xr + k0 + u * NW * F::KS + F::PER * g);
        b[u] = ld_global<typename F::V>(wr + k0 + u * NW * F::KS + F::PER * g);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) acc = mma(a[u], b[u], acc);
    }
  for (; k0 < p.K; k0 += NW * F::KS) {
    const int k = k0 + F::PER * g;
    acc = mma(load_frag<T>(xr, k, p.K, xv, vx), load_frag<T>(wr, k, p.K, wv, vw), acc);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) red[(wave * 4 + e) * 64 + lane] = acc[e];
  __syncthreads();
  if (wave != 0) return;
  const int col = col0 + r;
  if (col >= p.N) return;
  const float bv = bias ? (float)bias[col] : 0.0f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int row = row0 + 4 * g + e;
    if (row >= p.M) continue;
    float v = bv;
#pragma unroll
    for (int w = 0; w < NW; ++w) v += red[(4 * w + e) * 64 + lane];
    if (p.act == 1) v = gelu_tanh(v);
    const int64_t o = (int64_t)z * p.obs + (int64_t)row * p.ldo + col;
    if (p.out_f32) reinterpret_cast<float*>(p.out)[o] = v;
    else reinterpret_cast<T*>(p.out)[o] = (T)v;
  }
}

template <typename T, int TM, int TN, int WGM, int WGN>
hipError_t launch(const GemmRmParams& p, hipStream_t st) {
  dim3 grid((p.N + WGN * TN * 16 - 1) / (WGN * TN * 16), (p.M + WGM * TM * 16 - 1) / (WGM * TM * 16), p.batch);
  hipLaunchKernelGGL((gemm_rm_kernel<T, TM, TN, WGM, WGN>), grid, dim3(256), 0, st, p);
  return hipGetLastError();
}

int64_t lds_tiles(const GemmRmParams& p, int tile) {
  return (int64_t)((p.M + tile - 1) / tile) * ((p.N + tile - 1) / tile);
}

template <typename T, int WS, int KG>
hipError_t launch_lds(const GemmRmParams& p, hipStream_t st) {
  constexpr int kLds = kStages * KG * 2 * 32 * WS * 128;
  static bool attr_set = false;
  if (!attr_set) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_rm_lds_kernel<T, WS, KG>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    attr_set = true;
  }
  hipLaunchKernelGGL((gemm_rm_lds_kernel<T, WS, KG>), dim3((unsigned)lds_tiles(p, 32 * WS), 1, p.batch),
                     dim3(64 * WS * WS * KG), kLds, st, p);
  return hipGetLastError();
}

// 64 x 64 tiles or strips of 48 or 80 rows, whichever are through first
hipError_t launch_rows(const GemmRmParams& p, hipStream_t st) {
  const int rows = gemm_rm_form_rows(p.M, p.N, p.batch);
  return rows == 64 ? launch_lds<float, 2, 1>(p, st) : gemm_rm_strip(rows, p, st);
}

// Whole 128-byte chunks of 16-byte-aligned rows, each operand inside a 2 GiB buffer range
template <typename T>
bool lds_ok(const GemmRmParams& p) {
  const int64_t range = (int64_t)1 << 31, size = sizeof(T);
  return p.vecx && p.vecw && p.K * size % 128 == 0 && p.ldx >= 0 && p.ldw >= 0 &&
         ((int64_t)(p.M - 1) * p.ldx + p.K) * size < range && ((int64_t)(p.N - 1) * p.ldw + p.K) * size < range;
}

template <typename T>
hipError_t dispatch(const GemmRmParams& p, hipStream_t st) {
  if (p.M <= 16 || (p.N <= 64 && p.K >= 256)) {
    const dim3 grid((p.N + 15) / 16, (p.M + 15) / 16, p.batch);
    if ((int64_t)grid.x * grid.y * grid.z <= 256 && p.K >= 64 * Frag<T>::KS)
      hipLaunchKernelGGL((gemm_rm_skinny_kernel<T, 16>), grid, dim3(1024), 0, st, p);
    else
      hipLaunchKernelGGL((gemm_rm_skinny_kernel<T, 4>), grid, dim3(256), 0, st, p);
    return hipGetLastError();
  }
  if (lds_ok<T>(p)) {
    if constexpr (sizeof(T) == 4) {
      if (gemm_rm_split_pays(p.M, p.N, p.K, p.batch)) return gemm_rm_split(p, st);
    }
    // 64 x 64 tiles (fp32: or strips, gemm_rm_form_rows) while they fill the CUs; two wave groups per tile when there is one tile per CU at most (nothing else
    // would run while a wave waits for its fragments: 400 rows of 2048 x 2048 in fp32 45.4 -> 42.2 us); 32 x 32 tiles, four
    // groups each, while those make one round (64 rows of 2048 x 8192 in fp32 157 -> 50 us, 400 rows of 576 x 4096 in bf16
    // 19 -> 11 us).  A second round of them pays in fp32 (bound by the matrix rate) where the groups have four chunks each;
    // with fewer, filling and joining them is most of the time: mean of 256..512 tiles against the kernel above, 64 x 64 / 32 x
    // 32 tiles, 1 chunk 0.84 / 1.39, 4 chunks 0.70 / 0.92, 8 chunks 0.60 / 0.69, 16 chunks 0.52 / 0.52.
    const int chunks = (int)(p.K * sizeof(T) / 128);
    const int64_t small = lds_tiles(p, 32) * p.batch;
    if (chunks >= 2 && small <= (sizeof(T) == 4 && chunks >= 16 ? 512 : 256)) return launch_lds<T, 1, 4>(p, st);
    if (lds_tiles(p, 64) * p.batch <= 256 && chunks >= 8) return launch_lds<T, 2, 2>(p, st);
    // one or two chunks and many rows: the store is all there is to wait for (3000 rows of 512 x 128, 32 slices: 68 us here,
    // 76 us through LDS)
    if constexpr (sizeof(T) == 4) {
      if (chunks >= 3 || p.M < 1024) return launch_rows(p, st);
    } else if (chunks >= 3 || p.M < 1024) {
      return launch_lds<T, 2, 1>(p, st);
    }
  }
  if (p.M >= 256 && p.N >= 256) return launch<T, 4, 4, 2, 2>(p, st);
  return launch<T, 2, 2, 2, 2>(p, st);
}

}  // namespace

// LDS holds two workgroups of each form per CU, so a launch runs in rounds of 512, and what is left for the last one counts: 257
// workgroups and more take a round's time; fewer share no CU and take more than half of it, since a workgroup alone on its CU waits for its
// fragments; from some 160 on they go in pairs to the CUs that are free first, except for the longest ones.  Units: 1 us at K = 2048.  Over 171
// products (K 512, 2048 and 4096, 2048 to 16384 columns, 80 to 800 rows) the choice is within 0.3 % of the best of the three forms, 4 %
// at the worst.  us at K = 2048, 48 rows / 64 x 64 / 80 rows: 8192 columns, 330 rows 108 / 136 / 140, 400 rows 140 / 138 / 141; 12288, 130
// rows 89 / 108 / 91, 240 rows 110 / 130 / 140; 16384, 130 rows 99 / 135 / 92, 330 rows 194 / 209 / 228, 400 rows 247 / 247 / 228; one round of
// K = 224 (longer ones of 64 x 64 tiles are split over wave groups): 330 x 2048 7.6 / 9.0 / 10.6, 400 x 2048 10.4 / 9.1 / 10.7.  Strips of 96
// rows were the faster form nowhere by more than 3 %.
namespace {
int rows_us(int M, int N, int batch, int64_t& least) {
  struct Form {
    int rows, round, alone, paired, only;  // a round; up to 160, up to 256 workgroups behind full rounds; up to 256 and no others
  };
  static constexpr Form kForms[3] = {{64, 69, 39, 62, 53}, {48, 54, 34, 40, 52}, {80, 90, 50, 50, 55}};
  int best = 0;
  for (const Form& f : kForms) {
    const int64_t tiles = (int64_t)((M + f.rows - 1) / f.rows) * ((N + 63) / 64) * batch, full = tiles / 512, left = tiles % 512;
    int64_t t = full * f.round;
    if (left > 256) t += f.round;
    else if (left > 0) t += full == 0 ? f.only : (left > 160 ? f.paired : f.alone);
    if (!best || t < least) best = f.rows, least = t;
  }
  return best;
}
}  // namespace

// Whether the tiles of gemm_rm_split.hip are through before the forms below.  From K = 512 on by what both take, in us at K = 2048 (`rows_us`; tiles of
// 32 x 32 one round 16.5 and two 32, 64 x 64 tiles with two wave groups 41), with 3 % for the figures' own error: over 552 products of
// 20 to 1500 rows, 128 to 16384 columns, K 128 to 8192, others / chosen 1.10 in the mean (1.64 at the most: 257 to 512 tiles of 32 x 32), 0.93 at the least.  With
// 4 to 15 chunks by tiles of 32 x 32: K = 128 up to 512 of them 1.12 to 1.27, up to 1024 0.90 to 1.04; K = 256 up to 1024 0.96 to 1.54, more 0.78 to 1.03.
bool gemm_rm_split_pays(int M, int N, int K, int batch) {
  const int chunks = K / 32;
  auto tiles = [&](int t) { return (int64_t)((M + t - 1) / t) * ((N + t - 1) / t) * batch; };
  const int64_t small = tiles(32);
  if (chunks < 16) return chunks >= 4 && small <= (chunks < 8 ? 512 : 1024);
  int64_t us;
  if (small <= 512) us = small <= 256 ? 16 : 32;
  else if (tiles(64) <= 256) us = 41;
  else rows_us(M, N, batch, us);
  return 100 * gemm_rm_split_us(M, N, batch) < 97 * us;
}

int gemm_rm_form_rows(int M, int N, int batch) {
  int64_t us = 0;
  return rows_us(M, N, batch, us);
}

}  // namespace dsse

extern "C" hipError_t dsse_gemm_rm(const dsse::GemmRmParams* p, hipStream_t st) {
  if (p->M <= 0 || p->N <= 0 || p->batch <= 0) return hipSuccess;
  return p->f32 ? dsse::dispatch<float>(*p, st) : dsse::dispatch<bf16>(*p, st);
}
