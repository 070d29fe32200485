// Prefill / wide-batch GEMM on the engine's tiled weight layout:  Y[M, N] = X[M, K] · W[N, K]ᵀ, M >= 128.
//
// The decode GEMMs (gemm_stream / gemm_wide) stream weights once into registers and are built for M <= 256.
// Prefill (thousands of rows) is compute-bound: here both operands go through LDS and every fragment read
// from LDS feeds several MFMAs (register blocking), the classic CDNA GEMM structure:
//
//   * workgroup tile BM x BN = (WM·MT·16) x (WN·NT·16), WM x WN waves, each wave an (MT·16) x (NT·16)
//     sub-tile of v_mfma_f32_16x16x32_bf16 accumulators; K steps of 64 (half a 128-deep weight chunk);
//   * LDS-DMA staging (global_load_lds_dwordx4: no VGPR round trip) into a 3-deep ring of stages with a
//     counted `s_waitcnt vmcnt` -- the loads of step t+1 stay in flight across the barrier that publishes
//     step t, and step t+2 is issued right after it (one barrier per K step, never vmcnt(0) in the loop);
//   * the weight tile needs no swizzle: a (16-column tile, 32-deep K step) block of the tiled layout is
//     1 KiB in MFMA B-fragment order (api.h kTileChunk), staged by one lane-linear DMA instruction and read
//     back lane-linearly (bank-conflict free);
//   * X rows (128 B per stage) are staged with an XOR swizzle on the SOURCE address (the DMA writes LDS
//     lane-linearly) and read with the same XOR: conflict-free A-fragment reads;
//   * the contraction order inside a 128-deep chunk is the tiled layout's (k-step s of lane group g covers
//     K = 32g + 8s + j), applied identically to X;
//   * XCD-aware, L2-grouped tile order: consecutive logical tiles (8 row blocks x a run of column blocks)
//     land on one XCD, so its L2 serves the shared X and W panels;
//   * the epilogues of the decode GEMMs (gemm_epilogue.h): bf16 / fp32 store, residual add, SiLU·mul of the
//     interleaved gate/up columns, QKV + RoPE + paged KV write -- prefill writes its outputs once, no
//     intermediate [T, N] tensors; split-K (grid.z = S) writes fp32 slabs for the wide decode path.
//
// Replaces the library GEMMs of round 1's prefill and wide decode path, which needed a second, standard
// layout copy of every weight (engine/weights.py).
#include "gemm_epilogue.h"
#include "lds_dma.h"

namespace dsse {

template <int WM, int WN, int MT, int NT, int NS>
struct TiledGeom {
  static constexpr int BM = WM * MT * 16, BN = WN * NT * 16, NTHR = 64 * WM * WN;
  static constexpr int A_BYTES = (BM + 8 * WM * WN - 1) / (8 * WM * WN) * (8 * WM * WN) * 128;  // 64 bf16 per row
  static constexpr int B_BYTES = (BN / 16) * 2048;    // two 1 KiB k-step blocks per 16-column tile
  static constexpr int STAGE = A_BYTES + B_BYTES;
  static constexpr int A_INS = A_BYTES / 1024 / (WM * WN);  // 1 KiB DMA instructions per wave per stage
  static constexpr int B_INS = B_BYTES / 1024 / (WM * WN);
  static_assert(A_BYTES % (1024 * WM * WN) == 0 && B_BYTES % (1024 * WM * WN) == 0, "stage not divisible");
  static constexpr size_t LDS = (size_t)NS * STAGE;
};

DEV void glds16(const void* src, char* lds_base) {
  __builtin_amdgcn_global_load_lds(const_cast<void*>(src),
                                   reinterpret_cast<__attribute__((address_space(3))) void*>(
                                       reinterpret_cast<uintptr_t>(lds_base)),
                                   16, 0, 0);
}


// NS: LDS stages (3: one stage's DMA stays in flight across the publishing barrier; 2: the next stage is issued
// after the barrier and waited for at the next one).  FB: 2 = both k sub-steps' fragments are read before the
// first MFMA (the second read's latency hides under the first MFMA cluster), 1 = one sub-step at a time.
#ifndef DSSE_TILED_BURST
#define DSSE_TILED_BURST 0
#endif
constexpr bool kBurst = DSSE_TILED_BURST;  // A/B build only: every tile issues its stage in one burst

// ROWS: one tile holds all rows (65 to 256, MT of 3 to 8 sub-tiles per wave row) and 128 columns, so that every weight is fetched
// once, non-temporal, and no row that is not there is fetched; four stages where they fit.  What bounds it is the LDS fill, 45 GB/s
// per CU of rows from L2 and weights from memory together: (rows + 128) x 128 bytes per K step.  Mistral's gate_up at 160 rows: 57 us (0.86 us per step) against
// 69 with two row blocks of 128 x 256; with 192 rows computed for 160 the same, with 256 66.  A column
// block begins at a K step of its own and wraps around: X has just been written on other XCDs, and workgroups that ask for different
// parts of it bring it into their XCD's L2 for each other (160-stream decode step 6201 -> 6075 us, 200-row prompt 6277 -> 6108).

template <int WM, int WN, int MT, int NT, int NS, int FB, int MODE, bool ROWS = false>
__global__ void __launch_bounds__(64 * WM * WN)
gemm_tiled_kernel(const bf16* __restrict__ X, int ldx, int M, const bf16* __restrict__ W, int K, int N, int Kr,
                  GemmEpi ep, float* __restrict__ part) {
  using G = TiledGeom<WM, WN, MT, NT, NS>;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
  const int r = lane & 15, g = lane >> 4;
  const int wm = w / WN, wn = w % WN;

  // ---- tile order: XCD remap (bijective), then groups of 8 row blocks swept column by column
  const int nbm = (M + G::BM - 1) / G::BM, nbn = N / G::BN, ntile = nbm * nbn;
  const int nwg = gridDim.x;
  const int bid = blockIdx.x, xcd = bid % 8, q8 = nwg / 8, rem = nwg % 8;
  const int lid = (xcd < rem ? xcd * (q8 + 1) : rem * (q8 + 1) + (xcd - rem) * q8) + bid / 8;
  const int ks = lid / ntile, tl = lid % ntile;
  constexpr int GM = 8;
  const int grp = tl / (GM * nbn), first = grp * GM, gsz = min(GM, nbm - first);
  const int bm = first + (tl % (GM * nbn)) % gsz, bn = (tl % (GM * nbn)) / gsz;

  const int m0 = bm * G::BM, n0 = bn * G::BN;
  const int k0 = ks * Kr, nk = Kr >> 6;
  const int KC = K >> 7;

  // ---- per-thread DMA sources (stage-invariant parts)
  // A: instruction i of this wave covers LDS rows 8·(w·A_INS + i) .. +8; lane -> (row, slot q)
  const bf16* a_src[G::A_INS];
  int a_koff[G::A_INS];
#pragma unroll
  for (int i = 0; i < G::A_INS; ++i) {
    const int row = (w * G::A_INS + i) * 8 + (lane >> 3);
    const int p = (lane & 7) ^ piece_swizzle(row);  // X piece p = 2g' + s' -> K offset 32g' + 8s' (+16h per half chunk)
    a_src[i] = X + (size_t)min(m0 + row, M - 1) * ldx;
    a_koff[i] = 32 * (p >> 1) + 8 * (p & 1);
  }
  // B: instruction i covers (tile, k-step) block j = w·B_INS + i of the stage: tile j >> 1, sub-step j & 1
  const bf16* b_src[G::B_INS];
#pragma unroll
  for (int i = 0; i < G::B_INS; ++i) {
    const int j = w * G::B_INS + i;
    b_src[i] = W + ((size_t)(n0 / 16 + (j >> 1)) * KC) * kTileChunk + (j & 1) * 512 + lane * 8;
  }

  // ROWS: the same places as offsets into buffers, where rows that do not exist land as zeros without traffic
  const __amdgpu_buffer_rsrc_t xr = make_rsrc(X, (uint32_t)((size_t)M * ldx * 2));
  const __amdgpu_buffer_rsrc_t wr = make_rsrc(W + (size_t)(n0 / 16) * KC * kTileChunk, (uint32_t)(G::BN / 16) * KC * kTileChunk * 2);
  uint32_t a_vo[G::A_INS], b_vo[G::B_INS];
#pragma unroll
  for (int i = 0; i < G::A_INS; ++i) {
    const int row = m0 + (w * G::A_INS + i) * 8 + (lane >> 3);
    a_vo[i] = row < M ? (uint32_t)(row * ldx + a_koff[i]) * 2 : kOOB;
  }
#pragma unroll
  for (int i = 0; i < G::B_INS; ++i) {
    const int j = w * G::B_INS + i;
    b_vo[i] = (uint32_t)((j >> 1) * KC * kTileChunk + (j & 1) * 512 + lane * 8) * 2;
  }
  const int turn = ROWS ? bn % nk : 0;  // the K step this workgroup begins at; it wraps around
  auto issue_a = [&](int stage, int t) {
    t = t + turn < nk ? t + turn : t + turn - nk;
    const int kk = k0 + 64 * t, c = kk >> 7, h = (kk >> 6) & 1;
    char* base = smem + stage * G::STAGE;
    if constexpr (ROWS) {
#pragma unroll
      for (int i = 0; i < G::A_INS; ++i) lds_dma(xr, base + (w * G::A_INS + i) * 1024, a_vo[i], (uint32_t)(c * 128 + 16 * h) * 2);
      return;
    }
#pragma unroll
    for (int i = 0; i < G::A_INS; ++i)
      glds16(a_src[i] + c * 128 + 16 * h + a_koff[i], base + (w * G::A_INS + i) * 1024);
  };
  auto issue_b = [&](int stage, int t) {
    t = t + turn < nk ? t + turn : t + turn - nk;
    const int kk = k0 + 64 * t, c = kk >> 7, h = (kk >> 6) & 1;
    char* base = smem + stage * G::STAGE;
    if constexpr (ROWS) {
#pragma unroll
      for (int i = 0; i < G::B_INS; ++i)
        lds_dma<kAuxNT>(wr, base + G::A_BYTES + (w * G::B_INS + i) * 1024, b_vo[i], (uint32_t)(c * kTileChunk + h * 1024) * 2);
      return;
    }
#pragma unroll
    for (int i = 0; i < G::B_INS; ++i)
      glds16(b_src[i] + (size_t)c * kTileChunk + h * 1024, base + G::A_BYTES + (w * G::B_INS + i) * 1024);
  };
  auto issue = [&](int stage, int t) {
    issue_a(stage, t);
    issue_b(stage, t);
  };

  f32x4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

  // A-fragment LDS offsets (row-dependent swizzle) for k sub-step s' of a stage: piece 2g + s'
  int a_off[MT][2];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int row = wm * MT * 16 + 16 * mt + r;
#pragma unroll
    for (int sp = 0; sp < 2; ++sp) a_off[mt][sp] = row * 128 + (((2 * g + sp) ^ piece_swizzle(row)) << 4);
  }

  constexpr int INS = G::A_INS + G::B_INS;
  static_assert(NS >= 2 && NS <= 4, "2-4 LDS stages");
  issue(0, 0);
  if (NS >= 3 && nk > 1) issue(1, 1);
  if (NS == 4 && nk > 2) issue(2, 2);
  for (int t = 0; t < nk; ++t) {
    // step t's DMA done on this wave (steps t+1 .. t+NS-2 may stay in flight) and its fragments of step t-1 in registers, then
    // everyone's: publish step t
    const int younger = min(NS - 2, nk - 1 - t);
    if (NS == 4 && younger == 2) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * INS) : "memory");
    else if (NS >= 3 && younger >= 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(INS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // the stage step t+NS-1 overwrites was last read in step t-1, which every wave finished before this barrier.
    // 128x256 tile (the weight-heavy 129-256-row decode buckets): its X half goes out now, its weight half between
    // the two MFMA clusters, so the DMA issue is spread over the step (the order gemm_pipe.hip measured faster):
    // gate_up at 256 rows 74.9 vs 80.0 us, down 52.7 vs 54.9.  The 128x128 tile measured slower spread (qkv 256
    // rows 36.5 vs 33.6, o 26.6 vs 25.2) and 256x128 even, so those issue the stage in one burst
    // (profiles/r5/gemm_pipe_r5.md, tiled_ab_r5.log)
    constexpr bool spread = FB == 2 && WM == 2 && WN == 4 && !kBurst;
    const bool more = t + NS - 1 < nk;
    if (more) {
      if constexpr (spread) issue_a((t + NS - 1) % NS, t + NS - 1);
      else issue((t + NS - 1) % NS, t + NS - 1);
    }
    const char* As = smem + (t % NS) * G::STAGE;
    const char* Bs = As + G::A_BYTES;
    auto read = [&](int sp, bf16x8 (&a)[MT], bf16x8 (&b)[NT]) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        b[nt] = *reinterpret_cast<const bf16x8*>(Bs + (wn * NT + nt) * 2048 + sp * 1024 + lane * 16);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) a[mt] = *reinterpret_cast<const bf16x8*>(As + a_off[mt][sp]);
    };
    auto mma = [&](const bf16x8 (&a)[MT], const bf16x8 (&b)[NT]) {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = mfma16x16x32(a[mt], b[nt], acc[mt][nt]);
      __builtin_amdgcn_s_setprio(0);
    };
    if constexpr (FB == 2) {
      bf16x8 a0[MT], b0[NT], a1[MT], b1[NT];
      read(0, a0, b0);
      read(1, a1, b1);
      mma(a0, b0);
      if (spread && more) issue_b((t + NS - 1) % NS, t + NS - 1);
      mma(a1, b1);
    } else {
#pragma unroll
      for (int sp = 0; sp < 2; ++sp) {
        bf16x8 a[MT], b[NT];
        read(sp, a, b);
        mma(a, b);
      }
    }
  }

  float* part_ks = partial_of(ep, part, ks, M, N);
  const int row0 = m0 + wm * MT * 16, tile0 = n0 / 16 + wn * NT;
  if constexpr (MODE == kSiluMul) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) silu_epilogue4(ep, M, row0 + 16 * mt + 4 * g, tile0 + nt, r, acc[mt][nt]);
    return;
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = acc[mt][nt][i];
        const float partner = (MODE == kSiluMul || MODE == kQkvRope) ? __shfl_xor(v, 8) : 0.f;
        epilogue<MODE>(ep, part_ks, M, N, row0 + 16 * mt + 4 * g + i, tile0 + nt, r, v, partner);
      }
}

template <int WM, int WN, int MT, int NT, int NS, int FB, int MODE, bool ROWS = false>
static hipError_t launch_t(const bf16* X, int ldx, int M, const bf16* W, int K, int N, int S, const GemmEpi& ep,
                           float* part, hipStream_t st) {
  using G = TiledGeom<WM, WN, MT, NT, NS>;
  static bool attr_set = false;
  if (!attr_set) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_tiled_kernel<WM, WN, MT, NT, NS, FB, MODE, ROWS>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)G::LDS);
    attr_set = true;
  }
  const int nbm = (M + G::BM - 1) / G::BM, nbn = N / G::BN;
  hipLaunchKernelGGL((gemm_tiled_kernel<WM, WN, MT, NT, NS, FB, MODE, ROWS>), dim3(nbm * nbn * S), dim3(G::NTHR), G::LDS, st,
                     X, ldx, M, W, K, N, K / S, ep, part);
  return hipGetLastError();
}

template <int MODE>
static hipError_t launch_t_mode(int cfg, const bf16* X, int ldx, int M, const bf16* W, int K, int N, int S,
                                const GemmEpi& ep, float* part, hipStream_t st) {
  switch (cfg) {
    // measured on MI355X (profiles/r2/gemm_tiled_v*.log); other tile / ring shapes tried and removed are listed
    // in profiles/experiments_r2.md; the 256 x 256 configurations moved to gemm_pipe.hip (cfg 8, round 5)
    case 0: return launch_t<4, 2, 4, 4, 3, 2, MODE>(X, ldx, M, W, K, N, S, ep, part, st);  // 256 x 128, 8 waves
    case 1: return launch_t<2, 2, 4, 4, 3, 2, MODE>(X, ldx, M, W, K, N, S, ep, part, st);  // 128 x 128, 4 waves
    case 2:  // 65-256 rows, all in one tile x 128 columns, 8 waves
      switch ((M + 31) / 32) {
        case 3: return launch_t<2, 4, 3, 2, 4, 2, MODE, true>(X, ldx, M, W, K, N, S, ep, part, st);
        case 4: return launch_t<2, 4, 4, 2, 4, 2, MODE, true>(X, ldx, M, W, K, N, S, ep, part, st);
        case 5: return launch_t<2, 4, 5, 2, 4, 2, MODE, true>(X, ldx, M, W, K, N, S, ep, part, st);
        case 6: return launch_t<2, 4, 6, 2, 4, 2, MODE, true>(X, ldx, M, W, K, N, S, ep, part, st);
        case 7: return launch_t<2, 4, 7, 2, 3, 2, MODE, true>(X, ldx, M, W, K, N, S, ep, part, st);
        case 8: return launch_t<2, 4, 8, 2, 3, 2, MODE, true>(X, ldx, M, W, K, N, S, ep, part, st);
      }
      return hipErrorInvalidValue;
    case 5: return launch_t<2, 4, 4, 4, 3, 2, MODE>(X, ldx, M, W, K, N, S, ep, part, st);  // 128 x 256, 8 waves
  }
  return hipErrorInvalidValue;
}

}  // namespace dsse

// cfg: 0 = 256 x 128 tile (8 waves, 3 LDS stages), 1 = 128 x 128 (4 waves), 2 = 65-256 rows x 128 (8 waves, 4 or 3 stages), 5 = 128 x 256 (8 waves, 3 stages of 16
// KiB X + 32 KiB W: twice the weight bytes in flight per CU of cfg 0, for the weight-streaming 129-256-row decode
// GEMMs; the two row blocks of a column block share an XCD and its L2).  (256 x 256 configurations are
// gone: gemm_pipe.hip, cfg 8, replaces them.)
// (Round 3 also tried 4-stage rings and separate X / W loader rings for the 129-512-row decode buckets: all
// slower in the 256-stream step, removed; profiles/r3/experiments_r3.md.)
// Shape contract (checked by the caller): N % BN == 0, K % (64 S) == 0, the tiled weight layout (api.h).
// S > 1: fp32 slabs [S, M, N] into `part`, reduced by launch_splitk_reduce unless partial_only.
extern "C" hipError_t dsse_gemm_tiled(int mode, int cfg, int S, int partial_only, const void* X, int ldx, int M,
                                      const void* W, int K, int N, const dsse::GemmEpi* ep, float* part,
                                      hipStream_t st) {
  using namespace dsse;
  const bf16* x = reinterpret_cast<const bf16*>(X);
  const bf16* w = reinterpret_cast<const bf16*>(W);
  if (S == 1 && !partial_only) {
    switch (mode) {
      case kStoreBf16: return launch_t_mode<kStoreBf16>(cfg, x, ldx, M, w, K, N, 1, *ep, nullptr, st);
      case kStoreF32: return launch_t_mode<kStoreF32>(cfg, x, ldx, M, w, K, N, 1, *ep, nullptr, st);
      case kResidAdd: return launch_t_mode<kResidAdd>(cfg, x, ldx, M, w, K, N, 1, *ep, nullptr, st);
      case kSiluMul: return launch_t_mode<kSiluMul>(cfg, x, ldx, M, w, K, N, 1, *ep, nullptr, st);
      case kQkvRope: return launch_t_mode<kQkvRope>(cfg, x, ldx, M, w, K, N, 1, *ep, nullptr, st);
    }
    return hipErrorInvalidValue;
  }
  hipError_t e = launch_t_mode<kPartial>(cfg, x, ldx, M, w, K, N, S, *ep, part, st);
  if (e != hipSuccess || partial_only) return e;
  return launch_splitk_reduce(mode, part, S, M, N, *ep, st);
}

DSSE_CHECK_READER(dsse_check_gemm_tiled)
