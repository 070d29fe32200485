// Prefill / wide GEMM, 256 (or 192 / 128) x 256 tile, deep LDS-DMA pipeline:  Y[M, N] = X[M, K] · W[N, K]ᵀ on the
// engine's tiled weight layout (api.h kTileChunk), M >= 128 (few tiles: split K, grid.z-style slices in the tile
// index).
//
// Why a new schedule (profiles/r4/pmc_gemm_r4.md): gemm_phased (gemm_tiled.hip cfg 4) issued the last A half of step
// t+1 one phase before the counted wait that needed it, so every K step waited ~a full L2/HBM round trip -- 44 %
// MFMA-busy, 42 % of wave time waiting on a dependency at 8192 rows.  Here every half-tile is in flight for five
// phases (~2,500 cycles) before any wave waits for it:
//
//   * 8 waves = 2 wave rows (128 rows each) x 4 wave columns (64 columns each); a wave's 128 x 64 tile is four
//     64 x 32 quadrants; a K step of 64 runs as four phases, one quadrant (16 MFMAs 16x16x32) per phase:
//         phase 0  quadrant (0, 0)   reads A rows q0 + B cols q0   issue  B-half 1 of step t+1
//         phase 1  quadrant (0, 1)   reads B cols q1                issue  A-half 1 of step t+1
//         phase 2  quadrant (1, 1)   reads A rows q1                issue  A-half 0 of step t+2
//         phase 3  quadrant (1, 0)   (operands in registers)        issue  B-half 0 of step t+2
//     one half-tile per phase (round 5: +1-5 % at 8192 rows, +2-10 % at 2048 over the round-5 first form that issued
//     0 / 1 / 2 / 1 half-tiles in phases 1 / 0 / 2 / 3, profiles/r5/pipe_even_ab_r5.log),
//     each phase = [fragment reads, DMA issue, counted vmcnt] s_barrier lgkmcnt(0) [16 MFMAs, prio 1] s_barrier,
//     with the two wave rows one barrier apart, so on every SIMD one wave's MFMA cluster overlaps the other's LDS
//     reads (the 8-phase template of the CDNA HIP guide, §5; the half-tile order is this kernel's own);
//   * a "half-tile" is what one phase's quadrant reads across the workgroup: A-half q = the 64-row quadrant q of
//     BOTH wave rows (128 rows x 128 B = 16 KiB), B-half q = the 32-column quadrant q of all four wave columns
//     (8 column tiles x 2 KiB); each is 16 one-KiB LDS-DMA instructions, two per wave;
//   * WAR: a half is re-staged >= 2 phases after its last read (A0 / B0 of buffer t & 1 read in phase 0 of t,
//     re-staged for t+2 in phases 2 / 3; B1 of buffer (t+1) & 1 last read in phase 1 of t-1, re-staged in phase 0 of
//     t; A1 read in phase 2 of t-1, re-staged in phase 1 of t) -- the lagging wave row is then still >= 1 barrier
//     past its lgkmcnt(0);
//   * RAW: counted waits, 8 in each of phases 0, 1 and 3 (four half-tiles of 2 instructions each younger than the
//     one retired): phase 0 retires B-half 1 of step t, phase 1 A-half 1 of t, phase 3 A0 / B0 of t+1 -- each in the
//     phase before its first read, so the lagging row has passed it one barrier before the leading row reads (never
//     vmcnt(0) in the steady loop);
//   * buffer-load LDS-DMA: one SGPR offset per K step, per-lane offsets fixed for the whole loop (no per-step VALU
//     address arithmetic); rows past M read as zeros (out-of-range offsets, no memory traffic); the last two steps
//     issue nothing past the end and count their waits exactly;
//   * XCD-aware tile order (bijective remap, groups of 8 row blocks swept by column) as gemm_tiled.hip;
//   * epilogues: bf16 results and SiLU / GELU·mul through a wave's own 4 KiB of LDS (16-byte row stores), fp32 / residual / QKV+RoPE /
//     split-K partial slabs through gemm_epilogue.h;
//   * from three rounds of tiles on most workgroups take two (pairs_of): the requests past the first tile's last step are the second
//     one's first, and the first one's results leave while they are under way.  One tile each / this, one MI355X, us: 8192 x 28672 x 4096 SiLU
//     1410 / 1397, 8192 x 28672 x 2048 775 / 765, x 1024 466 / 446; 3000 x 28672 x 4096 565 / 564, 3000 x 16384 x 2048 GELU 167 / 164.
#include <algorithm>
#include <type_traits>

#include "gemm_epilogue.h"
#include "lds_dma.h"

#ifndef DSSE_PIPE_STAMPS
#define DSSE_PIPE_STAMPS 0
#endif

namespace dsse {
namespace gp {

// Diagnostic build only (_build.py variant "stamps"): workgroup-level s_memrealtime stamps (100 MHz, one clock for
// every CU) of the FIX path's phases after the fix-up counters: [wg][8] u64 (tools/pipe_stamps.py)
DEV void stamp(const GemmEpi& ep, int k, unsigned long long v) {
  if constexpr (DSSE_PIPE_STAMPS) {
    if (threadIdx.x == 0 && ep.fix_cnt)
      reinterpret_cast<unsigned long long*>(ep.fix_cnt + kStampOff)[(size_t)blockIdx.x * 8 + k] = v;
  }
}
DEV unsigned long long now() { return DSSE_PIPE_STAMPS ? __builtin_amdgcn_s_memrealtime() : 0ull; }

constexpr int kA = 256 * 128;     // A image of one K step: 256 rows x 64 bf16, swizzled 16-byte pieces
constexpr int kB = 16 * 2048;     // B image: 16 column tiles x two 1 KiB k-step blocks
constexpr int kBuf = kA + kB;     // 64 KiB per K step
constexpr int kStage = 4096;      // a wave's rows of the result on their way to 16-byte stores, beside the two images
constexpr int kCUs = 256;

// bf16 results: products with the weights as their first operand, so that a lane has four columns of a row, and rows that leave through LDS as 16-byte
// stores, this many per tile and wave, those of rows and columns that are not there included (past their descriptor's range).  0: fp32 results and
// scattered ones, a row's 16 columns in 16 lanes.  (fp32 slabs as 16-byte stores, straight or through LDS: 1024 x 2048 x 2048 17.3 / 20.0 / 17.9 us, 2048 x
// 4096 x 4096 61.5 / 63.7 / 59.7.)
template <int MODE, int QI>
constexpr int stores() {
  return MODE == kStoreBf16 ? 4 * QI : MODE == kSiluMul ? 2 * QI : 0;
}

// How many times kCUs workgroups of a launch of n tiles take two tiles each: as long as a round of single tiles follows.  Which CU a workgroup gets is decided
// when one is free, so a CU that another stream holds (the collectives beside a tensor-parallel prompt) costs what it does without pairs: with one workgroup
// per CU for all rounds, 8192 x 28672 x 4096 beside 16 held CUs took 2417 us and not 1574, 3000 rows 983 and not 633; with pairs up to the last
// tile, 8192 x 4096 x 4096 332 and not 267.  In time units of a tile, no count of tiles from 512 to 4096 ends later beside 8 to 64 held CUs than without pairs.
inline int pairs_of(int n) { return n < kCUs ? 0 : (n - kCUs) / (2 * kCUs); }

template <int MODE, int QI>
constexpr size_t lds() {
  return 2 * (size_t)kBuf + (stores<MODE, QI>() > 0 ? 8 * kStage : 0);
}

// Whether 16 bytes of a bf16 result row are one aligned store
__host__ __device__ inline bool wide_results(const GemmEpi& ep) {
  return reinterpret_cast<uintptr_t>(ep.out) % 16 == 0 && ep.ldo % 8 == 0;
}

}  // namespace gp

// BM: rows per workgroup tile, 256, 192 or 128.  192 / 128 keep the 256-row LDS image and schedule and fill 48 / 32
// of every 64-row quadrant (the other slot rows load as zeros, no traffic, and no MFMA reads them): 12 / 8 MFMAs per
// phase instead of 16, for row counts that leave a 256-row block partly empty (the mixed prefill + decode steps'
// 320-384 rows: 192; the 161-256-row decode buckets' qkv / down: 192 / 128).  Slot row s of quadrant q, wave row wr
// holds X row m0 + wr * BM / 2 + q * BM / 4 + s.
// FIX (round 6): split-K with the slices of a tile combined inside the launch, no reduce kernel and no slabs for the
// consumer.  Ticket first: after its K loop every workgroup takes a ticket on the tile's arrival counter; the
// first S - 1 store their fp32 accumulators (16-byte stores in the MFMA register order, 1 KiB per wave instruction,
// read back by the same lanes) into slot `ticket` of the tile's workspace, drain, release, and count themselves
// done (a tile's slices are adjacent in the remapped order, so they share an XCD and its L2); the workgroup that draws ticket S - 1 waits (bounded) until the others are done -- they are
// running already and wait for nothing, so this cannot deadlock whatever the residency -- adds their slots into
// its registers and runs the normal epilogue.  The slab round trip costs (S - 1) x the tile's fp32 bytes once, on
// the tile's last arriver (profiles/r6/gemm_fix_r6.md).
template <int MODE, int BM, bool FIX = false>
__global__ void __launch_bounds__(512)
gemm_pipe_kernel(const bf16* __restrict__ X, int ldx, int M, const bf16* __restrict__ W, int K, int N, int Kr,
                 GemmEpi ep, float* __restrict__ part, int pairs) {
  using namespace gp;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int wm = w >> 2, wn = w & 3;
  if constexpr (FIX) stamp(ep, 0, now());

  // ---- tile order: bijective XCD remap, then groups of 8 row blocks swept column by column (L2 panel reuse)
  constexpr int QR = BM / 4, QI = QR / 16;  // X rows per quadrant, MFMA row tiles per quadrant
  static_assert(BM == 256 || BM == 192 || BM == 128, "row tile");
  const int nbm = (M + BM - 1) / BM, nbn = (N + 255) / 256, ntile = nbm * nbn;
  // split slices: FIX keeps a tile's S slices adjacent in the remapped order, so they run on one XCD and the last
  // arriver reads the other slices' plain-stored slots from its own L2; the slab form (consumer-reduced) keeps
  // them ntile apart
  const int S_ = K / Kr, nwg = ntile * S_, nk = Kr >> 6, KC = K >> 7;
  struct Tile {
    int m0, n0, ks, tl;
  };
  auto decode = [&](int bid) {
    constexpr int GM = 8;
    const int xcd = bid % 8, q8 = nwg / 8, rem = nwg % 8;
    const int lid = (xcd < rem ? xcd * (q8 + 1) : rem * (q8 + 1) + (xcd - rem) * q8) + bid / 8;
    const int ks = FIX ? lid % S_ : lid / ntile, tl = FIX ? lid / S_ : lid % ntile;
    const int grp = tl / (GM * nbn), first = grp * GM, gsz = min(GM, nbm - first);
    return Tile{(first + (tl % (GM * nbn)) % gsz) * BM, (tl % (GM * nbn)) / gsz * 256, ks, tl};
  };
  // the first `pairs` times kCUs workgroups take two tiles each, kCUs apart, the others one
  const bool two = (int)blockIdx.x < pairs * kCUs;
  int bid = two ? blockIdx.x + blockIdx.x / kCUs * kCUs : blockIdx.x + pairs * kCUs;
  const int second = bid + kCUs;
  Tile at = decode(bid);

  const __amdgpu_buffer_rsrc_t xr = make_rsrc(X, (uint32_t)(((size_t)(M - 1) * ldx + K) * 2));
  const __amdgpu_buffer_rsrc_t wr = make_rsrc(W, (uint32_t)((size_t)N * K * 2));

  // ---- per-lane DMA offsets (bytes), fixed for a tile's K loop: [half q][instruction i] of this wave
  uint32_t a_vo[2][2], b_vo[2][2];
  int a_lo[2][2], b_lo[2][2];  // LDS byte offsets inside a buffer
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int j = 2 * w + i;  // instruction j of the 16 of this half
      a_lo[q][i] = ((j >> 3) * 128 + q * 64 + (j & 7) * 8) * 128;
      b_lo[q][i] = kA + ((j >> 2) * 4 + q * 2 + ((j >> 1) & 1)) * 2048 + (j & 1) * 1024;
    }
  auto offsets = [&](const Tile& to) {
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int j = 2 * w + i;
        const int row = (j >> 3) * 128 + q * 64 + (j & 7) * 8 + (lane >> 3), sr = (j & 7) * 8 + (lane >> 3);  // LDS slot row, slot row in the quadrant
        const int xrow = to.m0 + (j >> 3) * (BM / 2) + q * QR + sr;                                       // the X row it holds
        const int pc = (lane & 7) ^ piece_swizzle(row);
        a_vo[q][i] = sr < QR && xrow < M ? (uint32_t)(((size_t)xrow * ldx + 32 * (pc >> 1) + 8 * (pc & 1)) * 2) : kOOB;
        const int tb = (j >> 2) * 4 + q * 2 + ((j >> 1) & 1), sub = j & 1;  // column tile of the block, k sub-step
        b_vo[q][i] = to.n0 + 16 * tb < N ? (uint32_t)((((size_t)(to.n0 / 16 + tb) * KC) * kTileChunk + sub * 512 + lane * 8) * 2) : kOOB;
      }
  };
  offsets(at);
  // K steps count on from tile to tile; step t lies at column kk: X columns 128c + 16h + (piece offsets), W chunk c, k sub-steps 2h, 2h+1
  int k_at = at.ks * Kr;  // column of step 0, had the tile begun there
  auto issue_a = [&](int q, int t) {
    char* base = smem + (t & 1) * kBuf;
    const int kk = k_at + 64 * t;
    const uint32_t so = __builtin_amdgcn_readfirstlane((uint32_t)(((kk >> 7) * 128 + 16 * ((kk >> 6) & 1)) * 2));
#pragma unroll
    for (int i = 0; i < 2; ++i) lds_dma(xr, base + a_lo[q][i], a_vo[q][i], so);
  };
  auto issue_b = [&](int q, int t) {
    char* base = smem + (t & 1) * kBuf;
    const int kk = k_at + 64 * t;
    const uint32_t so = __builtin_amdgcn_readfirstlane((uint32_t)(((kk >> 7) * kTileChunk + ((kk >> 6) & 1) * 1024) * 2));
#pragma unroll
    for (int i = 0; i < 2; ++i) lds_dma(wr, base + b_lo[q][i], b_vo[q][i], so);
  };

  // ---- fragment reads: A rows wm*128 + 64 qm + 16 i + r (the swizzle is the same for every i), B column tiles
  // wn*4 + 2 qn + i, k sub-step sp of the step
  int a_rd[2];
#pragma unroll
  for (int sp = 0; sp < 2; ++sp) {
    const int row = wm * 128 + r;
    a_rd[sp] = row * 128 + (((2 * g + sp) ^ piece_swizzle(row)) << 4);
  }
  constexpr bool kTurned = stores<MODE, QI>() > 0;
  f32x4 acc[8][4];
  bf16x8 a[4][2], b[4][2];
  auto read_a = [&](const char* buf, int qm) {
#pragma unroll
    for (int i = 0; i < QI; ++i)
#pragma unroll
      for (int sp = 0; sp < 2; ++sp)
        a[i][sp] = *reinterpret_cast<const bf16x8*>(buf + a_rd[sp] + (64 * qm + 16 * i) * 128);
  };
  auto read_b = [&](const char* buf, int qn) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int sp = 0; sp < 2; ++sp)
        b[2 * qn + i][sp] =
            *reinterpret_cast<const bf16x8*>(buf + kA + (wn * 4 + 2 * qn + i) * 2048 + sp * 1024 + lane * 16);
  };
  auto mma = [&](int qm, int qn) {
    asm volatile("s_barrier\n\ts_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int sp = 0; sp < 2; ++sp)
#pragma unroll
      for (int i = 0; i < QI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[4 * qm + i][2 * qn + j] = kTurned ? mfma16x16x32(b[2 * qn + j][sp], a[i][sp], acc[4 * qm + i][2 * qn + j])
                                                : mfma16x16x32(a[i][sp], b[2 * qn + j][sp], acc[4 * qm + i][2 * qn + j]);
    __builtin_amdgcn_s_setprio(0);
    asm volatile("s_barrier" ::: "memory");
  };

  // prologue: step 0 whole, then A0 / B0 of step 1 (its B1 / A1 go out in phases 0 / 1 of step 0)
  issue_a(0, 0);
  issue_b(0, 0);
  issue_b(1, 0);
  issue_a(1, 0);
  issue_a(0, 1);
  issue_b(0, 1);
  asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory");  // A0 / B0 of step 0 landed everywhere
  if (wm == 1) asm volatile("s_barrier" ::: "memory");  // wave row 1 runs one barrier behind row 0
  // A workgroup goes on to its second tile without a pause: the requests past the first one's last step are those of the second one's first, and the
  // first one's results leave while they are under way.
  int t0 = 0;  // the tile's first step
  for (;; t0 += nk) {
    const bool more = !FIX && stores<MODE, QI>() > 0 && two && bid < second;  // uniform
    const Tile next = decode(more ? second : bid);
#pragma unroll
    for (int mt = 0; mt < 8; ++mt)
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    // TAIL 0 = steady, 1 = step t+1 exists but t+2 does not, 2 = last step.  RAW: B1(t) waited in phase 0 and read
    // in phase 1, A1(t) waited in 1 and read in 2, A0 / B0(t+1) waited in 3 and read in phase 0 of t+1 (the
    // barrier that opens the reading phase follows every wave's wait).  WAR: B1 of buffer (t+1)&1 was last read in
    // phase 1 of t-1, A1 in phase 2 of t-1, A0 / B0 of buffer t&1 in phase 0 of t -- each restaged >= 2 phases later.
    // OUT: stores of the tile before, which the wave has issued between the requests that are waited for here and the younger ones.
    auto step_even = [&](int t, auto tail_tag, auto out_tag) {
      constexpr int TAIL = decltype(tail_tag)::value, OUT = decltype(out_tag)::value;
      const char* buf = smem + (t & 1) * kBuf;
      read_a(buf, 0);
      read_b(buf, 0);
      if constexpr (TAIL < 2) {
        issue_b(1, t + 1);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 + OUT) : "memory");  // B-half 1 of step t
      } else {
        asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
      }
      mma(0, 0);
      read_b(buf, 1);
      if constexpr (TAIL < 2) {
        issue_a(1, t + 1);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 + OUT) : "memory");  // A-half 1 of step t
      } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      mma(0, 1);
      read_a(buf, 1);
      if (TAIL == 0 && OUT == 0 && t == t0 + nk - 2) {  // step t + 2 is the next tile's first
        offsets(next);
        k_at = next.ks * Kr - 64 * (t + 2);
      }
      if constexpr (TAIL == 0) issue_a(0, t + 2);
      mma(1, 1);
      if constexpr (TAIL == 0) {
        issue_b(0, t + 2);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 + OUT) : "memory");  // A0 / B0 of step t+1
      } else if constexpr (TAIL == 1) {
        asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      }
      mma(1, 0);
    };
    typedef std::integral_constant<int, 0> None;
    int t = t0;
    if constexpr (stores<MODE, QI>() > 0 && !FIX) {
      if (t0 > 0) step_even(t++, None{}, std::integral_constant<int, stores<MODE, QI>()>{});  // nk >= 4 (host contract)
    }
    const int end = t0 + (more ? nk : nk - 2);
    for (; t < end; ++t) step_even(t, None{}, None{});
    if (!more) {
      step_even(t++, std::integral_constant<int, 1>{}, None{});  // nk >= 2 (host contract)
      step_even(t, std::integral_constant<int, 2>{}, None{});
      // balance the barrier count of the two rows
      if (wm == 0) asm volatile("s_barrier" ::: "memory");
    }

  if constexpr (FIX) {
    const int S = S_;
    if (S > 1) {
      constexpr int kSlotF4 = 8 * 8 * QI * 64;  // f32x4 per slot: [wave][qm][i < QI][nt][lane]
      typedef __attribute__((address_space(1))) int gint;  // shared words: global agent-scope accesses, never flat
      gint* cnt = (gint*)(ep.fix_cnt) + 4;   // tickets [tl], done [kFixTiles + tl]; timeouts at [0]
      __syncthreads();  // every wave past its last LDS read: word 0 of the LDS carries the ticket
      stamp(ep, 1, now());
      int* sflag = reinterpret_cast<int*>(smem);
      if (threadIdx.x == 0) sflag[0] = __hip_atomic_fetch_add(cnt + at.tl, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      const int ticket = __builtin_amdgcn_readfirstlane(sflag[0]);  // wave-uniform: no waterfall around the rsrc
      stamp(ep, 2, now());
      if constexpr (DSSE_PIPE_STAMPS) {
        unsigned xcc;
        asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
        stamp(ep, 6, ((unsigned long long)ticket << 32) | (xcc & 0xF));
      }
      f32x4* slots = reinterpret_cast<f32x4*>(part) + (size_t)at.tl * (S - 1) * kSlotF4;
      const int lane_off = w * (8 * QI * 64) + lane;
      if (ticket < S - 1) {
        // plain stores (they stay in this XCD's L2 for the same-XCD reader), every wave drained, then ONE agent-scope
        // release and the done count (the CDNA guide's split-K recipe: fence before the count, wait after the fence)
        f32x4* dst = slots + (size_t)ticket * kSlotF4 + lane_off;
#pragma unroll
        for (int qm = 0; qm < 2; ++qm)
#pragma unroll
          for (int i = 0; i < QI; ++i)
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) dst[((qm * QI + i) * 4 + nt) * 64] = acc[4 * qm + i][nt];
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        stamp(ep, 3, now());
        if (threadIdx.x == 0) {
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          __hip_atomic_fetch_add(cnt + kFixTiles + at.tl, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        stamp(ep, 4, now());
        return;
      }
      if (threadIdx.x == 0) {
        unsigned spins = 0;
        while (__hip_atomic_load(cnt + kFixTiles + at.tl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < S - 1) {
          __builtin_amdgcn_s_sleep(2);
          if (++spins > (1u << 22)) {  // ~0.1 s: a writer never counted itself (cannot happen); flag, do not hang
            __hip_atomic_fetch_add(cnt - 4, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        // every other slice already took its ticket and counted itself: nothing touches this pair again in
        // this launch, so the last arriver leaves it zero for the next one
        __hip_atomic_store(cnt + at.tl, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(cnt + kFixTiles + at.tl, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      stamp(ep, 3, now());
      for (int s = 0; s < S - 1; ++s) {
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(slots + (size_t)s * kSlotF4, kSlotF4 * 16);
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          // 2 QI accumulators in flight at once (quadrant row h / 2, column pair h % 2), then the adds
          const int qm = h >> 1, n0 = 2 * (h & 1);
          f32x4 t[QI][2];
#pragma unroll
          for (int i = 0; i < QI; ++i)
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
              t[i][nt] = __builtin_bit_cast(
                  f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                             rs, (uint32_t)((lane_off + ((qm * QI + i) * 4 + n0 + nt) * 64) * 16), 0, 0));
#pragma unroll
          for (int i = 0; i < QI; ++i)
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) acc[4 * qm + i][n0 + nt] += t[i][nt];
        }
      }
      if constexpr (DSSE_PIPE_STAMPS) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        stamp(ep, 4, now());
      }
    }
  }

    // acc[4 qm + i][nt]: X rows row0 + QR qm + 16 i (i < QI), column tile tile0 + nt; turned, lane (r, g) has row r, columns 4 g .. 4 g + 3
    const int row0 = at.m0 + wm * (BM / 2), tile0 = at.n0 / 16 + wn * 4;
    const bool cols = tile0 * 16 < N;  // uniform; N % 128 == 0: a wave's 64 columns are all there or none is
    auto mt_of = [](int k) { return k / QI * 4 + k % QI; };  // k < 2 QI
    auto row_of = [&](int k) { return row0 + QR * (k / QI) + 16 * (k % QI); };
    if constexpr (MODE == kPartial || MODE == kStoreF32) {
      // a row's offset once for its four column tiles; rows that are not there are past the descriptor's range (a branch and an address per value / this, us:
      // 384 x 4096 x 4096 24.0 / 23.5, 300 x 2048 x 2048 12.6 / 12.3, 1500 x 2048 x 2048 21.4 / 21.1, 2048 x 4096 x 4096 63 / 61.5)
      if (!cols) return;
      const int ldo = MODE == kPartial ? (ep.parts ? ep.parts : 1) * N : ep.ldo;
      float* out = MODE == kPartial ? partial_of(ep, part, at.ks, M, N) : reinterpret_cast<float*>(ep.out);
      // a weight of up to 2 GiB has 2^23 columns at K = 128 (slices and all): a wave's rows span up to 127 * 4 * 2^23 bytes, so nearly all of a descriptor's 4 GiB
      constexpr uint32_t kPast = 0xfffffe00u;
      const __amdgpu_buffer_rsrc_t to = make_rsrc(out + (size_t)min(row0, M - 1) * ldo + tile0 * 16, kPast);
#pragma unroll
      for (int k = 0; k < 2 * QI; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = row_of(k) + 4 * g + i;
          const uint32_t row = m < M ? (uint32_t)(m - row0) * (uint32_t)ldo * 4 + 4 * r : kPast;
#pragma unroll
          for (int nt = 0; nt < 4; ++nt) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[mt_of(k)][nt][i]), to, row + 64 * nt, 0, 0);
        }
      if constexpr (FIX) stamp(ep, 5, now());
      return;
    }
    if (!kTurned || !wide_results(ep)) {  // uniform; such a launch has a workgroup per tile
      if (!cols) return;
      float* part_ks = partial_of(ep, part, at.ks, M, N);
#pragma unroll
      for (int k = 0; k < 2 * QI; ++k)
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float v = acc[mt_of(k)][nt][i];
            const float partner = MODE == kQkvRope || MODE == kSiluMul ? __shfl_xor(v, kTurned ? 32 : 8) : 0.f;
            epilogue<MODE>(ep, part_ks, M, N, row_of(k) + (kTurned ? r : 4 * g + i), tile0 + nt, kTurned ? 4 * g + i : r, v, partner);
          }
      if constexpr (FIX) stamp(ep, 5, now());
      return;
    }
    bf16* st = reinterpret_cast<bf16*>(smem + 2 * kBuf + w * kStage);
    // the wave's rows, from its first column on
    const int col0 = MODE == kSiluMul ? tile0 * 8 : tile0 * 16;
    const __amdgpu_buffer_rsrc_t to = make_rsrc(reinterpret_cast<bf16*>(ep.out) + (size_t)min(row0, M - 1) * ep.ldo + (cols ? col0 : 0), 0x7fffffffu);
    auto put = [&](const bf16x8& v, int m, int piece) {
      typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), to,
                                             cols && m < M ? (uint32_t)(m - row0) * (uint32_t)ep.ldo * 2 + 16 * piece : kOOB, 0, 0);
    };
    if constexpr (MODE == kStoreBf16) {
      // through the wave's LDS, 32 rows at a time: 16-byte row stores, 8 lanes per 128-byte row, 8 rows per instruction
#pragma unroll
      for (int k = 0; k < 2 * QI; k += 2) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int nt = 0; nt < 4; ++nt) {
            bf16x4 v;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = f2bf(acc[mt_of(k + u)][nt][i]);
            // piece 2 nt + g / 2 of row r at piece slot ^ (r & 7): conflict-spread writes and reads
            *reinterpret_cast<bf16x4*>(st + (16 * u + r) * 64 + (((2 * nt + (g >> 1)) ^ (r & 7)) << 3) + 4 * (g & 1)) = v;
          }
#pragma unroll
        for (int it = 0; it < 4; ++it) {
          const int rr = 8 * it + (lane >> 3), ch = lane & 7;
          const bf16x8 v = *reinterpret_cast<const bf16x8*>(st + rr * 64 + ((ch ^ (rr & 7)) << 3));
          put(v, row_of(k + (it >> 1)) + (rr & 15), ch);
        }
      }
    } else if constexpr (MODE == kSiluMul) {
      // gate rows 0-7 and up rows 8-15 of a column tile: lanes 0-31 and 32-63.  Of two row tiles, the lower lanes take the first and the upper ones the second.
#pragma unroll
      for (int k = 0; k < 2 * QI; k += 2) {
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
          bf16x4 v;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[mt_of(k)][nt][i]), __float_as_uint(acc[mt_of(k + 1)][nt][i]), false, false);
            v[i] = f2bf(gate_act(ep, __uint_as_float(x[0])) * __uint_as_float(x[1]));
          }
          const int rr = 16 * (g >> 1) + r;  // 32 rows of four 16-byte pieces
          *reinterpret_cast<bf16x4*>(st + rr * 32 + ((nt ^ (rr >> 1 & 3)) << 3) + 4 * (g & 1)) = v;
        }
#pragma unroll
        for (int it = 0; it < 2; ++it) {
          const int rr = 16 * it + (lane >> 2), ch = lane & 3;
          const bf16x8 v = *reinterpret_cast<const bf16x8*>(st + rr * 32 + ((ch ^ (rr >> 1 & 3)) << 3));
          put(v, row_of(k + it) + (rr & 15), ch);
        }
      }
    }
    if constexpr (FIX) stamp(ep, 5, now());
    if (!more) return;
    bid = second;
    at = next;
  }
}

template <int MODE, int BM, bool FIX>
static hipError_t launch_pipe_bm(const bf16* X, int ldx, int M, const bf16* W, int K, int N, int S, const GemmEpi& ep,
                                 float* part, hipStream_t st) {
  constexpr size_t kLDS = gp::lds<MODE, BM / 64>();
  static bool attr_set = false;
  if (!attr_set) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_pipe_kernel<MODE, BM, FIX>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLDS);
    attr_set = true;
  }
  const int nbm = (M + BM - 1) / BM, nbn = (N + 255) / 256, n = nbm * nbn * S;
  const int pairs = !FIX && gp::stores<MODE, BM / 64>() > 0 && K / S >= 256 && gp::wide_results(ep) && kernel_cfg_int("pipe_stay", 1) ? gp::pairs_of(n) : 0;
  hipLaunchKernelGGL((gemm_pipe_kernel<MODE, BM, FIX>), dim3(n - pairs * gp::kCUs), dim3(512), kLDS, st, X, ldx, M, W, K,
                     N, K / S, ep, part, pairs);
  return hipGetLastError();
}
template <int MODE, bool FIX = false>
static hipError_t launch_pipe(int bm, const bf16* X, int ldx, int M, const bf16* W, int K, int N, int S,
                              const GemmEpi& ep, float* part, hipStream_t st) {
  if (bm == 128) return launch_pipe_bm<MODE, 128, FIX>(X, ldx, M, W, K, N, S, ep, part, st);
  return bm == 192 ? launch_pipe_bm<MODE, 192, FIX>(X, ldx, M, W, K, N, S, ep, part, st)
                   : launch_pipe_bm<MODE, 256, FIX>(X, ldx, M, W, K, N, S, ep, part, st);
}

}  // namespace dsse

// Shape contract (checked here): N % 128 == 0 (the last column block may be half empty: zeros loaded, nothing stored), K % (128 S) == 0 (>= 2 K steps of 64 per slice), the tiled weight
// layout (api.h), X rows of ldx >= K elements.  S > 1: partial_only 0 = fp32 slabs [S, M, N] into `part` reduced by
// launch_splitk_reduce, 1 = the slabs only (the consumer reduces them), 2 = in-launch fix-up (FIX above): `part`
// holds dsse_gemm_pipe_fix_floats() floats and ep->fix_cnt the counters (api.h), tiles <= kFixTiles.
extern "C" hipError_t dsse_gemm_pipe(int mode, int bm, int S, int partial_only, const void* X, int ldx, int M,
                                     const void* W, int K, int N, const dsse::GemmEpi* ep, float* part, hipStream_t st) {
  using namespace dsse;
  if (M < 1 || N % 128 != 0 || S < 1 || K % (128 * S) != 0 || ldx < K || (bm != 256 && bm != 192 && bm != 128))
    return hipErrorInvalidValue;
  const bf16* x = reinterpret_cast<const bf16*>(X);
  const bf16* w = reinterpret_cast<const bf16*>(W);
  if (S == 1 && !partial_only) {
    switch (mode) {
      case kStoreBf16: return launch_pipe<kStoreBf16>(bm, x, ldx, M, w, K, N, 1, *ep, nullptr, st);
      case kStoreF32: return launch_pipe<kStoreF32>(bm, x, ldx, M, w, K, N, 1, *ep, nullptr, st);
      case kResidAdd: return launch_pipe<kResidAdd>(bm, x, ldx, M, w, K, N, 1, *ep, nullptr, st);
      case kSiluMul: return launch_pipe<kSiluMul>(bm, x, ldx, M, w, K, N, 1, *ep, nullptr, st);
      case kQkvRope: return launch_pipe<kQkvRope>(bm, x, ldx, M, w, K, N, 1, *ep, nullptr, st);
    }
    return hipErrorInvalidValue;
  }
  if (partial_only == 2) {
    if (ep->fix_cnt == nullptr || (size_t)((M + bm - 1) / bm) * ((N + 255) / 256) > (size_t)kFixTiles) return hipErrorInvalidValue;
    switch (mode) {
      case kStoreBf16: return launch_pipe<kStoreBf16, true>(bm, x, ldx, M, w, K, N, S, *ep, part, st);
      case kStoreF32: return launch_pipe<kStoreF32, true>(bm, x, ldx, M, w, K, N, S, *ep, part, st);
      case kResidAdd: return launch_pipe<kResidAdd, true>(bm, x, ldx, M, w, K, N, S, *ep, part, st);
      case kSiluMul: return launch_pipe<kSiluMul, true>(bm, x, ldx, M, w, K, N, S, *ep, part, st);
      case kQkvRope: return launch_pipe<kQkvRope, true>(bm, x, ldx, M, w, K, N, S, *ep, part, st);
    }
    return hipErrorInvalidValue;
  }
  hipError_t e = launch_pipe<kPartial>(bm, x, ldx, M, w, K, N, S, *ep, part, st);
  if (e != hipSuccess || partial_only) return e;
  return launch_splitk_reduce(mode, part, S, M, N, *ep, st);
}

extern "C" int dsse_gemm_pipe_pairs(int tiles) { return dsse::gp::pairs_of(tiles); }

// Workspace floats of the in-launch fix-up (partial_only = 2): S - 1 register-order slots per tile.
extern "C" size_t dsse_gemm_pipe_fix_floats(int bm, int S, int M, int N) {
  const int nbm = (M + bm - 1) / bm, qi = bm / 64;
  return (size_t)nbm * ((N + 255) / 256) * (S - 1) * (8 * 8 * qi * 64) * 4;
}
