// Expert GEMMs of decode steps and short prompts (bf16): the weights as one stream through per-wave LDS rings.
//
// What bounds it: a few rows per expert, so nearly every weight of the layer is read once for them (311 MB at 2048 x 1408 of
// 16 experts and a shared one of 2816, 1.59 GB at 4096 x 3584 and 7168), and what counts is how many bytes of weights are in
// flight.  256-row tiles (moe_pipe.hip) hold 32 KiB per CU for a step and a quarter and fill 136 to 198 of the 256 CUs at the
// smaller size; loads straight into MFMA operands touch 16 lines per quarter wave.  Here
//
//   * every wave streams its own 32 (gate / up) or 16 (down) weight rows through its own LDS ring, three to six 64-element
//     steps deep, whole 128-byte lines per eight lanes, two workgroups per CU: some 96 KiB of weights in flight;
//   * X comes through a ring that the four waves share, one barrier per step; its requests are spread over the waves, so a
//     counted vmcnt covers both rings;
//   * weights are non-temporal, and a column block starts at a K step of its own and wraps around: rows lie a power of two
//     apart, and workgroups that walk K in step ask a few memory channels at a time;
//   * sub-tiles of 16 rows: a workgroup takes the body for 16, 32 or 64 rows that its list tile needs, deeper for fewer;
//   * narrow tiles for the down product (64 columns): its K axis is the hidden width, twice that for a shared expert, and it
//     is the longest tile that ends last.
//
// Measured (one MI355X, work list and both products; weights of 700 MB and more read in turn; before: register-direct to 32
// rows, moe_pipe.hip above).  2048 x 1408, 16 experts, top 2, shared 2816: 1 row 33 -> 27 us, 8 68 -> 56, 32 84 -> 65,
// 64 105 -> 74, 160 106 -> 81.  4096 x 3584, shared 7168: 1 row 94 -> 67 us, 8 241 -> 202, 32 308 -> 237 (6.7 TB/s),
// 64 320 -> 259, 160 323 -> 314.  On the way (32 rows, the two sizes): without its own first step and the non-temporal
// hint 79 / 288, with the hint 73 / 261, with both 69 / 250, narrow down tiles 65 / 237; narrow gate / up tiles 64 / 251.
#include <algorithm>
#include <cmath>

#include "lds_dma.h"
#include "moe_rows.h"

namespace dsse {
namespace {
namespace ms {

constexpr int kWaves = 4;
constexpr int kStep = 64;         // K elements per step: 128 bytes of every row
constexpr int kTile = 16 * 128;   // 16 weight rows of one step
// By kind: weight tiles per wave, hidden units or output columns of a workgroup
constexpr int wave_tiles(int mode) { return mode == 1 ? 1 : 2; }
constexpr int columns(int mode) { return mode == 2 ? 128 : 64; }
// By kind and sub-tiles of 16 rows: ring depth, X's DMA instructions (8 rows each) per wave and step
constexpr int depth(int mode, int subs) { return mode == 1 ? (subs == 4 ? 5 : 6) : (subs == 4 ? 3 : 4); }
constexpr int x_dma(int subs) { return subs == 4 ? 2 : 1; }
constexpr int x_slot(int subs) { return x_dma(subs) * kWaves * 1024; }
constexpr int lds_bytes(int mode, int subs) { return depth(mode, subs) * (kWaves * wave_tiles(mode) * kTile + x_slot(subs)); }
constexpr int kLDS = 80 * 1024;   // two workgroups per CU

}  // namespace ms

// MODE 0: h = silu(gate x) * (up x); 1: o = weight * down h; 2: h = relu(up x)^2.  The column block cb of the list tile whose
// ids the lanes hold in `mine`, the first `rows` of them real.
template <int MODE, int SUBS>
DEV void stream_tile(const MoeGroupedParams& p, char* smem, int e, int cb, int mine, int rows, int slice) {
  using namespace ms;
  constexpr int CT = wave_tiles(MODE), D = depth(MODE, SUBS), NX = x_dma(SUBS), NW = 2 * CT;
  static_assert(lds_bytes(MODE, SUBS) <= kLDS);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const bool sh = e >= p.E;
  const int Fe = sh ? p.Fs : p.F;
  const int K = MODE == 1 ? Fe : p.W, N = MODE == 1 ? p.W : Fe;
  const int cut = MODE == 1 && sh ? p.parts - p.S + 1 : 1;  // the shared expert's hidden units in slices
  const int begin = K / kStep * slice / cut, nk = K / kStep * (slice + 1) / cut - begin, first = cb % nk;
  const bf16* X = reinterpret_cast<const bf16*>(MODE == 1 ? p.h : p.x);
  const int ldx = MODE == 1 ? p.ldh : p.W;

  auto weights = [&](const void* routed_w, const void* shared_w) {
    return reinterpret_cast<const bf16*>(sh ? shared_w : routed_w) + (sh ? 0 : (int64_t)e * p.F * p.W);
  };
  const bf16* w0 = MODE == 1 ? weights(p.down, p.sdown) : (MODE == 0 ? weights(p.gate, p.sgate) : weights(p.up, p.sup));
  const bf16* w1 = MODE == 0 ? weights(p.up, p.sup) : w0;
  const __amdgpu_buffer_rsrc_t xr = make_rsrc(X, (uint32_t)((size_t)(MODE == 1 ? p.M * p.S : p.M) * ldx * 2));
  const __amdgpu_buffer_rsrc_t wr0 = make_rsrc(w0, (uint32_t)((size_t)N * K * 2));
  const __amdgpu_buffer_rsrc_t wr1 = make_rsrc(w1, (uint32_t)((size_t)N * K * 2));
  const int n0 = cb * columns(MODE) + w * (columns(MODE) / kWaves);  // the wave's first hidden unit or column

  uint32_t xo[NX], wo[NW];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int row = (w * NX + i) * 8 + (lane >> 3);
    const int id = __shfl(mine, row);
    xo[i] = row < rows && row < 16 * SUBS
                ? (uint32_t)(((size_t)(MODE == 1 ? id : id / p.S) * ldx + 8 * ((lane & 7) ^ piece_swizzle(row))) * 2)
                : kOOB;
  }
#pragma unroll
  for (int j = 0; j < NW; ++j) {  // instruction j: 8 rows of weight tile j / 2 (gate and up are tiles of the same units)
    const int br = (j & 1) * 8 + (lane >> 3);
    const int n = n0 + br + (MODE == 0 ? 0 : 16 * (j >> 1));
    wo[j] = n < N ? (uint32_t)(((size_t)n * K + 8 * ((lane & 7) ^ piece_swizzle(br))) * 2) : kOOB;
  }
  char* wring = smem + w * D * CT * kTile;
  char* xring = smem + kWaves * D * CT * kTile;
  // byte offset of step c in every row; a step past the last lands as zeros, without traffic
  auto place = [&](int c) {
    const int k = c + first < nk ? c + first : c + first - nk;
    return c < nk ? (uint32_t)(begin + k) * 128 : kOOB;
  };
  auto issue_w = [&](int c, int slot) {
    const uint32_t at = place(c);
#pragma unroll
    for (int j = 0; j < NW; ++j)
      lds_dma<kAuxNT>(MODE == 0 && j >= 2 ? wr1 : wr0, wring + slot * CT * kTile + j * 1024, wo[j] | (at & kOOB), at & ~kOOB);
  };
  auto issue_x = [&](int c, int slot) {
    const uint32_t at = place(c);
#pragma unroll
    for (int i = 0; i < NX; ++i)
      lds_dma(xr, xring + slot * x_slot(SUBS) + (w * NX + i) * 1024, xo[i] | (at & kOOB), at & ~kOOB);
  };
  f32x4 acc[SUBS][CT];
#pragma unroll
  for (int i = 0; i < SUBS; ++i)
#pragma unroll
    for (int n = 0; n < CT; ++n) acc[i][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  int rd[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) rd[s] = r * 128 + (((2 * g + s) ^ piece_swizzle(r)) << 4);

  // Step c's X is requested D - 1 steps ahead, into the slot of step c - 1 once the barrier of step c says that every wave
  // has read it; its weights D steps ahead, into the wave's own ring once this wave has read them.  Younger than step c's X
  // when step c opens: the weights of step c + 1 and D - 2 whole steps.
  issue_w(0, 0);
#pragma unroll
  for (int c = 1; c < D; ++c) issue_x(c - 1, c - 1), issue_w(c, c);
  int slot = 0;
  for (int c = 0; c < nk; ++c) {
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(NW + (D - 2) * (NX + NW)) : "memory");
    const char* wb = wring + slot * CT * kTile;
    const char* xb = xring + slot * x_slot(SUBS);
    bf16x8 b[CT][2], a[SUBS][2];
#pragma unroll
    for (int n = 0; n < CT; ++n)
#pragma unroll
      for (int s = 0; s < 2; ++s) b[n][s] = *reinterpret_cast<const bf16x8*>(wb + n * kTile + rd[s]);
#pragma unroll
    for (int i = 0; i < SUBS; ++i)
      if (16 * i < rows)  // uniform
#pragma unroll
        for (int s = 0; s < 2; ++s) a[i][s] = *reinterpret_cast<const bf16x8*>(xb + i * 2048 + rd[s]);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    issue_x(c + D - 1, slot == 0 ? D - 1 : slot - 1);
    issue_w(c + D, slot);
#pragma unroll
    for (int i = 0; i < SUBS; ++i) {
      if (16 * i >= rows) continue;  // uniform
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int n = 0; n < CT; ++n) acc[i][n] = mfma16x16x32(a[i][s], b[n][s], acc[i][n]);
    }
    slot = slot + 1 == D ? 0 : slot + 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no piece lands in LDS that this workgroup has given back

#pragma unroll
  for (int i = 0; i < SUBS; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int id = __shfl(mine, 16 * i + 4 * g + j);
      if (id < 0) continue;
      const int row = id / p.S;
      const float wt = MODE == 1 ? out_weight(p, row, id - row * p.S) : in_weight(p, id);
      if (MODE == 0) {
        const int f = n0 + r;
        const float gv = acc[i][0][j] * wt;
        if (f < N)
          reinterpret_cast<bf16*>(p.h)[(int64_t)id * p.ldh + f] = (bf16)(gv / (1.0f + expf(-gv)) * (acc[i][CT - 1][j] * wt));
      } else {
#pragma unroll
        for (int n = 0; n < CT; ++n) {
          const int f = n0 + 16 * n + r;
          if (f >= N) continue;
          const float v = acc[i][n][j] * wt;
          if (MODE == 1) p.o[((int64_t)row * (p.parts - p.S) + id + slice) * p.W + f] = v;
          else reinterpret_cast<bf16*>(p.h)[(int64_t)id * p.ldh + f] = (bf16)(v > 0.0f ? v * v : 0.0f);
        }
      }
    }
}

// A workgroup per (list tile, column block): the shared expert's tiles, the last of the list, come first
template <int MODE>
__global__ void __launch_bounds__(256, 2) moe_stream_kernel(MoeGroupedParams p, int shared_tiles, int cols_s, int cols_r) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int v = blockIdx.x, each = shared_tiles * cols_s, head = MODE == 1 ? each * (p.parts - p.S + 1) : each;
  const int tiles = __builtin_amdgcn_readfirstlane(ld_global<int>(p.num_tiles));
  int t, cb, slice = 0;
  if (v < head) slice = v / each, t = max(tiles - shared_tiles, 0) + v % each / cols_s, cb = v % cols_s;
  else t = (v - head) / cols_r, cb = (v - head) % cols_r;
  // a routed tile's expert and ids are requested together with the tile count: the list has room for every t of the grid
  const int e = __builtin_amdgcn_readfirstlane(ld_global<int>(p.tile_expert + t));
  const int mine = ld_global<int>(p.sorted + t * kMoeRows + (threadIdx.x & 63));
  if (e < 0 || (v >= head && t >= tiles - shared_tiles)) return;
  if (cb * ms::columns(MODE) >= (MODE == 1 ? p.W : (e >= p.E ? p.Fs : p.F))) return;
  const int rows = __popcll(__ballot(mine >= 0));  // an expert's ids fill its tiles from the front
  if (rows <= 16) stream_tile<MODE, 1>(p, smem, e, cb, mine, rows, slice);
  else if (rows <= 32) stream_tile<MODE, 2>(p, smem, e, cb, mine, rows, slice);
  else stream_tile<MODE, 4>(p, smem, e, cb, mine, rows, slice);
}

template <int MODE>
hipError_t launch_moe_stream(const MoeGroupedParams& p, hipStream_t st) {
  static bool attr_set = false;
  if (!attr_set) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&moe_stream_kernel<MODE>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, ms::kLDS);
    attr_set = true;
  }
  // a multiple of 8 column blocks: the row tiles of a weight panel meet on one XCD
  auto blocks = [&](int F) {
    constexpr int cols = ms::columns(MODE);
    return (((MODE == 1 ? p.W : F) + cols - 1) / cols + 7) / 8 * 8;
  };
  const int shared = p.S > p.top ? (p.M + kMoeRows - 1) / kMoeRows : 0;
  const int64_t ids = (int64_t)p.M * p.top;
  // most list tiles that the routed experts can make
  const int64_t routed = std::min((ids + (int64_t)(kMoeRows - 1) * p.E) / kMoeRows, ids);
  const int cols_s = shared ? blocks(p.Fs) : 1, cols_r = blocks(p.F);
  const int64_t grid = (int64_t)shared * cols_s * (MODE == 1 ? p.parts - p.S + 1 : 1) + routed * cols_r;
  hipLaunchKernelGGL(moe_stream_kernel<MODE>, dim3((unsigned)grid), dim3(256), ms::kLDS, st, p, shared, cols_s, cols_r);
  return hipGetLastError();
}

}  // namespace

// The form of the expert GEMMs by cost, in us.  Up to 32 rows: the stream takes 7.7, 0.36 a list tile (to 16), and for each product the longer of
// its K steps, 0.19 each, and its bytes, 170 per GB where 119 workgroups and more ask for them; the register-direct kernels 8.6, 0.25 a
// list tile, and the root of the sum of 0.17 a K step and 200 per GB, each to the power of 1.34, a tenth less without gates.  Above,
// with S a form's K steps and G the GB it reads, a list tile's weights at a time: the stream 17.6 + max(0.067 S, 148 G) + 2.05 min(..), the
// direct kernels 10.6 + max(0.315 S, 237 G) + 1.16 min(..), the pipeline 20.4, 81 per GB of the weights and 0.683 per K step of its rounds
// of 256 workgroups.  Fitted over 57 sizes of 1 to 255 rows whose weights were last read 700 MB and more ago (choices of few experts are
// otherwise timed from the last-level cache); of 711 choices 8 are for a form that is slower by more than 3 %, by 8 % at most.
// Direct / stream, top 2 unless said: 1 row of 16 experts of 2048 x 2048 25 / 25, 2 rows 34 / 28, without gates 21 / 24, 26 / 26; of 4096 x
// 4096 59 / 45, without gates 41 / 42 (Dironex-wide's step 943 / 888); 4096 x 512 1 row 26 / 30, 4 rows 34 / 35; 8 of 1024 x 512 4 rows
// 16 / 16, 32 18 / 18; 4 of 512 x 256, top 1, 16 rows 13 / 14, 192 19 / 22 (pipeline 28); 16 of 2048 x 1408 and a shared one of 2816 1 row
// 36 / 28, 32 rows 89 / 67.
// Stream / pipeline at 96, 129, 160, 192 rows: 16 of 4096 x 3584 and 7168 285 / 296, 302 / 301, 315 / 303, 313 / 308; 2048 x 1408 and 2816 73 / 95,
// 78 / 95, 81 / 95, 80 / 96; 5120 x 3584 and 7168 367 / 353, 391 / 364, 406 / 370, 411 / 376; 4 of 4096 x 14336 251 / 363, 398 / 375, 470 / 372, 479 / 374;
// 8 of them 442 / 539 .. 481 / 566; 4 of 4096 x 3584 and 7168 147 / 170, 217 / 173, 231 / 175, 232 / 176; top 8 of 16 of 4096 x 3584 258 / 240,
// 387 / 252, 485 / 260, 485 / 264.  Above 192 rows the stream is not asked (255 rows of 2048 x 1408 and 2816 101 / 99).
MoeForm moe_form(const MoeGroupedParams& p) {
  const bool shared = p.S > p.top;
  const bool direct_ok = !p.lds_tiles, stream_ok = p.M <= 3 * kMoeRows, pipe_ok = p.M > 32;
  if (p.form == 1 && stream_ok) return MoeForm::kStream;
  if (p.form == 2) return MoeForm::kPipe;
  if (p.form == 3 && direct_ok) return MoeForm::kDirect;
  const int Fs = shared ? p.Fs : 0, long_f = std::max(p.F, Fs);
  const int mats = p.gate ? 3 : 2;
  const double unit = 2e-9 * mats * p.W;  // GB per hidden unit
  const double hit = p.E * (1.0 - std::pow(1.0 - (double)p.top / p.E, p.M));  // experts that some row chooses
  const double near = std::min(hit, 16.0), steps = (p.W + long_f) / 64.0;
  double direct, stream, pipe = 0;
  if (!pipe_ok) {
    const double gb = unit * (p.F * hit + Fs), down = gb / mats, up = gb - down;
    auto product = [](double gbs, int K, double wgs) { return std::max(0.193 * K / 64, 170 * gbs * std::max(1.0, 119 / wgs)); };
    stream = 7.7 + 0.36 * near + product(up, p.W, (hit * p.F + Fs) / (p.gate ? 64 : 128)) + product(down, long_f, (hit + shared) * p.W / 64);
    direct = 8.6 + 0.25 * near + (p.gate ? 1.0 : 0.89) * std::pow(std::pow(0.17 * steps, 1.34) + std::pow(200 * gb, 1.34), 1 / 1.34);
  } else {
    // list tiles of a routed expert: one, and a second and third as far as its rows' spread reaches over 64 and 128
    const double rows = std::max(1.0, (double)p.M * p.top / p.E), spread = 3 * std::sqrt(rows);
    double tiles_r = 1;
    for (int i = 1; i <= 2; ++i) tiles_r += std::min(1.0, std::max(0.0, 0.5 + (rows - i * kMoeRows) / spread));
    const int tiles_s = (p.M + kMoeRows - 1) / kMoeRows;
    const double gb = unit * (p.F * hit * tiles_r + Fs * (double)tiles_s);
    auto both = [](double a, double b, double part) { return std::max(a, b) + part * std::min(a, b); };
    stream = 17.6 + both(0.067 * steps, 148 * gb, 2.05);
    direct = 10.6 + both(0.315 * steps, 237 * gb, 1.16);
    // the pipeline's K steps: tiles of 256 weight rows, the down product's of a shared expert counted by their length
    auto blocks = [](int rows_w) { return (rows_w + 255) / 256; };
    const int per = p.gate ? 2 : 1;
    const int64_t up = (int64_t)p.E * blocks(per * p.F) + blocks(per * Fs);
    const double down = (double)blocks(p.W) * (p.E + (double)Fs / p.F);
    const double rounds = (double)((up + 255) / 256) * p.W / 64 + std::max(std::ceil(down / 256) * p.F, (double)Fs) / 64;
    pipe = 20.4 + 81 * unit * (p.F * hit + Fs) + 0.683 * rounds;
  }
  MoeForm best = stream_ok ? MoeForm::kStream : MoeForm::kPipe;
  double least = stream_ok ? stream : pipe;
  if (pipe_ok && pipe < least) best = MoeForm::kPipe, least = pipe;
  if (direct_ok && direct < least) best = MoeForm::kDirect;
  return best;
}

}  // namespace dsse

extern "C" hipError_t dsse_moe_stream(const dsse::MoeGroupedParams* p, hipStream_t st) {
  const hipError_t e = p->gate ? dsse::launch_moe_stream<0>(*p, st) : dsse::launch_moe_stream<2>(*p, st);
  return e != hipSuccess ? e : dsse::launch_moe_stream<1>(*p, st);
}
