// Expert GEMMs of prompt-sized steps (bf16): up to 256 rows of one expert x 256 weight rows per workgroup, deep LDS-DMA
// pipeline.
//
// What bounds it: at hundreds of rows per expert both products are compute-sized (muderax-wide, 3000 rows: 705 + 352 GFLOP
// per layer on 0.7 GB of weights).  The 64-row tiles of moe.hip re-read each weight panel once per 64 rows and wait for
// their register-staged loads at every chunk; here the schedule of gemm_pipe.hip runs on gathered rows and row-major
// expert weights:
//
//   * 8 waves = 2 wave rows x 4 wave columns of 64; a K step of 64 is four phases, one quadrant of the wave's tile each,
//     with one half-tile of LDS-DMA issued per phase and retired five phases later by a counted vmcnt, the two wave rows
//     one barrier apart (one row's MFMA cluster covers the other's LDS reads);
//   * both operands are row-major, so both LDS images are [row][64 k] with 16-byte pieces swizzled by (row >> 1) & 5 on the
//     source address (conflict-free fragment reads); rows and columns that do not exist load as zeros without traffic;
//   * a tile's height follows its expert: the expert's T = ceil(rows / 256) tiles take ceil(k / T) of its k 64-row list
//     tiles each, and a tile of 64 q rows fills 16 q of every 64-row quadrant: q of the four MFMA row tiles per phase, none
//     for rows that are not there;
//   * MODE 0: a column tile pair is (gate rows, up rows) of the same 16 hidden units, so silu(gate) * up needs no exchange;
//   * order: the shared expert's tiles first (the tallest), then the routed ones; each XCD owns a contiguous eighth of both,
//     row tiles fastest within groups of 8, so a weight panel's readers share an L2 at about the same time;
//   * a few tiles past an XCD's last whole round are cut over K, so that the launch does not wait for one of them.
//
// Every workgroup finds its tile by itself from the work list of 64-row tiles (the experts ascend, so ballots over the list
// give every expert's place); the host knows only a bound of the tile count.
//
// Measured (one MI355X, work list and both products, against the 64-row tiles of moe.hip): 3000 rows of 4096 x 3584, 16
// experts, top 2, shared 7168: 2369 -> 1005 us (1052 TFLOP/s); 2048 rows: 1695 -> 757; 1024 rows of 2048 x 1408, shared
// 2816: 245 -> 154; 1024 rows of 1024 x 512, 8 experts: 49 -> 39.  Up to 192 rows moe_stream.hip takes
// the sizes whose weights it need not read twice, or the kernels of moe.hip a few rows of small experts (moe_form).
#include <algorithm>
#include <cmath>
#include <vector>

#include "lds_dma.h"
#include "moe_cut.h"
#include "moe_rows.h"

namespace dsse {
namespace {
namespace mp {
using namespace moe_cut;

constexpr int kA = 256 * 128;   // row image of one K step: 256 rows x 64 bf16
constexpr int kB = 256 * 128;   // weight image: 16 column tiles x 16 rows x 64 bf16
constexpr int kBuf = kA + kB;
constexpr int kIds = 2 * kBuf;  // the tile's ids (256 ints), their weights (256 floats), their rows of the result (256 ints)
constexpr int kSay = kIds + 3 * 256 * 4;  // one word: whether this workgroup ends a cut tile
constexpr int kStage = kSay + 16;  // 2 KiB per wave: 16 rows of its hidden units on their way to 16-byte stores
constexpr size_t kLDS = kStage + 8 * 2048;

// Tiles cut over K (moe_cut.h): the counters are 16-bit halves of the first of the 64 ints behind the work list
constexpr int kSlot = 8 * 32 * 64;    // f32x4 of one piece: [wave][row tile, column tile][lane]
static_assert(8 * kPieces * kSlot * 4 == kMoeCutFloats && 8 * kCutTiles <= 2 * 64, "workspace and counters");

struct Place {
  int first;  // the expert's first list tile
  int tiles;  // its list tiles
  int at;     // workgroup index inside the expert
};

// The list's experts in chunks of 64 tiles, a tile per lane: the first four chunks stay in registers
struct List {
  const int* tile_expert;
  int n, lane;
  int v[4];
  DEV int chunk(int c) const {
    const int i = 64 * c + lane;
    return i < n ? ld_global<int>(tile_expert + i) : 0x7fffffff;
  }
  template <typename F>
  DEV void each(F f) const {
#pragma unroll
    for (int c = 0; c < 4; ++c) f(c, v[c]);
    for (int c = 4; 64 * c < n; ++c) f(c, chunk(c));
  }
};

}  // namespace mp

// MODE 0: h = silu(gate x) * (up x); 1: o = weight * down h; 2: h = relu(up x)^2
// ONCE: most weight panels have one row tile: they are non-temporal, and a column block starts at a K step of its own and wraps
// around, since rows a power of two apart ask a few memory channels at a time when every workgroup walks K in step
template <int MODE, bool ONCE>
__global__ void __launch_bounds__(512) moe_pipe_kernel(MoeGroupedParams p, int tall) {
  using namespace mp;  // tall: most list tiles in a row tile, 1, 2 or 4
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  constexpr int kCols = MODE == 0 ? 128 : 256;  // hidden units or output columns per tile
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int wm = w >> 2, wn = w & 3;
  auto blocks = [&](int F) { return ((MODE == 1 ? p.W : F) + kCols - 1) / kCols; };

  List list{p.tile_expert, __builtin_amdgcn_readfirstlane(ld_global<int>(p.num_tiles)), lane, {}};
  auto read_list = [&]() {
#pragma unroll
    for (int c = 0; c < 4; ++c) list.v[c] = list.chunk(c);
  };
  read_list();
  // list tiles of routed experts, and the row tiles they make: one per started `tall` list tiles of an expert
  int routed = 0, row_tiles = 0;
  auto walk = [&](auto f) {  // f(tile, its expert, its index inside the expert, it opens a row tile, row tiles before it)
    int last = -1, first = 0, before = 0;
    list.each([&](int c, int v) {
      const int i = 64 * c + lane;
      int prev = __shfl_up(v, 1);
      if (lane == 0) prev = last;
      const uint64_t starts = __ballot(v != prev && i < list.n), upto = starts & (~0ull >> (63 - lane));
      const int mine = upto ? 64 * c + 63 - __clzll((long long)upto) : first;
      const bool opens = v < p.E && ((i - mine) & (tall - 1)) == 0;
      const uint64_t open = __ballot(opens);
      f(i, v, i - mine, opens, before + __popcll(open & ((1ull << lane) - 1)));
      before += __popcll(open);
      last = __builtin_amdgcn_readlane(v, 63);
      first = starts ? 64 * c + 63 - __clzll((long long)starts) : first;
    });
    return before;
  };
  row_tiles = walk([&](int, int v, int, bool, int) { routed += __popcll(__ballot(v < p.E)); });
  const int shared = list.n - routed;
  const int nb_r = blocks(p.F), nb_s = blocks(p.Fs);
  const int slices = MODE == 1 ? p.parts - p.S + 1 : 1;  // of the shared expert's hidden units
  const int tiles_s = (shared + tall - 1) / tall * nb_s, total_s = tiles_s * slices, total_r = row_tiles * nb_r;
  const int steps_r = (MODE == 1 ? p.F : p.W) >> 6, steps_s = total_s ? (MODE == 1 ? p.Fs / slices : p.W) >> 6 : steps_r;  // (as may_cut)
  const Cut most = most_cut(steps_r, steps_s, p.ws ? p.cut : 1);

  // One tile; a second round only if a choice list is not what it should be (the list is read again for it: no registers for it in the K loop)
  for (int v = blockIdx.x; ; v += gridDim.x, read_list()) {
    const int x = v & 7, item = v >> 3;
    const int s0 = total_s * x / 8, ns = total_s * (x + 1) / 8 - s0;
    const int r0 = total_r * x / 8, nr = total_r * (x + 1) / 8 - r0;
    if (item >= (total_s + 7) / 8 + (total_r + 7) / 8 + pieces_room(most)) return;  // past every XCD's share
    Item it = item_of(item, ns + nr, most);
    const int u = it.u;
    if (u >= ns + nr) continue;
    const bool sh = u < ns;
    Place pl;
    int e;
    if (sh) {
      pl = Place{routed, shared, (s0 + u) % tiles_s};
      e = p.E;
    } else {
      const int at = r0 + u - ns, want = at / nb_r;
      int found = 0, opener = 0;
      walk([&](int i, int ve, int idx, bool opens, int before) {
        const uint64_t hit = __ballot(opens && before == want);
        if (hit) {
          const int l = __builtin_ctzll(hit);
          found = __builtin_amdgcn_readlane(ve, l);
          pl.first = __builtin_amdgcn_readlane(i - idx, l);
          opener = want - __builtin_amdgcn_readlane(idx, l) / tall;  // row tiles before this expert
        }
      });
      e = found;
      pl.tiles = 0;
      list.each([&](int, int ve) { pl.tiles += __popcll(__ballot(ve == e)); });
      pl.at = at - opener * nb_r;
    }
    const int T = (pl.tiles + tall - 1) / tall, q = (pl.tiles + T - 1) / T;
    const Spot spot = spot_of(pl.at, T, sh ? nb_s : nb_r);
    const int rt = spot.row_tile, n0 = spot.block * kCols;
    const int t0 = pl.first + rt * q;
    const int rows64 = min(q, pl.tiles - rt * q);  // list tiles of this row tile: 1..4, or none (T q > tiles + q)
    if (rows64 <= 0) continue;

    const int Fe = sh ? p.Fs : p.F;
    const int K = MODE == 1 ? Fe : p.W, N = MODE == 1 ? p.W : Fe;
    const int slice = sh ? (s0 + u) / tiles_s : 0, parts = sh ? slices : 1;
    const int k0 = (K >> 6) * slice / parts, kn = (K >> 6) * (slice + 1) / parts - k0;  // its K steps
    if (!cuts(it, kn, ns, ns + nr, rt, T)) {  // its first piece takes it whole
      if (it.piece) continue;
      it.of = 1;
    }
    const Walk mine = walk_of(k0, kn, it.piece, it.of);  // this piece's
    const int first = mine.first, nk = mine.steps;
    const int off = ONCE ? n0 / kCols % nk : 0;
    const bf16* X = reinterpret_cast<const bf16*>(MODE == 1 ? p.h : p.x);
    const int ldx = MODE == 1 ? p.ldh : p.W;
    auto weights = [&](const void* routed_w, const void* shared_w) {
      return reinterpret_cast<const bf16*>(sh ? shared_w : routed_w) + (sh ? 0 : (int64_t)e * p.F * p.W);
    };
    // the wave's weight DMA is of one kind: column tiles alternate gate / up, and wave w stages tiles of parity w & 1
    const bf16* Wp = MODE == 1 ? weights(p.down, p.sdown)
                               : (MODE == 0 && !(w & 1) ? weights(p.gate, p.sgate) : weights(p.up, p.sup));
    const __amdgpu_buffer_rsrc_t xr = make_rsrc(X, (uint32_t)((size_t)(MODE == 1 ? p.M * p.S : p.M) * ldx * 2));
    const __amdgpu_buffer_rsrc_t wr = make_rsrc(Wp, (uint32_t)((size_t)N * K * 2));

    int* s_id = reinterpret_cast<int*>(smem + kIds);
    float* s_w = reinterpret_cast<float*>(smem + kIds + 256 * 4);
    int* s_o = reinterpret_cast<int*>(smem + kIds + 2 * 256 * 4);
    __syncthreads();  // a second tile: every wave is past the first one's epilogue
    if ((int)threadIdx.x < rows64 * 64) {
      const int id = ld_global<int>(p.sorted + t0 * 64 + threadIdx.x);
      const int row = id >= 0 ? id / p.S : 0;
      s_id[threadIdx.x] = id;
      s_o[threadIdx.x] = row * (p.parts - p.S) + id + slice;
      s_w[threadIdx.x] = id < 0 ? 0.0f : (MODE == 1 ? out_weight(p, row, id - row * p.S) : in_weight(p, id));
    }
    __syncthreads();

    const int QI = rows64, QR = 16 * QI;  // MFMA row tiles and rows per quadrant
    uint32_t a_vo[2][2], b_vo[2][2];
    int a_lo[2][2], b_lo[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int j = 2 * w + i;                                          // instruction j of this half's 16
        const int rb = (j >> 3) * 128 + h * 64 + (j & 7) * 8;             // first of its 8 LDS rows
        const int row = rb + (lane >> 3), sr = (j & 7) * 8 + (lane >> 3);  // LDS row, row inside the quadrant
        int id = -1;
        if (sr < QR) id = s_id[((j >> 3) * 2 + h) * QR + sr];
        a_lo[h][i] = rb * 128;
        a_vo[h][i] = id >= 0 ? (uint32_t)(((size_t)(MODE == 1 ? id : id / p.S) * ldx + 8 * ((lane & 7) ^ piece_swizzle(row))) * 2)
                             : kOOB;
        const int tb = (j >> 2) * 4 + h * 2 + ((j >> 1) & 1);             // column tile
        const int br = (j & 1) * 8 + (lane >> 3);                         // row inside it
        const int n = MODE == 0 ? n0 + (tb >> 1) * 16 + br : n0 + tb * 16 + br;
        b_lo[h][i] = kA + (tb * 16 + (j & 1) * 8) * 128;
        b_vo[h][i] = n < N ? (uint32_t)(((size_t)n * K + 8 * ((lane & 7) ^ piece_swizzle(br))) * 2) : kOOB;
      }
    auto place = [&](int t) { return (uint32_t)(first + (t + off < nk ? t + off : t + off - nk)) * 128; };
    auto issue_a = [&](int h, int t) {
      char* base = smem + (t & 1) * kBuf;
#pragma unroll
      for (int i = 0; i < 2; ++i) lds_dma(xr, base + a_lo[h][i], a_vo[h][i], place(t));
    };
    auto issue_b = [&](int h, int t) {
      char* base = smem + (t & 1) * kBuf;
#pragma unroll
      for (int i = 0; i < 2; ++i) lds_dma<ONCE ? kAuxNT : 0>(wr, base + b_lo[h][i], b_vo[h][i], place(t));
    };
    int a_rd[2], b_rd[2];
#pragma unroll
    for (int sp = 0; sp < 2; ++sp) {
      const int piece = ((2 * g + sp) ^ piece_swizzle(r)) << 4;
      a_rd[sp] = (wm * 128 + r) * 128 + piece;
      b_rd[sp] = kA + (wn * 64 + r) * 128 + piece;
    }
    f32x4 acc[8][4];
#pragma unroll
    for (int m = 0; m < 8; ++m)
#pragma unroll
      for (int n = 0; n < 4; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    bf16x8 a[4][2], b[4][2];
    auto read_a = [&](const char* buf, int qm) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (i < QI)  // uniform
#pragma unroll
          for (int sp = 0; sp < 2; ++sp)
            a[i][sp] = *reinterpret_cast<const bf16x8*>(buf + a_rd[sp] + (64 * qm + 16 * i) * 128);
    };
    auto read_b = [&](const char* buf, int qn) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int sp = 0; sp < 2; ++sp)
          b[2 * qn + i][sp] = *reinterpret_cast<const bf16x8*>(buf + b_rd[sp] + (2 * qn + i) * 2048);
    };
    auto mma = [&](int qm, int qn) {
      asm volatile("s_barrier\n\ts_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (i >= QI) continue;  // uniform (one copy of the loop per height keeps no accumulators in registers)
#pragma unroll
        for (int sp = 0; sp < 2; ++sp)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[4 * qm + i][2 * qn + j] = mfma16x16x32(b[2 * qn + j][sp], a[i][sp], acc[4 * qm + i][2 * qn + j]);
      }
      __builtin_amdgcn_s_setprio(0);
      asm volatile("s_barrier" ::: "memory");
    };
    // Half-tiles of two instructions, in the order A0 B0 B1 A1 of a step.  A wait for 8 leaves the four youngest in flight and
    // has the half-tile that the next phase reads: B1 of step t in phase 0, A1 in phase 1, A0 and B0 of step t + 1 in phase 3,
    // each followed by the barrier that opens the reading phase.  A slot is refilled two phases or more after its last read.
    issue_a(0, 0);
    issue_b(0, 0);
    issue_b(1, 0);
    issue_a(1, 0);
    issue_a(0, 1);
    issue_b(0, 1);
    asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory");
    if (wm == 1) asm volatile("s_barrier" ::: "memory");
    auto step = [&](int t, auto tail_tag) {  // TAIL 0: steady; 1: no step t + 2; 2: the last step
      constexpr int TAIL = decltype(tail_tag)::value;
      const char* buf = smem + (t & 1) * kBuf;
      read_a(buf, 0);
      read_b(buf, 0);
      if constexpr (TAIL < 2) {
        issue_b(1, t + 1);
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");  // B-half 1 of step t
      } else {
        asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
      }
      mma(0, 0);
      read_b(buf, 1);
      if constexpr (TAIL < 2) {
        issue_a(1, t + 1);
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");  // A-half 1 of step t
      } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      mma(0, 1);
      read_a(buf, 1);
      if constexpr (TAIL == 0) issue_a(0, t + 2);
      mma(1, 1);
      if constexpr (TAIL == 0) {
        issue_b(0, t + 2);
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");  // A0 / B0 of step t + 1
      } else if constexpr (TAIL == 1) {
        asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      }
      mma(1, 0);
    };
    int t = 0;
    for (; t < nk - 2; ++t) step(t, std::integral_constant<int, 0>{});
    step(t++, std::integral_constant<int, 1>{});  // nk >= 2: a tile's (moe_lines_ok; bindings for slices), a piece's (cuts)
    step(t, std::integral_constant<int, 2>{});
    if (wm == 0) asm volatile("s_barrier" ::: "memory");  // the two rows' barrier counts meet

    if (it.of > 1) {
      const int of = it.of;
      f32x4* slots = reinterpret_cast<f32x4*>(p.ws) + (size_t)(x * kPieces + (u - it.whole) * of) * kSlot;
      int at = w * 32 * 64 + lane;
      asm volatile("" : "+v"(at));  // addresses of this part are not made before the K loop, whose registers are full
#pragma unroll
      for (int m = 0; m < 8; ++m)
        if ((m & 3) < QI)  // uniform
#pragma unroll
          for (int n = 0; n < 4; ++n) slots[(size_t)it.piece * kSlot + at + (4 * m + n) * 64] = acc[m][n];
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      int* say = reinterpret_cast<int*>(smem + kSay);
      if (threadIdx.x == 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        const int c = x * kCutTiles + u - it.whole, shift = 16 * (c & 1);
        int* count = p.sorted + (size_t)list.n * 64 + (c >> 1);
        const int before = __hip_atomic_fetch_add(count, 1 << shift, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >> shift & 0xffff;
        *say = before == of - 1;
        if (before == of - 1) __hip_atomic_fetch_sub(count, of << shift, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __syncthreads();
      if (!__builtin_amdgcn_readfirstlane(*say)) continue;
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      const __amdgpu_buffer_rsrc_t rs = make_rsrc(slots, (uint32_t)(of * kSlot * 16));
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        if ((m & 3) >= QI) continue;  // uniform
#pragma unroll
        for (int c0 = 0; c0 < kMostCut; c0 += 4) {
          if (c0 >= of) continue;  // uniform
          f32x4 t[4][4];
#pragma unroll
          for (int c = 0; c < 4; ++c)  // pieces that do not exist read as zeros, without traffic
#pragma unroll
            for (int n = 0; n < 4; ++n)
              t[c][n] = __builtin_bit_cast(
                  f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                             rs, c0 + c < of ? (uint32_t)(((c0 + c) * kSlot + at + (4 * m + n) * 64) * 16) : kOOB, 0, 0));
#pragma unroll
          for (int n = 0; n < 4; ++n) acc[m][n] = (c0 ? acc[m][n] + t[0][n] : t[0][n]) + t[1][n] + t[2][n] + t[3][n];
        }
      }
    }

    int ln = lane;
    asm volatile("" : "+v"(ln));  // addresses of this part are not made before the K loop either
    const int r = ln & 15, g = ln >> 4;
    char* st = smem + kStage + w * 2048;
    if constexpr (MODE != 1) {
      // The weights were the products' first operand: a lane has four hidden units of a row, which leaves through the wave's LDS in pieces of 16 bytes.
      // Two-byte stores from 16 lanes a row (the down product's: four bytes, 64 of four rows) / this, work list and both products, no tile cut, us: 1024
      // rows of 2048 x 1408 166 / 164, 400 111 / 108; 4096 x 3584, 1300 rows 564 / 553, 2048 769 / 756, 3000 1029 / 1017.
      constexpr int kPer = MODE == 0 ? 4 : 8;  // pieces of a row
      const int f0 = n0 + wn * 8 * kPer;
      if (f0 < N)  // uniform: N % 64 == 0
#pragma unroll
        for (int m = 0; m < 8; ++m) {
          if ((m & 3) >= QI) continue;  // uniform
          const int first_row = (wm * 2 + (m >> 2)) * QR + 16 * (m & 3);
          const float wt = s_w[first_row + r];
#pragma unroll
          for (int q = 0; q < kPer / 2; ++q) {
            bf16x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              if (MODE == 0) {
                const float gv = acc[m][2 * q][e] * wt;
                v[e] = (bf16)(gv / (1.0f + expf(-gv)) * (acc[m][2 * q + 1][e] * wt));
              } else {
                const float z = acc[m][q][e] * wt;
                v[e] = (bf16)(z > 0.0f ? z * z : 0.0f);
              }
            }
            *reinterpret_cast<bf16x4*>(st + r * 16 * kPer + (((2 * q + (g >> 1)) ^ (r >> (MODE == 0 ? 1 : 0) & (kPer - 1))) << 4) + 8 * (g & 1)) = v;
          }
#pragma unroll
          for (int it = 0; it < kPer / 4; ++it) {
            const int rr = it * 8 + ln / kPer, piece = ln % kPer;
            const bf16x8 v = *reinterpret_cast<const bf16x8*>(st + rr * 16 * kPer + ((piece ^ (rr >> (MODE == 0 ? 1 : 0) & (kPer - 1))) << 4));
            const int id = s_id[first_row + rr];
            if (id >= 0) *reinterpret_cast<bf16x8*>(reinterpret_cast<bf16*>(p.h) + (int64_t)id * p.ldh + f0 + 8 * piece) = v;
          }
        }
      continue;
    }
    // fp32 rows, 128 bytes of 16 of them at a time, wherever o begins (memory takes 16 bytes at any multiple of four)
    typedef f32x4 __attribute__((aligned(4))) f32x4_any;
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      if ((m & 3) >= QI) continue;  // uniform
      const int first_row = (wm * 2 + (m >> 2)) * QR + 16 * (m & 3);
      const float wt = s_w[first_row + r];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int f0 = n0 + wn * 64 + 32 * q;
        if (f0 >= N) continue;  // uniform: N % 64 == 0
#pragma unroll
        for (int n = 0; n < 2; ++n) *reinterpret_cast<f32x4*>(st + r * 128 + (((4 * n + g) ^ (r & 7)) << 4)) = acc[m][2 * q + n] * wt;
#pragma unroll
        for (int it = 0; it < 2; ++it) {
          const int rr = it * 8 + (ln >> 3), piece = ln & 7, at = first_row + rr;
          const f32x4 v = *reinterpret_cast<const f32x4*>(st + rr * 128 + ((piece ^ (rr & 7)) << 4));
          if (s_id[at] >= 0) *reinterpret_cast<f32x4_any*>(p.o + (int64_t)s_o[at] * p.W + f0 + 4 * piece) = v;
        }
      }
    }
  }
}

// Most workgroup tiles that the routed experts (the shared expert) can make: sum of ceil(rows / (64 tall)) over experts
int64_t col_blocks(const MoeGroupedParams& p, int mode, int F) {
  const int cols = mode == 0 ? 128 : 256;
  return ((mode == 1 ? p.W : F) + cols - 1) / cols;
}
int64_t routed_tiles(const MoeGroupedParams& p, int mode, int tall) {
  const int64_t rows = 64 * tall, ids = (int64_t)p.M * p.top;
  return std::min((ids + (rows - 1) * p.E) / rows, ids) * col_blocks(p, mode, p.F);
}
int64_t shared_tiles(const MoeGroupedParams& p, int mode, int tall) {
  const int64_t slices = mode == 1 ? p.parts - p.S + 1 : 1;
  return p.S > p.top ? (p.M + 64 * (int64_t)tall - 1) / (64 * tall) * col_blocks(p, mode, p.Fs) * slices : 0;
}
// The row tiles' greatest height in the gate / up product: the one whose tiles finish first by a simple model, rounds of 256
// workgroups (one per CU) times the tiles' mean time.  A tile of 1 / 2 / 3 / 4 list tiles takes 0.5 / 0.7 / 0.85 / 1 of the tallest one's
// time (0.75 to 1.7 us per K step, measured at 2048 x 1024, 8 experts); choices spread evenly over the experts but for one
// standard deviation, which is what decides whether a round is full.
int moe_pipe_height(const MoeGroupedParams& p, int mode) {
  static const double kTime[5] = {0.0, 0.5, 0.7, 0.85, 1.0};
  const double each = (double)p.M * p.top / p.E;
  const int64_t nb_r = col_blocks(p, mode, p.F), nb_s = p.S > p.top ? col_blocks(p, mode, p.Fs) : 0;
  const int64_t k_r = std::max<int64_t>(1, (int64_t)((each + std::sqrt(each) + 63.0) / 64.0)), k_s = (p.M + 63) / 64;
  int best = 4;
  double least = 0.0;
  for (int tall = 4; tall >= 1; tall /= 2) {
    const int64_t t_r = (k_r + tall - 1) / tall, t_s = (k_s + tall - 1) / tall;
    const int64_t q_r = (k_r + t_r - 1) / t_r, q_s = (k_s + t_s - 1) / t_s;
    const int64_t n_r = t_r * p.E * nb_r, n_s = t_s * nb_s;
    const double mean = (n_r * kTime[q_r] + n_s * kTime[q_s]) / (double)(n_r + n_s);
    const double time = (double)((n_r + n_s + 255) / 256) * mean;
    if (tall == 4 || time < least) best = tall, least = time;
  }
  return best;
}

// The down product's row tiles and what it takes with them.  Here tiles differ in length: a shared expert's K axis is its hidden
// width, most often twice a routed one's, and with its tiles first the rest may wait for the last of them: 700 rows of 2048 x 1408, 16
// experts, took 52 us with a shared expert of 2816 and 34 without.  So its hidden units may be cut into slices, each a part of its own
// in o, which the norm that follows adds.
struct Height {
  int tall;
  double us;
};

// What is asked: when the last of 256 CUs is done if every tile goes to the one that is free first, tiles in the order of the kernel (6 us each
// and 1.3 per K step of the tallest, 0.54 / 0.72 / 0.86 of it for 1 / 2 / 3 list tiles); the weights at 160 us per GB, three tenths of that where another
// row tile reads them again; 0.3 of the shorter one of the two; 400 us per GB of further parts, written and read.  Rows per expert: normal about
// their mean.
Height down_height(const MoeGroupedParams& p, int slices) {
  static const double kTime[5] = {0.0, 0.54, 0.72, 0.86, 1.0};
  const bool shared = p.S > p.top;
  const int cols = (p.W + 255) / 256;
  const double each = (double)p.M * p.top / p.E, sd = std::sqrt(each);
  const double hit = p.E * (1.0 - std::pow(1.0 - (double)p.top / p.E, p.M));
  auto below = [&](int k) { return 0.5 * std::erfc((each - 64.0 * k) / (1.4142135623730951 * sd)); };  // share of experts of k list tiles at most
  const int lo = std::max(1, (int)std::ceil((each - 2 * sd) / 64)), hi = std::max(lo, (int)std::ceil((each + 2 * sd) / 64));
  Height best{4, 0.0};
  for (int tall = 4; tall >= 1; tall /= 2) {
    struct {
      double until, cus;
    } g[32] = {{0.0, 256.0}};
    int n = 1;
    double last = 0.0, again = 0.0;
    auto tiles = [&](double count, double steps, int q) {
      const double t = 6.0 + 1.3 * steps * kTime[q];
      while (count > 1e-6) {
        int first = 0;
        for (int i = 1; i < n; ++i)
          if (g[i].until < g[first].until) first = i;
        const double take = std::min(count, g[first].cus), until = g[first].until + t;
        g[first].cus -= take;
        count -= take;
        int at = first;
        if (g[first].cus > 1e-6) {
          for (at = 0; at < n && std::abs(g[at].until - until) > 1e-6; ++at) {}
          if (at == n) {
            if (n < 32) g[n++] = {until, 0.0};
            else at = first;  // (never seen) the classes are few
          }
        }
        g[at].until = until;
        g[at].cus += take;
        last = std::max(last, until);
      }
    };
    auto expert = [&](double count, int k, double steps) {  // `count` times the tiles of an expert of k list tiles
      const int T = (k + tall - 1) / tall, q = (k + T - 1) / T;
      tiles(count * (k / q), steps, q);
      if (k % q) tiles(count, steps, k % q);
      return T - 1;
    };
    if (shared) again += (double)p.Fs * expert((double)cols * slices, (p.M + 63) / 64, p.Fs / 64.0 / slices);
    for (int k = lo; k <= hi; ++k) {
      const double share = (k < hi ? below(k) : 1.0) - (k > lo ? below(k - 1) : 0.0);
      if (share * hit > 0.05) again += share * hit * p.F * expert(share * hit * cols, k, p.F / 64.0);
    }
    const double gb = 2e-9 * p.W * (p.F * hit + (shared ? p.Fs : 0) + 0.3 * again);
    const double us = std::max(last, 160.0 * gb) + 0.3 * std::min(last, 160.0 * gb) + 400 * 8e-9 * p.M * p.W * (slices - 1);
    if (tall == 4 || us < best.us) best = Height{tall, us};
  }
  return best;
}

// The rule of the kernel, for every list that the step may have
moe_cut::Cut may_cut(const MoeGroupedParams& p, int mode) {
  const int steps_r = (mode == 1 ? p.F : p.W) >> 6, steps_s = mode == 1 && p.S > p.top ? p.Fs / (p.parts - p.S + 1) >> 6 : steps_r;
  return moe_cut::most_cut(steps_r, steps_s, p.cut);
}

template <int MODE, bool ONCE>
hipError_t launch_moe_pipe(const MoeGroupedParams& p, hipStream_t st) {
  static bool attr_set = false;
  if (!attr_set) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&moe_pipe_kernel<MODE, ONCE>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)mp::kLDS);
    attr_set = true;
  }
  const int tall = MODE == 1 ? down_height(p, p.parts - p.S + 1).tall : moe_pipe_height(p, MODE);
  const int64_t grid = 8 * ((routed_tiles(p, MODE, tall) + 7) / 8 + (shared_tiles(p, MODE, tall) + 7) / 8 + (p.ws ? moe_cut::pieces_room(may_cut(p, MODE)) : 0));
  hipLaunchKernelGGL((moe_pipe_kernel<MODE, ONCE>), dim3((unsigned)grid), dim3(512), mp::kLDS, st, p, tall);
  return hipGetLastError();
}

template <bool ONCE>
hipError_t launch_moe_pipes(const MoeGroupedParams& p, hipStream_t st) {
  const hipError_t e = p.gate ? launch_moe_pipe<0, ONCE>(p, st) : launch_moe_pipe<2, ONCE>(p, st);
  return e != hipSuccess ? e : launch_moe_pipe<1, ONCE>(p, st);
}

bool sixteens(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace

bool moe_pipe_cuts(const MoeGroupedParams& p) {
  return moe_cut::pieces_room(may_cut(p, p.gate ? 0 : 2)) > 0 || moe_cut::pieces_room(may_cut(p, 1)) > 0;
}

bool moe_lines_ok(const MoeGroupedParams& p) {
  constexpr int64_t kRange = (int64_t)1 << 31;
  const int64_t ids = (int64_t)p.M * p.S, widest = p.F > p.Fs ? p.F : p.Fs;
  const bool shared = p.S > p.top;
  if (p.f32 || p.W % 64 || p.W < 128 || p.F % 64 || p.F < 128 || (shared && (p.Fs % 64 || p.Fs < 128)) || p.ldh % 8)
    return false;
  if ((int64_t)p.M * p.W * 2 >= kRange || ids * p.ldh * 2 >= kRange || widest * p.W * 2 >= kRange) return false;
  if (!sixteens(p.x) || !sixteens(p.h) || !sixteens(p.up) || !sixteens(p.down) || (p.gate && !sixteens(p.gate))) return false;
  return !shared || (sixteens(p.sgate) && sixteens(p.sup) && sixteens(p.sdown));
}

// What every workgroup of a product takes, rows[e] rows of expert e: {XCD, expert (E: the shared one), row tile, column block, slice, piece, of,
// first K step, K steps}, by the kernel's own rules on the host
std::vector<int> moe_pipe_walks(const MoeGroupedParams& p, int mode, const int* rows) {
  using namespace moe_cut;
  const int tall = mode == 1 ? down_height(p, p.parts - p.S + 1).tall : moe_pipe_height(p, mode);
  const int nb_r = (int)col_blocks(p, mode, p.F), nb_s = (int)col_blocks(p, mode, p.Fs), slices = mode == 1 ? p.parts - p.S + 1 : 1;
  const int shared = p.S > p.top ? (p.M + 63) / 64 : 0, tiles_s = (shared + tall - 1) / tall * nb_s, total_s = tiles_s * slices;
  auto row_tiles = [&](int e) { return ((rows[e] + 63) / 64 + tall - 1) / tall; };
  int total_r = 0;
  for (int e = 0; e < p.E; ++e) total_r += row_tiles(e) * nb_r;
  const int steps_r = (mode == 1 ? p.F : p.W) >> 6, steps_s = total_s ? (mode == 1 ? p.Fs / slices : p.W) >> 6 : steps_r;
  const Cut most = most_cut(steps_r, steps_s, p.cut);
  std::vector<int> out;
  for (int x = 0; x < 8; ++x) {
    const int s0 = total_s * x / 8, ns = total_s * (x + 1) / 8 - s0, r0 = total_r * x / 8, nr = total_r * (x + 1) / 8 - r0;
    for (int item = 0; item < (total_s + 7) / 8 + (total_r + 7) / 8 + pieces_room(most); ++item) {
      Item it = item_of(item, ns + nr, most);
      if (it.u >= ns + nr) continue;
      const bool sh = it.u < ns;
      int e = p.E, at = sh ? (s0 + it.u) % tiles_s : r0 + it.u - ns;
      if (!sh)
        for (e = 0; at >= row_tiles(e) * nb_r; ++e) at -= row_tiles(e) * nb_r;
      const int slice = sh ? (s0 + it.u) / tiles_s : 0, parts = sh ? slices : 1, K = mode == 1 ? (sh ? p.Fs : p.F) : p.W;
      const int k0 = (K >> 6) * slice / parts, kn = (K >> 6) * (slice + 1) / parts - k0;
      const int T = sh ? (shared + tall - 1) / tall : row_tiles(e);
      const Spot spot = spot_of(at, T, sh ? nb_s : nb_r);
      if (!cuts(it, kn, ns, ns + nr, spot.row_tile, T)) {
        if (it.piece) continue;
        it.of = 1;
      }
      const Walk mine = walk_of(k0, kn, it.piece, it.of);
      out.insert(out.end(), {x, e, spot.row_tile, spot.block, slice, it.piece, it.of, mine.first, mine.steps});
    }
  }
  return out;
}

// Two slices where they end sooner.  One / two, work list, both products and the norm that adds the parts, in us: 2048 x 1408, 16 experts,
// top 2, shared 2816: 200 rows 103 / 90, 700 125 / 111, 1500 203 / 182, 2048 222 / 238; 1024 x 2048, 8 of them, 4096: 256 rows 94 / 71, 2500
// 221 / 189; 4096 x 3584, 4 of them, 7168: 300 rows 218 / 183, 1300 490 / 488; 16 of them, bound by their bytes: 200 rows 317 / 321, 3000
// 1083 / 1104.  Three and four are behind two.  Over 200 sizes of 12 widths the geometric mean is 1.045, one of them 5 % behind (1000 rows of the
// third: 384 / 403).  The stream up to 192 rows (moe_form): two where the shared expert's K steps, 0.45 us each, outlast the bytes, 170 us per GB:
// 1 row of the first 31 / 28, 64 77 / 72, 192 85 / 89; 96 rows of the third 150 / 137, 128 153 / 158; 64 rows of the second 56 / 48.
int moe_parts(const MoeGroupedParams& p) {
  if (p.S == p.top || p.Fs < 4 * 64 || !moe_lines_ok(p)) return p.S;
  const MoeForm form = moe_form(p);
  if (form == MoeForm::kDirect) return p.S;
  if (form == MoeForm::kPipe) return down_height(p, 2).us < down_height(p, 1).us ? p.S + 1 : p.S;
  const double rows = (double)p.M * p.top / p.E, hit = p.E * (1.0 - std::pow(1.0 - (double)p.top / p.E, p.M));
  const double tiles = std::max(1.0, 0.5 + rows / 64), gb = 2e-9 * p.W * (p.F * hit * tiles + (double)p.Fs * ((p.M + 63) / 64));
  return 0.45 * p.Fs / 64 > 170 * gb ? p.S + 1 : p.S;
}

}  // namespace dsse

// The line lies at a mean of 128 rows per expert.  Plain / ONCE at 16 experts, top 2 and a shared one: 2048 x 1408 + 2816: 400 rows
// 116 / 110 us, 1000 173 / 166, 1500 185 / 182 (but a whole prompt of 1649 rows in four 2708 / 2748), 3000 259 / 261; 4096 x 3584 +
// 7168: 256 rows 333 / 314, 700 407 / 404, 1000 471 / 465, 3000 1038 / 1068.  And where the weights are 40 MB and more: 300 rows, 8 of 512 x 2048
// (50 MB) 1.05 times, 16 of 1024 x 1024 (100 MB) 1.02, 16 of 2048 x 2048 1.07; 8 of 1024 x 512 (25 MB) 0.98, 16 of 768 x 384 and 768 (32 MB)
// 0.97, 4 of 512 x 256 (3 MB) 0.92.
extern "C" hipError_t dsse_moe_pipe(const dsse::MoeGroupedParams* p, hipStream_t st) {
  const int64_t weights = (int64_t)(p->gate ? 6 : 4) * p->W * ((int64_t)p->F * p->E + (p->S > p->top ? p->Fs : 0));
  const bool once = p->once ? p->once == 1 : (int64_t)p->M * p->top <= 128 * (int64_t)p->E && weights >= 40000000;
  return once ? dsse::launch_moe_pipes<true>(*p, st) : dsse::launch_moe_pipes<false>(*p, st);
}
