// Flash prefill of one (64-query tile, kv head) as a device function: attention_prefill.hip runs one per workgroup, attention_mixed.hip
// beside decode rows.  Layout and schedule are described in attention_prefill.hip.
#pragma once
#include "api.h"
#include "lds_dma.h"

#include <type_traits>

namespace dsse {
namespace flash {
namespace {
constexpr int kD = 128;
constexpr int kBQ = 64;    // query tokens per workgroup
constexpr int kBK = 64;    // keys per block (2 pages)
constexpr int kKBytes = kBK * kD * 2;  // 16 KiB
constexpr int kStage = 2 * kKBytes;    // K + Vᵀ of one block
constexpr int kRing = 4;               // LDS blocks
constexpr float kRescaleThr = 8.f;     // deferred online-softmax rescale threshold (log2 units)

// KV block of page `pg` (clamped to the last page: pages past the context are a harmless, masked re-read).
// The index is workgroup-uniform, so this is a scalar load: waiting for it (lgkmcnt) does not drain the
// vector loads of the K/V blocks already in flight, as a per-lane block-table load's vmcnt(0) did.
// (The block table is read-only for the kernel's lifetime, so reading it through the constant address space
// is safe and lets the compiler issue s_load_dword.)
DEV int page_block(const int* bt, int pg, int npages, const AttnParams& p) {
  pg = __builtin_amdgcn_readfirstlane(min(pg, npages - 1));
  const __attribute__((address_space(4))) int* cbt = (const __attribute__((address_space(4))) int*)bt;
  return DSSE_IDX(cbt[DSSE_IDX(pg, p.max_blocks, 0)], p.num_blocks, 0);
}
// G = q heads per kv head; HG = the q heads one workgroup takes (HG < G splits a kv head's q heads over G / HG
// workgroups: short prompts, where one workgroup per (tile, kv head) leaves most CUs idle -- a 512-token prompt is 64
// workgroups; each then stages its K/V itself, which the L2 serves)
// STAMP (diagnostic build, DSSE_FLASH_STAMPS): every wave of the first kStampWgs workgroups records the shader clock at
// six points of each key block (before / after the barrier in front of the products, before / after the barrier in front of
// the softmax, after the softmax, after the issue of the last Vᵀ reads) into 24 KiB of LDS past the ring, copied to `stamps` at the end; tools/flash_stamps.py reads them.
constexpr int kStampBlocks = 128, kStampWgs = 32, kStampsPerBlock = 6;
template <int G, int HG, bool STAMP>
DEV void flash_prefill(const AttnParams& p, unsigned* stamps, int block, char* smem) {  // smem: kRing blocks of kStage
  constexpr int NW = 2 * HG;
  constexpr int NSPLIT = G / HG;

  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
  const int r = lane & 15, g = lane >> 4;
  const int wh = w % HG, wq = w / HG;
  // flat grid, head fastest: workgroup b runs on XCD b % 8, so with Hkv = 8 every XCD serves ONE kv head and
  // its 4 MiB of 8k-context K/V stays in that XCD's L2 for all the head's query tiles (a (tile, head) grid put
  // consecutive tiles on different XCDs and every XCD streamed all 8 heads); the work list is heaviest-first
  // globally, not per head
  const int h = block % p.hkv, rest = block / p.hkv;
  const int hs = rest % NSPLIT, item = rest / NSPLIT;
  const int b = p.work_seq[item];
  const int qlen = p.q_len[b], ctx = p.ctx_len[b];
  const int pos0 = ctx - qlen;                 // absolute position of query 0 of this chunk
  const int tile = p.work_tile[item];
  const int q0 = tile * kBQ + wq * 32;         // this wave's first query (within the chunk)
  const int wg_last_q = min(qlen, (tile + 1) * kBQ) - 1;
  if (tile * kBQ >= qlen) return;              // uniform
  const int kmax = pos0 + wg_last_q + 1;       // keys [0, kmax) are visible to some query of the WG
  const int nblk = (kmax + kBK - 1) / kBK;
  // key split (round 6): this item's key blocks [jb, je) and its partial slot (-1: the whole range, final output)
  const int jb = p.work_kb ? p.work_kb[2 * item] : 0;
  const int je = p.work_kb ? min(nblk, p.work_kb[2 * item + 1]) : nblk;
  const int pslot = p.work_slot ? p.work_slot[item] : -1;
  const int w_first_pos = pos0 + q0, w_last_pos = pos0 + min(qlen, q0 + 32) - 1;
  // Key blocks from jv on (the tile's last one, or none) are after all of this wave's queries: skipped, since a weight of zero does not keep a value that is
  // not finite out of the sum
  const int jv = min(je, w_last_pos / kBK + 1);
  const int head = h * G + hs * HG + wh;
  const int* bt = p.block_tables + (size_t)b * p.max_blocks;
  const int npages = (kmax + kBS - 1) / kBS;

  // Q fragments (B operand of Sᵀ = K·Qᵀ): lane (r, g) holds Q[query 16qt + r][d = 32g + 8s + j]
  bf16x8 qf[2][4];
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    const int qi = min(q0 + 16 * qt + r, qlen - 1);
    const bf16* qp = p.q + ((size_t)(p.q_start[b] + qi) * p.hq + head) * kD + 32 * g;
#pragma unroll
    for (int s = 0; s < 4; ++s) qf[qt][s] = ld_bf16x8(qp + 8 * s);
  }
  // retire the Q loads here, before any DMA is issued: otherwise the compiler's wait for them at the first QKᵀ
  // MFMA (behind an unknown number of loop-carried DMAs) is a vmcnt(0) inside the loop, draining the prefetch
#pragma unroll
  for (int qt = 0; qt < 2; ++qt)
#pragma unroll
    for (int s = 0; s < 4; ++s) asm volatile("" ::"v"(qf[qt][s]));

  // LDS-DMA: a block is 32 x 1 KiB DMA instructions, IPW per wave, each a contiguous KiB of one page of this kv head.  Instruction q < 16 fills
  // keys 4q..4q+3 (lane -> key 4q + lane / 16, LDS slot lane % 16 = chunk ^ swz(key)); q >= 16 fills 16 rows d of one page's Vᵀ image (lane -> row
  // lane / 4, slot lane % 4 = chunk ^ vswz(row)).  The swizzles sit on the source address because the DMA writes LDS lane-linearly.  Blocks past
  // the last are issued too (pages clamp to the context, nobody reads them): a branch around the DMA made the compiler's waitcnt
  // placement drain every load in flight.  A wave's instructions are all K or all Vᵀ, of one page (of both where a wave has 16).
  constexpr int IPW = 32 / NW, NP = IPW > 8 ? 2 : 1;
  static_assert(IPW % 4 == 0, "a lane's offset inside the KiB repeats every 4 instructions");
  auto vswz = [](int row) { return (4 - (row >> 2)) & 3; };  // reads of lane (r, g): 16 distinct slots in every group of lanes that LDS serves together
  const bool kpiece = w * IPW < 16;  // wave-uniform
  uint32_t loff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    loff[i] = kpiece ? (lane >> 4) * 256 + (((lane & 15) ^ swz(4 * i + (lane >> 4))) << 4) : (lane >> 2) * 64 + (((lane & 3) ^ vswz(lane >> 2)) << 4);
  const size_t pstride = (size_t)p.hkv * kBS * kD;  // elements per page block (all kv heads)
  const bf16* head_pages = (kpiece ? p.k_cache : p.v_cache) + (size_t)h * kBS * kD;
  // Page-table entries are read one block ahead: the scalar load of block j + 1's page is in flight while block j
  // is issued and retired by the next LDS wait, not by a dependent wait in front of this block's DMA.
  const int par = (w * IPW & 15) >> 3;  // the block's page that the wave begins in
  int pg[NP];
  auto next_pages = [&](int j) {
#pragma unroll
    for (int n = 0; n < NP; ++n) pg[n] = page_block(bt, 2 * j + par + n, npages, p);
  };
  next_pages(jb);
  int jn = jb;  // next block to issue (blocks are issued in order)
  auto issue_block = [&](int slot) {
    __amdgpu_buffer_rsrc_t page[NP];
#pragma unroll
    for (int n = 0; n < NP; ++n) page[n] = make_rsrc(head_pages + (size_t)pg[n] * pstride, kBS * kD * 2);
    next_pages(++jn);
    char* base = smem + slot * kStage + w * IPW * 1024;
#pragma unroll
    for (int i = 0; i < IPW; ++i) lds_dma(page[i / 8], base + i * 1024, loff[i & 3], ((w * IPW + i) & 7) * 1024);
  };

  f32x4 o[8][2];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt)
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) o[dt][qt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run[2] = {-1e30f, -1e30f};
  // per-lane partial row sums (packed pairs): reduced over the 4 lane groups of a query once, after the last block
  f32x2 l_part[2] = {f32x2{0.f, 0.f}, f32x2{0.f, 0.f}};
  const float sc = p.scale_log2;
  f32x4 s4[4][2];  // Sᵀ[key tile kt][query tile qt] of the current block, live across the mid-block barrier

  // Lane-constant parts of the fragment addresses: K row 16 kt + r, chunk (4g + s) ^ swz(r) = kt * 4096 + kofs[s];
  // Vᵀ page t, row d = 16 dt + r, chunk g ^ vswz(r) = t * 8192 + dt * 1024 + vofs.  With the
  // slot a compile-time constant (the block loop is unrolled by the ring) every read is one base VGPR + an immediate.
  int kofs[4];
#pragma unroll
  for (int s2 = 0; s2 < 4; ++s2) kofs[s2] = r * 256 + (((4 * g + s2) ^ swz(r)) << 4);
  const int vofs = kKBytes + r * 64 + ((g ^ vswz(r)) << 4);

  unsigned* st_lds = reinterpret_cast<unsigned*>(smem + kRing * kStage) + w * kStampsPerBlock * kStampBlocks;
  auto stamp = [&](int j, int i) {
    if constexpr (STAMP) {
      if (lane == 0 && j < kStampBlocks) st_lds[kStampsPerBlock * j + i] = (unsigned)__builtin_amdgcn_s_memtime();
    }
  };
  bf16x8 vf[2][8];  // Vᵀ fragments of a block's two pages, read while its softmax is computed: a wave by itself gets 16 bytes per lane out of
                    // LDS every 46 clocks, the time of three MFMAs, so the reads of a block are spread over both its phases
  bf16x8 pf[2][2];  // Pᵀ fragments [query tile][page] of the block whose products come next
  bf16x8 kf[4][4];
  auto read_k = [&](int buf, int kt) {
    const char* kb = smem + buf * kStage;
#pragma unroll
    for (int s2 = 0; s2 < 4; ++s2) kf[kt][s2] = *reinterpret_cast<const bf16x8*>(kb + kt * 4096 + kofs[s2]);
  };
  auto read_v = [&](int buf, int t) {
    const char* vb0 = smem + buf * kStage;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) vf[t][dt] = *reinterpret_cast<const bf16x8*>(vb0 + t * 8192 + dt * 1024 + vofs);
  };
  // Oᵀ[d tile][query tile] += Vᵀ · Pᵀ of one page
  auto pv = [&](int t) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) o[dt][qt] = mfma16x16x32(vf[t][dt], pf[qt][t], o[dt][qt]);
    __builtin_amdgcn_sched_barrier(0);
  };
  // Sᵀ = K·Qᵀ of the block in LDS slot `buf`, whose first two tiles' fragments are read
  auto qk = [&](int buf) {
    read_k(buf, 2);
    read_k(buf, 3);
#pragma unroll
    for (int k2 = 0; k2 < 4; k2 += 2) {  // two key tiles at a time: four chains of products
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s2 = 0; s2 < 4; ++s2)
#pragma unroll
        for (int kt = k2; kt < k2 + 2; ++kt)
#pragma unroll
          for (int qt = 0; qt < 2; ++qt)
            s4[kt][qt] = mfma16x16x32(kf[kt][s2], qf[qt][s2], s2 ? s4[kt][qt] : f32x4{0.f, 0.f, 0.f, 0.f});
    }
  };
  // Online softmax of block j.  The running max (log2 units) only moves when a score exceeds it by more than kRescaleThr, so after the first blocks
  // O and l are not rescaled at all (P <= 2^thr stays well inside bf16 / fp32 range; the final O / l is unchanged).  Decided per wave (any
  // lane, each for the keys that it holds), and off the critical chain: the first half of the exponentials is made from the max as it was
  // and made again where it moved.
  auto softmax = [&](int j) {
    const int key0 = j * kBK;
    if (key0 + kBK - 1 > w_first_pos) {  // some key of the block is after some query: masked scores become -1e30
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) {
        const int qpos = q0 + 16 * qt + r < qlen ? pos0 + q0 + 16 * qt + r : -1;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
          for (int i = 0; i < 4; ++i) s4[kt][qt][i] = key0 + 16 * kt + 4 * g + i <= qpos ? s4[kt][qt][i] : -1e30f;
      }
    }
    // raw v_exp_f32 (no denormal range reduction: arguments are <= thr and underflow to 0 is wanted), the scale folded into one FMA; a
    // query with no visible key yet keeps m = -1e30 and must produce p = 0, not exp2(0)
    f32x4 e[2][2];
    auto make = [&](f32x4& to, int kt, int qt) {
      const float m_use = m_run[qt] < -1e29f ? 0.f : m_run[qt];
#pragma unroll
      for (int i = 0; i < 4; ++i) to[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s4[kt][qt][i], sc, -m_use));
    };
    auto half = [&]() {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) make(e[kt][qt], kt, qt);
    };
    float mx[2];
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {  // over the raw scores (scale_log2 > 0 commutes with max)
      float a = s4[0][qt][0], b = s4[2][qt][0];
#pragma unroll
      for (int i = 1; i < 8; ++i) {
        a = fmaxf(a, s4[i >> 2][qt][i & 3]);
        b = fmaxf(b, s4[2 + (i >> 2)][qt][i & 3]);
      }
      mx[qt] = fmaxf(a, b);
    }
    half();
    if (__any(mx[0] * sc > m_run[0] + kRescaleThr || mx[1] * sc > m_run[1] + kRescaleThr)) {
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) {
        const float m_new = fmaxf(m_run[qt], rows4_max(mx[qt]) * sc);
        const float alpha = __builtin_amdgcn_exp2f(m_run[qt] - (m_new < -1e29f ? 0.f : m_new));
        l_part[qt] *= alpha;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[dt][qt][i] *= alpha;
        m_run[qt] = m_new;
      }
      half();
    }
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) {
        if (kt < 2) s4[kt][qt] = e[kt][qt];
        else make(s4[kt][qt], kt, qt);
        // Pᵀ fragments: page t = key tiles 2t (keys 4g+i) and 2t+1 (keys 16+4g+i)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          l_part[qt][i & 1] += s4[kt][qt][i];
          pf[qt][kt >> 1][4 * (kt & 1) + i] = f2bf(s4[kt][qt][i]);
        }
      }
  };

  // Two phases per block, the products PV(j - 1), QKᵀ(j) and the softmax of block j, with a barrier before each.  Barrier accounting
  // (absolute barriers, counted from the loop entry of the leading half; the lagging half, wq = 1, passes one extra barrier first and
  // one fewer at the end).  Leading half: products of j in interval 2j, softmax in 2j + 1; lagging half one interval later.  So block j
  // is read from interval 2j (its K, leading) to 2j + 3 (its Vᵀ, lagging):
  //   RAW  every wave's DMA of block j has retired (its own counted vmcnt) before barrier 2j;
  //   WAR  block j + 4 reuses j's slot; its DMA is issued among the products of j + 2, in interval 2j + 4 or 2j + 5.
  // At barrier 2j either half has blocks up to j + 1 issued and waits for j: all but the youngest.
  const bool lag = wq == 1;
  issue_block(0);
  issue_block(1);
  if (lag) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(IPW) : "memory");
  auto step = [&](int j, auto slot, auto first) {  // slot: (j - jb) % kRing
    constexpr int k = decltype(slot)::value;
    stamp(j, 0);
    if (!lag) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(IPW) : "memory");
    else asm volatile("s_barrier" ::: "memory");
    stamp(j, 1);
    __builtin_amdgcn_s_setprio(1);
    if constexpr (!decltype(first)::value) {
      pv(0);
      read_k(k, 0);
      read_k(k, 1);
      issue_block((k + 2) % kRing);  // block j + 2
      pv(1);
    } else {
      read_k(k, 0);
      read_k(k, 1);
      issue_block((k + 2) % kRing);
    }
    qk(k);
    __builtin_amdgcn_s_setprio(0);
    stamp(j, 2);
    if (!lag) asm volatile("s_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(IPW) : "memory");
    stamp(j, 3);
    read_v(k, 0);
    softmax(j);
    stamp(j, 4);
    __builtin_amdgcn_sched_barrier(0);
    read_v(k, 1);
    stamp(j, 5);
  };
  // unrolled by the ring size: each block's LDS slot is a compile-time offset (no per-read address arithmetic)
  if (jb < jv) step(jb, std::integral_constant<int, 0>{}, std::true_type{});
  for (int j = jb + 1; j < jv; j += kRing) {
    step(j, std::integral_constant<int, 1>{}, std::false_type{});
    if (j + 1 < jv) step(j + 1, std::integral_constant<int, 2>{}, std::false_type{});
    if (j + 2 < jv) step(j + 2, std::integral_constant<int, 3>{}, std::false_type{});
    if (j + 3 < jv) step(j + 3, std::integral_constant<int, 0>{}, std::false_type{});
  }
  for (int j = max(jb, jv); j < je; ++j) {  // the barriers and the DMA of a step
    if (!lag) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(IPW) : "memory");
    else asm volatile("s_barrier" ::: "memory");
    issue_block((j - jb + 2) % kRing);
    if (!lag) asm volatile("s_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(IPW) : "memory");
  }
  if (!lag) asm volatile("s_barrier" ::: "memory");
  if (jb < jv) {
    pv(0);
    pv(1);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no DMA may still write this workgroup's LDS after it exits
  if constexpr (STAMP) {
    if (block < kStampWgs) {
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's stamp writes have landed
      unsigned* dst = stamps + ((size_t)block * NW + w) * kStampsPerBlock * kStampBlocks;
      for (int i = lane; i < kStampsPerBlock * kStampBlocks; i += 64) dst[i] = i < kStampsPerBlock * nblk ? st_lds[i] : 0u;
    }
  }

  // ---- epilogue: lane (r, g) holds O[query 16qt + r][d = 16dt + 4g + i]
  if (pslot >= 0) {  // one key range of a split tile: unnormalised O and (max, sum) for flash_combine_kernel
    const size_t sb = ((size_t)(pslot * p.hkv + h) * G + hs * HG + wh) * kBQ;
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      const int qrow = wq * 32 + 16 * qt + r;
      if (q0 + 16 * qt + r >= qlen) continue;
      const float l = rows4_sum(l_part[qt][0] + l_part[qt][1]);
      float* po = p.part_o + (sb + qrow) * kD + 4 * g;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) *reinterpret_cast<f32x4*>(po + 16 * dt) = o[dt][qt];
      if (g == 0) p.part_ml[sb + qrow] = make_float2(m_run[qt] < -1e29f ? 0.f : m_run[qt], l);
    }
    return;
  }
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    const int qi = q0 + 16 * qt + r;
    if (qi >= qlen) continue;
    const float l = rows4_sum(l_part[qt][0] + l_part[qt][1]);
    const float inv = l > 0.f ? 1.f / l : 0.f;
    bf16* op = p.out + ((size_t)(p.q_start[b] + qi) * p.hq + head) * kD + 4 * g;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      bf16x4 v;
      v[0] = f2bf(o[dt][qt][0] * inv);
      v[1] = f2bf(o[dt][qt][1] * inv);
      v[2] = f2bf(o[dt][qt][2] * inv);
      v[3] = f2bf(o[dt][qt][3] * inv);
      *reinterpret_cast<bf16x4*>(op + 16 * dt) = v;
    }
  }
}

}  // namespace
}  // namespace flash
}  // namespace dsse
