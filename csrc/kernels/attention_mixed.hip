// Attention of a mixed step in one launch: prompt tiles (attention_flash.h) and decode rows (attention_decode.h) of one layer.
//
// What bounds it: a step of 64 streams and 300 prompt rows has 40 prompt tiles, each a chain of key blocks on one of 256 CUs, and decode rows,
// which are bound by their pages.  One after the other they take 16 and 30 us; here the tiles' workgroups are the first of the grid and the
// other CUs read pages meanwhile.  A workgroup has the tile kernel's 8 waves and LDS, so a CU holds one: its waves take 8 / KWV (row, kv head, key
// partition) items of KWV waves each.
//
// Two launches / one, us, one MI355X, 32 heads over 8: 64 streams of 512 keys + 300 rows 47.5 / 37.8, + 64 rows 42.1 / 33.3, 32 + 300 37.0 / 31.3, 16
// of 500 + 200 27.9 / 19.2, 4 of 300 + 100 18.2 / 13.5, 2 of 64 + 32 12.4 / 8.1, 128 of 500 + 300 74.5 / 61.1, 128 of 128 + 384 37.2 / 27.7, 192 of
// 300 + 256 65.3 / 56.4, 16 of 4000 + 256 75.1 / 63.8, 64 of 512 + 256 rows behind 3000 112 / 80; one kv head, 64 + 256 26.5 / 21.2.
#include "attention_decode.h"
#include "attention_flash.h"

namespace dsse {
namespace {

constexpr int kWaves = 8;
constexpr int kLds = flash::kRing * flash::kStage;

template <int KWV>
__global__ void __launch_bounds__(64 * kWaves) mixed_attention_kernel(AttnParams d, AttnParams f, int tiles, int rows) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  if ((int)blockIdx.x < tiles) {
    flash::flash_prefill<4, 4, false>(f, nullptr, blockIdx.x, smem);
    return;
  }
  constexpr int kItems = kWaves / KWV;
  typedef DecodeLds<1, KWV, 0> Lds;
  static_assert(sizeof(Lds) * kItems <= kLds, "the tile kernel's LDS");
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), sub = w / KWV;
  const int i = ((int)blockIdx.x - tiles) * kItems + sub;
  const int items = rows * d.hkv * d.nparts, at = min(i, items - 1);
  decode_attention<1, KWV, 1, 0, true>(d, at % rows, at / rows % d.hkv, i < items ? at / (rows * d.hkv) : d.nparts, w % KWV,
                                        reinterpret_cast<Lds*>(smem)[sub]);
}

template <int KWV>
hipError_t launch(int tiles, int rows, const AttnParams& d, const AttnParams& f, hipStream_t st) {
  static bool attr_set = false;
  if (!attr_set) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&mixed_attention_kernel<KWV>), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    attr_set = true;
  }
  const int items = rows * d.hkv * d.nparts, per = kWaves / KWV;
  hipLaunchKernelGGL((mixed_attention_kernel<KWV>), dim3(tiles + (items + per - 1) / per), dim3(64 * kWaves), kLds, st, d, f, tiles, rows);
  return hipGetLastError();
}

}  // namespace
}  // namespace dsse

// Waves per (row, kv head, key partition) item of the one launch; 0: the step goes in two.  By the count of items, since how many keys an item has is known on
// the device only.  2 / 4 / 8, us: 1024 items of 500 keys 61.1 / 62.4 / 66.4, 800 of 300 31.1 / 33.7 / 37.2; 512 of 512 43.6 / 37.8 / 41.2, of 1000
// (16 rows of 4000 in four partitions) 85.0 / 63.8 / 67.1, of 375 37.9 / 35.5 / 36.4; 384 of 170 22.2 / 19.0 / 19.2, 128 of 75 15.3 / 15.1 / 13.5.  What the
// rule gives away: 512 of 256 keys 29.2 / 31.3 / 29.4.  (Two pages in flight per wave are 0 to 5 us behind one; one wave per item 73 us at 512 keys.)
extern "C" int dsse_mixed_attention_waves(int group, int rows, int hkv, int nparts, int num_work, int forced) {
  if (group != 4 || rows <= 0 || num_work <= 0) return 0;
  const int items = rows * hkv * nparts, kwv = forced ? forced : items > 640 ? 2 : items > 384 ? 4 : 8;
  return kwv < 2 ? 2 : kwv;
}

extern "C" hipError_t dsse_mixed_attention(int rows, const dsse::AttnParams* d, int num_work, const dsse::AttnParams* f, hipStream_t st) {
  using namespace dsse;
  const int kwv = f->group == d->group ? dsse_mixed_attention_waves(d->group, rows, d->hkv, d->nparts, num_work, d->kwv) : 0;
  if (!kwv) return hipErrorNotSupported;
  const int tiles = num_work * f->hkv;
  const hipError_t e = kwv == 2 ? launch<2>(tiles, rows, *d, *f, st) : kwv == 4 ? launch<4>(tiles, rows, *d, *f, st) : launch<8>(tiles, rows, *d, *f, st);
  return e == hipSuccess && d->nparts > 1 ? dsse_attn_combine(rows, d, st) : e;
}

DSSE_CHECK_READER(dsse_check_attention_mixed)
