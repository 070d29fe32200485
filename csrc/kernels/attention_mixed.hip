// Attention of a mixed step in one launch: prompt tiles (attention_flash.h) and decode rows (attention_decode.h) of one layer.
//
// What bounds it: a step of 64 streams and 300 prompt rows has 40 prompt tiles, each a chain of key blocks on one of 256 CUs, and decode rows,
// which are bound by their pages.  One after the other they took 20 and 30 us; here the tiles' workgroups are the first of the grid and the
// other CUs read pages meanwhile.  A workgroup has the tile kernel's 8 waves and LDS, so a CU holds one: its waves take 8 / KWV (row, kv head, key
// partition) items of KWV waves each.
//
// Two launches / one, us, one MI355X, 32 heads over 8: 64 streams of 512 keys + 300 rows 50.9 / 40.2, + 64 rows 43.1 / 34.5, 32 + 300 40.2 / 32.2, 16
// of 500 + 200 30.3 / 19.9, 4 of 300 + 100 19.7 / 14.9, 2 of 64 + 32 13.4 / 9.1, 128 of 500 + 300 78.1 / 63.0, 128 of 128 + 384 41.3 / 28.0, 192 of
// 300 + 256 68.0 / 55.9, 16 of 4000 + 256 77.5 / 65.8, 64 of 512 + 256 rows behind 3000 148 / 117; one kv head, 64 + 256 29.5 / 24.4.
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

extern "C" hipError_t dsse_mixed_attention(int rows, const dsse::AttnParams* d, int num_work, const dsse::AttnParams* f, hipStream_t st) {
  using namespace dsse;
  if (d->group != 4 || f->group != 4 || rows <= 0 || num_work <= 0) return hipErrorNotSupported;
  const int tiles = num_work * f->hkv, items = rows * d->hkv * d->nparts;
  // Waves per item, 2 / 4 / 8, us: 1024 items of 500 keys 63.0 / 65.2 / 65.7, 800 of 300 31.0 / 34.0 / 37.0; 512 of 512 43.7 / 40.2 / 41.7, of 1000
  // (16 rows of 4000 in four partitions) 83.8 / 65.8 / 68.3, of 375 37.7 / 38.4 / 36.9, of 256 29.5 / 32.2 / 30.0; 384 of 170 22.3 / 21.2 / 19.9, 128 of
  // 75 16.7 / 16.5 / 14.9.  (Two pages in flight per wave are 0 to 5 us behind one; one wave per item 73 us at 512 keys.)
  const int kwv = d->kwv ? d->kwv : items > 640 ? 2 : items > 384 ? 4 : 8;
  const hipError_t e = kwv <= 2 ? launch<2>(tiles, rows, *d, *f, st) : kwv == 4 ? launch<4>(tiles, rows, *d, *f, st) : launch<8>(tiles, rows, *d, *f, st);
  return e == hipSuccess && d->nparts > 1 ? dsse_attn_combine(rows, d, st) : e;
}

DSSE_CHECK_READER(dsse_check_attention_mixed)
