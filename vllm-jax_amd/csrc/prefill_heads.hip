// The tiled ping-pong prefill (prefill_run in prefill_impl.h) at head sizes
// other than 128, over pages its scalar tile bases can address.
//
// Against the generic kernel of any_head.hip, which stages K and V through
// registers a 32-token step at a time with two barriers a step, the tiles
// come straight into a four-stage LDS ring and one wave of a SIMD feeds the
// matrix cores while the other takes its softmax.  16 sequences of 1000 to
// 3000 tokens, 32 / 8 heads, generic -> this (one MI355X): 64 391 -> 351 us,
// 96 522 -> 511 (soft cap 852 -> 653), 256 1927 -> 1316 (soft cap 2037 ->
// 1326); one sequence of 32768 tokens: 64 4.82 -> 4.31 ms, 256 25.1 -> 16.7.
// Bound by the softmax's VALU work at 64, by MFMA and LDS reads at 256, and
// by the ~7 us an item spends outside its loop at these lengths.  80 gained
// nothing (492 us against 478, its generic kernel also fits two workgroups a
// CU) and stays generic, as do the sizes between.
#include <algorithm>
#include <type_traits>

#include "any_head.h"
#include "prefill_impl.h"

namespace pa {
namespace {

constexpr int kCUs = 256;

// Tile paging of a launch at head size D; kPageLane: not one of the forms
// built here (pages of other sizes, or rows too far apart for 32-bit offsets).
template <int D, bool kSoftCap>
int tiled_paging(int32_t page_size, int64_t slot_stride) {
  using A = PrefillDims<D, kSoftCap>;
  if (!prefill_offsets_fit(slot_stride, A::kN, D)) return kPageLane;
  if (page_size % A::kN == 0) return kPageTile;
  if (page_size == 16 || page_size == 32) return kPageWave;
  return kPageLane;
}

template <int D, bool kSoftCap>
int launch(const char* name, const PrefillParams& p, hipStream_t s) {
  const int paging = tiled_paging<D, kSoftCap>(p.page_size, p.slot_stride);
  const int64_t items = (int64_t)p.n_qtiles * p.batch * p.num_kv_heads;
  // without a list, workgroups past the items zero the rows no item writes,
  // 512 tokens each
  const int64_t blocks = items + (p.plan ? 0 : ((int64_t)p.num_tokens + kThreads - 1) / kThreads);
  if (blocks > 0x7fffffff)
    return fail(PA_ERR_UNSUPPORTED, "%s: grid of %lld workgroups too large", name, (long long)blocks);
  const dim3 g((unsigned)blocks), b(kThreads);
  auto run = [&](auto pg) {
    constexpr int kPg = decltype(pg)::value;
    if (p.plan) prefill_kernel<kSoftCap, kPg, false, D><<<g, b, 0, s>>>(p);
    else prefill_kernel<kSoftCap, kPg, true, D><<<g, b, 0, s>>>(p);
  };
  if (paging == kPageTile) run(std::integral_constant<int, kPageTile>{});
  else run(std::integral_constant<int, kPageWave>{});
  return launch_status(name);
}

template <int D>
int paging_of(const PrefillParams& p) {
  return p.soft_cap > 0.f ? tiled_paging<D, true>(p.page_size, p.slot_stride)
                          : tiled_paging<D, false>(p.page_size, p.slot_stride);
}

}  // namespace

bool prefill_tiled(const PrefillParams& p, int head_dim) {
  if (p.batch == 0 || p.max_seqlen_q == 0) return false;
  const int64_t tile_tokens = kRows / p.group;
  const int64_t pairs = p.batch * ((p.max_seqlen_q + tile_tokens - 1) / tile_tokens);
  // At 256 the generic kernel's items are half as long (128 rows): while they
  // fit one round on the CUs it is faster (3 x 299 tokens, 32 / 8 heads, 29.1
  // us against 31.7; 2 x 300 behind 4000 cached 203 against 260), from there
  // on this one (4 x 511 tokens 47 us against 52, 8 x 512 64 against 96).
  const int64_t live = std::min<int64_t>(pairs, p.num_tokens / tile_tokens + p.batch);
  switch (head_dim) {
    case 64: return paging_of<64>(p) != kPageLane;
    case 96: return paging_of<96>(p) != kPageLane;
    case 256: return p.group <= 128 && paging_of<256>(p) != kPageLane && live * p.num_kv_heads >= kCUs / 2;
    default: return false;
  }
}

int prefill_tiled_launch(const char* name, const PrefillParams& prm, int head_dim, hipStream_t s) {
  if (!prefill_tiled(prm, head_dim)) return kPrefillNotTiled;
  PrefillParams p = prm;
  p.pool = nullptr;
  p.tile_tokens = kRows / p.group;
  p.n_qtiles = (p.max_seqlen_q + p.tile_tokens - 1) / p.tile_tokens;
  const bool cap = p.soft_cap > 0.f;
  switch (head_dim) {
    case 64: return cap ? launch<64, true>(name, p, s) : launch<64, false>(name, p, s);
    case 96: return cap ? launch<96, true>(name, p, s) : launch<96, false>(name, p, s);
    case 256: return cap ? launch<256, true>(name, p, s) : launch<256, false>(name, p, s);
    default: return kPrefillNotTiled;
  }
}

}  // namespace pa
