// The tiled ping-pong prefill (prefill_run in prefill_impl.h) at head sizes
// other than 128, over pages its scalar tile bases can address.
//
// Against the generic kernel of any_head.hip, which stages K and V through
// registers a 32-token step at a time with two barriers a step, the tiles
// come straight into a four-stage LDS ring and one wave of a SIMD feeds the
// matrix cores while the other takes its softmax.  16 sequences of 1000 to
// 3000 tokens, 32 / 8 heads, generic -> this with the work list (one MI355X):
// 64 360 -> 316 us (soft cap 481 -> 422), 96 489 -> 440 (828 -> 575), 256 1682
// -> 1083 (1771 -> 1110); one sequence of 32768 tokens: 64 4.83 -> 4.21 ms, 96
// 6.55 -> 5.94, 256 24.5 -> 16.6.
// Bound by the softmax's VALU work at 64, by MFMA and LDS reads at 256, and
// by the ~7 us an item spends outside its loop at these lengths.  80 gained
// nothing (492 us against 478, its generic kernel also fits two workgroups a
// CU) and stays generic, as do the sizes between.
#include <algorithm>
#include <cmath>
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

// Items of `tokens`-token tiles a launch has, about: a sequence of n tokens has
// ceil(n / tokens) of them per kv head, half a tile more than its tokens fill.
static double items_of(const PrefillParams& p, int64_t tokens) {
  const double grid = (double)p.batch * ((p.max_seqlen_q + tokens - 1) / tokens);
  return std::min(grid, (double)p.num_tokens / tokens + .5 * p.batch) * p.num_kv_heads;
}

// Whether a launch at head size 256 is faster tiled than in the generic
// kernel.  The generic kernel's items are half as long (128 rows against 256)
// and each is done sooner: 12 us and 44 ns a kv token on a CU of its own,
// against 10 us and 57 ns.  So a launch whose generic items fit one round on
// the CUs stays generic, unless its sequences fill at most half a tile, where
// the tiled kernel's other waves skip their work; a launch of several rounds
// is tiled, and in between the two estimates decide: the longest item, or all
// of them over the CUs.  kv lengths are on the device.  The longest is taken
// from the table's width (its last page half full), or, where cu_seqlens_k says that nothing is cached
// (and in a mixed launch, whose table is as wide as its decode sequences),
// from max_seqlen_q; the others are taken to be as long, or, up to max_seqlen_q,
// to have nothing cached.
// Generic -> tiled, 32 / 8 heads unless said, us (both kernels timed at 740
// shapes, 400 of them with the soft cap as well; in all but three this rule is
// within 2.3 % of the generic one or faster, at worst 1.2 us of 23 behind): generic
// 3 x 299 tokens 28.0 -> 31.5, 1 x 2000 118 -> 131, 1 x 1000 behind 4000
// cached 237 -> 302, 16 / 8 heads 1 x 4000 211 -> 246; tiled 4 x 511 50.3 ->
// 46.6, 1 x 3000 258 -> 190, 4 x 300 behind 4000 384 -> 265, 8 / 8 heads 8 x 64
// behind 4000 223 -> 175.
static bool tiled_256_pays(const PrefillParams& p) {
  const int rows = 128;  // of a generic item
  const double mean = (double)p.num_tokens / p.batch;
  const double span = (double)p.pages_per_seq * p.page_size;
  const int64_t seq_rows = (int64_t)p.max_seqlen_q * p.group;
  if (seq_rows > 32 && seq_rows <= rows) return true;
  if (seq_rows > 32 && seq_rows <= kRows && p.max_seqlen_q <= 64 && span <= 256) return true;
  const double generic = items_of(p, rows / p.group), tiled = items_of(p, kRows / p.group);
  if (generic <= kCUs && (int64_t)p.num_tokens * p.num_heads < (int64_t)kCUs * rows) return false;
  const bool fresh = p.kv_lens || !p.cu_k || p.cu_k == p.cu_q;
  const double longest = fresh ? std::min<double>(span, p.max_seqlen_q) : std::max(span - .5 * p.page_size, mean);
  // over a sequence's items
  const double average = longest <= p.max_seqlen_q ? longest / 2 : longest - std::min(mean, longest) / 2;
  double rounds = generic / kCUs;
  // mostly cached tokens: items of about one length, so whole rounds
  if (longest > 2 * (p.batch == 1 ? mean : (double)p.max_seqlen_q)) rounds = std::ceil(rounds);
  const double t_generic = std::max(12 + .044 * longest, rounds * (12 + .044 * average) + (generic > kCUs ? 5 : 0));
  const double t_tiled = std::max(10 + .057 * longest, tiled / kCUs * (10 + .057 * average));
  return t_tiled < t_generic;
}

bool prefill_tiled(const PrefillParams& p, int head_dim) {
  if (p.batch == 0 || p.max_seqlen_q == 0) return false;
  switch (head_dim) {
    case 64: return paging_of<64>(p) != kPageLane;
    case 96: return paging_of<96>(p) != kPageLane;
    case 256: return p.group <= 128 && paging_of<256>(p) != kPageLane && tiled_256_pays(p);
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
