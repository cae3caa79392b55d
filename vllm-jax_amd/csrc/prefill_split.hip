// Prefill of few, long items: split over the kv range, then merged.
//
// One (q tile, sequence, kv head) item per workgroup leaves most of the chip
// idle when there are few of them: two new turns of 128 to 400 tokens behind
// 6 000 to 15 000 cached ones are 72 items of up to 240 kv tiles on 256 CUs.
// Here every workgroup first counts the launch's kv tiles (one thread per
// (sequence, q tile) pair, as prefill_plan estimates them), finds a part
// length with which the parts fill the chip once, and runs one part of one
// item.  A part leaves its unnormalised O, reference max
// and row sums in f32; prefill_split_merge_kernel adds the parts up.  That
// call: 217 us unsplit, 92 us so (131 with parts of an even share,
// whose 288 parts took two rounds).  What is left: about 1.1 us a tile and 10
// us around the loop, and 32 MB of partials written and read.
//
// A split pays where the parts are shorter than the longest item by more than
// the count, the partials and the merge cost.  The kernel knows the lengths
// and splits nothing where it does not; the host knows an upper bound of the
// items and takes the longest kv length from the table's width (from the new
// tokens where cu_seqlens_k says that nothing is cached), and launches the
// plain kernel where a split cannot be told to pay (prefill_splits).
#include <algorithm>
#include <climits>

#include "prefill_impl.h"
#include "prefill_split.h"

namespace pa {
namespace {

constexpr int kSplitCUs = 256;
// Pairs the in-kernel count takes.
constexpr int kSplitMaxPairs = 256;
static_assert(kSplitMaxPairs % 64 == 0 && kSplitMaxPairs <= kThreads, "one thread per pair, whole waves");
// No part below this many tiles is made: a part costs about 7 us outside its
// loop, and a tile about 1 us.
constexpr int kSplitMinTiles = 8;
// Shortest table span (in kv tiles) of a launch that splits.
constexpr int kSplitMinSpan = 24;
// From this longest kv length (in tiles) on several sequences are looked at by
// the kernel even where equal ones would gain nothing.  Where it then splits
// nothing, the count and the merge launch cost 4 to 7 us of 105 to 240; where
// it splits, such launches gain 20 % on average and up to 70.
constexpr int kSplitTryLongest = 80;
// Items that run at an item's own speed; more share the chip's power (a kv
// tile takes 1.04 us with up to 150 items at once, 1.45 us with 240).
constexpr float kSplitBusy = 165.f;
// What a split costs, in tiles: the count, the partials, the merge.
constexpr float kSplitCost = 9.f;
// Time, in tiles, of `parts` parts of `total` tiles in all, the longest of
// `len`: all but the longest as if they ended together.
__host__ __device__ inline float split_time(float len, float parts, float total) {
  return parts <= kSplitBusy ? len : fmaxf(len, total / kSplitBusy + len - total / parts);
}
// At least the time of the launch unsplit.
__host__ __device__ inline float whole_time(float longest, float total) { return fmaxf(longest, total / kSplitBusy); }
// Largest grid (n_qtiles x batch x kv heads) that is looked at.
constexpr int64_t kSplitMaxGrid = 1024;

// Slots of a launch: sum over pairs of ceil(tiles / L) with L at
// least an even share, tiles * kv heads / kSplitCUs, is at most kSplitCUs / kv
// heads + pairs; only split pairs (two parts or more, so longer than L, so at
// most kSplitCUs / kv heads of them) take slots.
int64_t split_max_slots(int64_t pairs, int32_t hkv) {
  const int64_t share = kSplitCUs / hkv;
  return (share + std::min(pairs, share)) * hkv;
}
// Split pairs of a launch: longer than L, so fewer than kSplitCUs / kv heads.
int64_t split_max_pairs(int64_t pairs, int32_t hkv) { return std::min<int64_t>(pairs, kSplitCUs / hkv); }
// The number of split pairs, then a record of four ints for each (fewer than
// 256, so that the number and they fit).
constexpr size_t kSplitHeader = kSplitMaxPairs * 4 * sizeof(int32_t);

template <bool kSoftCap, int kPaging>
__global__ void __launch_bounds__(kThreads, 1)
prefill_split_kernel(PrefillParams p, int grid_parts) {
  if ((int)blockIdx.x >= grid_parts) {  // uniform over the workgroup
    prefill_zero_rows<kPHeadDim>(p, ((int64_t)blockIdx.x - grid_parts) * kThreads);
    return;
  }
  __shared__ unsigned long long s_total;
  __shared__ int32_t s_tiles[kSplitMaxPairs];
  __shared__ float s_count[kWaves][64], s_longest[kWaves];
  __shared__ uint32_t s_before[kSplitMaxPairs / 64];
  __shared__ int32_t s_work[9];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hkv = p.num_kv_heads;
  const int nq = p.n_qtiles;
  const int pairs = p.batch * nq;
  const int mine = blockIdx.x / hkv;  // part of the launch's list; kv head bid % hkv (one XCD per head)
  if (tid == 0) {
    s_total = 0;
    s_work[0] = -1;
  }
  __syncthreads();
  int4 g = {};
  int tiles = -1, b = 0, qt = 0;
  if (tid < pairs) {
    int lag;
    b = tid / nq;
    qt = tid - b * nq;
    prefill_seq_geometry(p, b, g, lag);
    tiles = prefill_pair_tiles(g, lag, qt, p.tile_tokens);  // -1: no rows
    if (tiles > 0) atomicAdd(&s_total, (unsigned long long)tiles);
  }
  if (tid < kSplitMaxPairs) s_tiles[tid] = tiles;
  __syncthreads();
  // The part length: an even share of the launch's tiles leaves more parts
  // than CUs (every pair rounds up), so lane k of each wave counts the parts
  // of the wave's share of the pairs at a share times 2^(k / 10), and the
  // shortest length that fits one round is taken.  If none does (one pair 78
  // times the share, or more), nothing is split.
  const int64_t share = ((int64_t)s_total * hkv + kSplitCUs - 1) / kSplitCUs;
  const float cand = ceilf((float)max((int64_t)kSplitMinTiles, share) * exp2f(.1f * (float)lane));
  const float inv = 1.f / cand;
  float count = 0.f, longest = 0.f;
  const int per_wave = (pairs + kWaves - 1) / kWaves;
#pragma unroll 4
  for (int j = wave * per_wave; j < min(pairs, (wave + 1) * per_wave); ++j) {
    const float tj = (float)s_tiles[j];
    count += tj < 0.f ? 0.f : fmaxf(1.f, ceilf(tj * inv));
    longest = fmaxf(longest, tj);
  }
  s_count[wave][lane] = count;
  s_longest[wave] = longest;  // the same in every lane
  __syncthreads();
  count = 0.f;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) {
    count += s_count[i][lane];
    longest = fmaxf(longest, s_longest[i]);
  }
  const uint64_t fits = __ballot(count * (float)hkv <= (float)kSplitCUs);
  float len = (float)INT_MAX;
  if (fits) {
    const int first = __ffsll((unsigned long long)fits) - 1;
    const float at = __shfl(cand, first), total = (float)s_total * (float)hkv;
    const float split = split_time(at, __shfl(count, first) * (float)hkv, total) + kSplitCost;
    if (split < whole_time(longest, total)) len = at;
  }
  const int parts = tiles < 0 ? 0 : max(1, (int)ceilf((float)tiles * (1.f / len)));  // as counted
  // parts, partial slots and split pairs of the pairs before this one, ten
  // bits each: at most kSplitCUs of them
  const uint32_t own = (uint32_t)parts | (parts > 1 ? (uint32_t)parts << 10 | 1u << 20 : 0u);
  uint32_t upto = wave_scan(own);
  if (lane == 63 && wave < kSplitMaxPairs / 64) s_before[wave] = upto;
  __syncthreads();
  uint32_t all = 0;
#pragma unroll
  for (int i = 0; i < kSplitMaxPairs / 64; ++i) {
    upto += i < wave ? s_before[i] : 0;
    all += s_before[i];
  }
  const uint32_t before = upto - own;
  const int at = (int)(before & 0x3ff), slot = (int)(before >> 10 & 0x3ff);
  if (mine >= at && mine < at + parts) {
    const int k = mine - at;
    s_work[0] = b;
    s_work[1] = qt;
    s_work[2] = g.x;
    s_work[3] = g.y;
    s_work[4] = g.z;
    s_work[5] = g.w;
    s_work[6] = (int)((int64_t)tiles * k / parts);
    s_work[7] = k + 1 == parts ? INT_MAX : (int)((int64_t)tiles * (k + 1) / parts);
    s_work[8] = parts > 1 ? (slot + k) * hkv : -1;
  }
  if (blockIdx.x == 0) {  // for the merge
    if (tid == 0) p.split[0] = (int)(all >> 20);
    if (parts > 1)
      st16(p.split + 4 * (1 + (before >> 20)), u32x4{(uint32_t)parts | (uint32_t)qt << 16, (uint32_t)(slot * hkv),
                                                     (uint32_t)g.x, (uint32_t)g.y});
  }
  __syncthreads();
  auto work = [&](int i) { return __builtin_amdgcn_readfirstlane(s_work[i]); };
  PrefillWork w;
  w.b = work(0);
  if (w.b < 0) return;  // past the list; uniform over the workgroup
  w.qt = work(1);
  w.kvh = (int)blockIdx.x - mine * hkv;
  w.q0 = work(2);
  w.lq_rows = work(3);
  w.lk = work(4);
  w.kv_pos_off = work(5);
  PrefillPart part;
  part.lo = work(6);
  part.hi = work(7);
  part.slot = work(8);
  if (part.slot >= 0) part.slot += w.kvh;
  prefill_run<kSoftCap, kPaging, kPHeadDim, true>(p, w, part);
}

// out = sum_k o_k 2^(m_k - M) / sum_k l_k 2^(m_k - M) over an item's parts k,
// M their largest reference max.
// One workgroup per (split pair, kv head, 32-row block), one wave per 32 d: the
// lanes hold what the part's accumulators held.
__global__ void __launch_bounds__(256)
prefill_split_merge_kernel(PrefillParams p) {
  const int hkv = p.num_kv_heads;
  const int item = blockIdx.x / kWaves;
  const int block = blockIdx.x - item * kWaves;
  const int rank = item / hkv;
  const int kvh = item - rank * hkv;
  if (rank >= p.split[0]) return;
  const int4 rec = *reinterpret_cast<const int4*>(p.split + 4 * (1 + rank));  // parts and q tile, first slot, q0, rows
  const int parts = rec.x & 0xffff;
  const float* src = p.parts + (int64_t)(rec.y + kvh) * kPartFloats<kPHeadDim>;
  const int64_t step = (int64_t)hkv * kPartFloats<kPHeadDim>;
  const int lane = threadIdx.x & 63;
  const int dt = threadIdx.x >> 6;
  const int n = lane & 31, h = lane >> 5;
  const int row = 32 * block + n;
  const int rtok = (rec.x >> 16) * p.tile_tokens + row / p.group;
  const float* ml = src + kPartO<kPHeadDim> + 2 * row;
  const float* po = src + 4 * ((block * 4 + dt) * 4 * 64 + lane);
  f32x4 o[4] = {};
  float m_run = -INFINITY, lsum = 0.f;
  // the sums follow a running max, so that no load waits for another part's
#pragma unroll 4
  for (int k = 0; k < parts; ++k) {
    const f32x2 v = *reinterpret_cast<const f32x2*>(ml + k * step);
    const float m_new = fmaxf(m_run, v[0]);
    const float ms = m_new == -INFINITY ? 0.f : m_new;
    const float old = fast_exp2(m_run - ms), wgt = fast_exp2(v[0] - ms);
    m_run = m_new;
    lsum = lsum * old + v[1] * wgt;
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4)
      o[q4] = o[q4] * old + *reinterpret_cast<const f32x4*>(po + k * step + 256 * q4) * wgt;
  }
  if (row >= p.tile_tokens * p.group || rtok >= rec.w) return;
  const float inv = lsum > 0.f ? 1.f / lsum : 0.f;  // rows that see no key are zeros
  uint16_t* orow = p.out + (int64_t)(rec.z + rtok) * p.o_ts +
                   (int64_t)(kvh * p.group + row - row / p.group * p.group) * p.o_hs + 32 * dt + 4 * h;
#pragma unroll
  for (int q4 = 0; q4 < 4; ++q4)
    *reinterpret_cast<u32x2*>(orow + 8 * q4) =
        u32x2{pack_bf16x2(o[q4][0] * inv, o[q4][1] * inv), pack_bf16x2(o[q4][2] * inv, o[q4][3] * inv)};
}

}  // namespace

size_t prefill_split_bytes(int32_t batch, int32_t n_qtiles, int32_t num_kv_heads, int64_t span) {
  const int64_t pairs = (int64_t)batch * n_qtiles;
  if (pairs <= 0 || pairs > kSplitMaxPairs || pairs * num_kv_heads > kSplitMaxGrid ||
      span < (int64_t)kSplitMinSpan * kTileN)
    return 0;
  return kSplitHeader + (size_t)split_max_slots(pairs, num_kv_heads) * kPartFloats<kPHeadDim> * sizeof(float);
}

// With N items, the longest of T tiles (N an upper bound, T a lower one), a
// split surely pays if it does where every sequence is as long as the longest:
// to bring that down to L tiles each sequence has at most 64 (T - L) /
// tile_tokens items a kv head cut in two; or all N items are cut in 256 / N.
// Unsplit -> split, 32 / 8 heads unless said, us: 64 new tokens behind 1500
// cached 35.4 -> 22.4, 4 x 100 behind 1500 36.0 -> 30.4, 800 behind 8000 153.6
// -> 111.5, fresh 2400 at 16 / 8 heads 50.4 -> 43.8.  Split before this rule,
// and slower: fresh 1792 41.9 -> 47.7, fresh 3500 at 16 / 8 heads 72.0 -> 77.0,
// 1100 behind 8000 160.9 -> 178.9, 3 x 400 behind 2000 54.7 -> 60.5.
bool prefill_splits(const PrefillParams& p) {
  const int64_t tile = p.tile_tokens, batch = p.batch, hkv = p.num_kv_heads;
  if (batch == 0 || p.n_qtiles == 0 || batch * p.n_qtiles * hkv >= kSplitMaxGrid) return false;
  // pairs with rows: a sequence of n tokens has ceil(n / tile)
  const int64_t items = std::min<int64_t>(batch * p.n_qtiles, (p.num_tokens + batch * (tile - 1)) / tile) * hkv;
  if (items == 0 || items >= kSplitCUs) return false;
  const int64_t span = (int64_t)p.pages_per_seq * p.page_size, mean = (p.num_tokens + batch - 1) / batch;
  const bool fresh = !p.cu_k || p.cu_k == p.cu_q;
  const int64_t kv = fresh ? std::min(span, mean) : std::max(span - p.page_size + 1, mean);
  const int64_t longest = (kv + kTileN - 1) / kTileN;
  if (longest == 0) return false;
  const float t = (float)longest, n = (float)items;
  // the items of a sequence are tile / 64 tiles apart
  const float total = n * std::max(.5f * t, t - (n / (float)(batch * hkv) - 1.f) * (float)tile / (2 * kTileN));
  // (one cost more than the kernel's: the bounds round to whole tiles)
  const float whole = (batch == 1 ? whole_time(t, total) : t) - kSplitCost - 1.f;
  const float step = (float)(batch * kTileN * hkv) / (float)tile;
  const float half = std::max(.5f * t, t - ((float)kSplitCUs - n) / step);
  if (half < t && split_time(std::max(half, (float)kSplitMinTiles), n + std::min(n, step * (t - half)), total) < whole)
    return true;
  const int64_t ways = kSplitCUs / items;
  const int64_t len = std::max<int64_t>(kSplitMinTiles, (longest + ways - 1) / ways);
  if (split_time((float)len, n * (float)((longest + len - 1) / len), total) < whole) return true;
  return batch > 1 && longest >= kSplitTryLongest;
}

int prefill_split_launch(const char* name, const PrefillParams& prm, int paging, void* workspace, hipStream_t s) {
  PrefillParams p = prm;
  p.split = reinterpret_cast<int32_t*>(workspace);
  p.parts = reinterpret_cast<float*>((char*)workspace + kSplitHeader);
  const int64_t pairs = (int64_t)p.batch * p.n_qtiles;
  // the parts fit one round, and so do the pairs with rows (prefill_splits)
  const int grid_parts = kSplitCUs / p.num_kv_heads * p.num_kv_heads;
  // workgroups past the parts zero the rows no item writes, 512 tokens each
  const int64_t blocks = grid_parts + ((int64_t)p.num_tokens + kThreads - 1) / kThreads;
  const dim3 grid((unsigned)blocks), blk(kThreads);
  auto launch = [&](auto cap) {
    constexpr bool kCap = decltype(cap)::value;
    if (paging == kPageTile) prefill_split_kernel<kCap, kPageTile><<<grid, blk, 0, s>>>(p, grid_parts);
    else if (paging == kPageWave) prefill_split_kernel<kCap, kPageWave><<<grid, blk, 0, s>>>(p, grid_parts);
    else prefill_split_kernel<kCap, kPageLane><<<grid, blk, 0, s>>>(p, grid_parts);
  };
  if (p.soft_cap > 0.f) launch(std::true_type{});
  else launch(std::false_type{});
  const int rc = launch_status(name);
  if (rc) return rc;
  const int64_t merges = split_max_pairs(pairs, p.num_kv_heads) * p.num_kv_heads * kWaves;
  if (merges > 0) prefill_split_merge_kernel<<<dim3((unsigned)merges), dim3(256), 0, s>>>(p);
  return launch_status(name);
}

}  // namespace pa
