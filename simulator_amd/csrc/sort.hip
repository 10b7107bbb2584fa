// sort.hip -- Morton codes of the triangles' boxes and their stable sort on
// gfx950, for one body or for all bodies of a batch together.
//
// LSD radix sort of (code, primitive) pairs by code, three passes of 10-bit
// digits (the Morton codes have 30 bits).  Because the primitives enter in
// ascending order and every pass is stable, the result is ordered by the
// full 64-bit key (code << 32 | primitive).
//
// A pass cuts every body's keys into tiles of SORT_TILE, one workgroup each:
// the tile's digit counts (by k_morton for the first pass, k_radix_count for
// the others), then k_radix_scatter.  For a body of up to SORT_SUM_TILES tiles
// there is no scan launch between the two: the counts lie tile after tile
// and every scatter workgroup sums the ones before its own and all of them
// itself (at most 64 x 2 KB, coalesced).  The counts of a larger body are
// scanned by k_tile_scan first, because the tiles' own sums grow with the
// square of their number.
//
// What bounds it: for one body the chain of small launches (its lanes run
// beside the step, and other simulators' work queues behind them); for a
// batch the ranking and the scattered stores.  50,688 triangles, three frames
// in a chain: 33 us from codes to sorted keys in six launches, against
// 68 us in eleven (separate counts of the first pass, scans and key / leaf
// writing; one row of 256 keys at a time between barriers); four rows per wave
// instead of two: 33 us of scatters against 27.  The 4.2 M
// triangles of 256 bodies: 156 us, against 244 us with one workgroup per
// body (bound by the largest body, 36,096 keys on one CU).
#include "cc_device.h"
#include "cc_lbvh.h"

namespace cc {

constexpr int SORT_THREADS = 512;
constexpr int SORT_WAVES = SORT_THREADS / 64;
constexpr int SORT_ROWS = SORT_TILE / SORT_THREADS;   // rows of 64 consecutive keys per wave
constexpr int RADIX_BITS = 10;
constexpr int RADIX_DIGITS = 1 << RADIX_BITS;
constexpr int RADIX_PASSES = 3;
// a tile's counts are 16-bit pairs; a scatter workgroup reads them in
// SORT_GROUPS groups of lanes, each summing every SORT_GROUPS-th tile,
// SORT_LOADS of them in flight
constexpr uint32_t SORT_WORDS = RADIX_DIGITS / 2;
constexpr uint32_t SORT_GROUPS = SORT_THREADS * 4 / SORT_WORDS;
constexpr uint32_t SORT_LOADS = 8;
static_assert(SORT_THREADS * 2 == RADIX_DIGITS, "two digits per thread");
static_assert(SORT_SUM_TILES / SORT_GROUPS * SORT_TILE < 65536, "a group's sums fit 16 bits");

// A tile's entry {body, tile, tiles of the body, its first tile}; a big body's
// third word is TILES_BIG + the number of its row of totals.
constexpr uint32_t TILES_BIG = 1u << 31;

__device__ inline void put_counts(const uint32_t* h, uint32_t* __restrict__ counts, uint4 t) {
  counts[(size_t)(t.w + t.y) * SORT_WORDS + threadIdx.x] = h[2 * threadIdx.x] | (h[2 * threadIdx.x + 1] << 16);
}

// root box (sentinel U the body's partials, recomputed per tile), then the
// code of each box centroid (compute_morton_bbox, bvh.cu:71-79) of a tile and
// the first pass's digit counts
__global__ __launch_bounds__(SORT_THREADS) void k_morton(const BodyDesc* __restrict__ desc,
                                                         const uint4* __restrict__ tiles, PF<const float> boxes_f,
                                                         PF<const float> partial_f, PF<uint2> kv_f,
                                                         PF<uint32_t> counts_f, PF<float> root_f) {
  __shared__ float red[SORT_WAVES][6], sroot[6];
  __shared__ uint32_t h[RADIX_DIGITS];
  const uint4 t = tiles[blockIdx.x];
  const BodyDesc d = desc[t.x];
  const float* __restrict__ boxes = pick(boxes_f) + 6 * (size_t)d.t0;
  const float* __restrict__ partial = pick(partial_f) + 6 * (size_t)d.p0;
  const uint32_t m = d.m, npart = (m + BOX_BLOCK - 1) / BOX_BLOCK;
  const uint32_t tid = threadIdx.x, base = t.y * SORT_TILE;
  float bx[SORT_ROWS][6];
#pragma unroll
  for (int r = 0; r < SORT_ROWS; ++r) {
    const float* b = boxes + 6 * (size_t)min(base + r * SORT_THREADS + tid, m - 1);
#pragma unroll
    for (int c = 0; c < 6; ++c) bx[r][c] = b[c];
  }
  float mn[3], mx[3];
  box_sentinel(mn, mx);
  for (uint32_t q = tid; q < npart; q += SORT_THREADS) unite(mn, mx, partial + 6 * (size_t)q);
  h[tid] = h[tid + SORT_THREADS] = 0;
  const float v = block_box<SORT_WAVES>(mn, mx, red);
  if (tid < 6) {
    sroot[tid] = v;
    if (t.y == 0) pick(root_f)[6 * (size_t)t.x + tid] = v;
  }
  __syncthreads();
  const float rmin[3] = {sroot[0], sroot[1], sroot[2]};
  const float rext[3] = {sroot[3] - sroot[0], sroot[4] - sroot[1], sroot[5] - sroot[2]};
  // the first pass's values are the primitives themselves: codes alone,
  // packed at the body's place
  uint32_t* __restrict__ codes = reinterpret_cast<uint32_t*>(pick(kv_f) + d.t0);
#pragma unroll
  for (int r = 0; r < SORT_ROWS; ++r) {
    const uint32_t i = base + r * SORT_THREADS + tid;
    if (i >= m) continue;
    const uint32_t c = box_morton(bx[r], bx[r] + 3, rmin, rext);
    codes[i] = c;
    atomicAdd(&h[c & (RADIX_DIGITS - 1)], 1u);
  }
  __syncthreads();
  put_counts(h, pick(counts_f), t);
}

__global__ __launch_bounds__(SORT_THREADS) void k_radix_count(const BodyDesc* __restrict__ desc,
                                                              const uint4* __restrict__ tiles, PF<const uint2> kv_f,
                                                              int shift, PF<uint32_t> counts_f) {
  __shared__ uint32_t h[RADIX_DIGITS];
  const uint4 t = tiles[blockIdx.x];
  const BodyDesc d = desc[t.x];
  const uint2* __restrict__ kv = pick(kv_f) + d.t0;
  const uint32_t tid = threadIdx.x, base = t.y * SORT_TILE;
  uint32_t k[SORT_ROWS];
#pragma unroll
  for (int r = 0; r < SORT_ROWS; ++r) k[r] = kv[min(base + r * SORT_THREADS + tid, d.m - 1)].x;
  h[tid] = h[tid + SORT_THREADS] = 0;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < SORT_ROWS; ++r)
    if (base + r * SORT_THREADS + tid < d.m) atomicAdd(&h[(k[r] >> shift) & (RADIX_DIGITS - 1)], 1u);
  __syncthreads();
  put_counts(h, pick(counts_f), t);
}

// Places of the digits of every tile of a big body, without the digits' own
// bases (first), and its keys per digit (total).  A workgroup takes 64 words
// (128 digits) and cuts the tiles into eight runs, one per wave: sums of the
// runs, then their prefixes tile by tile.
constexpr uint32_t SCAN_WORDS = 64, SCAN_PARTS = SORT_WORDS / SCAN_WORDS;
__global__ __launch_bounds__(SORT_THREADS) void k_tile_scan(const uint4* __restrict__ big,
                                                            PF<const uint32_t> counts_f, PF<uint32_t> first_f,
                                                            PF<uint32_t> total_f) {
  __shared__ uint32_t sum[SORT_WAVES][2][SCAN_WORDS];
  const uint4 t = big[blockIdx.x / SCAN_PARTS];     // {body, -, tiles, first tile}
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  const uint32_t word = (blockIdx.x % SCAN_PARTS) * SCAN_WORDS + lane;
  const uint32_t* __restrict__ counts = pick(counts_f) + (size_t)t.w * SORT_WORDS + word;
  uint32_t* __restrict__ first = pick(first_f) + (size_t)t.w * RADIX_DIGITS + 2 * word;
  const uint32_t per = (t.z + SORT_WAVES - 1) / SORT_WAVES;
  const uint32_t b0 = min(w * per, t.z), b1 = min(b0 + per, t.z);
  uint32_t lo = 0, hi = 0;
#pragma unroll 8
  for (uint32_t b = b0; b < b1; ++b) {
    const uint32_t c = counts[(size_t)b * SORT_WORDS];
    lo += c & 0xffffu;
    hi += c >> 16;
  }
  sum[w][0][lane] = lo;
  sum[w][1][lane] = hi;
  __syncthreads();
  uint32_t f0 = 0, f1 = 0;
  for (uint32_t q = 0; q < w; ++q) {
    f0 += sum[q][0][lane];
    f1 += sum[q][1][lane];
  }
  if (w == SORT_WAVES - 1) {
    uint32_t* total = pick(total_f) + (size_t)(blockIdx.x / SCAN_PARTS) * RADIX_DIGITS + 2 * word;
    total[0] = f0 + lo;
    total[1] = f1 + hi;
  }
#pragma unroll 8
  for (uint32_t b = b0; b < b1; ++b) {
    const uint32_t c = counts[(size_t)b * SORT_WORDS];
    *reinterpret_cast<uint2*>(first + (size_t)b * RADIX_DIGITS) = make_uint2(f0, f1);
    f0 += c & 0xffffu;
    f1 += c >> 16;
  }
}

// Scatter with stable ranks.  Wave w owns SORT_ROWS rows of 64 consecutive
// keys; within a row the lanes of a digit are matched with RADIX_BITS
// ballots, and a running per-digit count of the wave's rows is kept in LDS,
// so a tile takes four barriers.  Element order = (wave, row, lane) order.
// FIRST: the values are the primitives themselves.  LAST: the sorted keys are
// written instead of the pairs, and the leaf triangles where the level build
// does not write them (there in leaf order; here they are scattered: 74 us of
// the last pass of 4.2 M keys against 38 without them).
template <bool FIRST, bool LAST>
__global__ __launch_bounds__(SORT_THREADS) void k_radix_scatter(const BodyDesc* __restrict__ desc,
                                                                const uint4* __restrict__ tiles,
                                                                PF<const uint2> in_f, int shift,
                                                                PF<const uint32_t> counts_f,
                                                                PF<const uint32_t> first_f,
                                                                PF<const uint32_t> total_f, PF<uint2> out_f,
                                                                const uint32_t* __restrict__ tris,
                                                                PF<uint64_t> keys_f, PF<uint4> leaf_tri_f) {
  __shared__ __align__(16) uint32_t wcnt[SORT_WAVES][RADIX_DIGITS];
  __shared__ uint32_t wsum[SORT_WAVES];
  const uint4 t = tiles[blockIdx.x];
  const BodyDesc d = desc[t.x];
  const uint32_t n = d.m;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
  const uint32_t base = t.y * SORT_TILE;
  const uint2* __restrict__ in = pick(in_f) + d.t0;
  uint32_t key[SORT_ROWS], val[SORT_ROWS], loc[SORT_ROWS];
  bool ok[SORT_ROWS];
#pragma unroll
  for (int r = 0; r < SORT_ROWS; ++r) {
    const uint32_t e = base + (w * SORT_ROWS + r) * 64 + lane;
    ok[r] = e < n;
    if constexpr (FIRST) {
      key[r] = reinterpret_cast<const uint32_t*>(in)[min(e, n - 1)];
      val[r] = e;
    } else {
      const uint2 kv = in[min(e, n - 1)];
      key[r] = kv.x;
      val[r] = kv.y;
    }
  }

  // the tile's first place of each of the thread's digits 2 tid, 2 tid + 1
  uint32_t tot[2], first[2];
  if (t.z <= SORT_SUM_TILES) {
    uint4* part = reinterpret_cast<uint4*>(&wcnt[0][0]);      // [2][SORT_GROUPS][SORT_WORDS] words
    const uint32_t g = tid / (SORT_WORDS / 4), q = tid % (SORT_WORDS / 4);
    const uint4* h4 = reinterpret_cast<const uint4*>(pick(counts_f) + (size_t)t.w * SORT_WORDS) + q;
    uint4 all = make_uint4(0, 0, 0, 0), pre = make_uint4(0, 0, 0, 0);   // sums of 16-bit pairs
    for (uint32_t b0 = g; b0 < t.z; b0 += SORT_LOADS * SORT_GROUPS) {
      uint4 c[SORT_LOADS];
#pragma unroll
      for (uint32_t j = 0; j < SORT_LOADS; ++j)
        c[j] = h4[(size_t)min(b0 + j * SORT_GROUPS, t.z - 1) * (SORT_WORDS / 4)];
#pragma unroll
      for (uint32_t j = 0; j < SORT_LOADS; ++j) {
        const uint32_t b = b0 + j * SORT_GROUPS;
        const uint32_t is = b < t.z ? ~0u : 0u, be = b < t.y ? ~0u : 0u;
        all.x += c[j].x & is; all.y += c[j].y & is; all.z += c[j].z & is; all.w += c[j].w & is;
        pre.x += c[j].x & be; pre.y += c[j].y & be; pre.z += c[j].z & be; pre.w += c[j].w & be;
      }
    }
    part[g * (SORT_WORDS / 4) + q] = all;
    part[(SORT_GROUPS + g) * (SORT_WORDS / 4) + q] = pre;
    __syncthreads();
    const uint32_t* pw = &wcnt[0][0] + tid;
    tot[0] = tot[1] = first[0] = first[1] = 0;
#pragma unroll
    for (uint32_t k = 0; k < SORT_GROUPS; ++k) {
      const uint32_t a = pw[k * SORT_WORDS], p = pw[(SORT_GROUPS + k) * SORT_WORDS];
      tot[0] += a & 0xffffu; tot[1] += a >> 16;
      first[0] += p & 0xffffu; first[1] += p >> 16;
    }
  } else {
    const uint32_t bigno = t.z - TILES_BIG;
    const uint2 t2 = reinterpret_cast<const uint2*>(pick(total_f) + (size_t)bigno * RADIX_DIGITS)[tid];
    const uint2 f2 = reinterpret_cast<const uint2*>(pick(first_f) + (size_t)(t.w + t.y) * RADIX_DIGITS)[tid];
    tot[0] = t2.x; tot[1] = t2.y;
    first[0] = f2.x; first[1] = f2.y;
  }
  {
    const uint32_t v = tot[0] + tot[1];
    uint32_t incl = v;
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t u = __shfl_up(incl, off, 64);
      if (lane >= (uint32_t)off) incl += u;
    }
    if (lane == 63) wsum[w] = incl;
    __syncthreads();                       // also: the parts have been read
    uint32_t s = incl - v;
    for (uint32_t q = 0; q < w; ++q) s += wsum[q];
    first[0] += s;
    first[1] += s + tot[0];
  }
  for (uint32_t q = lane; q < (uint32_t)RADIX_DIGITS / 4; q += 64)
    reinterpret_cast<uint4*>(wcnt[w])[q] = make_uint4(0, 0, 0, 0);
  wave_order_lds();

  const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
#pragma unroll
  for (int r = 0; r < SORT_ROWS; ++r) {
    const uint32_t dg = (key[r] >> shift) & (RADIX_DIGITS - 1);
    uint64_t msk = __ballot(ok[r]);
#pragma unroll
    for (int b = 0; b < RADIX_BITS; ++b) {
      const bool on = (dg >> b) & 1u;
      const uint64_t bb = __ballot(on);
      msk &= on ? bb : ~bb;
    }
    // the wave's count of this digit in its earlier rows, then this row's
    // lanes of the digit; the lowest such lane adds the row's count
    const uint32_t prior = wcnt[w][dg], rank = __popcll(msk & lt);
    loc[r] = prior + rank;
    if (ok[r] && rank == 0) wcnt[w][dg] = prior + (uint32_t)__popcll(msk);
    wave_order_lds();
  }
  __syncthreads();
#pragma unroll
  for (int v = 0; v < SORT_WAVES; ++v) {   // per digit: offsets of the waves' runs
    uint2& p = reinterpret_cast<uint2*>(wcnt[v])[tid];
    const uint2 c = p;
    p = make_uint2(first[0], first[1]);
    first[0] += c.x;
    first[1] += c.y;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < SORT_ROWS; ++r) {
    const uint32_t pos = wcnt[w][(key[r] >> shift) & (RADIX_DIGITS - 1)] + loc[r];
    if (!ok[r] || pos >= n) continue;      // pos < n always; the test keeps stores in the body
    if constexpr (LAST) {
      pick(keys_f)[(size_t)d.t0 + pos] = ((uint64_t)key[r] << 32) | val[r];
      if (uint4* leaf = pick(leaf_tri_f)) {
        const uint32_t* tr = tris + 3 * ((size_t)d.t0 + min(val[r], n - 1));
        leaf[(size_t)d.t0 + pos] = make_uint4(tr[0], tr[1], tr[2], val[r]);
      }
    } else {
      pick(out_f)[(size_t)d.t0 + pos] = make_uint2(key[r], val[r]);
    }
  }
}

// ------------------------------------------------------------ host side
void SortTable::init(const std::vector<BodyDesc>& h, const std::vector<uint32_t>& bodies, hipStream_t s,
                     const std::function<void(std::vector<uint4>&)>& arrange) {
  std::vector<uint4> t, g;
  uint32_t at = 0;
  for (uint32_t j : bodies) {
    const uint32_t k = sort_tiles(h[j].m);
    const bool is_big = k > SORT_SUM_TILES;
    const uint32_t z = is_big ? TILES_BIG + (uint32_t)g.size() : k;
    for (uint32_t q = 0; q < k; ++q) t.push_back(make_uint4(j, q, z, at));
    if (is_big) g.push_back(make_uint4(j, 0u, k, at));
    at += k;
  }
  if (arrange) arrange(t);
  ntiles = (uint32_t)t.size();
  nbig = (uint32_t)g.size();
  if (ntiles) tiles.upload(t.data(), t.size(), s);
  if (nbig) big.upload(g.data(), g.size(), s);
}

void SortScratch::alloc(size_t tiles, size_t nbig) {
  counts.alloc(tiles * SORT_WORDS);
  first.alloc(nbig ? tiles * RADIX_DIGITS : 0);
  total.alloc(nbig * RADIX_DIGITS);
}

void launch_sort(const BodyDesc* desc, const SortTable& t, const uint32_t* tris, const SortFrame* frames, int nframes,
                 hipStream_t s) {
  CC_REQUIRE(nframes >= 1 && nframes <= MAX_FRAMES, "sort: frame count");
  if (!t.ntiles) return;
  PF<const float> boxes{}, partial{};
  PF<uint2> kv[2] = {};
  PF<const uint2> kv_c[2] = {};
  PF<uint32_t> counts{}, first{}, total{};
  PF<const uint32_t> counts_c{}, first_c{}, total_c{};
  PF<uint64_t> keys{};
  PF<uint4> leaf{};
  PF<float> root{};
  for (int f = 0; f < nframes; ++f) {
    const SortFrame& F = frames[f];
    boxes.p[f] = F.boxes;
    partial.p[f] = F.partial;
    for (int b = 0; b < 2; ++b) {
      kv[b].p[f] = F.kv[b];
      kv_c[b].p[f] = F.kv[b];
    }
    counts.p[f] = F.sort->counts.p;
    counts_c.p[f] = F.sort->counts.p;
    first.p[f] = F.sort->first.p;
    first_c.p[f] = F.sort->first.p;
    total.p[f] = F.sort->total.p;
    total_c.p[f] = F.sort->total.p;
    keys.p[f] = F.keys;
    leaf.p[f] = F.leaf_tri;
    root.p[f] = F.root;
  }
  const unsigned nf = (unsigned)nframes;
  const dim3 grid(t.ntiles, nf);
  k_morton<<<grid, SORT_THREADS, 0, s>>>(desc, t.tiles.p, boxes, partial, kv[0], counts, root);
  CC_LAUNCHED();
  for (int pass = 0, shift = 0; pass < RADIX_PASSES; ++pass, shift += RADIX_BITS) {
    const int src = pass & 1, dst = src ^ 1;
    if (pass) k_radix_count<<<grid, SORT_THREADS, 0, s>>>(desc, t.tiles.p, kv_c[src], shift, counts);
    if (t.nbig) k_tile_scan<<<dim3(t.nbig * SCAN_PARTS, nf), SORT_THREADS, 0, s>>>(t.big.p, counts_c, first, total);
    auto scatter = pass == 0 ? k_radix_scatter<true, false>
                   : pass + 1 < RADIX_PASSES ? k_radix_scatter<false, false> : k_radix_scatter<false, true>;
    scatter<<<grid, SORT_THREADS, 0, s>>>(desc, t.tiles.p, kv_c[src], shift, counts_c, first_c, total_c, kv[dst], tris,
                                          keys, leaf);
    CC_LAUNCHED();
  }
}

}  // namespace cc
