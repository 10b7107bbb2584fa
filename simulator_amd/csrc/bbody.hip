// bbody.hip -- the bodies of a batch, posed and rebuilt together.
//
// Per frame, for all bodies at once:
//   k_bb_deform  grid over body vertices      capsule breathing + rigid motion
//   k_bb_boxes   grid over triangles          expanded boxes + per-block root boxes
//   launch_sort  tiles of 1024 keys           root box, Morton codes, sort (sort.hip)
//   k_bb_level   chunks of 1024 leaves, then  tree and boxes by splits, in LDS
//                of unfinished nodes
// and for refitted bodies, after the pose:
//   launch_refit_levels                       boxes by levels (refit.hip)
// Poses, keys, topology and boxes equal the single-body path bit for bit:
// the arithmetic is the shared routines of cc_lbvh.h, the sort is stable
// from ascending primitive order (so it orders the full 64-bit key), and
// box unions are exact.
#include <algorithm>
#include <cstring>
#include <numeric>

#include "cc_bbody.h"
#include "cc_lbvh.h"

namespace cc {

constexpr int BB_BLOCK = 256;       // vertices / triangles / nodes per block of the grid kernels
constexpr uint32_t BB_MAX_M = 1u << 19;   // triangles per batched body
static_assert(BB_BLOCK == BOX_BLOCK, "one partial root box per BOX_BLOCK triangles");

// ------------------------------------------------------------ pose
__global__ __launch_bounds__(BB_BLOCK) void k_bb_deform(const BodyDesc* __restrict__ desc,
                                                        const uint4* __restrict__ blk,
                                                        const float* __restrict__ rest, float* __restrict__ verts,
                                                        const uint32_t* __restrict__ capv,
                                                        const float* __restrict__ capp0,
                                                        const float* __restrict__ capp1,
                                                        const float* __restrict__ motion, uint32_t nb, int k) {
  __shared__ float sP0[3 * MAX_CAPS], sP1[3 * MAX_CAPS], sM[BB_MF];
  __shared__ uint32_t sV[MAX_CAPS + 1];
  const uint4 b = blk[blockIdx.x];    // {body, first vertex, count, -}
  const BodyDesc d = desc[b.x];
  const uint32_t tid = threadIdx.x;
  for (uint32_t q = tid; q < 3 * d.ncaps; q += BB_BLOCK) {
    sP0[q] = capp0[3 * (size_t)d.c0 + q];
    sP1[q] = capp1[3 * (size_t)d.c0 + q];
  }
  for (uint32_t q = tid; q <= d.ncaps; q += BB_BLOCK) sV[q] = capv[d.cv0 + q];
  const float* mf = motion + ((size_t)k * nb + b.x) * BB_MF;
  for (uint32_t q = tid; q < 12 + d.ncaps; q += BB_BLOCK) sM[q] = mf[q];
  __syncthreads();
  if (tid >= b.z) return;
  const uint32_t v = b.y + tid;
  const uint32_t c = capsule_of(sV, d.ncaps, v);
  const size_t g = (size_t)d.v0 + v;
  deform_point(ld3(rest + 3 * g), ld3(sP0 + 3 * c), ld3(sP1 + 3 * c), sM[12 + c], sM, sM + 9, verts + 3 * g);
}

// ------------------------------------------------------------ boxes
__global__ __launch_bounds__(BB_BLOCK) void k_bb_boxes(const BodyDesc* __restrict__ desc,
                                                       const uint4* __restrict__ blk,
                                                       const float* __restrict__ verts,
                                                       const uint32_t* __restrict__ tris, float* __restrict__ boxes,
                                                       float* __restrict__ partial) {
  __shared__ float red[BB_BLOCK / 64][6];
  const uint4 b = blk[blockIdx.x];    // {body, first triangle, count, partial index}
  const BodyDesc d = desc[b.x];
  const uint32_t tid = threadIdx.x;
  float mn[3], mx[3];
  box_sentinel(mn, mx);
  if (tid < b.z) {
    const size_t i = (size_t)d.t0 + b.y + tid;
    const uint32_t* t = tris + 3 * i;
    const float* V = verts + 3 * (size_t)d.v0;
    prim_box(ld3(V + 3 * (size_t)t[0]), ld3(V + 3 * (size_t)t[1]), ld3(V + 3 * (size_t)t[2]), d.depth, mn, mx);
    put6(boxes + 6 * i, mn, mx);
  }
  const float v = block_box<BB_BLOCK / 64>(mn, mx, red);
  if (tid < 6) partial[6 * (size_t)b.w + tid] = v;
}

// ------------------------------------------------------------ tree + boxes
// The Karras tree (processInternalNode, cudaBRT.cu:9-161) with its boxes
// (calculateBoudingBox, cudaBRT.cu:166-206), by splits.  Every boundary between
// adjacent sorted leaves i, i + 1 is the split of exactly one internal node:
// the leaves that share the first delta(i, i + 1) bits of their keys, a range
// [l, r] found by two binary searches.  All else follows from the range: the
// children are [l, i] and [i + 1, r], their Karras indices i and i + 1 (a left
// child's index is its last leaf, a right child's its first, the root's 0),
// and the node's own side is where its boundary pair shares the longer
// prefix (delta(r, r+1) > delta(l-1, l): it is a left child; with unique keys
// the two never tie).
//
// A workgroup takes up to LV_C adjacent "items" (leaves at level 0, else the
// nodes its input chunks could not finish) into LDS and builds every node
// whose range lies inside them.  A node or item whose parent is not built
// inside the chunk is passed to the next level (at most 2 x 63 per chunk: the
// children of the nodes crossing the chunk's two boundaries), LV_G chunks of
// it per workgroup, until one chunk holds the whole body.  The items of a
// chunk partition its leaf range in order, and a node's range never cuts an
// item, so one key per item decides whether it belongs to a range.
constexpr int LV_CAP = 128;
constexpr int LV_G = LV_C / LV_CAP;
// One level of the build: one thread per item, and per split between two
// items.  Boxes of ranges are unions of two overlapping power-of-two runs: in
// round q the workgroup holds the box of every run of 2^q items in LDS (each
// thread doubles its own run from a neighbour's), and the nodes whose
// children's lengths lie in [2^q, 2^(q+1)) read theirs.  Ten rounds of one
// LDS read and a barrier for 1024 items, every lane at work, where climbing
// from the leaves node by node took up to twenty dependent steps of an LDS
// atomic and a read with fewer lanes at each.  Bound by latency for one body
// (the loads, the searches, the barriers) and by the vector instructions at
// level 0 of a batch, hence the rounds written out and the searches on byte
// offsets.  Three frames of 50,688 triangles: 16.4 us at level 0 and
// 9.6 at each of the two above, against 22.8 and 19.0 climbing; the 4.2 M
// triangles of 256 bodies: 159 us at level 0 against 199 (3.3 TB/s of keys,
// gathered boxes and triangles, leaves and nodes written).
template <bool LEAVES>
__global__ __launch_bounds__(LV_C) void k_bb_level(const LvBlock* __restrict__ blk, PF<const uint64_t> keys_f,
                                                   const uint32_t* __restrict__ tris, PF<const float> boxes_f,
                                                   PF<uint4> leaf_f, PF<const BItem> items_in_f,
                                                   PF<const uint32_t> cnt_in_f, PF<BItem> items_out_f,
                                                   PF<uint32_t> cnt_out_f, PF<Node> nodes_f, PF<float> root_f,
                                                   PF<float> leaf0_f) {
  __shared__ uint64_t sK[LV_C + 2];      // [1 + k] a key of item k; no key on either side
  __shared__ float2 U[2][LV_C][3];       // boxes of the runs of 2^q items from item k
  __shared__ int32_t sD[LV_C];           // delta at the boundary right of item k
  __shared__ int32_t sR[LV_C];           // last leaf of item k
  __shared__ uint8_t built[LV_C];        // the node of the split right of item k lies in the chunk
  __shared__ BItem pend[LV_CAP];
  __shared__ uint32_t npend;
  __shared__ int32_t qmax, sfirst, sdl;  // rounds needed; first leaf, and the delta left of it
  const LvBlock b = blk[blockIdx.x];
  const uint32_t tid = threadIdx.x;
  Node* N = pick(nodes_f) + b.n0;
  float* R = pick(root_f) + 6 * (size_t)b.body;
  const float* box_src = nullptr;        // this thread's item's box
  int32_t n, k, gl = 0, gr = 0, dl = -1, dr = -1;
  uint64_t key = 0;
  Box6 run{};
  bool have;
  if constexpr (LEAVES) {
    const int32_t m = (int32_t)b.n_in, c0 = (int32_t)b.q * LV_C;
    n = min(LV_C, m - c0);
    k = (int32_t)tid;
    have = k < n;
    gl = gr = min(c0 + k, m - 1);
    const uint64_t* K = pick(keys_f) + b.t0;
    const uint64_t ka = K[max(gl - 1, 0)], kc = K[min(gl + 1, m - 1)];
    key = K[gl];
    const size_t prim = (size_t)b.t0 + (uint32_t)key;   // the key's low half is its primitive
    box_src = pick(boxes_f) + 6 * prim;
    for (int c = 0; c < 6; ++c) run.v[c] = box_src[c];
    if (b.write_leaves) {
      const uint32_t* t = tris + 3 * prim;
      if (have) pick(leaf_f)[(size_t)b.t0 + gl] = make_uint4(t[0], t[1], t[2], (uint32_t)key);
    }
    dl = gl > 0 ? __clzll(ka ^ key) : -1;
    dr = gl + 1 < m ? __clzll(key ^ kc) : -1;
    if (m == 1) {                          // a single leaf: no internal node
      if (tid == 0) {
        const Box6 r = box_node(run);
        put6(pick(leaf0_f) + 6 * (size_t)b.body, run.v, run.v + 3);
        put6(R, r.v, r.v + 3);
      }
      return;
    }
  } else {
    // counts of the LV_G input chunks (every lane needs them all) and the
    // item at this thread's place, loaded together
    const uint32_t g = tid / LV_CAP, at = tid % LV_CAP, slot0 = b.q * LV_G;
    const uint32_t* cnt = pick(cnt_in_f) + b.in_base;
    uint32_t c[LV_G];
#pragma unroll
    for (int j = 0; j < LV_G; ++j) c[j] = cnt[min(slot0 + j, b.n_in - 1)];
    const BItem* src = pick(items_in_f) + ((size_t)b.in_base + min(slot0 + g, b.n_in - 1)) * LV_CAP + at;
    const BItem it = *src;
    uint32_t acc = 0, before = 0, mine = 0;
#pragma unroll
    for (int j = 0; j < LV_G; ++j) {
      const uint32_t cj = slot0 + j < b.n_in ? min(c[j], (uint32_t)LV_CAP) : 0u;
      before = (uint32_t)j == g ? acc : before;
      mine = (uint32_t)j == g ? cj : mine;
      acc += cj;
    }
    n = (int32_t)acc;
    k = (int32_t)(before + at);
    have = at < mine;
    gl = it.l;
    gr = it.r;
    dl = it.dl;
    dr = it.dr;
    key = it.key;
    box_src = src->box;
    for (int q = 0; q < 6; ++q) run.v[q] = it.box[q];
  }
  if (tid == 0) {
    npend = 0;
    qmax = -1;
    sK[0] = sK[n + 1] = ~0ull;             // differs from every key (30-bit codes) in the top bit
  }
  if (have) {
    sK[1 + k] = key;
    sD[k] = dr;
    if (!LEAVES) sR[k] = gr;
    lds_box_put(U[0], k, run);
    if (k == 0) {
      sfirst = gl;
      sdl = dl;
    }
  }
  __syncthreads();

  // the range [l, r] of the split right of this item: the keys that differ
  // from this one in the bits of `rest` only
  int32_t l = k, r = k, ndl = 0, ndr = 0;
  bool node = false;
  if (have && k < n - 1) {
    const uint64_t rest = ~0ull >> dr;
    const char* K8 = reinterpret_cast<const char*>(sK);
    int32_t a = 8 * (1 + k), z = a + 8;    // byte offsets of l's and r's keys
    const int32_t last = 8 * (n + 1);
#pragma unroll
    for (int32_t step = 4 * LV_C; step >= 8; step >>= 1) {
      const int32_t na = max(a - step, 0), nz = min(z + step, last);
      const uint64_t xa = *reinterpret_cast<const uint64_t*>(K8 + na) ^ key;
      const uint64_t xz = *reinterpret_cast<const uint64_t*>(K8 + nz) ^ key;
      a = xa <= rest ? na : a;
      z = xz <= rest ? nz : z;
    }
    l = a / 8 - 1;
    r = z / 8 - 1;
    ndl = l > 0 ? sD[l - 1] : sdl;
    ndr = sD[r];
    node = ndl < dr && ndr < dr;
  }
  const int32_t qa = node ? 31 - __clz(k - l + 1) : -1, qb = node ? 31 - __clz(r - k) : -1;
  if (have) built[k] = node ? 1 : 0;
  {
    int32_t q = max(qa, qb);
    for (int off = 32; off > 0; off >>= 1) q = max(q, __shfl_xor(q, off, 64));
    if ((tid & 63u) == 0 && q >= 0) atomicMax(&qmax, q);
  }
  __syncthreads();
  Box6 A{}, B{};
  const int32_t rounds = qmax;
#define CC_ROUND(Q) \
  if (rounds >= Q) level_round<Q>(U[Q & 1], U[(Q & 1) ^ 1], have, k, n, l, r, qa, qb, rounds > Q, run, A, B)
  CC_ROUND(0); CC_ROUND(1); CC_ROUND(2); CC_ROUND(3); CC_ROUND(4);
  CC_ROUND(5); CC_ROUND(6); CC_ROUND(7); CC_ROUND(8); CC_ROUND(9);
#undef CC_ROUND
  // the node's links and boxes
  auto pend_put = [&](int32_t pl, int32_t pr, int32_t idx, int32_t pdl, int32_t pdr, uint64_t pkey, const float* bx) {
    BItem& o = pend[min(atomicAdd(&npend, 1u), (uint32_t)LV_CAP - 1)];
    o.l = pl;
    o.r = pr;
    o.idx = idx;
    o.dl = pdl;
    o.dr = pdr;
    o.key = pkey;
    for (int c = 0; c < 6; ++c) o.box[c] = bx[c];
  };
  if (node) {
    const int32_t s = gr, first = LEAVES ? sfirst + l : (l > 0 ? sR[l - 1] + 1 : sfirst);
    const int32_t last = LEAVES ? sfirst + r : sR[r];
    if (first < s) A = box_node(A);
    if (s + 1 < last) B = box_node(B);
    const bool root = (ndl & ndr) < 0, left = ndr > ndl;   // both deltas -1: [0, m)
    const int32_t me = root ? 0 : (left ? last : first);
    float4* o = reinterpret_cast<float4*>(N + me);
    o[0] = make_float4(A.v[0], A.v[1], A.v[2], A.v[3]);
    o[1] = make_float4(A.v[4], A.v[5], B.v[0], B.v[1]);
    o[2] = make_float4(B.v[2], B.v[3], B.v[4], B.v[5]);
    // no parent (the export derives the parents); the end of its range that
    // is not its index
    reinterpret_cast<int4*>(o)[3] = make_int4(first < s ? s : ~s, s + 1 < last ? s + 1 : ~(s + 1), -1,
                                              root || !left ? last : first);
    const int32_t p = left ? r : l - 1;    // the parent's split
    if (root || p < 0 || p >= n - 1 || !built[p]) {
      const Box6 box = box_node(box_or(A, B));
      if (root)
        put6(R, box.v, box.v + 3);
      else
        pend_put(first, last, me, ndl, ndr, sK[1 + l], box.v);
    }
  }
  // the item itself, when its parent is not built here
  if (have) {
    const int32_t p = dr > dl ? k : k - 1;
    if (p < 0 || p >= n - 1 || !built[p])
      pend_put(gl, gr, gl == gr ? ~gl : (dr > dl ? gr : gl), dl, dr, key, box_src);
  }
  __syncthreads();
  // the unfinished nodes, in leaf order, to this chunk's output slot
  BItem* __restrict__ items_out = pick(items_out_f);
  const uint32_t np = min(npend, (uint32_t)LV_CAP);
  if (tid < np) {
    const int32_t at = pend[tid].l;
    uint32_t rank = 0;
    for (uint32_t q = 0; q < np; ++q) rank += pend[q].l < at;
    items_out[((size_t)b.out_base + b.q) * LV_CAP + rank] = pend[tid];
  }
  if (tid == 0) pick(cnt_out_f)[b.out_base + b.q] = np;
}

// ------------------------------------------------------------ host side
size_t level_chunks0(uint32_t m) { return (m + LV_C - 1) / LV_C; }

std::vector<std::vector<LvBlock>> build_level_tables(const std::vector<BodyDesc>& h,
                                                     const std::vector<uint32_t>& bodies,
                                                     const std::function<bool(uint32_t)>& write_leaves) {
  // level 0 over the leaves, level L+1 over LV_G chunks of level L, until a
  // body's level has a single chunk; slot bases are per level, in list order
  std::vector<std::vector<LvBlock>> out;
  std::vector<uint32_t> chunks(h.size(), 0), prev_base(h.size(), 0), prev_n(h.size(), 0);
  for (uint32_t j : bodies) chunks[j] = (uint32_t)level_chunks0(h[j].m);
  for (int L = 0; L < BB_MAX_LEVELS; ++L) {
    std::vector<LvBlock> t;
    uint32_t base = 0;
    std::vector<uint32_t> next(h.size(), 0), base_of(h.size(), 0);
    for (uint32_t j : bodies) {
      if (chunks[j] == 0) continue;
      base_of[j] = base;
      for (uint32_t q = 0; q < chunks[j]; ++q) {
        LvBlock e{};
        e.body = j;
        e.q = q;
        e.in_base = prev_base[j];
        e.out_base = base;
        e.n_in = L == 0 ? h[j].m : prev_n[j];
        e.t0 = h[j].t0;
        e.n0 = h[j].n0;
        e.write_leaves = write_leaves(j) ? 1 : 0;
        t.push_back(e);
      }
      base += chunks[j];
      next[j] = chunks[j] > 1 ? (chunks[j] + LV_G - 1) / LV_G : 0;
    }
    if (t.empty()) break;
    out.push_back(std::move(t));
    prev_base = base_of;
    prev_n = chunks;
    chunks = next;
  }
  for (uint32_t j : bodies) CC_REQUIRE(chunks[j] == 0, "bottom-up build: too many levels");
  return out;
}

void launch_build_levels(const LvBlock* const* level, const uint32_t* n_level,
                         const LvFrame* frames, int nframes, hipStream_t s) {
  CC_REQUIRE(nframes >= 1 && nframes <= MAX_FRAMES, "level build: frame count");
  PF<const uint64_t> keys{};
  PF<const float> boxes{};
  PF<uint4> leaf{};
  PF<BItem> items[2] = {};
  PF<const BItem> items_c[2] = {};
  PF<uint32_t> nitems[2] = {};
  PF<const uint32_t> nitems_c[2] = {};
  PF<Node> nodes{};
  PF<float> root{}, leaf0{};
  for (int f = 0; f < nframes; ++f) {
    const LvFrame& F = frames[f];
    keys.p[f] = F.keys;
    boxes.p[f] = F.boxes;
    leaf.p[f] = F.leaf_tri;
    for (int q = 0; q < 2; ++q) {
      items[q].p[f] = F.items[q];
      items_c[q].p[f] = F.items[q];
      nitems[q].p[f] = F.nitems[q];
      nitems_c[q].p[f] = F.nitems[q];
    }
    nodes.p[f] = F.nodes;
    root.p[f] = F.root;
    leaf0.p[f] = F.leaf0;
  }
  for (int L = 0; L < BB_MAX_LEVELS; ++L) {
    if (!n_level[L]) continue;
    const int in = (L + 1) & 1, out = L == 0 ? 0 : (L & 1);
    const dim3 grid(n_level[L], (unsigned)nframes);
    if (L == 0)
      k_bb_level<true><<<grid, LV_C, 0, s>>>(level[L], keys, frames[0].tris, boxes, leaf, items_c[in], nitems_c[in],
                                              items[out], nitems[out], nodes, root, leaf0);
    else
      k_bb_level<false><<<grid, LV_C, 0, s>>>(level[L], keys, frames[0].tris, boxes, leaf, items_c[in], nitems_c[in],
                                               items[out], nitems[out], nodes, root, leaf0);
    CC_LAUNCHED();
  }
}

BatchBodies::~BatchBodies() {
  for (int q = 0; q < 2; ++q) {
    if (ev_motion[q]) {
      (void)hipEventSynchronize(ev_motion[q]);
      (void)hipEventDestroy(ev_motion[q]);
    }
    if (h_motion[q]) (void)hipHostFree(h_motion[q]);
  }
}

namespace {

void append_blocks(std::vector<uint4>& t, uint32_t body, uint32_t count, uint32_t aux0, bool aux) {
  for (uint32_t f = 0, q = 0; f < count; f += BB_BLOCK, ++q)
    t.push_back(make_uint4(body, f, std::min<uint32_t>(BB_BLOCK, count - f), aux ? aux0 + q : 0u));
}

void upload_list(DBuf<uint4>& d, uint32_t& n, const std::vector<uint4>& h, hipStream_t s) {
  n = (uint32_t)h.size();
  d.upload(h.data(), std::max<size_t>(h.size(), 1), s);
  if (h.empty()) d.zero(s);
}

}  // namespace

void XcdMap::init(const std::vector<double>& a, const std::vector<double>& b) {
  double sa = 0.0, sb = 0.0;
  for (double v : a) sa += v;
  for (double v : b) sb += v;
  auto part = [&](size_t k) { return (sa > 0 ? a[k] / sa : 0.0) + (sb > 0 ? b[k] / sb : 0.0); };
  std::vector<uint32_t> order(a.size());
  std::iota(order.begin(), order.end(), 0u);
  std::stable_sort(order.begin(), order.end(), [&](uint32_t x, uint32_t y) { return part(x) > part(y); });
  double la[XCDS] = {}, lb[XCDS] = {};
  of.assign(a.size(), 0);
  for (uint32_t k : order) {
    size_t best = 0;
    double least = 1e300;
    for (size_t x = 0; x < XCDS; ++x) {
      const double w = std::max(sa > 0 ? (la[x] + a[k]) / sa : 0.0, sb > 0 ? (lb[x] + b[k]) / sb : 0.0);
      if (w < least) {
        least = w;
        best = x;
      }
    }
    la[best] += a[k];
    lb[best] += b[k];
    of[k] = (uint8_t)best;
  }
  const double ma = *std::max_element(la, la + XCDS), mb = *std::max_element(lb, lb + XCDS);
  if (ma * XCDS > 1.1 * sa || mb * XCDS > 1.1 * sb) of.clear();
}

void BatchBodies::init(const cc_body_desc* bodies, const cc_params* params, const std::vector<uint32_t>& cloth_n,
                       uint32_t count, hipStream_t s) {
  std::vector<float> h_rest, h_p0, h_p1;
  std::vector<uint32_t> h_tris, h_capv;
  uint32_t nv_sum = 0, m_sum = 0, n_sum = 0, c_sum = 0, cv_sum = 0, p_sum = 0;
  for (uint32_t k = 0; k < count; ++k) {
    const cc_body_desc* bd = bodies ? &bodies[k] : nullptr;
    if (!bd || bd->mode == CC_BODY_NONE) continue;
    CC_REQUIRE(bd->mode <= CC_BODY_REBUILD, "batch body: unknown mode");
    CC_REQUIRE(bd->verts && bd->tris && (bd->stride == 3 || bd->stride == 4) && bd->nv > 0 && bd->nf > 0,
               "batch body: vertices and triangles required");
    CC_REQUIRE(bd->nf <= BB_MAX_M, "batch body: at most 524288 triangles per body");
    for (size_t i = 0; i < 3 * (size_t)bd->nf; ++i)
      CC_REQUIRE(bd->tris[i] < bd->nv, "batch body: triangle index out of range");
    std::vector<float> bv;
    read_vec3_from(bd->verts, bd->stride, bd->nv, bv);
    if (bd->extend) {
      CC_REQUIRE(bd->normals3, "batch body: normals required for extend");
      int rc = cc_mesh_vertex_extend(bv.data(), 3, bd->nv, bd->tris, bd->nf, nullptr, bd->normals3,
                                     params[k].body_extend);
      if (rc) throw Error(rc, cc_last_error());
    }
    BodyDesc d{};
    d.nv = bd->nv;
    d.m = bd->nf;
    d.mode = bd->mode;
    d.depth = params[k].box_depth;
    d.v0 = nv_sum;
    d.t0 = m_sum;
    d.n0 = n_sum;
    d.c0 = c_sum;
    d.cv0 = cv_sum;
    d.p0 = p_sum;
    MotionParams mpk;
    std::vector<float> ph;
    if (bd->mode != CC_BODY_STATIC) {
      const cc_capsules* caps = bd->caps;
      CC_REQUIRE(caps && caps->ncaps >= 1 && caps->ncaps <= MAX_CAPS, "batch body: capsule layout required (1..64)");
      CC_REQUIRE(caps->vstart[0] == 0 && caps->vstart[caps->ncaps] == bd->nv,
                 "batch body: capsule ranges must cover vertices");
      for (uint32_t q = 0; q < caps->ncaps; ++q)
        CC_REQUIRE(caps->vstart[q] <= caps->vstart[q + 1], "batch body: capsule ranges must be ascending");
      d.ncaps = caps->ncaps;
      h_capv.insert(h_capv.end(), caps->vstart, caps->vstart + caps->ncaps + 1);
      h_p0.insert(h_p0.end(), caps->p0, caps->p0 + 3 * caps->ncaps);
      h_p1.insert(h_p1.end(), caps->p1, caps->p1 + 3 * caps->ncaps);
      ph.assign(caps->phase, caps->phase + caps->ncaps);
      mpk.amp = bd->amp;
      mpk.freq = bd->freq;
      mpk.rot_amp = bd->rot_amp;
      mpk.breath_amp = bd->breath_amp;
      mpk.breath_freq = bd->breath_freq;
      mpk.dx = bd->dir[0];
      mpk.dy = bd->dir[1];
      mpk.dz = bd->dir[2];
      mpk.px = bd->pivot[0];
      mpk.py = bd->pivot[1];
      mpk.pz = bd->pivot[2];
      mpk.dt = (double)params[k].dt;
      mpk.ncaps = d.ncaps;
      moving = true;
      c_sum += d.ncaps;
      cv_sum += d.ncaps + 1;
    }
    h_rest.insert(h_rest.end(), bv.begin(), bv.end());
    h_tris.insert(h_tris.end(), bd->tris, bd->tris + 3 * (size_t)bd->nf);
    CC_REQUIRE((uint64_t)nv_sum + d.nv < (1ull << 31) && (uint64_t)m_sum + d.m < (1ull << 31),
               "batch body: too many vertices or triangles in total");
    nv_sum += d.nv;
    m_sum += d.m;
    n_sum += std::max<uint32_t>(d.m, 2) - 1;
    p_sum += (d.m + BB_BLOCK - 1) / BB_BLOCK;
    h.push_back(d);
    inst.push_back(k);
    mp.push_back(mpk);
    phase.push_back(ph);
  }
  nb = (uint32_t)h.size();
  {
    std::vector<double> tri(count, 0.0), vert(cloth_n.begin(), cloth_n.end());
    for (uint32_t j = 0; j < nb; ++j) tri[inst[j]] = h[j].m;
    xcd.init(tri, vert);
  }
  if (nb == 0) return;
  desc.upload(h.data(), nb, s);
  rest.upload(h_rest.data(), h_rest.size(), s);
  for (auto& b : verts) b.upload(h_rest.data(), h_rest.size(), s);
  tris.upload(h_tris.data(), h_tris.size(), s);
  capv.upload(h_capv.data(), std::max<size_t>(h_capv.size(), 1), s);
  capp0.upload(h_p0.data(), std::max<size_t>(h_p0.size(), 1), s);
  capp1.upload(h_p1.data(), std::max<size_t>(h_p1.size(), 1), s);
  boxes.alloc(6 * (size_t)m_sum);
  partial.alloc(6 * (size_t)p_sum);
  for (auto& b : kv) b.alloc(m_sum);
  keys.alloc(m_sum);
  for (int q = 0; q < 2; ++q) {
    leaf_tri[q].alloc(m_sum);
    nodes[q].alloc(n_sum);
    nodes[q].zero(s);
    root[q].alloc(6 * (size_t)nb);
    root[q].zero(s);
    leaf0[q].alloc(6 * (size_t)nb);
    leaf0[q].zero(s);
  }
  motion.alloc((size_t)BB_FRAMES * nb * BB_MF);
  motion.zero(s);
  for (int q = 0; q < 2; ++q) {
    if (alloc_fault_now()) alloc_failed("hipHostMalloc: injected failure (cc_fault_inject)");
    CC_HIP(hipHostMalloc((void**)&h_motion[q], (size_t)BB_FRAMES * nb * BB_MF * sizeof(float), hipHostMallocDefault));
    std::memset(h_motion[q], 0, (size_t)BB_FRAMES * nb * BB_MF * sizeof(float));
    CC_HIP(hipEventCreate(&ev_motion[q]));
  }
  // work lists: largest body first for the per-body kernels
  std::vector<uint32_t> order(nb);
  std::iota(order.begin(), order.end(), 0u);
  std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) { return h[a].m > h[b].m; });
  size_t chunks0 = 0;
  for (uint32_t j = 0; j < nb; ++j) chunks0 += level_chunks0(h[j].m);
  for (auto& b : items) b.alloc(chunks0 * LV_CAP);
  for (auto& b : nitems) {
    b.alloc(chunks0);
    b.zero(s);
  }
  for (int which = 0; which < 2; ++which) {
    BodyPass& P = which == 0 ? all : step;
    std::vector<uint4> tdef, tbox;
    std::vector<uint32_t> lsort, lbuild;
    for (uint32_t j : order) {
      const BodyDesc& d = h[j];
      const bool mov = d.mode != CC_BODY_STATIC;
      if (!(which == 0 || mov)) continue;
      if (mov) append_blocks(tdef, j, d.nv, 0, false);
      if (which == 1 && by_refit(j)) {
        P.refit = true;
        continue;
      }
      append_blocks(tbox, j, d.m, d.p0, true);
      if (which == 0 || d.mode == CC_BODY_REBUILD) lsort.push_back(j);
      lbuild.push_back(j);
    }
    auto of_body = [&](const uint4& e) { return inst[e.x]; };
    upload_list(P.deform, P.n_deform, xcd.arrange(tdef, of_body), s);
    upload_list(P.boxes, P.n_boxes, xcd.arrange(tbox, of_body), s);
    P.sort.init(h, lsort, s, [&](std::vector<uint4>& tl) { tl = xcd.arrange(tl, of_body); });
    std::vector<std::vector<LvBlock>> t = build_level_tables(
        h, lbuild, [&](uint32_t j) { return which == 0 || h[j].mode == CC_BODY_REBUILD; });
    for (auto& lv : t) lv = xcd.arrange(lv, [&](const LvBlock& e) { return inst[e.body]; });
    for (int L = 0; L < BB_MAX_LEVELS; ++L) {
      P.n_level[L] = L < (int)t.size() ? (uint32_t)t[L].size() : 0u;
      if (P.n_level[L]) P.level[L].upload(t[L].data(), t[L].size(), s);
    }
  }
  scratch.alloc(all.sort.ntiles, all.sort.nbig);
  // frame 0 for every body, in both slots
  upload_motion(0, 1, s);
  launch(all, 0, 0, s);
  launch(all, 0, 1, s);
  if (step.refit) refit_setup(s);
}

// Against building them again from their sorted keys every frame (boxes, then
// keys searched and leaves gathered): 50 steps of 16 instances 3.35 -> 2.85 ms, 64
// steps of 256 36.8 -> 32.6.
void BatchBodies::refit_setup(hipStream_t s) {
  RefitTables t;
  std::vector<Node> nd;
  for (uint32_t j = 0; j < nb; ++j) {
    if (!by_refit(j)) continue;
    const BodyDesc& d = h[j];
    nd.resize(d.m - 1);
    copy_on(nd.data(), nodes[0].p + d.n0, nd.size() * sizeof(Node), hipMemcpyDeviceToHost, s);
    RefitGroup g{};
    g.v0 = d.v0;
    g.n0 = d.n0;
    g.body = j;
    g.depth = d.depth;
    t.add(nd.data(), d.m, d.t0, g, {});
  }
  for (int L = 0; L < t.nlevels; ++L)
    t.blk[L] = xcd.arrange(t.blk[L], [&](const RefitGroup& e) { return inst[e.body]; });
  t.upload(rl, s);
  nrl = t.nlevels;
  for (int L = 1; L < nrl; ++L) ritem[L].alloc(6 * (size_t)rl[L].nitems);
}

BvhView BatchBodies::view(uint32_t j, int slot) const {
  const BodyDesc& d = h[j];
  BvhView v;
  v.nodes = nodes[slot].p + d.n0;
  v.leaf_tri = leaf_tri[slot].p + d.t0;
  v.verts = verts[slot].p + 3 * (size_t)d.v0;
  v.leaf0_box = leaf0[slot].p + 6 * (size_t)j;
  v.m = d.m;
  return v;
}

void BatchBodies::upload_motion(uint64_t frame0, int nframes, hipStream_t s) {
  if (!moving) return;
  CC_REQUIRE(nframes >= 1 && nframes <= BB_FRAMES, "batch body: motion frames");
  CC_HIP(hipEventSynchronize(ev_motion[hm]));        // the staging buffer's last copy is done
  float* hmv = h_motion[hm];
  for (int f = 0; f < nframes; ++f)
    for (uint32_t j = 0; j < nb; ++j) {
      if (h[j].mode == CC_BODY_STATIC) continue;
      const MotionFrame mf = motion_of(mp[j], phase[j].data(), frame0 + (uint64_t)f);
      std::memcpy(hmv + ((size_t)f * nb + j) * BB_MF, mf.v, (12 + h[j].ncaps) * sizeof(float));
    }
  CC_HIP(hipMemcpyAsync(motion.p, hmv, (size_t)nframes * nb * BB_MF * sizeof(float), hipMemcpyHostToDevice, s));
  CC_HIP(hipEventRecord(ev_motion[hm], s));
  hm ^= 1;
}

void BatchBodies::pre(const BodyPass& P, int k, int slot, hipStream_t s) {
  if (nb == 0) return;
  if (P.n_deform)
    k_bb_deform<<<P.n_deform, BB_BLOCK, 0, s>>>(desc.p, P.deform.p, rest.p, verts[slot].p, capv.p, capp0.p,
                                                 capp1.p, motion.p, nb, k);
  if (P.n_boxes)
    k_bb_boxes<<<P.n_boxes, BB_BLOCK, 0, s>>>(desc.p, P.boxes.p, verts[slot].p, tris.p, boxes.p, partial.p);
  CC_LAUNCHED();
}

void BatchBodies::sort(const BodyPass& P, int slot, hipStream_t s) {
  if (nb == 0) return;
  const SortFrame f{boxes.p, partial.p, {kv[0].p, kv[1].p}, &scratch, keys.p, nullptr, root[slot].p};
  launch_sort(desc.p, P.sort, tris.p, &f, 1, s);
}

void BatchBodies::post(const BodyPass& P, int slot, hipStream_t s) {
  if (nb == 0) return;
  const LvBlock* tabs[BB_MAX_LEVELS];
  for (int L = 0; L < BB_MAX_LEVELS; ++L) tabs[L] = P.level[L].p;
  if (P.refit) {
    RefitFrame r{verts[slot].p, {}, nodes[slot].p, nullptr, root[slot].p};
    for (int L = 1; L < nrl; ++L) r.items[L] = ritem[L].p;
    launch_refit_levels(rl, nrl, leaf_tri[slot].p, nullptr, &r, 1, s);
  }
  const LvFrame f{keys.p, tris.p, boxes.p, leaf_tri[slot].p, {items[0].p, items[1].p}, {nitems[0].p, nitems[1].p},
                  nodes[slot].p, root[slot].p, leaf0[slot].p};
  launch_build_levels(tabs, P.n_level, &f, 1, s);
}

void BatchBodies::export_tree(uint32_t j, int slot, float* verts3, uint64_t* okeys, uint32_t* order,
                              int32_t* childA, int32_t* childB, int32_t* parent_int, int32_t* parent_leaf,
                              float* box_int, float* box_leaf, float* root6, hipStream_t s) {
  CC_REQUIRE(j < nb, "batch body: no such body");
  const BodyDesc& d = h[j];
  if (verts3)
    CC_HIP(hipMemcpyAsync(verts3, verts[slot].p + 3 * (size_t)d.v0, 3 * (size_t)d.nv * sizeof(float),
                          hipMemcpyDeviceToHost, s));
  export_tree_raw(d.m, keys.p + d.t0, leaf_tri[slot].p + d.t0, nodes[slot].p + d.n0,
                  root[slot].p + 6 * (size_t)j, leaf0[slot].p + 6 * (size_t)j, okeys, order, childA, childB,
                  parent_int, parent_leaf, box_int, box_leaf, root6, s);
}

}  // namespace cc
