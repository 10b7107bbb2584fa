// wide.hip -- the four-wide form of the body's LBVH.
//
// The collision query walks the Karras tree one node record per dependent
// memory round trip, and the slowest lanes of a step (points resting on the
// body) walk 50-70 nodes.  Folding every second level into its parent halves
// that chain: a wide node holds the entries of a binary node X and of X's
// internal children, four boxes and four links in one 128-byte record, and
// the traversal (wide_first_hit) tests all four at once.
//
// The entries are stored in the order the binary traversal considers them
// (D_BVH::intersect, cudaBRT.cu:239-285, returns an overlapped leaf child at
// once, A before B, before it descends into internal children), so the first
// hit, and with it the contact set, is the same leaf.  The binary tree stays
// the topology the refit walks.  The layout is computed once per topology on
// the host (Body::wide_setup), which writes the records in full from the
// binary boxes (k_fold_wide).  Later refits write each box straight into the
// wide entry that mirrors its binary child slot (through the tables of the
// refit by levels, or w_dst in a refit by chunks) and leave the binary
// boxes alone; export and the binary walk ask for a binary refit.
//
// A rebuilt body's topology changes every frame, so its wide form is folded
// on the device after each build (k_fold_grouped): one record per internal
// node at the node's own index, no host set-up, no bound to check (the
// split records keep the walk's deferrals within the tree depth).
#include <algorithm>
#include <cstring>
#include <vector>

#include "cc_lbvh.h"

namespace cc {

// Record w of the wide form: four 32-byte entries, entry e = floats
// [8e, 8e + 8) = {min xyz, max x, max yz, link, 0}.  src[w] names for each
// entry the binary record and side (record * 2 + side, side 0 = child A)
// that holds its box, ~0 for an empty entry (box +inf / -inf, link 0).
__global__ __launch_bounds__(256) void k_fold_wide(const Node* __restrict__ nodes, const uint4* __restrict__ src,
                                                   const int4* __restrict__ link, uint32_t nw,
                                                   float4* __restrict__ wide) {
  const uint32_t w = blockIdx.x * 256 + threadIdx.x;
  if (w >= nw) return;
  const uint4 s = src[w];
  const int4 l = link[w];
  const uint32_t e4[4] = {s.x, s.y, s.z, s.w};
  const int32_t l4[4] = {l.x, l.y, l.z, l.w};
  float4* o = wide + 8 * (size_t)w;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float b[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    if (e4[e] != ~0u) {
      const float* f = reinterpret_cast<const float*>(nodes + (e4[e] >> 1)) + 6 * (e4[e] & 1u);
      for (int c = 0; c < 6; ++c) b[c] = f[c];
    }
    o[2 * e] = make_float4(b[0], b[1], b[2], b[3]);
    o[2 * e + 1] = make_float4(b[4], b[5], __int_as_float(l4[e]), 0.0f);
  }
}

// The wide form of a rebuilt body, record x from internal node x: X's leaf
// children (A before B), then the children of its internal children (A's,
// then B's), each pair in its parent's order of consideration (a leaf child
// first, A before B).  With both children internal, entry 0's split word is
// B's index.  Four lanes per record, lane e writing entry e: bound by the 128
// bytes written and the lines read (nodes x, A and B), which the lanes of a
// quad share.  Three frames of 50,688 triangles: 9.9 us, against 14.8 with one
// lane per record (eight stores 128 bytes apart).
__global__ __launch_bounds__(256) void k_fold_grouped(PF<const Node> nodes_f, uint32_t mi, PF<float4> wide_f) {
  const uint32_t t = blockIdx.x * 256 + threadIdx.x, x = t >> 2;
  const int e = (int)(t & 3u);
  if (x >= mi) return;
  const float4* N = reinterpret_cast<const float4*>(pick(nodes_f));
  const int4 lx = reinterpret_cast<const int4*>(N)[4 * (size_t)x + 3];
  const bool la = lx.x < 0, lb = lx.y < 0;
  // the node whose child slot the entry is, and the entry's place in its pair
  int32_t y = (int32_t)x;
  int at = e;
  bool empty = false;
  if (la && lb) {
    empty = e > 1;
  } else if (la || lb) {
    empty = e == 3;
    if (e > 0) {
      y = la ? lx.y : lx.x;
      at = e - 1;
    } else {
      at = la ? 0 : 1;
    }
  } else {
    y = e < 2 ? lx.x : lx.y;
    at = e & 1;
  }
  const float4* ny = N + 4 * (size_t)y;
  const float4 q0 = ny[0], q1 = ny[1], q2 = ny[2];
  const int4 ly = reinterpret_cast<const int4*>(ny)[3];
  // a pair whose B alone is a leaf is considered B first
  const bool b_side = (y != (int32_t)x && ly.x >= 0 && ly.y < 0) ? at == 0 : at == 1;
  const float inf = INFINITY;
  float4 o0 = b_side ? make_float4(q1.z, q1.w, q2.x, q2.y) : q0;
  float4 o1 = b_side ? make_float4(q2.z, q2.w, 0.0f, 0.0f) : make_float4(q1.x, q1.y, 0.0f, 0.0f);
  o1.z = __int_as_float(b_side ? ly.y : ly.x);
  if (e == 0 && !la && !lb) o1.w = __int_as_float(lx.y);
  if (empty) {
    o0 = make_float4(inf, inf, inf, -inf);
    o1 = make_float4(-inf, -inf, 0.0f, 0.0f);
  }
  float4* o = pick(wide_f) + 2 * (size_t)t;
  o[0] = o0;
  o[1] = o1;
}

void Body::fold_static(int k, hipStream_t s) {
  if (!nwide || !wide_enabled) return;
  k_fold_wide<<<grid_for(nwide, 256), 256, 0, s>>>(slot[k].nodes.p, w_src.p, w_link.p, nwide, slot[k].wide.p);
  CC_LAUNCHED();
}

void Body::fold_frames(int F, const int* ks, hipStream_t s) {
  if (!grouped || !wide_enabled) return;
  PF<const Node> nodes{};
  PF<float4> wide{};
  for (int f = 0; f < F; ++f) {
    nodes.p[f] = slot[ks[f]].nodes.p;
    wide.p[f] = slot[ks[f]].wide.p;
  }
  k_fold_grouped<<<dim3(grid_for(4 * (size_t)(m - 1), 256), (unsigned)F), 256, 0, s>>>(nodes, m - 1, wide);
  CC_LAUNCHED();
}

void Body::wide_setup(int k, hipStream_t s) {
  nwide = 0;
  wide_stack = 0;
  if (mode == CC_BODY_NONE || mode == CC_BODY_REBUILD || m < 2) return;
  // (a vector: the pages are there before the copy, which takes twice as long otherwise)
  std::vector<Node> nd(m - 1);
  copy_on(nd.data(), slot[k].nodes.p, nd.size() * sizeof(Node), hipMemcpyDeviceToHost, s);
  std::vector<uint2> dst;
  const uint32_t nw = wide_layout(k, nd.data(), dst, s);
  if (mode == CC_BODY_REFIT && bottom_up) refit_setup(nd.data(), dst, s);
  nwide = nw;            // all of it is there
}

uint32_t Body::wide_layout(int k, const Node* nd, std::vector<uint2>& dst, hipStream_t s) {
  const uint32_t mi = m - 1;
  // Depth-first over the kept binary nodes (the root, then the internal entries
  // of each kept node), so that the nodes read next lie near those just read;
  // wid maps a kept binary node to its record.
  std::vector<int32_t> wid(mi, -1), order;
  std::vector<uint4> src;
  std::vector<int4> link;
  std::vector<uint32_t> acc;     // deferrable entries on the path to each record
  order.reserve(mi / 2 + 1);
  src.reserve(mi / 2 + 1);
  link.reserve(mi / 2 + 1);
  acc.reserve(mi / 2 + 1);
  std::vector<uint32_t> open;    // records not laid out yet
  auto keep = [&](int32_t x, uint32_t deferrable) {
    const uint32_t h = (uint32_t)order.size();
    wid[x] = (int32_t)h;
    order.push_back(x);
    acc.push_back(deferrable);
    src.push_back(make_uint4(~0u, ~0u, ~0u, ~0u));
    link.push_back(make_int4(0, 0, 0, 0));
    open.push_back(h);
    return (int32_t)h;
  };
  keep(0, 0);
  uint32_t worst = 0;
  while (!open.empty()) {
    const uint32_t h = open.back();
    open.pop_back();
    const int32_t x = order[h];
    uint32_t es[4], cnt = 0;
    int32_t ref[4];
    auto add = [&](int32_t rec, int side, int32_t child) {
      CC_REQUIRE(cnt < 4, "wide form: more than four entries");
      es[cnt] = (uint32_t)rec * 2u + (uint32_t)side;
      ref[cnt++] = child;
    };
    // X's children in its order of consideration (leaf children first),
    // then, while there is room, the internal entry with the largest box
    // surface is replaced in place by its own children in their order: an
    // in-place replacement keeps the whole list in the binary walk's order
    // of consideration.  (A CPU replay of a late frame of the large workload:
    // 7.44 wide visits per query and 12.4 per wave's slowest lane, against
    // 7.69 and 12.95 when every node folds exactly its children.)
    add(x, 0, nd[x].childA);
    add(x, 1, nd[x].childB);
    auto order_pair = [&](uint32_t e0) {        // leaf child of the pair first
      if (ref[e0] >= 0 && ref[e0 + 1] < 0) {
        std::swap(es[e0], es[e0 + 1]);
        std::swap(ref[e0], ref[e0 + 1]);
      }
    };
    order_pair(0);
    while (cnt < 4) {
      int best = -1;
      double best_area = -1.0;
      for (uint32_t e = 0; e < cnt; ++e) {
        if (ref[e] < 0) continue;
        const Node& P = nd[es[e] >> 1];
        const float* bmn = (es[e] & 1u) ? P.b_min : P.a_min;
        const float* bmx = (es[e] & 1u) ? P.b_max : P.a_max;
        const double dx = (double)bmx[0] - bmn[0], dy = (double)bmx[1] - bmn[1], dz = (double)bmx[2] - bmn[2];
        const double area = dx * dy + dy * dz + dz * dx;
        if (area > best_area) {
          best_area = area;
          best = (int)e;
        }
      }
      if (best < 0) break;
      const int32_t c = ref[best];
      CC_REQUIRE((uint32_t)c < mi, "wide form: link out of range");
      for (uint32_t e = cnt; e > (uint32_t)best + 1; --e) {
        es[e] = es[e - 1];
        ref[e] = ref[e - 1];
      }
      ++cnt;
      es[best] = (uint32_t)c * 2u;
      ref[best] = nd[c].childA;
      es[best + 1] = (uint32_t)c * 2u + 1u;
      ref[best + 1] = nd[c].childB;
      order_pair((uint32_t)best);
    }
    const uint32_t deferrable = acc[h] + (cnt - 1);
    worst = std::max(worst, deferrable);
    uint4 sv = make_uint4(~0u, ~0u, ~0u, ~0u);
    int4 lv = make_int4(0, 0, 0, 0);
    uint32_t* sp = &sv.x;
    int32_t* lp = &lv.x;
    for (uint32_t e = 0; e < cnt; ++e) {
      sp[e] = es[e];
      if (ref[e] < 0) {
        lp[e] = ref[e];
      } else {
        CC_REQUIRE((uint32_t)ref[e] < mi && wid[ref[e]] < 0, "wide form: node reached twice");
        lp[e] = keep(ref[e], deferrable);
      }
    }
    src[h] = sv;
    link[h] = lv;
  }
  // The traversal stack holds 64 entries; keep the binary form otherwise.
  if (worst > 64) return 0;
  // Renumber the records in the order of their binary nodes (Karras
  // indices; the root stays 0): the refit, which walks binary nodes in index
  // order, then writes each chunk's entries into a compact run of records.
  {
    const size_t nw = order.size();
    std::vector<int32_t> renum(nw);
    int32_t r = 0;
    for (uint32_t x = 0; x < mi; ++x)
      if (wid[x] >= 0) renum[wid[x]] = r++;
    std::vector<uint4> src2(nw);
    std::vector<int4> link2(nw);
    for (size_t w = 0; w < nw; ++w) {
      int4 l = link[w];
      int32_t* lp = &l.x;
      const uint32_t* e = &src[w].x;
      for (int q = 0; q < 4; ++q)
        if (e[q] != ~0u && lp[q] >= 0) lp[q] = renum[lp[q]];
      src2[renum[w]] = src[w];
      link2[renum[w]] = l;
    }
    src.swap(src2);
    link.swap(link2);
  }
  // for the refits: the one by levels takes it into its tables, the one by chunks
  // reads it as it is, and a static body built by levels is folded anew
  if (!bottom_up || mode == CC_BODY_REFIT) {
    dst.assign(2 * (size_t)mi, make_uint2(~0u, 0u));
    for (size_t w = 0; w < src.size(); ++w) {
      const uint32_t* e = &src[w].x;
      const int32_t* lk = &link[w].x;
      for (int q = 0; q < 4; ++q)
        if (e[q] != ~0u) dst[e[q]] = make_uint2((uint32_t)(4 * w + q), (uint32_t)lk[q]);
    }
  }
  w_src.upload(src.data(), src.size(), s);
  w_link.upload(link.data(), link.size(), s);
  if (!bottom_up) w_dst.upload(dst.data(), dst.size(), s);
  const uint32_t nw = (uint32_t)src.size();
  wide_stack = worst;
  for (int j = 0; j < nslots; ++j) slot[j].wide.alloc(8 * (size_t)nw);
  // Slot k's records in full (links, empty entries, boxes); the other slots
  // get theirs from share_topology, and every refit rewrites the boxes.
  k_fold_wide<<<grid_for(nw, 256), 256, 0, s>>>(slot[k].nodes.p, w_src.p, w_link.p, nw, slot[k].wide.p);
  CC_LAUNCHED();
  CC_HIP(hipStreamSynchronize(s));
  return nw;
}

}  // namespace cc
