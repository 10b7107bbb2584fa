// cc_bbody.h -- the collider bodies of a batch: every instance's body in
// concatenated arrays, posed and rebuilt (or refitted) for all instances
// together, a handful of launches per frame whatever the instance count.
#pragma once

#include <vector>

#include "cc_sim.h"

namespace cc {

constexpr int BB_MF = 12 + MAX_CAPS;   // floats per motion frame and body
constexpr int BB_FRAMES = 16;          // motion frames held on the device (one step graph)

// Where the instances' work runs.  Workgroups are dealt to the chip's eight
// XCDs in turn, and each XCD has an L2 of its own, so a table whose entry k
// belongs to an instance of XCD k % 8 keeps what one kernel of an instance
// writes in the L2 that the next one reads it from, and the scattered stores
// of the sort merge into whole lines there.  Instances are dealt out, the
// largest first, to the XCD with the least load; a batch whose loads come out
// uneven by more than a tenth (a few instances, or one far larger than the
// rest) keeps plain tables, which spread every instance over the whole chip.
// Measured at 256 instances: the sort's scatters 49 -> 38 us each and 97 -> 74
// with the leaves, the step 197 -> 189.
constexpr uint32_t XCDS = 8;
struct XcdMap {
  std::vector<uint8_t> of;            // XCD of each instance; empty: plain tables
  // a[k], b[k]: two loads of instance k (body triangles, cloth vertices)
  void init(const std::vector<double>& a, const std::vector<double>& b);
  // t in an order of its XCDs; key(entry): its instance
  template <class T, class K>
  std::vector<T> arrange(const std::vector<T>& t, K key) const {
    if (of.empty()) return t;
    std::vector<T> list[XCDS], out;
    for (const T& e : t) list[of[key(e)]].push_back(e);
    size_t at[XCDS] = {};
    out.reserve(t.size());
    while (out.size() < t.size()) {
      size_t x = out.size() % XCDS;
      if (at[x] == list[x].size())    // this XCD's list is done: the tail of the longest one left
        for (size_t y = 0; y < XCDS; ++y)
          if (list[y].size() - at[y] > list[x].size() - at[x]) x = y;
      out.push_back(list[x][at[x]++]);
    }
    return out;
  }
};

// Work lists of one kind of pass: block tables {body, first, count, aux} of
// the grid-wide kernels, the tiles of the sort, and the workgroups of each
// build level.
struct BodyPass {
  bool refit = false;                 // the REFIT bodies by levels (else built like the others)
  DBuf<uint4> deform, boxes;
  SortTable sort;
  DBuf<LvBlock> level[BB_MAX_LEVELS];
  uint32_t n_deform = 0, n_boxes = 0, n_level[BB_MAX_LEVELS] = {};
};

// What one cloth step of a batch reads and writes: per-instance step
// constants and LBVH view.
struct InstDesc {
  StepArgs a;
  BvhView bvh;
};

struct BatchBodies {
  uint32_t nb = 0;                    // bodies
  std::vector<BodyDesc> h;
  std::vector<uint32_t> inst;         // body -> instance
  std::vector<MotionParams> mp;
  std::vector<std::vector<float>> phase;
  bool moving = false;                // any REFIT / REBUILD body

  DBuf<BodyDesc> desc;
  DBuf<float> rest;                   // [3 * sum nv]
  // Two body slots: frame g lives in slot g % 2, so frame g + 1 is built
  // while the cloth steps against frame g.
  DBuf<float> verts[2];               // [3 * sum nv]
  DBuf<uint32_t> tris;                // [3 * sum m], body-local vertex indices
  DBuf<uint32_t> capv;                // [sum (ncaps + 1)]
  DBuf<float> capp0, capp1;           // [3 * sum ncaps]
  DBuf<float> boxes;                  // [6 * sum m] expanded box of each triangle
  DBuf<float> partial;                // [6 * sum ceil(m / 256)]
  DBuf<uint2> kv[2];                  // [sum m] (code, primitive) sort ping-pong
  SortScratch scratch;
  DBuf<uint64_t> keys;                // [sum m]
  DBuf<BItem> items[2];               // [level-0 chunks * 128] unfinished nodes between levels
  DBuf<uint32_t> nitems[2];           // [level-0 chunks] their count per chunk
  DBuf<uint4> leaf_tri[2];            // [sum m]
  DBuf<Node> nodes[2];                // [sum max(m - 1, 1)]
  DBuf<float> root[2], leaf0[2];      // [6 * nb]
  DBuf<float> motion;                 // [BB_FRAMES * nb * BB_MF]
  float* h_motion[2] = {nullptr, nullptr};   // pinned staging of the motion uploads
  hipEvent_t ev_motion[2] = {nullptr, nullptr};
  int hm = 0;

  // REFIT bodies of two or more triangles keep the topology of their frame-0
  // pose: refitted by levels (refit.hip) over tables of all of them
  RefitLevel rl[RL_MAX];
  int nrl = 0;
  DBuf<float> ritem[RL_MAX];          // [6 * items] boxes of each level's items

  BodyPass all;    // set-up: every body built from its frame-0 pose
  BodyPass step;   // per frame: moving bodies posed, REBUILD ones sorted and built, REFIT ones refitted

  BatchBodies() = default;
  BatchBodies(const BatchBodies&) = delete;
  BatchBodies& operator=(const BatchBodies&) = delete;
  ~BatchBodies();

  // bodies[k] of instance k (NULL or mode NONE: no body); extends the
  // vertices when asked, checks every layout, uploads, builds frame 0.
  // xcd: filled from the bodies' triangles and cloth_n[k], instance k's cloth
  // vertices.
  void init(const cc_body_desc* bodies, const cc_params* params, const std::vector<uint32_t>& cloth_n, uint32_t count,
            hipStream_t s);
  XcdMap xcd;
  BvhView view(uint32_t j, int slot) const;
  bool by_refit(uint32_t j) const { return h[j].mode == CC_BODY_REFIT && h[j].m >= 2; }
  void refit_setup(hipStream_t s);
  // motion of frames [frame0, frame0 + nframes) into the device table
  void upload_motion(uint64_t frame0, int nframes, hipStream_t s);
  // One pass into a slot, in three parts: pose + boxes (k selects the
  // motion frame in the table), the sort, the build by levels.
  void pre(const BodyPass& p, int k, int slot, hipStream_t s);
  void sort(const BodyPass& p, int slot, hipStream_t s);
  void post(const BodyPass& p, int slot, hipStream_t s);
  void launch(const BodyPass& p, int k, int slot, hipStream_t s) {
    pre(p, k, slot, s);
    sort(p, slot, s);
    post(p, slot, s);
  }
  void export_tree(uint32_t j, int slot, float* verts3, uint64_t* keys, uint32_t* order, int32_t* childA,
                   int32_t* childB, int32_t* parent_int, int32_t* parent_leaf, float* box_int, float* box_leaf,
                   float* root6, hipStream_t s);
};

}  // namespace cc
