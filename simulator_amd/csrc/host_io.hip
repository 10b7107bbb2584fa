// host_io.hip -- states, points and vertices to and from a caller's host arrays.
//
// A copy from or to pageable memory goes through the runtime's own staging, one
// blocking copy per array, and a query that allocates its device memory pays
// more for that than for the query.  Here the kernels themselves read and
// write pinned memory that the handle keeps (Stage, bounded by IO_CHUNK items),
// and the caller's arrays are copied from and to it by the host, the next
// chunk's kernel running beside the copy of this one.  Measured: a query of
// 20,000 points 175 -> 70 us (its kernel takes 17), the states of 256 instances
// 20 -> 13 ms, 262,144 vertices after 200 steps 0.8 ms less, 25,344 body vertices
// 8 us less.
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "cc_step.h"

namespace cc {

// items of a chunk: 2.4 MB of states, 2.7 MB of a query's points and results
// and the 15.7 MB of its spill area, the most a handle keeps (two chunks of
// pinned memory)
constexpr uint32_t IO_CHUNK = 65536;
constexpr size_t STATE_BYTES = 36;   // of a vertex: x_cur, x_prev, contact normal
constexpr uint32_t chunks_of(uint32_t n) { return n / IO_CHUNK + (n % IO_CHUNK ? 1 : 0); }
static_assert(chunks_of(1) == 1 && chunks_of(IO_CHUNK) == 1 && chunks_of(IO_CHUNK + 1) == 2 &&
                  chunks_of(~0u - IO_CHUNK) == (1u << 16) - 1 && chunks_of(~0u) == 1u << 16,
              "every count of points is covered, also those a chunk short of 2^32");

// {x_cur, x_prev} records and normals to three arrays of vec3, one after the
// other.  Bound by the link to the host (36 bytes per vertex).
__global__ __launch_bounds__(256) void k_state_out(const float* __restrict__ state, const float* __restrict__ contact,
                                                   uint32_t n, float* __restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const f3 p = ld3(state + 6 * (size_t)i), q = ld3(state + 6 * (size_t)i + 3), c = ld3(contact + 3 * (size_t)i);
  st3(out + 3 * (size_t)i, p);
  st3(out + 3 * ((size_t)n + i), q);
  st3(out + 3 * (2 * (size_t)n + i), c);
}

__global__ __launch_bounds__(256) void k_points_in(const float* __restrict__ in, uint32_t n, float* __restrict__ a,
                                                   float* __restrict__ b) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 3 * n) return;
  const float v = in[i];
  a[i] = v;
  b[i] = v;
}

namespace {
// pinned memory of a chunk (two alternate where there are several)
size_t chunk_bytes(uint32_t n, size_t bytes) { return (bytes * std::min(n, IO_CHUNK) + 255) / 256 * 256; }

// Chunks of [0, n): fill(o, k, h) before a chunk's launch(o, k, h), drain(o, k,
// h) after it has run, h the chunk's pinned memory (`bytes` per item).  Returns
// with every chunk drained, or, when there is nothing to drain, with the last
// ones still running.
struct Nothing {
  void operator()(uint32_t, uint32_t, char*) const {}
};
template <class Fill, class Launch, class Drain>
void by_chunks(Stage& st, uint32_t n, size_t bytes, hipStream_t s, Fill&& fill, Launch&& launch, Drain&& drain) {
  constexpr bool wait = !std::is_same_v<std::decay_t<Drain>, Nothing>;
  const uint32_t c = std::min(n, IO_CHUNK), chunks = chunks_of(n);
  const size_t half = chunk_bytes(n, bytes);
  char* h = st.host(half * std::min(chunks, 2u));
  if (chunks == 1) {
    fill(0u, n, h);
    launch(0u, n, h);
    if (wait) CC_HIP(hipStreamSynchronize(s));
    drain(0u, n, h);
    return;
  }
  Events<2> ev;
  auto start = [&](uint32_t k) {
    const uint32_t o = k * c, m = std::min(c, n - o);
    fill(o, m, h + (k & 1) * half);
    launch(o, m, h + (k & 1) * half);
    CC_HIP(hipEventRecord(ev[(int)(k & 1)], s));
  };
  start(0);
  for (uint32_t k = 0; k < chunks; ++k) {
    // (the half of chunk k + 1 was drained, or written from, at chunk k - 1)
    if (k + 1 < chunks) start(k + 1);
    if (wait || k + 2 < chunks) CC_HIP(hipEventSynchronize(ev[(int)(k & 1)]));
    drain(k * c, std::min(c, n - k * c), h + (k & 1) * half);
  }
}
}  // namespace

size_t state_bytes(uint32_t n) { return chunk_bytes(n, STATE_BYTES) * (n > IO_CHUNK ? 2 : 1); }

void read_state(Stage& st, const float* state, const float* contact, uint32_t n, float* x_cur, float* x_prev,
                float* contact_n, hipStream_t s) {
  std::lock_guard<std::mutex> g(st.m);
  by_chunks(
      st, n, STATE_BYTES, s, Nothing{},
      [&](uint32_t o, uint32_t k, char* h) {
        k_state_out<<<grid_for(k, 256), 256, 0, s>>>(state + 6 * (size_t)o, contact + 3 * (size_t)o, k,
                                                     reinterpret_cast<float*>(h));
        CC_LAUNCHED();
      },
      [&](uint32_t o, uint32_t k, char* h) {
        float* out[3] = {x_cur, x_prev, contact_n};
        for (int a = 0; a < 3; ++a)
          if (out[a]) std::memcpy(out[a] + 3 * (size_t)o, h + 12 * (size_t)k * a, 12 * (size_t)k);
      });
}

void write_points(Stage& st, const float* src, uint32_t n, float* a, float* b, hipStream_t s) {
  by_chunks(
      st, n, 12, s,
      [&](uint32_t o, uint32_t k, char* h) { std::memcpy(h, src + 3 * (size_t)o, 12 * (size_t)k); },
      [&](uint32_t o, uint32_t k, char* h) {
        k_points_in<<<grid_for(3 * (size_t)k, 256), 256, 0, s>>>(reinterpret_cast<const float*>(h), k,
                                                                 a + 3 * (size_t)o, b + 3 * (size_t)o);
        CC_LAUNCHED();
      },
      Nothing{});
}

uint32_t query_points(Stage& st, const BvhView& v, const float* pts, uint32_t n, int32_t* hit, uint8_t* inside,
                      float* out_pos, float* out_n, hipStream_t s) {
  std::lock_guard<std::mutex> g(st.m);
  const uint32_t c = std::min(n, IO_CHUNK);
  if (st.spill.n < (size_t)STACK_SPILL * c + SPILL_TAIL) st.spill.alloc((size_t)STACK_SPILL * c + SPILL_TAIL);
  // a chunk: points, positions, normals, hits, the fault word, insides
  uint32_t fault = 0;
  by_chunks(
      st, n, 41 + 4, s,
      [&](uint32_t o, uint32_t k, char* h) { std::memcpy(h, pts + 3 * (size_t)o, 12 * (size_t)k); },
      [&](uint32_t, uint32_t k, char* h) {
        float* f = reinterpret_cast<float*>(h);
        int32_t* hits = reinterpret_cast<int32_t*>(f + 9 * (size_t)k);
        int32_t* tail = st.spill.p + (size_t)STACK_SPILL * k;
        launch_spill_tail(tail, s);
        launch_collide_points(v, f, k, st.spill.p, hits, reinterpret_cast<uint8_t*>(hits + k + 1), f + 3 * (size_t)k,
                              f + 6 * (size_t)k, s);
        launch_spill_status(tail, reinterpret_cast<uint32_t*>(hits + k), s);
      },
      [&](uint32_t o, uint32_t k, char* h) {
        const float* f = reinterpret_cast<const float*>(h);
        const int32_t* hits = reinterpret_cast<const int32_t*>(f + 9 * (size_t)k);
        std::memcpy(out_pos + 3 * (size_t)o, f + 3 * (size_t)k, 12 * (size_t)k);
        std::memcpy(out_n + 3 * (size_t)o, f + 6 * (size_t)k, 12 * (size_t)k);
        std::memcpy(hit + o, hits, 4 * (size_t)k);
        std::memcpy(inside + o, hits + k + 1, k);
        fault |= (uint32_t)hits[k];
      });
  return fault;
}

}  // namespace cc
